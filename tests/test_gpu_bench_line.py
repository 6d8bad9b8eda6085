"""bench.py prints its line where the reference executable of its CPU leg is not built."""
import json
import sys

import pytest

import bench

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("argv", [["--workload", "periodic", "--steps", "2", "--warmup", "1"],
                                  ["--workload", "batch2f", "--steps", "5", "--warmup", "1"]])
def test_line_without_the_reference_executable(argv, monkeypatch, capsys, tmp_path):
    monkeypatch.setattr(bench, "REFERENCE", str(tmp_path / "absent"), raising=False)
    monkeypatch.setattr(sys, "argv", ["bench.py"] + argv)
    bench.main()
    out = json.loads(capsys.readouterr().out.splitlines()[-1])
    assert out["value"] > 0.0 and out["steps"] == int(argv[3]) and "cpu_baseline" not in out
