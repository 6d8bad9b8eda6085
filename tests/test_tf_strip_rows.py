"""The height of the two-fluid strips counts the blocks that can run at once: 1024 where a member has the
Maxwell curl terms (two wavefronts per SIMD), else 1536 (three)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spruce_amd", "csrc")
MAIN = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "tf_rows.hpp"
int main(int argc, char** argv) {
  std::vector<int> rows, tiles;
  for (int k = 2; k + 1 < argc; k += 2) { rows.push_back(atoi(argv[k])); tiles.push_back((atoi(argv[k + 1]) + 59) / 60); }
  printf("%d\\n", spruce::tf_strip_rows_default(rows.data(), tiles.data(), (int)rows.size(), atoi(argv[1]) != 0));
}
"""


@pytest.fixture(scope="module")
def rows_of(tmp_path_factory):
    d = tmp_path_factory.mktemp("rows")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I" + CSRC, "-o", str(d / "main"), str(d / "main.cpp")], check=True)
    return lambda curl, sizes: int(subprocess.run([str(d / "main"), str(int(curl))] + [str(v) for s in sizes for v in s],
                                                  check=True, capture_output=True, text=True).stdout)


@pytest.mark.parametrize("curl,resident", [(False, 1536), (True, 1024)])
@pytest.mark.parametrize("sizes", [[(5, 5)], [(192, 192)], [(256, 256)], [(384, 384)], [(512, 512)],
                                   [(160, 200)] * 8, [(192 + 16 * k, 208 + 24 * k) for k in range(16)]])
def test_height_has_the_least_rounds_times_cost(rows_of, curl, resident, sizes):
    def cost(R):
        blocks = sum(-(-ny // 60) * -(-nx // R) for nx, ny in sizes)
        return -(-blocks // resident) * (R + 3)
    best = min(cost(R) for R in range(1, 65))
    assert rows_of(curl, sizes) == max(R for R in range(1, 65) if cost(R) == best)
