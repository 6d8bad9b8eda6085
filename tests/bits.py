"""Bit for bit equality of floating-point results, the sign of a zero included."""
import numpy as np


def same_bits(a, b):
    """The same bits everywhere but in NaN, which has to stand in the same places (its payload is the
    machine's)."""
    a, b = np.ascontiguousarray(a, np.float64), np.ascontiguousarray(b, np.float64)
    if a.shape != b.shape:
        return False
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a.view(np.int64)[~nan], b.view(np.int64)[~nan])
