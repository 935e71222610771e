"""The comparison of the parity tests (tests/parity.py) on values that are not numbers."""
import numpy as np
import pytest

from parity import compare

NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("g, c, bad", [
    (1.0, 1.0 + 1e-11, False), (1.0, 1.0 + 1e-9, True), (0.0, 1e-13, False), (NAN, NAN, False), (NAN, 1.0, True),
    (1.0, NAN, True), (INF, INF, False), (-INF, INF, True), (INF, 1e308, True), (0.0, -INF, True), (INF, NAN, True)])
def test_compare(g, c, bad):
    got = compare({"soil": np.array([2.0, g])}, {"soil": np.array([2.0, c])})
    assert bool(got) == bad, got
    assert not got or got[0][2:4] == (1, 1)
