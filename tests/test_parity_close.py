"""The comparison of the parity cases (tests/parity_cases.py): what counts as out of tolerance."""
import numpy as np
import pytest

from tests.parity_cases import REL_TOL, close

NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("a,b,scale,bad", [
    ([1.0, 2.0], [1.0, 2.0], 1.0, 0),
    ([1.0 + 0.9 * REL_TOL], [1.0], 1.0, 0), ([1.0 + 2.1 * REL_TOL], [1.0], 1.0, 1),
    ([0.0, 0.0], [0.0, 0.0], 0.0, 0), ([1e-300], [0.0], 0.0, 1),
    ([NAN, 1.0], [1.0, 1.0], 1.0, 1), ([1.0], [NAN], 1.0, 1), ([NAN], [NAN], 1.0, 1), ([NAN], [0.0], 0.0, 1),
    ([1.0], [1.0], NAN, 0), ([1.5], [1.0], NAN, 1),
    ([INF], [1.0], 1.0, 1), ([INF], [INF], 1.0, 0), ([1.0], [INF], 1.0, 1), ([], [], 1.0, 0)])
def test_close(a, b, scale, bad):
    with np.errstate(all="raise"):
        n, err = close(a, b, scale)
    assert n == bad
    assert bad or err <= REL_TOL
