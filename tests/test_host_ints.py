"""Labels and dims at the boundary: what numpy's conversion to Int64 accepts,
refuses and gives is what a contraction passes on (CPU only)."""
import numpy as np
import pytest

import helpers  # noqa: F401  (puts the package on the path)
from itg import _lib

GOOD = [(), (3,), (1, -1, 2), [4, 5, 6, 7], tuple(range(40)), (1.0, -1.0), [2.0, 3],
        np.array([1, -2], dtype=np.int32), np.array([5.0, 6.0]), np.arange(6).reshape(2, 3),
        (np.int64(7), True), (2**63 - 1, -2**63)]
BAD = [(2**63,), (0, -2**63 - 1), (2**64 + 1,), ("a",), (None, 1), (1j,)]


@pytest.mark.parametrize("seq", GOOD, ids=[str(i) for i in range(len(GOOD))])
def test_same_values(seq):
    want = _lib.i64(seq)
    got = _lib.ints(seq)
    assert list(got)[:want.size] == want.tolist()
    assert len(got) == max(want.size, 1)  # never an empty array


@pytest.mark.parametrize("seq", BAD, ids=[str(i) for i in range(len(BAD))])
def test_same_refusals(seq):
    with pytest.raises(Exception) as want:
        _lib.i64(seq)
    with pytest.raises(want.type):
        _lib.ints(seq)
