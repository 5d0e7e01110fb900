"""Dims arguments of the calls on device tensors: the direct conversion to a C
int array accepts, refuses and yields what the general one does."""
import numpy as np
import pytest

import libconv as lc

TAKEN = [[3, 4, 5], (7,), [-1, 0, 1], [True, 2], [np.int64(9), 2], np.array([1, 2], dtype=np.int64), 5,
         np.int32(4), [2.0, 3.7], [2 ** 31 - 1, -2 ** 31], [], np.array([[4], [5]])]
REFUSED = [[2 ** 31], [-2 ** 31 - 1], ['x'], [None], [[1, 2], [3]]]


@pytest.mark.parametrize('v', TAKEN, ids=repr)
def test_same_values(v):
    want = lc._ints(v)
    got = lc._iv(v)
    assert list(got) == [int(k) for k in np.ravel(want)] and len(got) == len(want)


@pytest.mark.parametrize('v', REFUSED, ids=repr)
def test_same_refusals(v):
    with pytest.raises(Exception) as general:
        lc._ints(v)
    with pytest.raises(general.type):
        lc._iv(v)


def test_dtype_names_follow_str():
    torch = pytest.importorskip('torch')
    for dt in (torch.float32, torch.float64, torch.int32):
        for _ in range(2):
            assert lc._dtype_name(torch.zeros(1, dtype=dt)) == str(dt)
    assert lc._dtype_name(np.zeros(1, dtype=np.float32)) == 'float32'
    assert lc._is_f32(np.zeros(1, dtype=np.float32)) and not lc._is_f32(np.zeros(1))
