"""Dims arguments of the Python calls that are only passed on (the boundary
conditions, the coarse grid of the work size) are taken in memory order whatever
their shape, as the C array they become; those that are counted stay one
dimensional."""
import numpy as np
import pytest

import libconv as lc


@pytest.mark.parametrize('v', [[[8, 9, 10]], np.array([[8, 9, 10]]), np.array([[8], [9], [10]]), (8, 9, 10)], ids=repr)
def test_passed_on_in_memory_order(v):
    assert list(lc._iv(v, flat=True)) == [8, 9, 10]
    assert lc.local_hamiltonian_work(v) == lc.local_hamiltonian_work([8, 9, 10])


def test_counted_dims_stay_one_dimensional():
    with pytest.raises(TypeError):
        lc._iv([[8, 9, 10]])


@pytest.mark.parametrize('call', ['conv_md', 'conv_1ds', 'wavelet_md'])
def test_conditions_of_any_shape_reach_the_tensor_checks(call):
    torch = pytest.importorskip('torch')
    n = [4, 4, 4]
    x = torch.zeros(64 * 8, dtype=torch.float64)  # on the host: refused after the dims were taken
    args = {'conv_md': (lc.FIL_MD, n, [[0, 0, 0]], n, n, 1, x, x.clone()),
            'conv_1ds': (lc.FIL_D2, n, [[0, 0, 0]], n, n, 1, [1.0] * 3, 0.0, 0.0, x, x.clone()),
            'wavelet_md': (lc.WAV_SYM8, False, n, [[0, 0, 0]], n, n, 1, x, x.clone())}[call]
    with pytest.raises(lc.LibconvError, match='not in device memory'):
        getattr(lc, call)(*args)
