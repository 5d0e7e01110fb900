"""GPU: the three energies of lc_conv_1ds and of the local Hamiltonian reach
whatever memory the caller names: device memory, written by the summing kernel,
or host memory, pinned or not, which takes a copy; in a captured call too."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = [20, 17, 33]
A = (ctypes.c_double * 3)(-0.5, -0.4, -0.3)
I3 = ctypes.c_int * 3


def kinetic(lc, x, y, dot, stream=None):
    n, bc = I3(*N), I3(0, 0, 0)
    rc = lc.lib().lc_conv_1ds(8, lc.FIL_D2, 3, n, bc, n, n, 1, A, 0.0, 0.0, x.data_ptr(), y.data_ptr(), dot, stream)
    assert rc == 0


def test_energies_in_host_memory(gpu):
    import libconv as lc
    torch = gpu
    x = torch.rand(int(np.prod(N)), dtype=torch.float64, device='cuda') - 0.5
    y = torch.empty_like(x)
    dev = torch.full((4,), 7.0, dtype=torch.float64, device='cuda')
    pinned = torch.full((4,), 7.0, dtype=torch.float64, pin_memory=True)
    host = np.full(4, 7.0)
    kinetic(lc, x, y, dev.data_ptr())
    kinetic(lc, x, y, pinned.data_ptr())
    kinetic(lc, x, y, host.ctypes.data)
    torch.cuda.synchronize()
    want = dev.cpu().numpy()
    assert want[3] == 7.0 and np.all(want[:3] != 7.0)
    assert np.array_equal(pinned.numpy(), want) and np.array_equal(host, want)


def test_hamiltonian_energies_in_host_memory(gpu):
    import libconv as lc
    torch = gpu
    n = [6, 5, 7]
    m = int(np.prod([2 * v + 29 for v in n]))
    psi = torch.rand(8 * int(np.prod(n)), dtype=torch.float64, device='cuda')
    pot, h = torch.rand(m, dtype=torch.float64, device='cuda'), torch.empty_like(psi)
    work = torch.empty(lc.local_hamiltonian_work(n), dtype=torch.float64, device='cuda')
    dev, host = torch.zeros(3, dtype=torch.float64, device='cuda'), np.zeros(3)
    lc.local_hamiltonian(n, [-0.5, -0.4, -0.3], psi, h, pot, None, work, ekin=dev)
    rc = lc.lib().lc_local_hamiltonian(8, I3(*n), A, ctypes.c_void_p(psi.data_ptr()), ctypes.c_void_p(h.data_ptr()),
                                       ctypes.c_void_p(pot.data_ptr()), None, ctypes.c_void_p(work.data_ptr()),
                                       ctypes.c_void_p(host.ctypes.data), None)
    assert rc == 0
    torch.cuda.synchronize()
    assert np.array_equal(dev.cpu().numpy(), host) and np.all(host != 0.0)


def test_captured_energies(gpu):
    import libconv as lc
    torch = gpu
    x = torch.rand(int(np.prod(N)), dtype=torch.float64, device='cuda') - 0.5
    y, dot, want = torch.empty_like(x), torch.zeros(3, dtype=torch.float64, device='cuda'), torch.zeros(
        3, dtype=torch.float64, device='cuda')
    st = torch.cuda.Stream()
    kinetic(lc, x, y, dot.data_ptr(), st.cuda_stream)  # the stream's scratch
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        kinetic(lc, x, y, dot.data_ptr(), st.cuda_stream)
    for k in range(3):
        x.copy_(torch.rand_like(x) - 0.5)
        dot.zero_()
        g.replay()
        kinetic(lc, x, y, want.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(dot, want), k
