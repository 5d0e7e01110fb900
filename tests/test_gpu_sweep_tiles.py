"""GPU: the tiled 1D sweeps at the edges of their tiles: lines of 1 .. a few
chunks of outputs (8 lanes of 2, 4, 8 or 16 outputs each), columns around the
32 of a tile, lines shorter than the filter, several arrays and every epilogue
term, against the FP64 oracle (1e-13 relative, the bar of the parity tests).
FP32 lines along the contiguous dim equal the same lines along a strided dim
bit for bit: both kernels sum in the same order."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize('length', [1, 15, 16, 17, 33, 64, 65, 128, 129, 300])
@pytest.mark.parametrize('bc', [0, 1, -1])
@pytest.mark.parametrize('idim', [0, 1])
@pytest.mark.parametrize('lines', [1, 31, 33, 700])
def test_conv_lines(gpu, length, bc, idim, lines):
    import libconv as lc
    torch = gpu
    rng = np.random.default_rng(length * 7 + lines + idim)
    n = [length, lines] if idim == 0 else [lines, length]
    for fil in (O.MD, O.D2):
        nin, nout = O.conv_extents(fil, bc, length)
        nx, ny = list(n), list(n)
        nx[idim], ny[idim] = nin, nout
        narr = 2
        x = rng.uniform(-1, 1, nin * lines * narr)
        y0 = rng.uniform(-1, 1, nout * lines * narr)
        a, ax, ay = 0.75, 0.5, -0.25
        ref = y0.copy()
        rdot = O.s0s0_1d(fil, idim, n, bc, nx, ny, narr, x, ref, a, ax, ay, want_dot=True)
        y = torch.from_numpy(y0).cuda()
        dot = torch.zeros(1, dtype=torch.float64, device='cuda')
        lc.conv_1d(fil, idim, n, bc, nx, ny, narr, torch.from_numpy(x).cuda(), y, a=a, a_x=ax, a_y=ay, dot=dot)
        torch.cuda.synchronize()
        assert rel(y.cpu().numpy(), ref) < 1e-13, fil
        # a sum of up to lines * length products of cancelling signs
        assert abs(dot.item() - rdot) < 1e-12 * np.sqrt(lines * max(nin, nout)) * 4.0


@pytest.mark.parametrize('length', [1, 16, 17, 65, 129])
@pytest.mark.parametrize('bc', [0, 1, -1])
@pytest.mark.parametrize('lines', [2, 33, 500])
def test_contiguous_equals_strided_fp32(gpu, length, bc, lines):
    import libconv as lc
    torch = gpu
    g = torch.Generator(device='cuda').manual_seed(length + lines)
    nin, nout = O.conv_extents(O.D2, bc, length)
    x = torch.rand((lines, nin), device='cuda', generator=g) - 0.5
    y = torch.rand((lines, nout), device='cuda', generator=g)
    xt, yt = x.t().contiguous(), y.t().contiguous()
    kw = dict(a=0.75, a_x=0.5, a_y=-0.25)
    lc.conv_1d(lc.FIL_D2, 0, [length, lines], bc, [nin, lines], [nout, lines], 1, x, y, **kw)
    lc.conv_1d(lc.FIL_D2, 1, [lines, length], bc, [lines, nin], [lines, nout], 1, xt, yt, **kw)
    for wav, w in ((lc.WAV_SYM8, 8), (lc.WAV_SYMICOMB8, 16)):
        ni, no = length + (w - 1 if bc == -1 else 0), length + (w - 1 if bc == 1 else 0)
        for inverse in (False, True):
            v = torch.rand((2 * lines, 2 * ni), device='cuda', generator=g) - 0.5
            vt = v.t().contiguous()
            o = torch.empty((2 * lines, 2 * no), device='cuda')
            ot = torch.empty((2 * no, 2 * lines), device='cuda')
            lc.wavelet_1d(wav, inverse, 0, [length, lines], bc, [ni, lines], [no, lines], 1, v, o)
            lc.wavelet_1d(wav, inverse, 1, [lines, length], bc, [lines, ni], [lines, no], 1, vt, ot)
            torch.cuda.synchronize()
            assert torch.equal(o.t(), ot), (wav, inverse)
    assert torch.equal(y.t(), yt)


@pytest.mark.parametrize('length', [1, 7, 8, 16, 33, 65])
@pytest.mark.parametrize('bc', [0, 1, -1])
@pytest.mark.parametrize('idim', [0, 1])
@pytest.mark.parametrize('comb', [False, True])
def test_wavelet_lines(gpu, length, bc, idim, comb):
    import libconv as lc
    torch = gpu
    rng = np.random.default_rng(length + idim)
    wav, w = (O.SYMICOMB8, 16) if comb else (O.SYM8, 8)
    for lines in (1, 17, 400):
        n = [length, lines] if idim == 0 else [lines, length]
        nx, ny = list(n), list(n)
        nx[idim] += w - 1 if bc == -1 else 0
        ny[idim] += w - 1 if bc == 1 else 0
        x = rng.uniform(-1, 1, 4 * nx[0] * nx[1])
        y0 = rng.uniform(-1, 1, 4 * ny[0] * ny[1])
        for inverse in (False, True):
            ref = y0.copy()
            (O.s1s0_1d if inverse else O.s0s1_1d)(wav, idim, n, bc, nx, ny, 1, x, ref, 0.75, -0.5)
            y = torch.from_numpy(y0).cuda()
            lc.wavelet_1d(wav, inverse, idim, n, bc, nx, ny, 1, torch.from_numpy(x).cuda(), y, a=0.75, a_y=-0.5)
            torch.cuda.synchronize()
            assert rel(y.cpu().numpy(), ref) < 1e-13, (lines, inverse)
