"""GPU: every form and chunk of the 1D sweeps on calls large enough to take it.
The form follows from the number of lines and of outputs (256 CUs): tiles of 4,
8 and 16 outputs per lane want 1024 blocks, the forms without a tile want a few
outputs on many lines or a few long lines.

Each call is compared with the same lines in small calls, which run tiles of two
outputs per lane (tested against the oracle elsewhere): every form sums an
output over the same taps in the same order, so the bits are equal.  The energy
is the same products added in another order: a sum of n doubles in any order is
within (additions on the longest path) eps sum|terms| of the exact one, at most
8192 here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PART = 16  # slower-dim slices of a small call


def conv_ext(fil, bc, n):
    w = 15 if fil < 2 else 28
    return n + (w if bc == -1 else 0), n + (w if bc == 1 else 0)


def run_conv(lc, torch, fil, dt, fast, nout, slow, bc):
    """A sweep of `nout` outputs along dim 1 of (fast, line, slow), or along
    dim 0 of (line, slow) with fast = 0; whole or in slices of the slow dim."""
    w = 15 if fil < 2 else 28
    n = nout - w if bc == 1 else nout
    nin, no = conv_ext(fil, bc, n)
    assert no == nout
    L = max(fast, 1)
    g = torch.Generator(device='cuda').manual_seed(nout + slow)
    x = (torch.rand((slow, nin, L), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
    y0 = (torch.rand((slow, no, L), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
    outs, dots = [], []
    for whole in (True, False):
        for kw, dot in ((dict(a=0.75, a_x=0.5, a_y=-0.25), True), (dict(), False)):
            y = y0.clone()
            e = 0.0
            step = slow if whole else PART
            d = torch.zeros(1, dtype=torch.float64, device='cuda')
            parts = []
            for s in range(0, slow, step):
                m = min(step, slow - s)
                if fast:
                    a = ([fast, n, m], [fast, nin, m], [fast, no, m])
                else:
                    a = ([n, m], [nin, m], [no, m])
                lc.conv_1d(fil, 1 if fast else 0, a[0], bc, a[1], a[2], 1, x[s:s + m], y[s:s + m],
                           dot=d if dot else None, **kw)
                if dot:
                    parts.append(d.clone())
            torch.cuda.synchronize()
            outs.append(y)
            if dot:
                dots.append(sum(float(v) for v in parts))
    assert torch.equal(outs[0], outs[2]) and torch.equal(outs[1], outs[3])
    if bc == 0:
        bound = float((x.double().abs() * outs[1].double().abs()).sum()) * 0.75
        assert abs(dots[0] - dots[1]) <= 2 * 8192 * 2.0 ** -53 * bound


# 16384 columns = 512 tiles of 32: 33 .. 64 outputs take 4 per lane, 65 .. 128
# take 8, beyond that 16
@pytest.mark.parametrize('nout', [33, 63, 64, 65, 127, 128, 129, 255, 257])
@pytest.mark.parametrize('bc', [0, 1, -1])
@pytest.mark.parametrize('contig', [False, True])
@pytest.mark.parametrize('prec', [8, 4])
def test_tile_chunks(gpu, nout, bc, contig, prec):
    import libconv as lc
    dt = gpu.float64 if prec == 8 else gpu.float32
    for fil in (lc.FIL_MD, lc.FIL_D2):
        if contig:
            run_conv(lc, gpu, fil, dt, 0, nout, 16380, bc)
        else:
            run_conv(lc, gpu, fil, dt, 30, nout, 546, bc)


# many lines of a few outputs: one lane per column, or a segment per group of lanes
@pytest.mark.parametrize('nout', [1, 2, 4, 5, 11, 12, 13, 16, 24, 25])
@pytest.mark.parametrize('bc', [0, -1])
@pytest.mark.parametrize('contig', [False, True])
@pytest.mark.parametrize('prec', [8, 4])
def test_many_short_lines(gpu, nout, bc, contig, prec):
    import libconv as lc
    dt = gpu.float64 if prec == 8 else gpu.float32
    for fil in (lc.FIL_MD, lc.FIL_D2):
        if contig:
            run_conv(lc, gpu, fil, dt, 0, nout, 24591, bc)
        else:
            run_conv(lc, gpu, fil, dt, 77, nout, 641, bc)  # 49357 columns


@pytest.mark.parametrize('nout', [16, 17, 30])
def test_many_short_grown_lines(gpu, nout):
    """Lines of 1 and more inputs grown by the filter, on the form for many columns."""
    import libconv as lc
    run_conv(lc, gpu, lc.FIL_MD, gpu.float32, 77, nout, 641, 1)
    run_conv(lc, gpu, lc.FIL_MD, gpu.float64, 77, nout, 1705, 1)


@pytest.mark.parametrize('lines,nout', [(1, 60000), (1, 500001), (3, 65537), (4, 60000), (8, 500000)])
@pytest.mark.parametrize('prec', [8, 4])
def test_few_long_lines(gpu, lines, nout, prec):
    """A few long contiguous lines against the same lines along a strided dim
    beside others (tiles)."""
    import libconv as lc
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    g = torch.Generator(device='cuda').manual_seed(nout + lines)
    for fil in (lc.FIL_MD, lc.FIL_D2):
        x = (torch.rand((lines, nout), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
        wide = torch.zeros((nout, 40), device='cuda', dtype=dt)
        wide[:, :lines] = x.t()
        n, nw = [nout, lines], [40, nout]
        y, f, yw = torch.empty_like(x), torch.empty_like(x), torch.empty_like(wide)
        d = torch.zeros(2, dtype=torch.float64, device='cuda')
        lc.conv_1d(fil, 0, n, 0, n, n, 1, x, y, a=0.75, a_x=0.5, dot=d[:1])
        lc.conv_1d(fil, 0, n, 0, n, n, 1, x, f, a=0.75)
        lc.conv_1d(fil, 1, nw, 0, nw, nw, 1, wide, yw, a=0.75, a_x=0.5, dot=d[1:])
        torch.cuda.synchronize()
        assert torch.equal(y, yw[:, :lines].t())
        bound = float((x.double() * f.double()).abs().sum())
        assert abs(float(d[0] - d[1])) <= 2 * 8192 * 2.0 ** -53 * bound


def run_wav(lc, torch, wav, dt, fast, nout, slow, bc, inverse):
    w = 15 if wav == lc.WAV_SYMICOMB8 else 7
    n = nout - w if bc == 1 else nout
    nin = n + (w if bc == -1 else 0)
    L = max(2 * fast, 1)
    g = torch.Generator(device='cuda').manual_seed(nout + slow)
    x = (torch.rand((2 * slow, 2 * nin * L), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
    y0 = (torch.rand((2 * slow, 2 * nout * L), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
    for kw in (dict(), dict(a=0.75, a_y=-0.25)):
        outs = []
        for step in (slow, PART):
            y = y0.clone()
            for s in range(0, slow, step):
                m = min(step, slow - s)
                if fast:
                    a = ([fast, n, m], [fast, nin, m], [fast, nout, m])
                else:
                    a = ([n, m], [nin, m], [nout, m])
                lc.wavelet_1d(wav, inverse, 1 if fast else 0, a[0], bc, a[1], a[2], 1, x[2 * s:2 * (s + m)],
                              y[2 * s:2 * (s + m)], **kw)
            outs.append(y)
        torch.cuda.synchronize()
        assert torch.equal(*outs), kw


# (pairs along the fast dim, output pairs, pairs along the slow dim): tiles of 4
# and 8 output pairs per lane; one lane per column with one and several chunks;
# segments
WAV = [(8, 33, 512), (8, 64, 512), (8, 65, 512), (8, 129, 513), (8, 1, 1540), (8, 2, 1540), (8, 11, 1540),
       (8, 12, 1541), (8, 80, 770), (8, 150, 520), (8, 41, 1541), (4, 161, 1200), (0, 33, 8200), (0, 65, 8190),
       (0, 129, 8192), (0, 1, 12300), (0, 2, 12300), (0, 4, 131100), (0, 3, 12299), (0, 6, 12300)]


@pytest.mark.parametrize('shape', WAV, ids=lambda s: 'x'.join(map(str, s)))
@pytest.mark.parametrize('comb', [False, True])
@pytest.mark.parametrize('prec', [8, 4])
def test_wavelet_forms(gpu, shape, comb, prec):
    import libconv as lc
    fast, nout, slow = shape
    dt = gpu.float64 if prec == 8 else gpu.float32
    wav = lc.WAV_SYMICOMB8 if comb else lc.WAV_SYM8
    for inverse in (False, True):
        for bc in (0, -1, 1):
            if bc == 1 and nout <= (15 if comb else 7):
                continue
            run_wav(lc, gpu, wav, dt, fast, nout, slow, bc, inverse)


@pytest.mark.parametrize('lines,nout', [(1, 16999), (2, 17000), (1, 22000), (4, 25000), (5, 34567), (8, 50000),
                                        (12, 80001), (13, 80001)])
@pytest.mark.parametrize('prec', [8, 4])
def test_long_lines_among_others(gpu, lines, nout, prec):
    test_few_long_lines(gpu, lines, nout, prec)


@pytest.mark.parametrize('lines,nout', [(2, 33999), (4, 34001), (8, 49999), (8, 50000), (12, 80000), (16, 80001)])
@pytest.mark.parametrize('prec', [8, 4])
def test_wavelet_long_lines(gpu, lines, nout, prec):
    """The lines of a few-line call against the same lines among many."""
    import libconv as lc
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    g = torch.Generator(device='cuda').manual_seed(nout + lines)
    for wav in (lc.WAV_SYM8, lc.WAV_SYMICOMB8):
        for inverse in (False, True):
            wide = (torch.rand((32, 2 * nout), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
            y0 = (torch.rand((32, 2 * nout), device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
            for kw in (dict(), dict(a=0.75, a_y=-0.25)):
                y, yw = y0[:lines].clone(), y0.clone()
                n, nw = [nout, lines // 2], [nout, 16]
                lc.wavelet_1d(wav, inverse, 0, n, 0, n, n, 1, wide[:lines].contiguous(), y, **kw)
                lc.wavelet_1d(wav, inverse, 0, nw, 0, nw, nw, 1, wide, yw, **kw)
                torch.cuda.synchronize()
                assert torch.equal(y, yw[:lines])
