"""The z chunks of the fused 3D kernels, picked per grid from the expected time
of the busiest CU, and the magic filter with the potential step.

Chunking and tiling only split the work: every output is summed over the same
taps in the same order by every form, so the default kernels must give the
bits of the general forms (variants 12 and 8), whose chunks are long.  Sizes:
grids of one short chunk, chunks of the least length with a remainder, ragged
tiles, grids near one and two blocks per CU, and marches of hundreds of planes.

Energies are sums of the same products, regrouped by chunk.  A sum of n
doubles in any order is within (depth) eps sum|terms| of the exact one, where
depth counts the additions on the longest path: at most 4096 here (rows and
planes of a lane, lanes, partials of 1024 threads).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(3, 5, 4), (17, 33, 9), (33, 17, 64), (31, 34, 63), (40, 40, 130), (96, 90, 101), (129, 65, 48),
         (12, 9, 300), (160, 144, 33)]


@pytest.fixture(scope='module')
def lc(gpu):
    import libconv
    libconv.lib()
    return libconv


def _ext(n, bc, w):
    return [v + w if b == -1 else v for v, b in zip(n, bc)], [v + w if b == 1 else v for v, b in zip(n, bc)]


@pytest.mark.parametrize('bc', [(0, 0, 0), (1, 0, 1), (-1, -1, -1)])
@pytest.mark.parametrize('prec', [8, 4])
def test_default_chunks_equal_general_forms(lc, gpu, monkeypatch, prec, bc):
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    rng = np.random.default_rng(71 + prec)
    for n in SIZES:
        for fil, w in ((0, 15), (2, 28)):
            nx, ny = _ext(n, bc, w)
            x = torch.from_numpy(rng.uniform(-1, 1, int(np.prod(nx)))).to('cuda', dt)
            y0 = torch.from_numpy(rng.uniform(-1, 1, int(np.prod(ny)))).to('cuda', dt)
            got = []
            for v in (None, '12' if fil == 0 else '8'):
                key = 'LIBCONV_SEP3D_VARIANT' if fil == 0 else 'LIBCONV_SUM3D_VARIANT'
                monkeypatch.delenv(key, raising=False)
                if v:
                    monkeypatch.setenv(key, v)
                y = y0.clone()
                dot = torch.zeros(3, dtype=torch.float64, device='cuda')
                if fil == 0:
                    lc.conv_md(0, n, bc, nx, ny, 1, x, y, a=0.75, a_y=0.5)
                    y2 = y0.clone()
                    lc.conv_md(0, n, bc, nx, ny, 1, x, y2)
                else:
                    lc.conv_1ds(2, n, bc, nx, ny, 1, [-0.5, 0.25, 2.0], 0.5, 0.0, x, y, dot=dot)
                    y2 = y0.clone()
                    lc.conv_1ds(2, n, bc, nx, ny, 1, [-0.5, 0.25, 2.0], 0.0, 0.5, x, y2)
                got.append((y, y2, dot))
            torch.cuda.synchronize()
            (ya, y2a, da), (yb, y2b, db) = got
            assert torch.equal(ya, yb) and torch.equal(y2a, y2b), (n, bc, fil)
            if fil == 2 and bc == (0, 0, 0):
                for d, ad in enumerate((-0.5, 0.25, 2.0)):
                    a1 = [ad if k == d else 0.0 for k in range(3)]
                    t = torch.empty_like(x)
                    lc.conv_1ds(2, n, bc, nx, ny, 1, a1, 0.0, 0.0, x, t)
                    terms = float((x.double() * t.double()).abs().sum())
                    # FP32: the products are of values rounded to FP32 in both forms alike
                    assert abs(float(da[d] - db[d])) <= 2 * 4096 * 2.0 ** -53 * terms, (n, d)


@pytest.mark.parametrize('prec', [8, 4])
def test_potential_step_equals_general_form(lc, gpu, monkeypatch, prec):
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    rng = np.random.default_rng(5 + prec)
    for n in [(1, 1, 1), (2, 9, 3), (18, 3, 20), (33, 20, 41)]:
        m = int(np.prod([2 * v + 29 for v in n]))
        dev = lambda k: torch.from_numpy(rng.uniform(-1, 1, k)).to('cuda', dt)
        psi, pot, rho0 = dev(8 * int(np.prod(n))), dev(m), dev(m)
        work = torch.empty(lc.local_hamiltonian_work(n), dtype=dt, device='cuda')
        for with_rho in (True, False):
            got = []
            for v in (None, '12'):
                monkeypatch.delenv('LIBCONV_SEP3D_VARIANT', raising=False)
                if v:
                    monkeypatch.setenv('LIBCONV_SEP3D_VARIANT', v)
                rho, h = rho0.clone(), torch.full_like(psi, float('nan'))
                lc.local_hamiltonian(n, [-0.5, -0.4, -0.3], psi, h, pot, rho if with_rho else None, work)
                got.append((h, rho))
            torch.cuda.synchronize()
            assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), (n, with_rho)
