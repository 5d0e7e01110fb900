"""GPU: the z march of the Poisson operators at launch shapes that small grids
do not reach, against the one-point kernels (same taps, same order: equal bits):
the 32-row tiles of order 16, which need 512 tile-chunks of 16 planes, with the
last tile of 1, 3 and 31 rows (so that on a free dim its window is the shifted
one) and a last column tile of 1 and 3 points; and grids of several chunks per
tile whose arrays are beyond the last-level cache."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = [0.3, 0.4, 0.5]


def run(lc, torch, monkeypatch, n, nord, geocode, dt, ops):
    np3 = int(np.prod(n))
    g = torch.Generator(device='cuda').manual_seed(nord + n[1])
    rnd = lambda k: (torch.rand(k * np3, device='cuda', generator=g, dtype=torch.float32) - 0.5).to(dt)
    u, eps, dl, rho = rnd(3), rnd(1), rnd(3), rnd(1)
    outs = []
    for point in (False, True):
        if point:
            monkeypatch.setenv('LIBCONV_POISSON_POINT', '1')
        z = lambda k: torch.full((k * np3,), 7.0, device='cuda', dtype=dt)
        o = []
        if 'div' in ops:
            du, cc, d0 = z(1), z(1), z(1)
            lc.div_u_i(geocode, n, u, du, nord, H, cc)
            lc.div_u_i(geocode, n, u, d0, nord, H)
            o += [du, cc, d0]
        gr, gq, g2, sq, ge, rp = z(3), z(3), z(1), z(1), z(3), rho.clone()
        r2 = torch.zeros(1, device='cuda', dtype=torch.float64)
        lc.nabla_u(geocode, n, u, gr, nord, H)
        lc.nabla_u_and_square(geocode, n, u, gq, g2, nord, H)
        lc.nabla_u_square(geocode, n, u, sq, nord, H)
        lc.nabla_u_epsilon(geocode, n, u, ge, nord, H, eps)
        lc.update_rhopol(geocode, n, u, nord, H, 0.5, dl, rp, r2)
        torch.cuda.synchronize()
        outs.append((o + [gr, gq, g2, sq, ge, rp], float(r2)))
    monkeypatch.delenv('LIBCONV_POISSON_POINT')
    for k, (a, b) in enumerate(zip(outs[0][0], outs[1][0])):
        assert torch.equal(a, b), (n, k)
    # positive FP64 terms in another order: (additions on the longest path) eps
    assert abs(outs[0][1] - outs[1][1]) <= 2 * 8192 * 2.0 ** -53 * outs[1][1]


@pytest.mark.parametrize('n', [[257, 257, 130], [259, 255, 131], [131, 195, 300]], ids=lambda n: 'x'.join(map(str, n)))
@pytest.mark.parametrize('geocode', [1, 2, 3])
@pytest.mark.parametrize('prec', [8, 4])
def test_tall_tiles(gpu, monkeypatch, n, geocode, prec):
    import libconv as lc
    assert ((n[0] + 31) // 32) * ((n[1] + 31) // 32) * (n[2] // 16) >= 512
    run(lc, gpu, monkeypatch, n, 16, geocode, gpu.float64 if prec == 8 else gpu.float32, ())


@pytest.mark.parametrize('nord', [2, 4, 6, 8, 16])
@pytest.mark.parametrize('prec', [8, 4])
def test_chunks_beyond_the_cache(gpu, monkeypatch, nord, prec):
    import libconv as lc
    n, geocode = ([231, 190, 150], 1) if prec == 8 else ([297, 201, 190], 3)
    run(lc, gpu, monkeypatch, n, nord, geocode, gpu.float64 if prec == 8 else gpu.float32, ('div',))
