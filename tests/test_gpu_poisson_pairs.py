"""GPU: the z march with two columns per lane against the one-point kernels (same
taps, same order: equal bits) at the edges of its tiles: the smallest grids an
order takes, odd row lengths (a lane with one column), rows around the 32
columns of a tile, planes around the 16 rows, and z ranges with one to several
chunks and their border planes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shapes(nord):
    m = nord + 1
    return [[m, m, m], [m + 1, 17, m], [31, m, 2 * m], [32, 16 + m, m], [33, 31 + m, 40], [65, 33, m + 2],
            [max(m, 47), max(m, 15), 70]]


@pytest.mark.parametrize('nord', [2, 4, 6, 8, 16])
@pytest.mark.parametrize('geocode', [1, 2, 3])
@pytest.mark.parametrize('prec', [8, 4])
def test_pairs_equal_points(gpu, monkeypatch, nord, geocode, prec):
    import libconv as lc
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    h = [0.3, 0.4, 0.5]
    g = torch.Generator(device='cuda').manual_seed(nord)
    for n in shapes(nord):
        np3 = int(np.prod(n))
        rnd = lambda k: (torch.rand(k * np3, device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
        u, eps, dl, rho = rnd(3), rnd(1), rnd(3), rnd(1)
        outs = []
        for point in (False, True):
            if point:
                monkeypatch.setenv('LIBCONV_POISSON_POINT', '1')
            z = lambda k: torch.zeros(k * np3, device='cuda', dtype=dt)
            du, cc, d0, gr, g2, sq, ge, rp = z(1), z(1), z(1), z(3), z(1), z(1), z(3), rho.clone()
            r2 = torch.zeros(1, device='cuda', dtype=torch.float64)
            lc.div_u_i(geocode, n, u, du, nord, h, cc)
            lc.div_u_i(geocode, n, u, d0, nord, h)
            lc.nabla_u_and_square(geocode, n, u, gr, g2, nord, h)
            lc.nabla_u_square(geocode, n, u, sq, nord, h)
            lc.nabla_u_epsilon(geocode, n, u, ge, nord, h, eps)
            lc.update_rhopol(geocode, n, u, nord, h, 0.5, dl, rp, r2)
            torch.cuda.synchronize()
            outs.append((du, cc, d0, gr, g2, sq, ge, rp, r2))
        monkeypatch.delenv('LIBCONV_POISSON_POINT')
        for k, (a, b) in enumerate(zip(*outs)):
            if k == 8:  # FP64 sums of positive terms, grouped differently
                assert abs(a.item() - b.item()) <= 1e-12 * b.item(), n
            else:
                assert torch.equal(a, b), (n, k)
