"""GPU: the default route of single and batched sym8 transforms, whose tile and
z chunk follow from the grid, against the step-at-a-time kernel.  Both sum in
the same order, so the bits are equal; the sizes walk the edges of the tiles
(one step, one less and one more than 4, 8, 16), one-step chunks and grids
large enough for several chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [[1, 1, 1], [2, 3, 1], [4, 4, 9], [5, 17, 3], [8, 8, 8], [7, 9, 15], [16, 16, 16], [17, 15, 33],
          [65, 8, 4], [4, 71, 12], [40, 33, 25]]


@pytest.mark.parametrize('n', SHAPES, ids=lambda n: 'x'.join(map(str, n)))
@pytest.mark.parametrize('prec', [8, 4])
@pytest.mark.parametrize('bc', [0, 1, -1])
def test_default_tiles_equal_the_step_kernel(gpu, monkeypatch, n, prec, bc):
    import libconv as lc
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    rng = np.random.default_rng(sum(n) + 10 * (bc + 1))
    nx = [v + 7 if bc == -1 else v for v in n]
    ny = [v + 7 if bc == 1 else v for v in n]
    nin, nout = 8 * int(np.prod(nx)), 8 * int(np.prod(ny))
    for inverse in (False, True):
        for narr, a_y in ((1, 0.0), (2, -0.5)):
            x = torch.from_numpy(rng.uniform(-1, 1, nin * narr)).to('cuda', dt)
            y0 = torch.from_numpy(rng.uniform(-1, 1, nout * narr)).to('cuda', dt)
            got, want = y0.clone(), y0.clone()
            lc.wavelet_md(lc.WAV_SYM8, inverse, n, [bc] * 3, nx, ny, narr, x, got, a_y=a_y)
            monkeypatch.setenv('LIBCONV_WAV3D_VARIANT', '5')
            lc.wavelet_md(lc.WAV_SYM8, inverse, n, [bc] * 3, nx, ny, narr, x, want, a_y=a_y)
            monkeypatch.delenv('LIBCONV_WAV3D_VARIANT')
            torch.cuda.synchronize()
            assert torch.equal(got, want), (inverse, narr)


@pytest.mark.parametrize('count', [1, 40])
def test_batch_tiles_equal_single_calls(gpu, count):
    """A stage that fills the chip takes wider tiles than its items alone."""
    import libconv as lc
    torch = gpu
    rng = np.random.default_rng(count)
    items, single = [], []
    for k in range(count):
        n = [int(v) for v in rng.integers(20, 60, 3)]
        x = torch.from_numpy(rng.uniform(-1, 1, 8 * int(np.prod(n)))).cuda()
        y, z = torch.zeros_like(x), torch.zeros_like(x)
        items.append(dict(kind=lc.BATCH_DWT, op=lc.WAV_SYM8, n=n, bc=0, nx=n, ny=n, x=x, y=y,
                          a_y=0.25 if k == 3 else 0.0))
        lc.wavelet_md(lc.WAV_SYM8, False, n, [0] * 3, n, n, 1, x, z)
        single.append(z)
    plan = lc.Batch(items)
    plan.run()
    torch.cuda.synchronize()
    for it, z in zip(items, single):
        assert torch.equal(it['y'], z)
    plan.close()
