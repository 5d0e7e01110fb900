"""GPU: batched sym8 transforms, both directions, against one call per item, bit
for bit (the layout of a stage splits the work and leaves every output's sum as
it is): stages that fill the chip and take the wide block (131072 output steps
and more), stages of one to a dozen items laid out by the expected time, items
of every boundary condition beside each other, a and a_y on some of them with
y of random values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STAGES = {
    'one': [[33, 20, 17]],
    'flat': [[90, 70, 3], [4, 5, 60], [1, 1, 1]],
    'few': [[24, 40, 31], [31, 9, 50], [40, 40, 40], [17, 64, 8]],
    'dozen': [[16 + 3 * k, 50 - 2 * k, 20 + k] for k in range(12)],
    'wide': [[150 - k, 151 + 2 * k, 3 + k % 5] for k in range(7)],
    'many': [[20 + (7 * k) % 40, 20 + (11 * k) % 37, 6 + k % 9] for k in range(110)],
}


@pytest.mark.parametrize('name', list(STAGES))
@pytest.mark.parametrize('inverse', [False, True])
@pytest.mark.parametrize('acc', [False, True])
@pytest.mark.parametrize('prec', [8, 4])
def test_stage_equals_single_calls(gpu, name, inverse, acc, prec):
    import libconv as lc
    torch = gpu
    dt = torch.float64 if prec == 8 else torch.float32
    g = torch.Generator(device='cuda').manual_seed(len(name) + inverse)
    rnd = lambda k: (torch.rand(k, device='cuda', generator=g, dtype=torch.float64) - 0.5).to(dt)
    items, want = [], []
    for k, n in enumerate(STAGES[name]):
        bc = [(0, 0, 0), (1, 1, 1), (-1, -1, -1), (0, 1, -1)][k % 4]
        nx = [v + 7 if b == -1 else v for v, b in zip(n, bc)]
        ny = [v + 7 if b == 1 else v for v, b in zip(n, bc)]
        x, y0 = rnd(8 * int(np.prod(nx))), rnd(8 * int(np.prod(ny)))
        a, a_y = (0.75, [0.25, 0.0, -0.5][k % 3]) if acc else (1.0, 0.0)
        z = y0.clone()
        lc.wavelet_md(lc.WAV_SYM8, inverse, n, list(bc), nx, ny, 1, x, z, a=a, a_y=a_y)
        want.append(z)
        items.append(dict(kind=lc.BATCH_IDWT if inverse else lc.BATCH_DWT, op=lc.WAV_SYM8, n=n, bc=bc, nx=nx, ny=ny,
                          x=x, y=y0.clone(), a=a, a_y=a_y))
    plan = lc.Batch(items)
    wide = sum(i['ny'][0] * i['ny'][1] for i in items) >= 131072
    assert wide == (name in ('wide', 'many'))
    if wide:
        assert plan.stage_variant(0) == (9 if prec == 8 else 10)
    plan.run()
    torch.cuda.synchronize()
    for k, (it, z) in enumerate(zip(items, want)):
        assert torch.equal(it['y'], z), (k, it['n'], it['bc'])
    plan.close()
