"""GPU: a stage whose variant is chosen, by the tuner's table or by the
environment, keeps it, also where the stage is large enough for the wide
default block of the batched wavelets (items of 150^2 pairs: 22500 output steps
a plane, the default changes at 131072 a stage)."""
import json

import pytest

pytestmark = pytest.mark.gpu

N = [150, 150, 4]
COUNT = 6  # 135000 steps


def stage(lc, torch, dt, kind=None):
    x = torch.rand(8 * N[0] * N[1] * N[2], device='cuda', dtype=dt)
    ys = [torch.empty_like(x) for _ in range(COUNT)]
    items = [dict(kind=lc.BATCH_DWT if kind is None else kind, op=lc.WAV_SYM8, n=N, bc=0, nx=N, ny=N, x=x, y=y)
             for y in ys]
    plan = lc.Batch(items)
    v = plan.stage_variant(0)
    plan.run()
    torch.cuda.synchronize()
    plan.close()
    want = torch.empty_like(x)
    lc.wavelet_md(lc.WAV_SYM8, items[0]['kind'] == lc.BATCH_IDWT, N, [0] * 3, N, N, 1, x, want)
    torch.cuda.synchronize()
    assert all(torch.equal(y, want) for y in ys)
    return v


@pytest.mark.parametrize('prec', [8, 4])
@pytest.mark.parametrize('v', [5, 7, 12, 14])
def test_environment_choice_is_kept(gpu, monkeypatch, prec, v):
    import libconv as lc
    dt = gpu.float64 if prec == 8 else gpu.float32
    default = stage(lc, gpu, dt)
    assert default == (9 if prec == 8 else 10)  # the wide block: the stage is above the bound
    monkeypatch.setenv('LIBCONV_WAV3D_VARIANT', str(v))
    assert stage(lc, gpu, dt) == v
    assert stage(lc, gpu, dt, lc.BATCH_IDWT) == v


def test_tuned_choice_is_kept(gpu, tmp_path):
    import libconv as lc
    f = tmp_path / 'tuned.json'
    f.write_text(json.dumps({'prec': 8, 'form': lc.FORM_DWT, 'op': lc.WAV_SYM8, 'n': N, 'bc': [0, 0, 0], 'nx': N,
                             'ny': N, 'variant': 12, 'ms': 0.1}, separators=(',', ':')) + '\n')
    lc.tune_clear()
    try:
        lc.tune_load(str(f))
        assert stage(lc, gpu, gpu.float64) == 12
    finally:
        lc.tune_clear()
    assert stage(lc, gpu, gpu.float64) == 9
