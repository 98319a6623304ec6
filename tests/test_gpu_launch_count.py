"""The launches a step reports are the launches it makes (the library's own
kernel timing counts them)."""
import pytest

from tests.test_gpu_batch import SPECS, _frames

pytestmark = pytest.mark.gpu


def _count(fn):
    import torch
    from vmbd_amd import _lib
    fn()  # (binds what a first call binds)
    torch.cuda.synchronize()
    _lib.prof_reset()
    _lib.prof_enable(True)
    try:
        fn()
        torch.cuda.synchronize()
        return sum(c for c, _, _ in _lib.prof_report().values())
    finally:
        _lib.prof_enable(False)
        _lib.prof_reset()


@pytest.mark.parametrize('grouped', [True, False])
def test_mixed_batch(cuda, grouped):
    from vmbd_amd.batch import MixedBatch
    print(f'case launches grouped={grouped}', flush=True)
    mb = MixedBatch(SPECS, grouped=grouped)
    mb.load(*_frames(cuda))
    assert _count(mb.step) == mb.kernel_launches


@pytest.mark.parametrize('separable', [True, False])
def test_plan_step(cuda, separable):
    import torch
    from vmbd_amd import _lib
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.ola import OlaPlan
    print(f'case launches separable={separable}', flush=True)
    sx, sf, csf = (96, 96), (9, 9), (3, 3)
    p = OlaPlan(sx, sf, win2winaux(sx, csf, 0.5), device=cuda, separable=separable)
    x, f, g = (torch.rand(s, device=cuda) for s in (sx, (9,) + sf, p.sy))
    n = _lib.lib().vmbd_plan_step_launches(p._h, 1)
    assert n == (6 if separable else 7)
    assert _count(lambda: (p.forward(x, f), p.adjoint_xf(g, x, f))) == n
    assert _lib.lib().vmbd_plan_step_launches(p._h, 2) < 0 and _lib.lib().vmbd_plan_step_launches(None, 1) < 0
