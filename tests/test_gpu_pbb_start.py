"""The start of the projected Barzilai-Borwein solver in two launches against
the dots and the selection in calls of their own: the same sums in the same
order, so every value is the same."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,m', [(1, 1), (255, 257), (2048, 1), (61504, 260100), (131073, 300000), (300000, 17)])
@pytest.mark.parametrize('second', [0.5, 2.0])
def test_pbb_start(cuda, n, m, second):
    # one block, one past it, past the 512 partials of one norm or of both;
    # a second point that is better (the pairs change places) or worse
    import torch
    from vmbd_amd import _lib
    print(f'case pbb start {n} {m} {second}', flush=True)
    rng = np.random.default_rng(n + m)

    def dev(a):
        return torch.as_tensor(a.astype(np.float32), device=cuda)

    x, u, g, og = (dev(rng.standard_normal(n)) for _ in range(4))
    r = dev(rng.standard_normal(m) + 1.0)
    r2, beta, st = r * second, 1e-3 if n < m else 0.0, _lib.stream_ptr()
    y = torch.empty_like(x)
    _lib.call('vmbd_pbb_start', _lib.ptr(y), _lib.ptr(u), _lib.ptr(x), n, st)
    assert torch.equal(y, (u - x) - 0.5)
    part = torch.empty(4 * _lib.lib().vmbd_reduce_blocks(max(n, m)), dtype=torch.float64, device=cuda)
    got = [x.clone(), y.clone(), g.clone(), og.clone()]
    _lib.call('vmbd_pbb_choose', *(_lib.ptr(t) for t in got), n, _lib.ptr(r), _lib.ptr(r2), m, beta, _lib.ptr(part), st)
    want, dots = [x.clone(), y.clone(), g.clone(), og.clone()], torch.zeros(4, dtype=torch.float64, device=cuda)
    for k, t in enumerate((r, x, r2, y)):
        out = ctypes.c_void_p(dots.data_ptr() + 8 * k)
        _lib.call('vmbd_dot', _lib.ptr(t), _lib.ptr(t), t.numel(), _lib.ptr(part), out, st)
    _lib.call('vmbd_pbb_select', *(_lib.ptr(t) for t in want), n, _lib.ptr(dots), beta, st)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    d = dots.cpu().numpy()
    assert torch.equal(got[0], y if d[0] + beta * d[1] >= d[2] + beta * d[3] else x)
