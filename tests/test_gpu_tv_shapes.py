"""Total variation of image stacks of any shape: values and gradients where a
tile holds several rows, several images, part of a row or its last, shorter
piece, and stacks of small images as fast as one large image of their size."""
import numpy as np
import pytest

from oracle import loss_oracle as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(300, 41, 41), (50, 7, 7), (1, 4096, 16), (1, 3, 5000), (3000, 1, 8), (40, 3, 100),
                                   (1, 1, 3000), (2, 2, 1025), (9, 4, 64), (3, 5, 63), (700, 2, 1), (2, 300, 255),
                                   (2, 300, 257), (1, 700, 1024)])
def test_values_and_gradients(cuda, shape):
    # value: a sum in double of roots rounded to 2^-23, 1e-6 with the final
    # rounding; gradient: three quotients of at most 1, a few roundings each
    import torch
    from vmbd_amd.autograd import tv
    print(f'case tv {shape}', flush=True)
    x = np.random.default_rng(sum(shape)).random(shape).astype(np.float32)
    t = torch.as_tensor(x, device=cuda).requires_grad_()
    v = tv(t, 0.05)
    v.backward()
    x64 = x.astype(np.float64)
    assert abs(v.item() - L.tv(x64, 0.05)) < 1e-6 * L.tv(x64, 0.05)
    assert np.abs(t.grad.cpu().numpy() - L.tv_grad(x64, 0.05)).max() < 1e-5


def test_accumulated_gradient(cuda):
    import torch
    from vmbd_amd import _lib
    print('case tv accumulate', flush=True)
    x = np.random.default_rng(1).random((20, 9, 11)).astype(np.float32)
    t = torch.as_tensor(x, device=cuda)
    g = torch.ones_like(t)
    s = torch.full((1,), 0.5, device=cuda)
    _lib.call('vmbd_tv_grad', _lib.ptr(g), _lib.ptr(t), 20, 9, 11, 0.05, _lib.ptr(s), 3.0, 1, _lib.stream_ptr())
    assert np.abs(g.cpu().numpy() - (1 + 1.5 * L.tv_grad(x.astype(np.float64), 0.05))).max() < 2e-5


@pytest.mark.parametrize('shape', [(3200, 41, 41), (1, 200000, 3), (1, 3, 200000), (20000, 7, 7)])
def test_stacks_cost_what_images_cost(cuda, shape):
    # the same number of pixels 1024 wide; a row per block of 256 threads, or
    # a tile of 64 x 4, took 3 to 25 times that
    import torch
    from vmbd_amd import _lib
    print(f'case tv time {shape}', flush=True)

    def times(K, H, W):
        x = torch.rand((K, H, W), device=cuda)
        g = torch.empty_like(x)
        part = torch.empty(2 * _lib.lib().vmbd_reduce_blocks(x.numel()), dtype=torch.float64, device=cuda)
        val = torch.empty(1, dtype=torch.float64, device=cuda)
        one = torch.ones(1, device=cuda)
        calls = (lambda: _lib.call('vmbd_tv', _lib.ptr(x), K, H, W, 0.05, _lib.ptr(part), _lib.ptr(val),
                                   _lib.stream_ptr()),
                 lambda: _lib.call('vmbd_tv_grad', _lib.ptr(g), _lib.ptr(x), K, H, W, 0.05, _lib.ptr(one), 1.0, 0,
                                   _lib.stream_ptr()))
        out = []
        for fn in calls:
            best = float('inf')
            for _ in range(6):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                for _ in range(20):
                    fn()
                b.record()
                b.synchronize()
                best = min(best, a.elapsed_time(b))
            out.append(best)
        return out
    wide = times(1, -(-int(np.prod(shape)) // 1024), 1024)
    for t, w in zip(times(*shape), wide):
        assert t < 2.5 * w, (t, w)
