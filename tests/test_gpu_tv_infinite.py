"""An infinite pixel makes the total variation infinite wherever it lies, also
in the last row and column, whose missing differences are zero (the oracle's
definition); only two infinite neighbours of one sign make it undefined."""
import numpy as np
import pytest

from oracle import loss_oracle as L

pytestmark = pytest.mark.gpu


# widths and row counts of the sum's forms: whole rows, tiles of several rows,
# tiles of part of a row
@pytest.mark.parametrize('shape', [(1, 700, 700), (2, 40, 41), (1, 3, 1500)])
def test_infinite_pixel(cuda, shape):
    import torch
    from vmbd_amd import _lib
    from vmbd_amd.autograd import tv
    print(f'case tv infinite {shape}', flush=True)
    K, H, W = shape
    for i, j in ((0, 0), (H // 2, W - 1), (H - 1, W // 2), (H - 1, W - 1)):
        x = np.random.default_rng(3).random(shape).astype(np.float32)
        x[K - 1, i, j] = np.inf
        assert L.tv(x.astype(np.float64), 0.05) == np.inf
        t = torch.as_tensor(x, device=cuda)
        assert tv(t, 0.05).item() == np.inf, (i, j)
        r = torch.zeros(5, device=cuda)
        part = torch.empty(2 * _lib.lib().vmbd_reduce_blocks(t.numel()), dtype=torch.float64, device=cuda)
        val = torch.empty(1, device=cuda)
        _lib.call('vmbd_loss', _lib.ptr(r), 5, _lib.ptr(t), K, H, W, 0.05, 0.3, _lib.ptr(part), _lib.ptr(val),
                  _lib.stream_ptr())
        assert val.item() == np.inf, (i, j)
