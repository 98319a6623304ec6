"""The bilateral filter's two tile shapes at their edges, against the FP64
oracle.  A weight 2^t is off by |t| 2^-24 (t rounded, |t| < 20 where it still
counts) and the hardware exponential's 2^-23; 2e-6 covers their weighted
mean."""
import numpy as np
import pytest

from oracle import filters_oracle as FO
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(1, 1), (3, 70), (70, 3), (16, 64), (17, 65), (26, 74), (128, 200),
                                   (512, 1024), (511, 1023), (515, 1030)])
def test_bilateral_tiles(cuda, shape):
    # smaller than the window, one tile, one past it, windows that just fit
    # (26 x 74: one inner workgroup of the one-pixel form), the switch to four
    # pixels per thread at 512 x 1024 and ragged sizes around it
    import torch
    from vmbd_amd import gputools as G
    print(f'case bilateral {shape}', flush=True)
    rng = np.random.default_rng(shape[0] + shape[1])
    a = (rng.random(shape) * 0.2 + (np.add.outer(np.arange(shape[0]), np.arange(shape[1])) // 9 % 2) * 0.7)
    t = torch.as_tensor(a.astype(np.float32), device=cuda)
    G.bfilter_gpu(t, w=5, sigma_d=3, sigma_r=0.1)
    ref = FO.bilateral(a.astype(np.float32).astype(np.float64), 5, 3.0, 0.1)
    assert rel_l2(t.cpu().numpy(), ref) < 2e-6
    assert np.abs(t.cpu().numpy() - ref).max() < 2e-6
