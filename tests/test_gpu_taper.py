"""Border tapers with the tables as kernel arguments, and the one-pass end of
'direct', against the oracle's filters.  A value takes at most the roundings of
its two table entries, two products, a clip and a division: 6 * 2^-24 < 4e-7."""
import numpy as np
import pytest

from oracle import filters_oracle as FO
from oracle import ola_oracle as O
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

TOL = 4e-7


@pytest.mark.parametrize('sf', [(1, 1), (2, 3), (3, 64), (82, 82), (126, 127), (255, 256), (257, 40), (300, 2)])
def test_edgetaper_sizes(cuda, sf):
    # tapers from none to half the image, to the last size passed as
    # arguments (256) and the first one that takes device tables (257)
    import torch
    from vmbd_amd import gputools as G
    print(f'case edgetaper {sf}', flush=True)
    y = np.random.default_rng(7).random((311, 290)).astype(np.float32)
    t = torch.as_tensor(y, device=cuda).clone()
    G.edgetaper_gpu(t, np.array(sf))
    ref = FO.edgetaper(y.astype(np.float64), np.array(sf))
    assert np.abs(t.cpu().numpy() - ref).max() <= TOL


@pytest.mark.parametrize('shape,sf,factor', [((96, 96), (9, 9), 3), ((70, 131), (6, 11), 3), ((64, 65), (5, 4), 1),
                                             ((40, 41), (13, 13), 2)])
def test_direct_ratio(cuda, shape, sf, factor):
    import torch
    from vmbd_amd import _lib
    print(f'case direct ratio {shape} {sf}', flush=True)
    rng = np.random.default_rng(8)
    num = rng.standard_normal(shape).astype(np.float32)
    den = (12 * rng.random(shape) - 1).astype(np.float32)  # both clips
    sfa = np.array(sf)
    m, n = (int(v) for v in np.array(shape) - factor * sfa - 1)
    o0, o1 = (int(v) for v in np.floor((factor * sfa - 1) / 2.0))
    a, b = (torch.as_tensor(v, device=cuda) for v in (num, den))
    out = torch.empty_like(a)
    _lib.call('vmbd_direct_ratio', _lib.ptr(out), _lib.ptr(a), _lib.ptr(b), shape[0], shape[1], 2 * sf[0], 2 * sf[1],
              o0, o1, m, n, _lib.stream_ptr())
    d = np.clip(FO.edgetaper(den.astype(np.float64), 2 * sfa), 0.01, 10.0)
    z = O.crop(np.maximum(num.astype(np.float64), 0) / d, (m, n), (o0, o1))
    assert rel_l2(out.cpu().numpy(), FO.impad(z, tuple(np.array(shape) - (m, n)))) <= TOL
    for bad in ((-1, o1, m, n), (o0, o1, 0, n), (o0, o1, shape[0], n)):
        with pytest.raises(_lib.VmbdError):
            _lib.call('vmbd_direct_ratio', _lib.ptr(out), _lib.ptr(a), _lib.ptr(b), shape[0], shape[1], 2 * sf[0],
                      2 * sf[1], *bad, _lib.stream_ptr())
