"""The fused Fourier divisions at every tile height and width they run at
(square and not; the last geometry's image columns are past the 6 MB from which
column passes store nontemporally), against the FP64 oracle.  The tolerance is
ten times the oracle's own distance from FP64 with its transforms and products
in float32, at least 1e-5."""
import numpy as np
import pytest

from oracle import deconv_oracle as DO
from oracle import ola_oracle as O
from tests.helpers import case_inputs, rel_l2

pytestmark = pytest.mark.gpu

GEOMS = [((20, 40), (3, 3), (4, 7), (16, 32)), ((40, 20), (3, 3), (7, 4), (32, 16)),
         ((300, 120), (2, 2), (31, 9), (256, 128)), ((90, 330), (3, 2), (9, 27), (64, 256)),
         ((600, 260), (2, 2), (41, 23), (512, 256)), ((250, 610), (2, 2), (15, 63), (256, 512)),
         ((700, 620), (3, 3), (31, 40), (512, 512))]


@pytest.mark.parametrize('sx,csf,sf,tile', GEOMS)
def test_divisions(cuda, sx, csf, sf, tile):
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.olaGPU import OlaGPU
    wa, owa = win2winaux(sx, csf, 0.5), O.Win2WinAux(sx, csf, 0.5)
    x, f, _ = case_inputs(51, sx, csf, sf)
    x32, f32 = x.astype(np.float32), f.astype(np.float32)
    y = O.forward(x32.astype(np.float64), f32.astype(np.float64), owa)
    y32 = (y + 0.01 * np.random.default_rng(52).standard_normal(y.shape)).astype(np.float32)
    x64, f64, y64 = (v.astype(np.float64) for v in (x32, f32, y32))
    F, X = OlaGPU(f32, np.array(sx), 'valid', wa), OlaGPU(x32, np.array(sf), 'valid', wa)
    assert F.plan.tile == tile
    if tile == (512, 512):
        assert csf[0] * csf[1] * F.plan.sw[0] * (tile[1] // 2) * 8 >= 6 << 20
    cases = [('xdirect image', F, dict(mode='xdirect', alpha=0.05, beta=0.01),
              lambda: DO.xdirect(O.OlaOracle(f64, sx, 'valid', owa), y64, 0.05, 0.01)),
             ('xdirect PSFs', X, dict(mode='xdirect', alpha=0.05, beta=0.01),
              lambda: DO.xdirect(O.OlaOracle(x64, sf, 'valid', owa), y64, 0.05, 0.01)),
             ('gdirect', X, dict(mode='gdirect', alpha=0.01, beta=0.01),
              lambda: DO.gdirect(O.OlaOracle(x64, sf, 'valid', owa), y64, 0.01, 0.01)),
             ('sparse', F, dict(mode='sparse', alpha=1e-4),
              lambda: DO.sparse(O.OlaOracle(f64, sx, 'valid', owa), y64, 1e-4))]
    for name, inst, kw, oracle in cases:
        print(f'case {name} tile {tile}', flush=True)
        got = inst.deconv(y32, **kw).cpu().numpy()
        ref = oracle()
        old = O.set_fft(1, True)
        try:
            d = rel_l2(oracle(), ref)
        finally:
            O.set_fft(*old)
        err = rel_l2(got, ref)
        print(f'{name} {tile}: gpu {err:.2e}, fp32 oracle {d:.2e}', flush=True)
        assert err <= max(10 * d, 1e-5), name
