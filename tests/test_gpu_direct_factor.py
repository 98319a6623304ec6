"""'direct' with a crop factor of its own for each axis, which is refused
nowhere: against the oracle at the operators' 1e-5."""
import numpy as np
import pytest

from oracle import deconv_oracle as DO
from oracle import ola_oracle as O
from tests.helpers import case_inputs, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('factor', [np.array([3, 2]), (1, 4), 2])
def test_factor_per_axis(cuda, factor):
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.olaGPU import OlaGPU
    print(f'case direct factor {factor}', flush=True)
    sx, csf, sf = (96, 80), (3, 3), (9, 7)
    x, f, _ = case_inputs(62, sx, csf, sf)
    f32 = f.astype(np.float32)
    owa = O.Win2WinAux(sx, csf, 0.5)
    y = O.forward(x, f32.astype(np.float64), owa).astype(np.float32)
    ref = DO.direct(O.OlaOracle(f32.astype(np.float64), sx, 'valid', owa), y.astype(np.float64), 0.05, 0.01,
                    factor=np.asarray(factor))
    got = OlaGPU(f32, np.array(sx), 'valid', win2winaux(sx, csf, 0.5)).deconv(y, mode='direct', alpha=0.05, beta=0.01,
                                                                             factor=factor)
    assert rel_l2(got.cpu().numpy(), ref) <= 1e-5
