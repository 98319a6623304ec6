"""OlaLoss with a forward-mode tangent on the observation: the derivative of
1/2 |B(x, f) - y|^2 along t is -(B(x, f) - y) . t."""
import numpy as np
import pytest

from oracle import ola_oracle as O
from tests.helpers import case_inputs

pytestmark = pytest.mark.gpu


def test_tangent_of_the_observation(cuda):
    import torch
    import torch.autograd.forward_ad as fwAD
    from vmbd_amd.autograd import OlaLoss
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.ola import OlaPlan
    print('case loss tangent', flush=True)
    sx, csf, sf = (64, 64), (2, 2), (5, 5)
    x, f, t = (v.astype(np.float32) for v in case_inputs(61, sx, csf, sf))
    y = np.full(t.shape, 0.25, np.float32)
    plan = OlaPlan(sx, sf, win2winaux(sx, csf, 0.5), device=cuda)
    X, F, Y, T = (torch.as_tensor(v, device=cuda) for v in (x, f, y, t))
    with fwAD.dual_level():
        out = fwAD.unpack_dual(OlaLoss(plan, 1e-3, 1e-2)(X, F, fwAD.make_dual(Y, T)))
    r = O.forward(x.astype(np.float64), f.astype(np.float64), O.Win2WinAux(sx, csf, 0.5)) - y
    # float32 products and their sum over 3600 values, the residual to 1e-6
    assert abs(out.tangent.item() + float((r * t).sum())) < 1e-5 * float(np.abs(r * t).sum())
    plain = OlaLoss(plan, 1e-3, 1e-2)(X, F, Y).item()
    assert abs(out.primal.item() - plain) < 1e-5 * plain
