"""Column passes store outputs of 4 MB and more with other store instructions
than smaller ones: batches on both sides of that size hold, frame by frame,
the bits of the frames run alone."""
import numpy as np
import pytest

from tests.helpers import case_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('sx,csf,sf', [((50, 50), (2, 2), (5, 5)), ((131, 97), (3, 4), (9, 7)),
                                       ((256, 256), (4, 4), (15, 15)), ((300, 410), (3, 3), (31, 40))])
def test_both_sides_of_the_line(cuda, sx, csf, sf):
    import torch
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.ola import OlaPlan
    wa = win2winaux(sx, csf, 0.5)
    p = OlaPlan(sx, sf, wa, device=cuda)
    ext, nbp = p.sw[0] + sf[0] - 1, -(-(p.tile[1] // 2 + 2) // 16) * 16
    n = (4 << 20) // (csf[0] * csf[1] * ext * nbp * 8)  # the forward's frames below the line
    assert n >= 1
    frames = n + 2
    print(f'case stores {sx} {csf} {sf}: {n} frames below the line', flush=True)
    x, f, g = (torch.as_tensor(np.asarray(v, np.float32), device=cuda) for v in case_inputs(3, sx, csf, sf))
    scale = torch.linspace(0.5, 1.5, frames, device=cuda)
    X, F, G = (v[None] * scale.view((-1,) + (1,) * v.dim()) for v in (x, f, g))
    p = OlaPlan(sx, sf, wa, max_frames=frames, device=cuda)
    p.set_tuning(image_rows=2)  # the same row transforms for every number of frames
    one = []
    for k in range(frames):
        y = p.forward(X[k], F[k])
        one.append((y,) + tuple(p.adjoint_xf(G[k], X[k], F[k])))
    for m in (n, n + 1, frames):
        y = p.forward(X[:m].contiguous(), F[:m].contiguous())
        xb, fb = p.adjoint_xf(G[:m].contiguous(), X[:m].contiguous(), F[:m].contiguous())
        for k in range(m):
            assert torch.equal(y[k], one[k][0]) and torch.equal(xb[k], one[k][1]) and torch.equal(fb[k], one[k][2])
