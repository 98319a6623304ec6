"""Where the column passes' stores change: every output of every operator just
below and just above its line (6 MB for one output, 64 MB for each of the
two-adjoint pass's) holds, frame by frame, the bits of batches far below it.
The first geometry's PSF rows take the unpruned store, the second's the one of
three slots."""
import numpy as np
import pytest

from tests.helpers import case_inputs

pytestmark = pytest.mark.gpu

ONE, TWO = 6 << 20, 64 << 20


@pytest.mark.parametrize('sx,csf,sf', [((96, 96), (2, 2), (60, 60)), ((131, 97), (3, 4), (9, 7))])
def test_lines(cuda, sx, csf, sf):
    import torch
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.ola import OlaPlan
    wa = win2winaux(sx, csf, 0.5)
    p0 = OlaPlan(sx, sf, wa, device=cuda)
    assert (sf[0] <= 3 * (p0.tile[0] // 16)) == (sf == (9, 7))
    nbp = -(-(p0.tile[1] // 2 + 2) // 16) * 16
    size = lambda rows: csf[0] * csf[1] * rows * nbp * 8  # bytes of one frame's output
    ext0, sw0, sf0 = int(p0.sw[0]) + sf[0] - 1, int(p0.sw[0]), sf[0]
    x, f, g = (torch.as_tensor(np.asarray(v, np.float32), device=cuda) for v in case_inputs(3, sx, csf, sf))
    cases = [('forward', ext0, ONE, lambda p, X, F, G: (p.forward(X, F),)),
             ('adjoint_x', sw0, ONE, lambda p, X, F, G: (p.adjoint_x(G, F),)),
             ('adjoint_f', sf0, ONE, lambda p, X, F, G: (p.adjoint_f(G, X),)),
             ('adjoint_xf image', sw0, TWO, lambda p, X, F, G: p.adjoint_xf(G, X, F)),
             ('adjoint_xf PSFs', sf0, TWO, lambda p, X, F, G: p.adjoint_xf(G, X, F))]
    for name, rows, line, call in cases:
        n = (line - 1) // size(rows)  # the most frames below the line
        assert n >= 4 and n * size(rows) < line <= (n + 1) * size(rows)
        print(f'case store line {name} {sx}: {n} frames below', flush=True)
        scale = torch.linspace(0.5, 1.5, n + 1, device=cuda)
        X, F, G = (v[None] * scale.view((-1,) + (1,) * v.dim()) for v in (x, f, g))
        p = OlaPlan(sx, sf, wa, max_frames=n + 1, device=cuda)
        p.set_tuning(image_rows=2)  # the same row transforms for every number of frames
        step = max(1, n // 4)
        parts = [call(p, X[k:k + step].contiguous(), F[k:k + step].contiguous(), G[k:k + step].contiguous())
                 for k in range(0, n + 1, step)]
        want = [torch.cat(o) for o in zip(*parts)]
        for m in (n, n + 1):
            got = call(p, X[:m].contiguous(), F[:m].contiguous(), G[:m].contiguous())
            for a, b in zip(got, want):
                assert torch.equal(a, b[:m]), (name, m)
