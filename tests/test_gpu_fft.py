"""The FFT core on its own (every length, both directions) and the operator at
the row counts where its column transforms change to a pruned first pass.

Tolerance: a transform of length N rounds each value about log2 N times, so a
chain of three length-64 transforms stays below 36 roundings of 2^-24 = 2.1e-6
even if they all add up."""
import numpy as np
import pytest

from oracle import ola_oracle as O
from tests.helpers import case_inputs, rel_l2

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.mark.parametrize('n', [16, 32, 64, 128, 256, 512, 1024])
def test_fft_lengths(cuda, n):
    import torch
    from vmbd_amd import _lib
    print(f'case fft {n}', flush=True)
    tw = torch.empty(2048, dtype=torch.float32, device=cuda)
    _lib.call('vmbd_twiddles', _lib.ptr(tw), _lib.stream_ptr())
    rng = np.random.default_rng(n)
    a = (rng.standard_normal((2, n, 16)) + 1j * rng.standard_normal((2, n, 16))).astype(np.complex64)
    a[1] = 0
    a[1, n - 1, 3] = 1  # an impulse: every output is a twiddle
    for x in (a, np.ascontiguousarray(a.swapaxes(1, 2))):
        for d, ref in ((-1, np.fft.fft2), (1, lambda v: np.fft.ifft2(v) * v[0].size)):
            got = torch.as_tensor(x, device=cuda)
            _lib.call('vmbd_fft2', _lib.ptr(got), 2, x.shape[1], x.shape[2], d, 1.0, _lib.ptr(tw), _lib.stream_ptr())
            want = ref(x.astype(np.complex128))
            for k in range(2):
                assert rel_l2(np.stack([got[k].real.cpu(), got[k].imag.cpu()]),
                              np.stack([want[k].real, want[k].imag])) < TOL, (d, k)


@pytest.mark.parametrize('sx,sf', [(72, 12), (72, 13), (75, 12), (75, 14), (69, 11)])
def test_pruned_column_transforms(cuda, sx, sf):
    # tile 64, four rows per slot: 12 or 13 PSF rows, 48, 50 or 46 image rows
    import torch
    from vmbd_amd.imagetools import win2winaux
    from vmbd_amd.ola import OlaPlan
    print(f'case pruned {sx} {sf}', flush=True)
    sx, sf, csf = (sx, sx), (sf, sf), (2, 2)
    x, f, g = (np.asarray(v, np.float32) for v in case_inputs(5, sx, csf, sf))
    wa, owa = win2winaux(sx, csf, 0.5), O.Win2WinAux(sx, csf, 0.5)
    p = OlaPlan(sx, sf, wa, device=cuda)
    assert p.tile == (64, 64)
    t = lambda v: torch.as_tensor(v, device=cuda)
    x64, f64, g64 = (v.astype(np.float64) for v in (x, f, g))
    y = p.forward(t(x), t(f))
    xb, fb = p.adjoint_xf(t(g), t(x), t(f))
    fb1 = p.adjoint_f(t(g), t(x))
    assert rel_l2(y.cpu().numpy(), O.forward(x64, f64, owa)) < TOL
    assert rel_l2(xb.cpu().numpy(), O.adjoint_x(g64, f64, owa, sx, exact=True)) < TOL
    assert rel_l2(fb.cpu().numpy(), O.adjoint_f(g64, x64, owa, sf, exact=True)) < TOL
    assert rel_l2(fb1.cpu().numpy(), O.adjoint_f(g64, x64, owa, sf, exact=True)) < TOL
