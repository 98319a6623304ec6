"""The frequency terms of the Fourier divisions, compiled for the host, are no
further from their 64-bit values than the same formulas on correctly rounded
sines and cosines (what per-frequency trigonometry gives): rms over the
frequencies of every tile length, plus 2 % for a rounding more or less."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'vmbd_amd', 'csrc')
f32 = np.float32


def test_rms_error(tmp_path):
    cxx = shutil.which('g++') or shutil.which('clang++')
    if cxx is None:
        pytest.skip('no host compiler')
    exe = str(tmp_path / 'div_terms')
    subprocess.run([cxx, '-O1', '-std=c++17', '-w', '-ffp-contract=off', '-I', os.path.join(HERE, 'host'), '-I', CSRC,
                    os.path.join(HERE, 'host', 'div_terms.cpp'), '-o', exe], check=True)
    out = np.loadtxt(subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines())
    for T in (16, 32, 64, 128, 256, 512):
        got = out[out[:, 0] == T]
        q = got[:, 1]
        assert np.array_equal(q, np.arange(T))
        w = 2 * np.pi * q / T
        exact = (4 * np.sin(w / 2) ** 2, (1 + 2 * np.cos(w)) ** 2, np.sqrt(0.5) * (np.cos(w) - 1),
                 -np.sqrt(0.5) * np.sin(w))
        s, c, c2, s2 = (f32(v) for v in (np.sin(w / 2), np.cos(w / 2), np.cos(w), np.sin(w)))
        plain = (f32(4) * s * s, (f32(1) + f32(2) * c2) ** 2, f32(np.sqrt(0.5)) * (c2 - f32(1)),
                 -f32(np.sqrt(0.5)) * s2)
        rms = lambda a, b: np.sqrt(np.mean((a.astype(np.float64) - b) ** 2))
        for k in range(4):
            assert rms(f32(got[:, 2 + k]), exact[k]) <= 1.02 * rms(plain[k], exact[k]), (T, k)
