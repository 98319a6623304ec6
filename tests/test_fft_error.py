"""Rounding error of the FFT core, its arithmetic compiled for the host.

The bounds are those of the textbook form of the same passes (radix-16 passes
of radix-4 butterflies, each input of a pass multiplied by its own twiddle from
the table): its relative rms against 64 bits in the same harness, plus 2 % for
the scatter of 51200 values (their rms varies by less than 1 %)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'vmbd_amd', 'csrc')

# length: (normal input, smooth windowed input), 1e-8
TEXTBOOK = {16: (6.25, 6.21), 32: (7.34, 7.17), 64: (8.07, 7.73), 128: (8.79, 8.49), 256: (9.53, 9.08),
            512: (10.25, 9.64), 1024: (11.55, 10.52)}


@pytest.fixture(scope='module')
def lines(tmp_path_factory):
    cxx = shutil.which('g++') or shutil.which('clang++')
    if cxx is None:
        pytest.skip('no host compiler')
    exe = str(tmp_path_factory.mktemp('fft') / 'fft_error')
    # one rounding per operation, FMAs where the source asks for them
    subprocess.run([cxx, '-O1', '-std=c++17', '-w', '-ffp-contract=off', '-I', os.path.join(HERE, 'host'), '-I', CSRC,
                    os.path.join(HERE, 'host', 'fft_error.cpp'), '-o', exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {(int(w[0]), int(w[1])): [float(v) for v in w[2:]] for w in map(str.split, out.splitlines())}


@pytest.mark.parametrize('smooth', [0, 1])
@pytest.mark.parametrize('n', sorted(TEXTBOOK))
def test_rms_error(lines, n, smooth):
    # forward and inverse, twiddles from a plan's table and from exponentials
    assert len(lines[n, smooth]) == 4
    assert max(lines[n, smooth]) < 1.02e-8 * TEXTBOOK[n][smooth], lines[n, smooth]
