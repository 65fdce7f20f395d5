"""WDM transforms at the sizes that choose their kernels: columns and rows of 512
to 4096 points (cut to series that a wave transforms), layers of 32 to 512 time
pixels on both sides of the line above which waves take them (2^19 samples for
up to 64 time pixels, 2^20 for more), and above.  Normwise 1e-12 against the
oracle; the largest against the layers of its own spectrum."""
import numpy as np
import pytest

from test_gpu_wdm import grids, normwise

pytestmark = pytest.mark.gpu


# ND/2 = 2^16 (256 x 256), 2^18 (512 x 512), 2^19 (512 x 1024), 2^21 (1024 x 2048), 3 2^18 (768 x 1024)
@pytest.mark.parametrize("NF,NT", [(4096, 32), (8192, 64), (4096, 128), (4096, 256), (8192, 512), (4096, 1024),
                                   (6144, 256)])
def test_forward_sizes(orc, gl, NF, NT):
    from glass_amd import wdm as W
    ow, gw = grids(orc, W, NF, NT)
    x = np.random.default_rng(NF + NT).standard_normal(NF * NT)
    ref = orc.wavelet_transform_timefreq(ow, x)
    got = W.wavelet_transform_timefreq(gw, x)
    assert normwise(got, ref) < 1e-12
    F = np.fft.rfft(x).view(np.float64)
    assert normwise(W.wavelet_transform_freq(gw, F), orc.wavelet_transform_freq(ow, F)) < 1e-12


def test_largest_against_the_spectrum(gl, orc):
    """2^24 points (4096 x 4096): the transform of a series against the layers
    of its own spectrum, which take no column or row pass."""
    from glass_amd import wdm as W
    NF, NT = 8192, 4096
    _, gw = grids(orc, W, NF, NT)
    x = np.random.default_rng(5).standard_normal(NF * NT)
    a = W.wavelet_transform_timefreq(gw, x)
    b = W.wavelet_transform_freq(gw, np.fft.rfft(x).view(np.float64))
    # the same pixels: neither entry normalises the spectrum
    assert normwise(a, b) < 1e-12


# the last below the line, 3 2^17 or 3 2^18 samples, and the first above it
@pytest.mark.parametrize("NF,NT", [(12288, 32), (16384, 32), (6144, 64), (6144, 128), (8192, 128), (3072, 256),
                                   (1536, 512), (2048, 512)])
def test_layers_on_both_sides_of_the_line(orc, gl, NF, NT):
    test_forward_sizes(orc, gl, NF, NT)
