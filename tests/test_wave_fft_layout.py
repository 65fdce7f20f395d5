"""The padded LDS layout of the wave-held transforms (glass_amd/csrc/fft_lds.h,
wave_fft_units): a unit of 512 points is read and written by one wave's lanes
with no workgroup barrier between the stages, and all places of a butterfly are
constants away from its first.  The layout's own functions are taken from the
headers (compiled for the host); the stages' butterfly -> lane assignment is
enumerated here:
  * a thread's place of a series (FdShape::place) lies in the template's LDS
    buffer for every thread of the workgroup;
  * the offsets add up: slot(j + m N/R) = slot(j) + slot(m N/R), slot(base + m
    Ns) = slot(base) + slot(m Ns);
  * every element of every series is read once and written once in each stage,
    by the wave that has its unit, and each unit has one wave;
  * the stages carried out on the padded buffer give the DFT."""
import json
import os
import shutil
import subprocess

import numpy as np
import pytest

from glass_amd import build

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None and not os.path.exists(build.HIPCC),
                                reason="hipcc not available")

SRC = r"""
#include <cstdio>
#include "fd_waveform.h"
using namespace glass;
template <int N> void shape()
{
    using S = FdShape<N>;
    printf("[%d, %d, %d, %d, %d, %d, [", N, S::NT, S::NTHR, S::PN, S::LDS, S::G);
    for (int t = 0; t < 2 * S::NTHR; t++) printf("%s%d", t ? "," : "", S::place(t));
    printf("], [");
    for (int s = 0; s < S::Q; s++)
        for (int t = 0; t < S::G * (N < 512 ? N : 512); t++)
            printf("%s%d", s || t ? "," : "", S::bin(t % 512, t / 512, s));
    printf("], [");
    for (int n = 0; n < N; n++) printf("%s%d", n ? "," : "", pos_soa_place(N, n));
    printf("]]");
}
int main()
{
    printf("{\"slot\": [");
    for (int n = 0; n < 1024; n++) printf("%s%d", n ? "," : "", wave_fft_slot(n));
    printf("], \"stride\": {");
    for (int N = 16; N <= 512; N *= 2) printf("%s\"%d\": %d", N > 16 ? "," : "", N, wave_fft_stride(N));
    printf("}, \"shapes\": [");
    shape<16>(); printf(",");
    shape<32>(); printf(",");
    shape<64>(); printf(",");
    shape<128>(); printf(",");
    shape<256>(); printf(",");
    shape<512>(); printf(",");
    shape<1024>(); printf(",");
    shape<2048>(); printf(",");
    shape<4096>();
    printf("]}\n");
}
"""


@pytest.fixture(scope="module")
def lay(tmp_path_factory):
    d = tmp_path_factory.mktemp("lay")
    src = d / "lay.hip"
    src.write_text(SRC)
    exe = d / "lay"
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-O3")]
    subprocess.run([build.HIPCC] + flags + ["-O1", "--offload-host-only", "-I", build.CSRC, str(src), "-o", str(exe)],
                   check=True)
    return json.loads(subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout)


def test_places_of_a_template(lay):
    """What every thread of the workgroup may read of each series without a
    test of its index: the adjoint's threads past a series of 32 points did
    read past the buffer."""
    assert [s[0] for s in lay["shapes"]] == [16 << k for k in range(9)]
    for N, NT, NTHR, PN, LDS, G, place, _, _ in lay["shapes"]:
        assert max(place) < PN and LDS == 5 * G * PN, N
        per = [p for t, p in enumerate(place) if t < NT]
        assert len(set(per)) == NT and place[:NT] == lay["slot"][:NT], N


def test_bins_of_a_template(lay):
    """Each bin has one thread and pass, each sample one place in the positions'
    rows.  At 4096 bins a wave's lanes take consecutive bins: eight apart, each
    of eight passes read every line of the window (2.67 against 1.42 ms)."""
    for N, NT, NTHR, PN, LDS, G, _, bins, pos in lay["shapes"]:
        assert sorted(bins) == list(range(N)) and sorted(pos) == list(range(N)), N
        if N == 4096:
            b = np.array(bins).reshape(-1, 64)
            assert np.all(np.diff(b, axis=1) == 1)
            # thread t of a group takes sample 8 t + p in pass p
            p = np.array(pos).reshape(512, 8)
            assert np.all(np.diff(p, axis=0) == 1)
