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


def schedule(N):
    """Radices of wave_fft_units: eights, then one or two fours."""
    log2 = N.bit_length() - 1
    n4 = {0: 0, 2: 1, 1: 2}[log2 % 3]
    return [8] * ((log2 - 2 * n4) // 3) + [4] * n4


def stage(N, NL, R, Ns, unit, slot, PN):
    """Every butterfly of a unit: (lane, reads, writes) as places of the buffer,
    its first place and the offsets from it as the kernel forms them."""
    SPW, NB, PER = 512 // N, N // R, 8 // R
    out = []
    for lane in range(64):
        for p in range(PER):
            b = lane + 64 * p
            l, j = unit * SPW + b // NB, b % NB
            if NL % SPW and l >= NL:
                continue
            base = (j // Ns) * Ns * R + j % Ns
            rd = [l * PN + slot[j] + slot[m * NB] for m in range(R)]
            wr = [l * PN + slot[base] + slot[m * Ns] for m in range(R)]
            assert rd == [l * PN + slot[j + m * NB] for m in range(R)]
            assert wr == [l * PN + slot[base + m * Ns] for m in range(R)]
            out.append((lane, j, rd, wr))
    return out


# (series, waves, padding, first wave) in use: the five or fifteen series of the
# templates and their derivatives, two groups' ten, the wavelet kernels' padded
# ones (whose half-length series start at another wave), the split transforms'
# eight and a layer pass' one wave
CASES = [(5, 1, 0, 0), (5, 4, 0, 0), (5, 8, 0, 0), (10, 16, 0, 0), (15, 8, 0, 0), (15, 1, 0, 0), (1, 1, 0, 0), (8, 8, 1, 0),
         (2, 8, 1, 2), (3, 8, 1, 3), (4, 8, 1, 4), (3, 4, 1, 2), (6, 8, 1, 0), (9, 8, 1, 0), (16, 1, 0, 0)]


@pytest.mark.parametrize("N", [16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("NL,waves,pad,first", CASES)
def test_stages_stay_within_a_wave(lay, N, NL, waves, pad, first):
    slot, PN = lay["slot"], lay["stride"][str(N)] + pad
    SPW = 512 // N
    units = (NL + SPW - 1) // SPW
    # u = wave - first (mod waves), striding by the waves
    owner = {}
    for w in range(waves):
        for u in range(w - first if w >= first else w - first + waves, units, waves):
            assert u not in owner
            owner[u] = w
    assert sorted(owner) == list(range(units))
    every = sorted(l * PN + slot[n] for l in range(NL) for n in range(N))
    assert len(set(every)) == NL * N and every[-1] < NL * PN
    Ns = 1
    for R in schedule(N):
        reads, writes, of = [], [], {}
        for u in range(units):
            for lane, j, rd, wr in stage(N, NL, R, Ns, u, slot, PN):
                reads += rd
                writes += wr
                for e in rd + wr:
                    assert of.setdefault(e, owner[u]) == owner[u]
        assert sorted(reads) == every and sorted(writes) == every
        Ns *= R
    assert Ns == N


@pytest.mark.parametrize("N", [16, 32, 64, 128, 256, 512])
def test_stages_give_the_transform(lay, N):
    slot, PN, NL = lay["slot"], lay["stride"][str(N)], 512 // N + 1
    rng = np.random.default_rng(N)
    x = rng.standard_normal((NL, N)) + 1j * rng.standard_normal((NL, N))
    buf = np.full(NL * PN, np.nan + 0j)
    for l in range(NL):
        buf[[l * PN + s for s in slot[:N]]] = x[l]
    Ns = 1
    for R in schedule(N):
        for u in range((NL * N + 511) // 512):
            done = []
            for lane, j, rd, wr in stage(N, NL, R, Ns, u, slot, PN):
                tw = np.exp(-2j * np.pi * (j % Ns) * np.arange(R) / (R * Ns))
                done.append((wr, np.fft.fft(buf[rd] * tw)))
            for wr, y in done:
                buf[wr] = y
        Ns *= R
    got = np.array([[buf[l * PN + slot[k]] for k in range(N)] for l in range(NL)])
    assert np.max(np.abs(got - np.fft.fft(x, axis=1))) < 1e-12 * np.sqrt(N)


def test_checker_sees_offsets_that_do_not_add_up(lay):
    slot = [n + n // 6 for n in range(512)]
    with pytest.raises(AssertionError):
        stage(64, 8, 8, 8, 0, slot, 80)
