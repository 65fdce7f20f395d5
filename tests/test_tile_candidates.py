"""The compiled launch shapes of the fused eval kernels are different kernels: an
autotuner that is offered copies chooses among them by noise, and a striding grid
is sized by waves that are not there.  Compiles the device code for gfx950 and
compares what the compiler allocated."""
import collections
import os
import re
import shutil

import pytest

from glass_amd import build
from test_kernel_stack import _device_asm

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None and not os.path.exists(build.HIPCC),
                                reason="hipcc not available")


def test_shapes_differ_and_have_their_waves(tmp_path):
    asm = _device_asm("fd_batch.hip", str(tmp_path / "b.s"))
    shapes = collections.defaultdict(list)
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", asm, re.S):
        m = re.match(r"_ZN5glass11eval_kernelILi(\d+)ELi(\d+)ELb([01])ELi(\d+)EE", name)
        if not m:
            continue
        N, nthr, loop, waves = (int(x) for x in m.groups())
        vgpr = int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1))
        scratch = int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", body).group(1))
        # waves a SIMD: 512 vector registers in units of 8
        if waves > 1:
            assert 512 // ((vgpr + 7) // 8 * 8) >= waves, name
        shapes[N, nthr, loop].append((vgpr, scratch))
    assert len({k[0] for k in shapes}) == 8
    for k, v in shapes.items():
        assert len(set(v)) == len(v), (k, v)
