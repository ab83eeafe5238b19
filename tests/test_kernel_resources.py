"""What the compiler makes of the copy kernels: registers decide how many wavefronts a SIMD holds, and scalar registers it runs out of wait in lanes of a vector register, which
each wavefront pays for although no result changes (28 of them made a workgroup per pair 3 - 10 % slower).  Compiled for gfx950 without a GPU, from the compiler's own remarks."""
import os
import re
import subprocess

import pytest

from rbruck_alltoallv_amd import build

# kernel, template arguments (all of them where None): wavefronts a SIMD at least, scalar registers in lanes at most
LIMITS = [
    ("vc_copy_blocks_batch_kernel", r"64, 4, .*", 6, 0),
    ("vc_copy_blocks_batch_kernel", None, 8, 0),
    ("vc_copy_blocks_quarter_kernel", None, 5, 6),
    ("vc_copy_blocks_kernel", r"64, .*", 6, 22),
    ("vc_copy_blocks_kernel", r"256, false, true, .*", 7, 8),
    ("vc_copy_blocks_kernel", None, 7, 0),
    ("vc_copy_chains_kernel", None, 8, 0),
    ("vc_copy_chains_quarter_kernel", None, 8, 0),
    ("vc_copy_items_kernel", None, 8, 0),
    ("vc_copy_items_quarter_kernel", None, 8, 0),
]


@pytest.fixture(scope="module")
def remarks(tmp_path_factory):
    cmd = [build.HIPCC, *[f for f in build.FLAGS if f != "-shared"], "--cuda-device-only", "-c", "-Rpass-analysis=kernel-resource-usage",
           os.path.join(build.CSRC, "vc_copy.hip"), "-o", str(tmp_path_factory.mktemp("resources") / "vc_copy.o")]
    out = subprocess.run(cmd, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    found = re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+).*?Occupancy \[waves/SIMD\]: (\d+).*?SGPRs Spill: (\d+).*?VGPRs Spill: (\d+)", out.stderr, re.S)
    names = subprocess.run(["c++filt"], input="\n".join(f[0] for f in found), capture_output=True, text=True, check=True).stdout.splitlines()
    return {name.replace("void ", "").split("(")[0]: tuple(map(int, f[1:])) for name, f in zip(names, found)}


def test_copy_kernels_keep_their_registers(remarks):
    seen = set()
    for name, (scratch, waves, scalars, vectors) in remarks.items():
        kernel, arguments = re.match(r"(\w+)(?:<(.*)>)?$", name).groups()
        assert scratch == 0 and vectors == 0, name
        for k, (of, pattern, at_least, at_most) in enumerate(LIMITS):
            if kernel == of and (pattern is None or re.fullmatch(pattern, arguments)):
                assert waves >= at_least and scalars <= at_most, (name, waves, scalars)
                seen.add(k)
                break
    assert seen == set(range(len(LIMITS)))
