"""What the chunked delta rule's kernels ask a compute unit for, read from the assembly the compiler makes of them."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: (vector registers of a lane, bytes of scratch)}"""
    spec = importlib.util.spec_from_file_location("mvllm_build_flags", os.path.join(ROOT, "micro-vllm_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not shutil.which(b._hipcc()):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("delta") / "delta.s")
    subprocess.run([b._hipcc()] + b._flags_for("delta.hip") + ["-S", "--cuda-device-only", os.path.join(b.CSRC, "delta.hip"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        text = f.read()
    found = {}
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", text, re.S):
        found[name] = tuple(int(re.search(rf"\.amdhsa_{key} (\d+)", body).group(1)) for key in ("next_free_vgpr", "private_segment_fixed_size"))
    return found


def test_two_workgroups_inside_a_chunk_share_a_unit(kernels):
    """Eight waves a workgroup: two of them are four waves a SIMD, of 128 registers a lane each."""
    intra = [v for n, v in kernels.items() if "delta_chunk_intra_kernel" in n]
    assert len(intra) == 1 and intra[0][0] <= 128 and intra[0][1] == 0, intra


def test_two_workgroups_of_the_carry_share_a_unit(kernels):
    """Two sets of operands in at most half of a SIMD's 512 registers, up to 128 state rows; three in all of them past those."""
    carry = {n: v for n, v in kernels.items() if "delta_chunk_carry_kernel" in n}
    assert len(carry) == 6 and all(v[1] == 0 for v in carry.values()), carry
    assert all(v[0] <= (512 if "ILi10E" in n else 256) for n, v in carry.items()), carry
