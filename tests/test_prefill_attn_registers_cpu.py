"""What the prefill attention's short-chunk kernels ask a compute unit for, read from the assembly the compiler makes of them."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_turning_its_own_queries_costs_the_attention_no_workgroup(tmp_path):
    """Four waves a workgroup: three of them to a unit are 168 registers a lane (heads of 64), two 256 (of 128), with and without the rotation."""
    spec = importlib.util.spec_from_file_location("mvllm_build_flags", os.path.join(ROOT, "micro-vllm_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not shutil.which(b._hipcc()):
        pytest.skip("no hipcc")
    out = str(tmp_path / "attn_prefill.s")
    subprocess.run([b._hipcc()] + b._flags_for("attn_prefill.hip") + ["-S", "--cuda-device-only", os.path.join(b.CSRC, "attn_prefill.hip"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        text = f.read()
    found = {}
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", text, re.S):
        shape = re.search(r"25paged_attn_prefill_kernelILi(\d+)ELi4ELb([01])E", name)
        if shape:
            found[int(shape.group(1)), shape.group(2) == "1"] = tuple(
                int(re.search(rf"\.amdhsa_{key} (\d+)", body).group(1)) for key in ("next_free_vgpr", "private_segment_fixed_size"))
    assert len(found) == 4 and all(scratch == 0 for _, scratch in found.values()), found
    assert all(regs <= (168 if d == 64 else 256) for (d, _), (regs, _) in found.items()), found
