"""What the pick's kernels keep out of registers, read from the assembly the compiler makes of them."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_selection_in_line_uses_no_scratch(tmp_path):
    """Picks past 256 candidates always take the radix selection or may fall back to it after the parts met: in line, no register of
    theirs goes to memory on the way (called, 60 a lane do: 128 rows of 128256 took 10 us longer)."""
    spec = importlib.util.spec_from_file_location("mvllm_build_flags", os.path.join(ROOT, "micro-vllm_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not shutil.which(b._hipcc()):
        pytest.skip("no hipcc")
    out = str(tmp_path / "sampler.s")
    subprocess.run([b._hipcc()] + b._flags_for("sampler.hip") + ["-S", "--cuda-device-only", os.path.join(b.CSRC, "sampler.hip"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        text = f.read()
    scratch = {name: int(size) for name, size in re.findall(r"\.name:\s+(\S+)\n(?:\s+\.[^\n]*\n|\s+-[^\n]*\n)*?\s+\.private_segment_fixed_size:\s+(\d+)", text)}
    kernels = [n for n in scratch if "sample" in n]
    assert len(kernels) == 4
    in_line = [n for n in kernels if "sample_parts_kernel" in n or "Lb0E" in n]
    assert len(in_line) == 2 and all(scratch[n] == 0 for n in in_line), scratch
