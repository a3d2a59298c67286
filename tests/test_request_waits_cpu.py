"""The hand-placed waits of the prefill product, checked in the assembly the compiler makes of it.

Its stages of x arrive by requests the compiler does not count, and the wait in front of a stage's barrier says how many younger
requests may still be on their way.  That number is only right if every request it counts was really made: what the
compiler removes (a refill nobody uses) must not be in it.  No GPU test shows such a fault reliably."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("mvllm_build_flags", os.path.join(ROOT, "micro-vllm_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not shutil.which(b._hipcc()):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "gemm_prefill.s")
    subprocess.run([b._hipcc()] + b._flags_for("gemm_prefill.hip") + ["-S", "--cuda-device-only", os.path.join(b.CSRC, "gemm_prefill.hip"),
                    "-o", out], check=True, capture_output=True)
    with open(out) as f:
        return f.read()


def _blocks(text, kernel):
    """The basic blocks of the kernel of these template arguments (all of them), each a list of 'x' (request of x into LDS), 'w'
    (load), wait counts and 'barrier'."""
    body = re.search(rf"^_ZN2mv19gemm_prefill_kernelI{kernel}EEEvNS_9PGemmArgsE:.*?^\.Lfunc_end", text, re.S | re.M).group(0)
    blocks = [[]]
    for line in map(str.strip, body.splitlines()):
        if re.match(r"\.LBB\d+_\d+:", line) or line.startswith(("s_cbranch", "s_branch")):
            blocks.append([])
        elif line.startswith("global_load_lds"):
            blocks[-1].append("x")
        elif line.startswith(("global_load", "global_store")):
            blocks[-1].append("w")
        elif line.startswith("s_waitcnt") and "vmcnt(" in line:
            blocks[-1].append(int(re.search(r"vmcnt\((\d+)\)", line).group(1)))
        elif line.startswith("s_barrier"):
            blocks[-1].append("barrier")
    return [b for b in blocks if "x" in b and "barrier" in b]


# (every epilogue is a compilation of its own: the plain one, max(v, 0)^2, the clamped gate)
@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("kernel,pieces", [("Li8ELi8ELi4ELi4", 4), ("Li4ELi8ELi4ELi4", 2)])
def test_a_stage_of_x_has_arrived_at_the_barrier_before_its_first_reader(assembly, kernel, pieces, act):
    """Four stages of x: behind a stage's barrier the next stage reads what was requested a stage before this one's own
    requests, so at the barrier only the latter may be on their way."""
    blocks = _blocks(assembly, f"{kernel}ELi{act}")
    prologue, loop = blocks[0], next(b for b in blocks if b.count("barrier") == 4)
    left = [b for b in blocks if b.count("barrier") == 1 and b is not prologue]
    assert prologue.count("x") == 3 * pieces and loop.count("x") == 4 * pieces
    assert len(left) == 3 and all(b.count("x") == pieces for b in left)

    def run(queue, events):
        queue, seen = list(queue), []
        for e in events:
            if isinstance(e, int):
                queue = queue[max(0, len(queue) - e):]
            elif e == "barrier":
                seen.append(queue.count("x"))
            else:
                queue.append(e)
        return queue, seen

    start, seen = run([], prologue)
    assert seen == [pieces]                      # two of three stages
    once, seen = run(start, loop)
    assert max(seen) <= pieces
    again, seen = run(once, loop)
    assert max(seen) <= pieces
    for b in left:                               # behind the prologue or behind whole passes
        for before in (start, again):
            assert run(before, b)[1] == [pieces]


@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("kernel", ["Li4ELi8ELi4ELi1", "Li4ELi8ELi4ELi2", "Li4ELi8ELi4ELi4"])
def test_tiles_of_fewer_strips_wait_for_no_less(assembly, kernel, act):
    """64-row tiles of one, two and four strips a wave: at every barrier, in any run through the loop and the stages behind it,
    at most the stage's own two requests of x are on their way.  (The compiler may wait for more in front of its own loads.)"""
    pieces = 2
    blocks = _blocks(assembly, f"{kernel}ELi{act}")
    prologue, loop = blocks[0], next(b for b in blocks if b.count("barrier") == 4)
    left = [b for b in blocks if b.count("barrier") == 1 and b is not prologue]
    assert prologue.count("x") == 3 * pieces and loop.count("x") == 4 * pieces
    assert len(left) == 3 and all(b.count("x") == pieces for b in left)

    def run(queue, events):
        queue, most = list(queue), 0
        for e in events:
            if isinstance(e, int):
                queue = queue[max(0, len(queue) - e):]
            elif e == "barrier":
                most = max(most, queue.count("x"))
            else:
                queue.append(e)
        return queue, most

    start, most = run([], prologue)
    assert most == pieces
    queue = start
    for _ in range(3):
        for tail in range(4):      # up to three stages are left
            q = queue
            for b in left[:tail]:
                q, most = run(q, b)
                assert most <= pieces
        queue, most = run(queue, loop)
        assert most <= pieces


def test_every_form_with_counted_waits_is_looked_at(assembly):
    """The forms above are all there are with four stages of x."""
    forms = set(re.findall(r"^_ZN2mv19gemm_prefill_kernelI(Li\d+ELi\d+ELi4ELi\d+ELi\d+)EEEvNS_9PGemmArgsE:", assembly, re.M))
    assert forms == {f"{k}ELi{act}" for k in ("Li8ELi8ELi4ELi4", "Li4ELi8ELi4ELi1", "Li4ELi8ELi4ELi2", "Li4ELi8ELi4ELi4") for act in range(3)}
