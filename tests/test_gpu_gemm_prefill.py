"""Many-row MFMA projection (mv_gemm_prefill) against the CPU oracle's linear_ref / swiglu_ref and
against the single-token kernel on the same tile image."""
import pytest
import torch

from conftest import assert_close_bf16, ulp_diff
from oracle.ref_ops import linear_ref, swiglu_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mk(m, n, k, seed, scale=0.05):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * scale).to(torch.bfloat16)
    return x, w, g


# ragged M (partial m-blocks), N that is not a multiple of the 256-column block, one k stage
@pytest.mark.parametrize("m", [1, 16, 127, 128, 129, 300, 1024])
@pytest.mark.parametrize("n,k", [(64, 64), (272, 2048), (4096, 1024), (2560, 2048)])
def test_gemm_prefill_vs_oracle(mv, m, n, k):
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    x, w, _ = _mk(m, n, k, seed=m + 3 * n + k)
    sw = StreamedWeight.from_linear(w.to(DEV))
    acc = gemm_prefill(x.to(DEV), sw, torch.empty(m, n, dtype=torch.float32, device=DEV))
    want32 = x.float() @ w.float().t()
    scale = max(1.0, want32.abs().max().item())
    assert (acc.cpu() - want32).abs().max().item() <= 1e-4 * scale
    y = gemm_prefill(x.to(DEV), sw, torch.empty(m, n, dtype=torch.bfloat16, device=DEV))
    want = linear_ref(x, w)
    assert_close_bf16(y, want, atol=1e-4 * scale, rtol=2 ** -7, what=f"gemm_prefill m={m} n={n} k={k}")
    assert float((ulp_diff(y, want) == 0).float().mean()) > 0.99


def test_gemm_prefill_epilogues(mv):
    """bias and residual rounding points, strided rows, fused SwiGLU (rows interleaved by 8)."""
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    m, n, k = 200, 512, 1024
    x, w, g = _mk(m, n, k, seed=5)
    bias = torch.randn(n, generator=g).to(torch.bfloat16)
    res = torch.randn(m, n, generator=g).to(torch.bfloat16)
    sw = StreamedWeight.from_linear(w.to(DEV))
    xb = torch.zeros(m, k + 64, dtype=torch.bfloat16, device=DEV)
    xb[:, :k] = x.to(DEV)
    yb = torch.full((m, n + 32), 7.0, dtype=torch.bfloat16, device=DEV)
    gemm_prefill(xb[:, :k], sw, yb[:, :n], bias=bias.to(DEV), residual=res.to(DEV))
    t = linear_ref(x, w, bias)
    want = (t.float() + res.float()).to(torch.bfloat16)
    # a one-ulp flip of an intermediate survives the cancellation in t + res: allow one ulp
    # of the larger operand
    err = (yb[:, :n].cpu().float() - want.float()).abs()
    tol = 1e-3 + 2 ** -7 * torch.maximum(t.float().abs(), want.float().abs())
    assert bool((err <= tol).all()), f"bias+residual: max err {err.max().item():.3e}"
    assert float((ulp_diff(yb[:, :n], want) == 0).float().mean()) > 0.99
    assert torch.all(yb[:, n:] == 7.0), "wrote past the row"

    inter = 768
    up = (torch.randn(inter, k, generator=g) * 0.05).to(torch.bfloat16)
    gate = (torch.randn(inter, k, generator=g) * 0.05).to(torch.bfloat16)
    gu = StreamedWeight.from_up_gate(up.to(DEV), gate.to(DEV))
    act = gemm_prefill(x.to(DEV), gu, torch.empty(m, inter, dtype=torch.bfloat16, device=DEV), swiglu=True)
    want = swiglu_ref(linear_ref(x, torch.cat([up, gate], 0)))
    # gate and up may each sit on a rounding boundary (one bf16 ulp apart between two fp32
    # summation orders); the product then moves by up to two ulps
    assert_close_bf16(act, want, atol=1e-3, rtol=2 ** -6, what="fused swiglu")
    assert float((ulp_diff(act, want) == 0).float().mean()) > 0.98


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


# tile width the planner gives each case on a 256-CU device: form 1 = 256 columns, 2 = 192, 3 = 224
WIDE_FORM = {(1000, 8208): 2, (2300, 4096): 2, (1300, 6144): 2, (1025, 8192): 2, (2048, 4096): 2,
             (700, 22016): 2, (2048, 28672): 3, (2048, 8192): 1, (2000, 7120): 3}


@pytest.mark.parametrize("m,n,k,mode", [(1000, 8208, 256, "plain"), (2300, 4096, 512, "residual"),
                                        (1300, 6144, 512, "bias"), (2048, 28672, 256, "swiglu"),
                                        (2048, 8192, 256, "plain"),
                                        # 224-column tiles, the last one 11 strips wide, the last m-block ragged
                                        (2000, 7120, 256, "residual"),
                                        (1025, 8192, 320, "bias"), (2048, 4096, 1024, "f32"),
                                        (700, 22016, 256, "swiglu"), (4096, 2048, 4096, "plain"),
                                        # tiles for half the CUs and a long k: two k-slices of the wide form
                                        (2000, 4096, 8192, "residual"), (1500, 4096, 8192, "bias")])
def test_gemm_prefill_wide_form(mv, m, n, k, mode):
    """Shapes whose 256 x 256 tiles fill at least half the CUs take the wide form (both operands
    through LDS, eight waves on a tile): ragged last m- and n-blocks, every epilogue, k from the
    shortest the form accepts to the model's."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    form = nv.lib().mv_gemm_prefill_form(m, n, k)
    assert form in (1, 2, 3), "this shape is meant to take the wide form"
    # all three tile widths are among the cases (the narrower ones where they fill the CUs in fuller rounds)
    if _cus() == 256:
        assert form == WIDE_FORM.get((m, n), 1), f"tile width of {(m, n, k)}: form {form}"
    if k >= 8192:
        assert nv.lib().mv_gemm_prefill_workspace_bytes(m, n, k) == 4096 + 2 * m * n * 4, "meant to be cut in two k-slices"
    x, w, g = _mk(m, n, k, seed=m + n + k, scale=0.03)
    bias = torch.randn(n, generator=g).to(torch.bfloat16) if mode == "bias" else None
    res = torch.randn(m, n, generator=g).to(torch.bfloat16) if mode == "residual" else None
    swiglu = mode == "swiglu"
    sw = (StreamedWeight.from_up_gate(w[:n // 2].to(DEV), w[n // 2:].to(DEV)) if swiglu
          else StreamedWeight.from_linear(w.to(DEV)))
    ncols = sw.out_features
    dt = torch.float32 if mode == "f32" else torch.bfloat16
    xb = torch.zeros(m, k + 64, dtype=torch.bfloat16, device=DEV)       # strided rows in
    xb[:, :k] = x.to(DEV)
    yb = torch.full((m, ncols + 32), 7.0, dtype=dt, device=DEV)         # and out
    gemm_prefill(xb[:, :k], sw, yb[:, :ncols], bias=None if bias is None else bias.to(DEV),
                 residual=None if res is None else res.to(DEV), swiglu=swiglu)
    assert torch.all(yb[:, ncols:] == 7.0), "wrote past the row"
    got = yb[:, :ncols].cpu()
    want32 = x.float() @ w.float().t()
    scale = max(1.0, want32.abs().max().item())
    if mode == "f32":
        assert (got - want32).abs().max().item() <= 1e-4 * scale
        return
    if swiglu:
        want = swiglu_ref(linear_ref(x, w))
        assert_close_bf16(got, want, atol=1e-3, rtol=2 ** -6, what="wide form, fused swiglu")
    else:
        t0 = linear_ref(x, w).float()
        t1 = linear_ref(x, w, bias).float()
        want = t1 if res is None else (t1 + res.float()).to(torch.bfloat16).float()
        mag = torch.maximum(torch.maximum(t0.abs(), t1.abs()), want.abs())
        # as for the k-sliced product below: each rounding point may flip by one unit at its own
        # magnitude between two fp32 summation orders, so two units of the largest intermediate
        err = (got.float() - want).abs()
        assert bool((err <= 1e-3 + 2 ** -6 * mag).all()), f"{mode}: max err {err.max().item():.3e}"
        want = want.to(torch.bfloat16)
    assert float((ulp_diff(got, want) == 0).float().mean()) > 0.98


@pytest.mark.parametrize("m,n,k,mode,strips", [
    (3072, 6144, 1024, "bias", 12),        # 48 tiles per XCD on 32 CUs: the 16 left over in two parts each
    (2560, 6144, 3072, "residual", 12),    # 40 tiles per XCD: the 8 left over in three parts each
    (4096, 6144, 2048, "swiglu", 16),      # the fused activation behind a cut tile
    (2300, 7168, 1024, "f32", 14),         # a ragged last m-block, fp32 out
    (3000, 7168, 1536, "residual", 16),    # 28 n-blocks: the eighth XCD owns none
])
def test_gemm_prefill_wide_form_cuts_left_over_tiles(mv, m, n, k, mode, strips):
    """With more tiles than CUs and a remainder of at most half a round, the left-over tiles are cut
    along k between workgroups inside the launch (the last part adds the others' sums in its
    epilogue).  Checked against the oracle, against the same launch with the cut switched off, and
    twice in a row (the parts count themselves in through counters that must be back at zero)."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    if _cus() != 256:
        pytest.skip("the cases are laid out for 32 CUs per XCD")
    L = nv.lib()
    x, w, g = _mk(m, n, k, seed=m + n + k + strips, scale=0.03)
    bias = torch.randn(n, generator=g).to(torch.bfloat16) if mode == "bias" else None
    res = torch.randn(m, n, generator=g).to(torch.bfloat16) if mode == "residual" else None
    swiglu = mode == "swiglu"
    sw = (StreamedWeight.from_up_gate(w[:n // 2].to(DEV), w[n // 2:].to(DEV)) if swiglu
          else StreamedWeight.from_linear(w.to(DEV)))
    ncols = sw.out_features
    dt = torch.float32 if mode == "f32" else torch.bfloat16

    def run():
        yb = torch.full((m, ncols + 32), 7.0, dtype=dt, device=DEV)
        gemm_prefill(x.to(DEV), sw, yb[:, :ncols], bias=None if bias is None else bias.to(DEV),
                     residual=None if res is None else res.to(DEV), swiglu=swiglu)
        assert torch.all(yb[:, ncols:] == 7.0), "wrote past the row"
        return yb[:, :ncols].cpu()

    try:
        L.mv_debug_prefill_options(1, strips)
        assert L.mv_gemm_prefill_workspace_bytes(m, n, k) == 4096 + 256 * 256 * 1024, "meant to cut its left-over tiles"
        cut, again = run(), run()
        L.mv_debug_prefill_options(0, strips)
        assert L.mv_gemm_prefill_workspace_bytes(m, n, k) == 0
        whole = run()
    finally:
        L.mv_debug_prefill_options(-1, -1)
    assert torch.equal(cut, again), "the second launch differs from the first"
    want32 = x.float() @ w.float().t()
    scale = max(1.0, want32.abs().max().item())
    if mode == "f32":
        assert (cut - want32).abs().max().item() <= 1e-4 * scale
        assert (cut - whole).abs().max().item() <= 1e-4 * scale
        return
    if swiglu:
        want = swiglu_ref(linear_ref(x, w))
        assert_close_bf16(cut, want, atol=1e-3, rtol=2 ** -6, what="cut tiles, fused swiglu")
        assert_close_bf16(cut, whole, atol=1e-3, rtol=2 ** -6, what="cut vs whole tiles, fused swiglu")
    else:
        t0 = linear_ref(x, w).float()
        t1 = linear_ref(x, w, bias).float()
        want = t1 if res is None else (t1 + res.float()).to(torch.bfloat16).float()
        mag = torch.maximum(torch.maximum(t0.abs(), t1.abs()), want.abs())
        for name, ref in (("oracle", want), ("whole tiles", whole.float())):
            err = (cut.float() - ref).abs()
            assert bool((err <= 1e-3 + 2 ** -6 * mag).all()), f"{mode} vs {name}: max err {err.max().item():.3e}"
        want = want.to(torch.bfloat16)
    assert float((ulp_diff(cut, want) == 0).float().mean()) > 0.98
    assert float((ulp_diff(cut, whole) == 0).float().mean()) > 0.98


def test_gemm_prefill_cut_tiles_replayed_from_a_captured_graph(mv):
    """The cut of left-over tiles keeps its counters inside the library and returns them to zero in
    the launch itself: a captured launch replays any number of times with the bits of the eager one."""
    import ctypes
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    if _cus() != 256:
        pytest.skip("the case is laid out for 32 CUs per XCD")
    L = nv.lib()
    m, n, k = 3072, 6144, 1024
    x, w, _ = _mk(m, n, k, seed=11, scale=0.03)
    xd, sw = x.to(DEV), StreamedWeight.from_linear(w.to(DEV))
    try:
        L.mv_debug_prefill_options(1, 12)
        need = L.mv_gemm_prefill_workspace_bytes(m, n, k)
        assert need == 4096 + 256 * 256 * 1024, "meant to cut its left-over tiles"
        ws = torch.zeros(need // 4, dtype=torch.float32, device=DEV)   # starts with the parts' counters
        eager = gemm_prefill(xd, sw, torch.empty(m, n, dtype=torch.bfloat16, device=DEV), workspace=ws).clone()
        out = torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            side.synchronize()
            nv.check("begin", L.mv_graph_begin_capture(side.cuda_stream))
            gemm_prefill(xd, sw, out, workspace=ws)
            h = ctypes.c_void_p()
            nv.check("end", L.mv_graph_end_capture(side.cuda_stream, ctypes.byref(h)))
            for replay in range(3):
                out.zero_()
                nv.check("launch", L.mv_graph_launch(h, side.cuda_stream))
                side.synchronize()
                assert torch.equal(out, eager), f"replay {replay} differs from the eager launch"
            L.mv_graph_destroy(h)
    finally:
        L.mv_debug_prefill_options(-1, -1)


def test_gemm_prefill_cut_tiles_on_two_streams_at_once(mv):
    """Two streams issue launches that cut their left-over tiles, back to back and unsynchronised: each
    stream has its own workspace (counters and accumulator slots), so neither sees the other's parts."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    if _cus() != 256:
        pytest.skip("the case is laid out for 32 CUs per XCD")
    L = nv.lib()
    m, n, k = 3072, 6144, 1024
    cases = []
    for seed in (21, 22):
        x, w, _ = _mk(m, n, k, seed=seed, scale=0.03)
        cases.append((x.to(DEV), StreamedWeight.from_linear(w.to(DEV))))
    try:
        L.mv_debug_prefill_options(1, 12)
        serial = [gemm_prefill(xd, sw, torch.empty(m, n, dtype=torch.bfloat16, device=DEV)).clone() for xd, sw in cases]
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        outs = [torch.zeros(m, n, dtype=torch.bfloat16, device=DEV) for _ in cases]
        for _ in range(4):
            for st, (xd, sw), out in zip(streams, cases, outs):
                with torch.cuda.stream(st):
                    gemm_prefill(xd, sw, out)
        torch.cuda.synchronize()
    finally:
        L.mv_debug_prefill_options(-1, -1)
    for i, (out, want) in enumerate(zip(outs, serial)):
        assert torch.equal(out, want), f"stream {i}: differs from the launch on its own"


_ONE_WORKGROUP_PER_TILE_CHILD = r"""
import sys, torch
sys.path.insert(0, sys.argv[1])
import micro_vllm_amd
from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill
g = torch.Generator().manual_seed(77)
m, n, k = 2500, 9216, 1024
x = (torch.randn(m, k, generator=g) * 0.5).to(torch.bfloat16)
w = (torch.randn(n, k, generator=g) * 0.03).to(torch.bfloat16)
y = gemm_prefill(x.cuda(), StreamedWeight.from_linear(w.cuda()), torch.empty(m, n, dtype=torch.bfloat16, device="cuda"))
torch.save(y.cpu(), sys.argv[2])
"""


def test_gemm_prefill_wide_form_one_workgroup_per_tile_gives_the_same_bits(mv, tmp_path):
    """MVLLM_PREFILL_PERSIST=0 (read once per process: a child process) launches one workgroup per tile
    where the default has one per CU walk several tiles and cut the left-over ones along k: a tile
    that is not cut is summed in the same order either way, so the outputs must be the same bits
    wherever the default did not cut, and within the usual bound where it did."""
    import os
    import subprocess
    import sys
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = str(tmp_path / "per_tile.pt")
    r = subprocess.run([sys.executable, "-c", _ONE_WORKGROUP_PER_TILE_CHILD, root, out], capture_output=True, text=True,
                       timeout=280, env=dict(os.environ, MVLLM_PREFILL_PERSIST="0"))
    assert r.returncode == 0, r.stdout[-1500:] + r.stderr[-1500:]
    per_tile = torch.load(out, weights_only=True)
    g = torch.Generator().manual_seed(77)
    m, n, k = 2500, 9216, 1024
    x = (torch.randn(m, k, generator=g) * 0.5).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * 0.03).to(torch.bfloat16)
    assert nv.lib().mv_gemm_prefill_form(m, n, k) in (1, 2, 3), "meant to take the wide form"
    walked = gemm_prefill(x.to(DEV), StreamedWeight.from_linear(w.to(DEV)),
                          torch.empty(m, n, dtype=torch.bfloat16, device=DEV)).cpu()
    same = float((ulp_diff(walked, per_tile) == 0).float().mean())
    assert same > 0.98, f"only {same:.4f} of the outputs agree bit for bit"
    err = (walked.float() - per_tile.float()).abs()
    assert bool((err <= 1e-3 + 2 ** -6 * per_tile.float().abs()).all())
    want = linear_ref(x, w)
    assert float((ulp_diff(walked, want) == 0).float().mean()) > 0.98


def test_gemm_prefill_agrees_with_single_token_kernel(mv):
    """Same weights, same rows: the two kernels differ only in fp32 summation order."""
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill, wgemm

    m, n, k = 48, 1024, 4096
    x, w, _ = _mk(m, n, k, seed=9, scale=0.02)
    sw = StreamedWeight.from_linear(w.to(DEV))
    a = gemm_prefill(x.to(DEV), sw, torch.empty(m, n, dtype=torch.bfloat16, device=DEV))
    b = wgemm(x.to(DEV), sw, torch.empty(m, n, dtype=torch.bfloat16, device=DEV))
    assert_close_bf16(a, b.cpu(), atol=1e-4 * max(1.0, float(b.float().abs().max())), rtol=2 ** -7,
                      what="prefill vs single-token kernel")
    assert float((ulp_diff(a, b) == 0).float().mean()) > 0.99


def test_gemm_prefill_rejects_bad_shapes(mv):
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    w = StreamedWeight.from_linear(torch.zeros(64, 96, dtype=torch.bfloat16, device=DEV))
    x = torch.zeros(4, 96, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(AssertionError):  # K = 96 is not a multiple of 64
        gemm_prefill(x, w, torch.empty(4, 64, dtype=torch.bfloat16, device=DEV))
    assert gemm_prefill(x[:0], w, torch.empty(0, 64, dtype=torch.bfloat16, device=DEV)).shape == (0, 64)


@pytest.mark.parametrize("m", [1, 32, 100, 128, 300, 512])
@pytest.mark.parametrize("n,k,mode", [(512, 4096, "plain"), (4096, 14336, "residual"), (1536, 4096, "swiglu"),
                                      (6144, 4096, "bias"), (256, 8192, "f32")])
def test_gemm_prefill_k_slices(mv, m, n, k, mode):
    """Few output tiles and a long k: the product is cut into k-slices that run side by side and are
    added by a second launch (with the epilogue).  Against the oracle as the unsplit product is,
    and against the unsplit product itself (the C entry without a workspace): the two differ only
    in fp32 summation order."""
    import ctypes

    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    L = nv.lib()
    assert L.mv_gemm_prefill_workspace_bytes(m, n, k) > 0, "this shape is meant to be split"
    x, w, g = _mk(m, n, k, seed=m + n + k, scale=0.03)
    bias = torch.randn(n, generator=g).to(torch.bfloat16) if mode == "bias" else None
    res = torch.randn(m, n, generator=g).to(torch.bfloat16) if mode == "residual" else None
    swiglu = mode == "swiglu"
    if swiglu:
        sw = StreamedWeight.from_up_gate(w[:n // 2].to(DEV), w[n // 2:].to(DEV))
    else:
        sw = StreamedWeight.from_linear(w.to(DEV))
    ncols = sw.out_features
    dt = torch.float32 if mode == "f32" else torch.bfloat16
    xd = x.to(DEV)
    split = gemm_prefill(xd, sw, torch.empty(m, ncols, dtype=dt, device=DEV),
                         bias=None if bias is None else bias.to(DEV),
                         residual=None if res is None else res.to(DEV), swiglu=swiglu)
    whole = torch.empty(m, ncols, dtype=dt, device=DEV)
    flags = (nv.MV_GEMM_SWIGLU if swiglu else 0) | (nv.MV_GEMM_OUT_F32 if mode == "f32" else 0)
    rd = None if res is None else res.to(DEV)
    bd = None if bias is None else bias.to(DEV)
    nv.check("mv_gemm_prefill", L.mv_gemm_prefill(
        xd.data_ptr(), k, sw.tiles.data_ptr(), nv.ptr(bd), nv.ptr(rd), n if rd is not None else 0,
        whole.data_ptr(), ncols, m, n, k, flags, nv.stream_ptr()))
    want32 = x.float() @ w.float().t()
    scale = max(1.0, want32.abs().max().item())
    if mode == "f32":
        assert (split.cpu() - want32).abs().max().item() <= 1e-4 * scale
        assert (split - whole).abs().max().item() <= 1e-4 * scale
        return
    if swiglu:
        want = swiglu_ref(linear_ref(x, w))
        assert_close_bf16(split, want, atol=1e-3, rtol=2 ** -6, what="k-sliced swiglu")
        assert_close_bf16(split, whole.cpu(), atol=1e-3, rtol=2 ** -6, what="k-sliced vs whole swiglu")
    else:
        # Every rounding point may flip by one unit in the last place AT ITS OWN MAGNITUDE between
        # two fp32 summation orders, and the flip survives where a later addend cancels most of
        # the value: the bound is taken at the largest intermediate, not at the result.
        t0 = linear_ref(x, w).float()
        t1 = linear_ref(x, w, bias).float()
        want = t1 if res is None else (t1 + res.float()).to(torch.bfloat16).float()
        mag = torch.maximum(torch.maximum(t0.abs(), t1.abs()), want.abs())
        tol = 1e-3 + 2 ** -6 * mag
        for other, name in ((want, "oracle"), (whole.cpu().float(), "whole")):
            err = (split.cpu().float() - other).abs()
            assert bool((err <= tol).all()), f"{mode} vs {name}: max err {err.max().item():.3e}"
        want = want.to(torch.bfloat16)
    assert float((ulp_diff(split, want) == 0).float().mean()) > 0.98
    assert float((ulp_diff(split, whole) == 0).float().mean()) > 0.98


@pytest.mark.parametrize("m", [1, 16, 17, 37, 48, 49, 64])
@pytest.mark.parametrize("n,k,mode", [(16, 2048, "plain"), (256, 8192, "f32"), (1280, 8192, "bias"),
                                      (2048, 5632, "residual"), (4096, 4096, "plain"), (11264, 2048, "swiglu"),
                                      (6160, 4096, "residual"), (8192, 1024, "plain"), (2560, 2048, "residual")])
def test_few_rows_add_the_slices_in_order(mv, m, n, k, mode):
    """Up to 16 rows, and with a short k up to 64, the k-slices are added within a workgroup.  The result is that of the slices' own products added in
    order, bit for bit (4, 8 and 16 slices, one to four blocks of rows, n that leaves a part of a workgroup's columns
    unused)."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    L = nv.lib()
    slices = (L.mv_gemm_prefill_workspace_bytes(m, n, k) - 4096) // (4 * m * n)
    assert slices in (4, 8, 16), "meant to be cut"
    x, w, g = _mk(m, n, k, seed=m + n + k, scale=0.03)
    wd = w.to(DEV)
    sw = StreamedWeight.from_up_gate(wd[:n // 2], wd[n // 2:]) if mode == "swiglu" else StreamedWeight.from_linear(wd)
    ncols, dt = sw.out_features, torch.float32 if mode == "f32" else torch.bfloat16
    bias = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if mode == "bias" else None
    res = torch.randn(m, n, generator=g).to(torch.bfloat16).to(DEV) if mode == "residual" else None
    xd = x.to(DEV)
    got = gemm_prefill(xd, sw, torch.full((m, ncols), float("nan"), dtype=dt, device=DEV), bias=bias, residual=res,
                       swiglu=mode == "swiglu")
    total = torch.zeros(m, n, device=DEV)
    kk = k // slices
    for i in range(slices):
        xs, part = xd[:, i * kk:(i + 1) * kk].contiguous(), torch.empty(m, n, device=DEV)
        ws = StreamedWeight.from_linear(wd[:, i * kk:(i + 1) * kk].contiguous())
        nv.check("mv_gemm_prefill", L.mv_gemm_prefill(xs.data_ptr(), kk, ws.tiles.data_ptr(), None, None, 0, part.data_ptr(),
                                                      n, m, n, kk, nv.MV_GEMM_OUT_F32, nv.stream_ptr()))
        total += part
    want = total if mode == "f32" else total.to(torch.bfloat16)
    if mode == "swiglu":   # (the activation's own rounding: one unit in the last place)
        assert_close_bf16(got, swiglu_ref(want.cpu()), atol=1e-6, rtol=2 ** -7, what="swiglu of the slices' sum")
        return
    for addend in (bias, res):
        want = want if addend is None else (want.float() + addend.float()).to(torch.bfloat16)
    assert torch.equal(got, want)


@pytest.mark.parametrize("m,n,k,mode", [(65, 6144, 2048, "bias"), (129, 16384, 1024, "swiglu"), (512, 4112, 2048, "residual"),
                                        (700, 2048, 64, "plain"), (700, 2048, 320, "f32"), (1000, 2048, 832, "plain"),
                                        (1000, 4096, 4096, "residual"), (768, 8192, 2048, "plain"),
                                        (700, 2048, 128, "plain"), (700, 2048, 192, "f32"), (700, 2048, 384, "plain"),
                                        (700, 2048, 448, "f32"), (1100, 4096, 1600, "f32"), (1100, 4096, 1664, "plain"),
                                        (1100, 4096, 1728, "f32"), (1100, 4096, 13824, "plain")])
def test_tiles_of_64_and_128_rows_give_the_same_sums(mv, m, n, k, mode):
    """Grids of less than a workgroup to a compute unit take 64-row tiles or the deep form (1100 rows, and 768 of 8192
    columns); the same rows inside a product of many take 128-row tiles.  The sums have the same order wherever neither is
    cut along k.  Both forms pass over k in fours of 64: every remainder, with whole passes before it (64-row tiles: k of
    320, 384, 448; deep form: 1600, 1664, 1728) and without (64, 128, 192)."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight

    x, w, g = _mk(m, n, k, seed=m + n + k, scale=0.03)
    sw = (StreamedWeight.from_up_gate(w[:n // 2].to(DEV), w[n // 2:].to(DEV)) if mode == "swiglu"
          else StreamedWeight.from_linear(w.to(DEV)))
    ncols, dt = sw.out_features, torch.float32 if mode == "f32" else torch.bfloat16
    flags = (nv.MV_GEMM_SWIGLU if mode == "swiglu" else 0) | (nv.MV_GEMM_OUT_F32 if mode == "f32" else 0)
    bias = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if mode == "bias" else None
    reps = 4096 // m + 1
    xd, res = x.to(DEV), torch.randn(m, n, generator=g).to(torch.bfloat16).to(DEV) if mode == "residual" else None
    outs = []
    for r in (1, reps):      # without a workspace: k whole in both
        xr, rr = xd.repeat(r, 1), None if res is None else res.repeat(r, 1)
        y = torch.full((m * r, ncols), float("nan"), dtype=dt, device=DEV)
        nv.check("mv_gemm_prefill", nv.lib().mv_gemm_prefill(
            xr.data_ptr(), k, sw.tiles.data_ptr(), nv.ptr(bias), nv.ptr(rr), n if rr is not None else 0, y.data_ptr(), ncols,
            m * r, n, k, flags, nv.stream_ptr()))
        outs.append(y)
    assert torch.equal(outs[0], outs[1][:m]) and torch.equal(outs[0], outs[1][-m:])


@pytest.mark.parametrize("mode", ["plain", "bias", "residual", "f32", "swiglu"])
@pytest.mark.parametrize("m,n,k", [(128, 8192, 1024), (128, 8208, 1024), (256, 4096, 1024), (256, 8192, 1024), (192, 8240, 1024),
                                   (65, 2064, 512), (300, 8208, 512),
                                   (37, 28672, 4096), (64, 28672, 4096)])
def test_narrow_tiles_give_the_sums_of_wide_ones(mv, m, n, k, mode):
    """64-row tiles of one and two n-tiles a wave (grids of up to a quarter and half of the compute units; n that leaves a part
    of a workgroup's columns unused) and, of up to 64 rows, in place of the 256-row form in two slices: the same rows as
    the first of many, whose plan cuts k the same way, bit for bit."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight

    rows, ks = (256, 2) if n == 28672 else (2048, 1)
    L = nv.lib()
    for r in (m, rows) if ks == 2 else (m,):
        assert L.mv_gemm_prefill_workspace_bytes(r, n, k) == (4096 + 8 * r * n if ks == 2 else 0)
    x, w, g = _mk(rows, n, k, seed=m + n + k, scale=0.03)
    wd, xd = w.to(DEV), x.to(DEV)
    sw = StreamedWeight.from_up_gate(wd[:n // 2], wd[n // 2:]) if mode == "swiglu" else StreamedWeight.from_linear(wd)
    bias = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if mode == "bias" else None
    res = torch.randn(rows, n, generator=g).to(torch.bfloat16).to(DEV) if mode == "residual" else None
    flags = {"swiglu": nv.MV_GEMM_SWIGLU, "f32": nv.MV_GEMM_OUT_F32}.get(mode, 0)
    # (unsliced products without a workspace: left-over tiles of the many rows are not cut along k either)
    ws = torch.zeros(1024 + 2 * rows * n, device=DEV) if ks == 2 else None

    def run(r):
        y = torch.full((r, sw.out_features), float("nan"), dtype=torch.float32 if mode == "f32" else torch.bfloat16, device=DEV)
        nv.check("mv_gemm_prefill_ws", L.mv_gemm_prefill_ws(
            xd.data_ptr(), k, sw.tiles.data_ptr(), nv.ptr(bias), nv.ptr(res), n, y.data_ptr(), sw.out_features, r, n, k, flags,
            nv.ptr(ws), 0 if ws is None else ws.numel() * 4, nv.stream_ptr()))
        return y

    assert torch.equal(run(m), run(rows)[:m])


# slices added in the workgroup: four, eight and sixteen slices, every count of 8-row blocks, k-tiles of a slice that are fewer than the
# stages in flight, as many, and a few more, strips left over: the sums of the sliced 64-row tiles, bit for bit where both are cut alike
@pytest.mark.parametrize("m", [5, 8, 9, 17, 25, 33, 40, 41, 49, 57, 64])
@pytest.mark.parametrize("n,k", [(4112, 1024), (8224, 1024), (11280, 2048), (16400, 1024), (2064, 2048), (1536, 4096), (6160, 4096)])
def test_short_prompts_add_their_slices_in_the_workgroup(mv, m, n, k):
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    sw = StreamedWeight.from_linear(w)
    got = gemm_prefill(x, sw, torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV))
    want = x.double() @ w.double().t()
    # fp32 sums of exact products: at most k roundings of 2^-24 of partial sums that the absolute products bound
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((got.double() - want).abs() <= bound).all())
    # a row among 65 goes through tiles, bit for bit the same where the plan cuts both into as many slices
    L, ks = nv.lib(), nv.lib().mv_linear_slab_count(65, n, k)
    counters = L.mv_gemm_prefill_workspace_bytes(65, n, k) - ks * 65 * n * 4
    if L.mv_gemm_prefill_workspace_bytes(m, n, k) - counters == ks * m * n * 4:
        more = torch.cat([x, torch.zeros(65 - m, k, dtype=torch.bfloat16, device=DEV)])
        assert torch.equal(gemm_prefill(more, sw, torch.empty(65, n, dtype=torch.float32, device=DEV))[:m], got)


# slices added in the workgroup: every instance of the kernel, that is four slices in groups of one to four strips, eight in one to four,
# sixteen in one and two, by every count of 8-row blocks; more k-tiles in a slice than stages in flight and fewer, strips left over.  The
# slices' own products added in order, bit for bit
@pytest.mark.parametrize("m", [5, 8, 9, 17, 25, 33, 40, 41, 49, 57, 64])
@pytest.mark.parametrize("n,k,slices,group", [(528, 1024, 4, 1), (4112, 1024, 4, 2), (8224, 1024, 4, 3), (12560, 1024, 4, 4),
                                              (528, 2048, 8, 1), (4112, 2048, 8, 2), (8208, 3072, 8, 3), (12304, 4096, 8, 4),
                                              (2560, 4096, 16, 1), (5120, 8192, 16, 2)])
def test_every_instance_adds_its_slices_in_order(mv, m, n, k, slices, group):
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.linear import StreamedWeight, gemm_prefill

    L = nv.lib()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (L.mv_gemm_prefill_workspace_bytes(m, n, k) - 4096) // (4 * m * n) == slices
        assert L.mv_gemm_prefill_group(m, n, k) == group
    g = torch.Generator().manual_seed(m + n + k)
    wide = torch.full((m, k + 24), float("nan"), dtype=torch.bfloat16, device=DEV)    # nothing beside the rows reaches a sum
    wide[:, :k] = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    x = wide[:, :k]
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    got = gemm_prefill(x, StreamedWeight.from_linear(w), torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV))
    total, kk = torch.zeros(m, n, device=DEV), k // slices
    for i in range(slices):
        xs, part = x[:, i * kk:(i + 1) * kk].contiguous(), torch.empty(m, n, device=DEV)
        ws = StreamedWeight.from_linear(w[:, i * kk:(i + 1) * kk].contiguous())
        nv.check("mv_gemm_prefill", L.mv_gemm_prefill(xs.data_ptr(), kk, ws.tiles.data_ptr(), None, None, 0, part.data_ptr(),
                                                      n, m, n, kk, nv.MV_GEMM_OUT_F32, nv.stream_ptr()))
        total += part
    assert torch.equal(got, total)
