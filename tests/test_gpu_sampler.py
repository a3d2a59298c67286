"""Device top-k / top-p sampling (mv_sample_topk_topp) against the CPU oracle on the same uniform
numbers: a deterministic function, so the picks must agree except where the uniform number falls
within float rounding of a CDF step."""
import pytest
import torch

from oracle.ref_sampler import distribution_ref, sample_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("v,top_k", [(512, 50), (32000, 50), (128256, 50), (128256, 1000), (4096, 5000)])
def test_sample_matches_oracle(mv, v, top_k):
    from micro_vllm_amd.core.layer.sampler import sample

    g = torch.Generator().manual_seed(v + top_k)
    bs = 24
    logits = (torch.randn(bs, v, generator=g) * 3).to(torch.bfloat16)   # bf16: plenty of exact ties
    temps = torch.rand(bs, generator=g) * 1.5 + 0.05
    temps[3] = 0.0                                                       # greedy limit inside a batch
    top_ps = torch.rand(bs, generator=g) * 0.6 + 0.4
    top_ps[5] = 1e-6
    top_ps[6] = 2.0
    u = torch.rand(bs, generator=g)
    u[7] = 0.0
    want = sample_ref(logits, temps, top_ps, top_k, u)
    got = sample(logits.to(DEV), temps, top_ps, top_k, uniforms=u).cpu()
    again = sample(logits.to(DEV), temps, top_ps, top_k, uniforms=u).cpu()
    assert torch.equal(got, again), "not deterministic"
    mism = (got != want).nonzero().flatten().tolist()
    for r in mism:   # tolerated only as a neighbour in the sorted candidate list with equal CDF to 1e-5
        idx, p = distribution_ref(logits[r], float(temps[r]), float(top_ps[r]), top_k)
        pos = {int(i): n for n, i in enumerate(idx.tolist())}
        assert abs(pos[int(got[r])] - pos[int(want[r])]) == 1, (r, got[r], want[r])
        cum = torch.cumsum(p, 0)
        j = min(pos[int(got[r])], pos[int(want[r])])
        assert abs(float(cum[j]) - float(u[r])) < 1e-5
    assert len(mism) <= 1


@pytest.mark.parametrize("v", [8, 64, 512, 8200, 131072, 131080, 151936])
@pytest.mark.parametrize("kind", ["random", "ties", "zeros", "sorted", "few"])
def test_selection_through_maxima_equals_radix_selection(mv, v, kind):
    """A NaN sorts below everything and sends its row through the radix selection; -inf in its place leaves the row on the
    selection through the threads' maxima (rows of mostly equal logits excepted, which overflow its list)."""
    from micro_vllm_amd.core.layer.sampler import sample

    g = torch.Generator().manual_seed(v)
    bs = 6
    x = torch.randn(bs, v, generator=g) * 3
    if kind == "ties":
        x = (x * 2).round() / 2
    elif kind == "zeros":       # zeros of both signs among the largest
        x = -x.abs().round()
    elif kind == "sorted":
        x = x.sort(dim=-1, descending=True).values
    elif kind == "few":
        x[:, 3:] = -float("inf")
    x = x.to(torch.bfloat16)
    at = torch.randint(0, v, (bs,), generator=g)
    a, b = x.clone(), x.clone()
    a[torch.arange(bs), at], b[torch.arange(bs), at] = -float("inf"), float("nan")
    temps, top_ps, u = torch.rand(bs, generator=g) + 0.5, torch.rand(bs, generator=g) * 0.5 + 0.5, torch.rand(bs, generator=g)
    for k in (1, 2, 50, 64, 65, 255, 256):
        if k > (3 if kind == "few" else v) - 1:
            continue        # the NaN itself would be among the k
        assert torch.equal(sample(a.to(DEV), temps, top_ps, k, uniforms=u), sample(b.to(DEV), temps, top_ps, k, uniforms=u)), k


@pytest.mark.parametrize("v,left", [(512, 1), (32000, 10), (32000, 64), (128256, 255), (131080, 300)])
def test_masked_rows_with_fewer_entries_than_k(mv, v, left):
    """All but `left` entries at -infinity (a constrained vocabulary): they have no weight, so asking for more entries than
    there are gives the pick among those there are, also where nothing is cut off by top-p."""
    from micro_vllm_amd.core.layer.sampler import sample

    g = torch.Generator().manual_seed(v + left)
    bs = 6
    x = torch.full((bs, v), -float("inf"))
    for b in range(bs):
        x[b, torch.randperm(v, generator=g)[:left]] = (torch.randn(left, generator=g) * 3).to(torch.bfloat16).float()
    x = x.to(torch.bfloat16).to(DEV)
    temps, u = torch.rand(bs, generator=g) + 0.5, torch.rand(bs, generator=g)
    temps[0] = 0.0
    for top_p in (0.7, 1.0, 1.5):
        want = sample(x, temps, torch.full((bs,), top_p), left, uniforms=u)
        assert bool(torch.isfinite(x[torch.arange(bs, device=DEV), want].float()).all())
        for k in (50, 256, 1000):
            if k > left:
                assert torch.equal(sample(x, temps, torch.full((bs,), top_p), k, uniforms=u), want), (top_p, k)


def test_sampler_class_uses_device_kernel_and_respects_top_k(mv):
    from micro_vllm_amd.core.layer.sampler import Sampler

    g = torch.Generator().manual_seed(1)
    logits = (torch.randn(64, 1024, generator=g) * 2).to(torch.bfloat16).to(DEV)
    temps = torch.full((64,), 0.9, device=DEV)
    topp = torch.full((64,), 0.95, device=DEV)
    torch.manual_seed(0)
    picks = Sampler()(logits, temps, topp, 10).cpu()
    top10 = logits.float().cpu().topk(10, dim=-1).indices
    assert all(int(picks[r]) in top10[r].tolist() for r in range(64))
    assert len(set(picks.tolist())) > 8          # actually random across rows


@pytest.mark.parametrize("rows,v", [(1, 128256), (1, 32000), (2, 151936), (4, 128256), (1, 8200),
                                    (1, 2048), (33, 32000), (40, 128256)])
def test_greedy_is_first_maximum(mv, rows, v):
    """mv_argmax: index of the largest logit, lowest index on ties, NaN never wins; the few-row
    form (several workgroups per row, merged by the last to arrive) and the one-workgroup-per-row
    form must agree with torch.  Bit exact (index work).  Called twice: the arrival tickets of the
    first call must be back at zero for the second."""
    from micro_vllm_amd.core.layer.sampler import greedy

    g = torch.Generator().manual_seed(rows * 7 + v)
    x = torch.randn(rows, v, generator=g).to(torch.bfloat16)
    for r in range(rows):                      # ties for the maximum, scattered over the row
        top = x[r].float().max().item()
        idx = torch.randint(0, v, (5,), generator=g)
        x[r, idx] = top
    x[0, v - 1] = float("nan")
    x[0, 0] = float("nan")
    want = torch.where(torch.isnan(x.float()), torch.tensor(float("-inf")), x.float())
    want = torch.stack([(row == row.max()).nonzero()[0, 0] for row in want])
    xd = x.to("cuda")
    for _ in range(2):
        got = greedy(xd)
        assert got.dtype == torch.long and torch.equal(got.cpu(), want)
    # the maximum in the last, shorter part and in the scalar tail (v not a multiple of 8 is rejected
    # by the vector path's callers; a multiple of 8 that does not divide into equal parts is not)
    y = torch.full((1, v), -3.0, dtype=torch.bfloat16)
    y[0, v - 3] = 5.0
    assert int(greedy(y.to("cuda")).item()) == v - 3


def test_greedy_on_two_streams_and_without_workspace(mv):
    """The parts of a long row meet in the caller's workspace: two picks in flight on two streams
    (each stream has its own default workspace) do not disturb each other, and a call without a
    workspace (one workgroup per row) returns the same ids."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.core.layer.sampler import greedy

    g = torch.Generator().manual_seed(5)
    xs = [torch.randn(2, 128256, generator=g).to(torch.bfloat16).to("cuda") for _ in range(2)]
    want = [x.float().argmax(-1) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for _ in range(50):
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                outs[i].append(greedy(xs[i]).clone())
    torch.cuda.synchronize()
    for i in (0, 1):
        assert all(torch.equal(o, want[i]) for o in outs[i])
        ids = torch.zeros(2, dtype=torch.long, device="cuda")
        nv.check("mv_argmax", nv.lib().mv_argmax(xs[i].data_ptr(), xs[i].stride(0), 2, 128256,
                                                 ids.data_ptr(), None, 0, nv.stream_ptr()))
        assert torch.equal(ids, want[i])


@pytest.mark.parametrize("v", [16376, 16384, 16392, 32000, 128256, 131080, 151936])
@pytest.mark.parametrize("kind", ["random", "ties", "equal", "zeros", "sorted", "few", "nan", "masked"])
def test_rows_over_several_workgroups_pick_what_one_picks(mv, v, kind):
    """The same ids with a workspace (rows of 16384 and more over several workgroups where there are more than 256 candidates; up
    to those, and of shorter rows, both sides take one) and without: few and many candidates (ranked, sorted, and too many of
    them: the radix selection), parts that end unevenly, entries of the largest maxima at the row's ends, rows whose greedy
    pick is given; twice, since the tickets have to be back at zero."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.core.layer.sampler import sample

    g = torch.Generator().manual_seed(v)
    bs = 9
    x = torch.randn(bs, v, generator=g) * 3
    if kind == "ties":
        x = (x * 2).round() / 2
    elif kind == "equal":
        x = torch.ones(bs, v)
    elif kind == "zeros":
        x = -x.abs().round()
    elif kind == "sorted":
        x = x.sort(dim=-1).values
    elif kind == "few":
        x[:, 3:-3] = -float("inf")
    elif kind == "nan":
        x[:, v // 2] = float("nan")
    elif kind == "masked":
        x[:] = -float("inf")
    x = x.to(torch.bfloat16).to(DEV)
    temps = (torch.rand(bs, generator=g) * 1.5 + 0.05).to(DEV)
    temps[2] = 0.0
    top_ps = (torch.rand(bs, generator=g) * 0.3 + 0.7).to(DEV)
    top_ps[4] = 2.0
    u = torch.rand(bs, generator=g).to(DEV)
    u[5] = 0.99999
    known = torch.arange(bs, device=DEV)
    L = nv.lib()
    for k in (1, 2, 50, 256, 257, 600, 1024, 4096):
        for greedy_ids in (None, known):
            want = torch.empty(bs, dtype=torch.long, device=DEV)
            nv.check("mv_sample_or_greedy", L.mv_sample_or_greedy(
                x.data_ptr(), v, bs, v, temps.data_ptr(), top_ps.data_ptr(), k, u.data_ptr(), nv.ptr(greedy_ids), want.data_ptr(),
                nv.stream_ptr()))
            for _ in range(2):
                assert torch.equal(sample(x, temps, top_ps, k, uniforms=u, greedy_ids=greedy_ids), want), (k, greedy_ids)


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("kind", ["random", "equal"])
def test_picks_of_as_many_rows_as_the_workspace_holds(mv, rows, kind):
    """Up to 64 rows the workspace has a ticket and a place for the maxima of each; more take one workgroup a row."""
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.core.layer.sampler import sample

    v, k, L = 16392, 600, nv.lib()
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, v, generator=g) * 3 if kind == "random" else torch.ones(rows, v)
    x = x.to(torch.bfloat16).to(DEV)
    temps, top_ps, u = ((torch.rand(rows, generator=g) * a + b).to(DEV) for a, b in ((1.5, 0.05), (0.3, 0.7), (1.0, 0.0)))
    want, got = (torch.empty(rows, dtype=torch.long, device=DEV) for _ in range(2))
    nv.check("mv_sample_or_greedy", L.mv_sample_or_greedy(
        x.data_ptr(), v, rows, v, temps.data_ptr(), top_ps.data_ptr(), k, u.data_ptr(), None, want.data_ptr(), nv.stream_ptr()))
    # a buffer of that size and not a byte more is written to (its tickets are back at zero, what lies behind it is as it was)
    size = L.mv_sample_workspace_bytes()
    room = torch.full((size + 4096,), 7, dtype=torch.uint8, device=DEV)
    room[:size] = 0
    for _ in range(2):
        nv.check("mv_sample_or_greedy_ws", L.mv_sample_or_greedy_ws(
            x.data_ptr(), v, rows, v, temps.data_ptr(), top_ps.data_ptr(), k, u.data_ptr(), None, got.data_ptr(),
            room.data_ptr(), size, nv.stream_ptr()))
        assert torch.equal(got, want)
    assert bool((room[size:] == 7).all()) and bool((room[:64 * 64 * 4] == 0).all())
    assert bool(room[64 * 64 * 4:size].any()) == bool(L.mv_sample_parts(rows, v, k)) == (rows <= 64)
    assert torch.equal(sample(x, temps, top_ps, k, uniforms=u), want)
