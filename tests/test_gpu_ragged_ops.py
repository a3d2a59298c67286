"""Each mechanism of the ragged family alone: the HIP kernel against the plain restatement in
oracle/ref_hybrid.py (fp64 on the CPU), on random inputs and on inputs built so that a fault shows
(one key made dominant just inside / just outside a window, far back, at a page border)."""
import math

import pytest
import torch

from oracle import ref_hybrid as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    import micro_vllm_amd  # noqa: F401
    from micro_vllm_amd.kernel import ragged_ops
    return ragged_ops


def make_cache(kv=None, state=None, pages=16, slots=3, dtype=torch.float32, page=64, max_tokens=512):
    from micro_vllm_amd.core.state_cache import HybridCacheManager
    return HybridCacheManager(pages, page, slots, kv or {}, state or {}, dtype=dtype, device=DEV, max_tokens=max_tokens,
                              max_rows=4, max_step_tokens=1024)


def step_of(cache, rows):
    cache.reserve([(sid, len(t)) for sid, t in rows])
    st = cache.plan(rows)
    cache.advance([(sid, len(t)) for sid, t in rows])
    return st


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 650, 200), (5, 37, 19), (70, 130, 288), (129, 64, 64), (3, 16, 2048)])
def test_linear_any(ops, f32, m, n, k):
    g = torch.Generator().manual_seed(m * 1000 + n)
    dt = torch.float32 if f32 else torch.bfloat16
    x = torch.randn(m, k, generator=g).to(dt)
    w = (torch.randn(n, k, generator=g) / math.sqrt(k)).to(dt)
    lin = ops.AnyLinear(w.to(DEV), wave_tiles=False)
    got = lin(x.to(DEV)).cpu().double()
    want = x.double() @ w.double().T
    assert (got - want).abs().max().item() <= (2e-5 if f32 else 2e-5) * max(1.0, want.abs().max().item()) * math.sqrt(k)
    # rows of a wider buffer, and a row's result does not depend on its neighbours
    wide = torch.zeros(m, k + 8, dtype=dt, device=DEV)
    wide[:, :k] = x.to(DEV)
    assert torch.equal(lin(wide[:, :k]).cpu().double(), got)
    assert torch.equal(lin(x[:1].to(DEV)).cpu().double(), got[:1])


@pytest.mark.parametrize("m,n,k,pad", [(1, 16, 4, 0), (8, 8200, 36, 4), (9, 8200, 36, 4), (16, 100, 1028, 0), (17, 100, 1028, 0),
                                       (33, 33, 31, 1), (64, 9000, 132, 0), (200, 9000, 132, 0), (700, 1100, 160, 4),
                                       (4100, 2100, 64, 0)])
def test_linear_any_f32_forms(ops, m, n, k, pad):
    """Streamed weights, tiles, vector and scalar loads: each within the bound of a 32-bit sum, and all of them the
    same sums bit for bit (a row on its own, behind its neighbours, in rows of a wider buffer)."""
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    wide = torch.full((m, k + pad), float("nan"), device=DEV)      # nothing beside the operand is read into a sum
    wide[:, :k] = x.to(DEV)
    out = torch.full((m, n + 3), 7.0, device=DEV)
    lin = ops.AnyLinear(w.to(DEV), wave_tiles=False)
    got = lin(wide[:, :k], out[:, :n])
    assert bool((out[:, n:] == 7.0).all())
    err = (got.cpu().double() - x.double() @ w.double().T).abs()
    # at most k roundings of 2^-24 of partial sums that the absolute products bound
    assert bool((err <= k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all())
    for rows in (slice(0, 1), slice(m - 1, m), slice(0, min(m, 20)), slice(m // 2, m)):
        assert torch.equal(lin(x[rows].to(DEV)), got[rows])


def test_wave_tile_and_plain_projection_agree(ops):
    g = torch.Generator().manual_seed(1)
    w = (torch.randn(96, 128, generator=g) / 11).to(torch.bfloat16).to(DEV)
    a, b = ops.AnyLinear(w), ops.AnyLinear(w, wave_tiles=False)
    assert a.tiles is not None and b.tiles is None
    for m in (1, 7, 64, 65, 200):
        x = torch.randn(m, 128, generator=g).to(torch.bfloat16).to(DEV)
        assert (a(x) - b(x)).abs().max().item() < 1e-4


@pytest.mark.parametrize("f32", [False, True])
def test_stream_ops(ops, f32):
    g = torch.Generator().manual_seed(2)
    dt = torch.float32 if f32 else torch.bfloat16
    rows, n, eps = 5, 203, 1e-5
    table = torch.randn(50, n, generator=g).to(dt)
    ids = torch.tensor([3, 49, 0, 7, 7], dtype=torch.int32)
    x, h = torch.empty(rows, n, device=DEV), torch.empty(rows, n, dtype=dt, device=DEV)
    ops.embed_scaled(table.to(DEV), ids.to(DEV), 2.5, x, h)
    assert torch.equal(x.cpu(), table.float()[ids.long()] * 2.5) and torch.equal(h.cpu(), (table.float()[ids.long()] * 2.5).to(dt))
    y1, y2, w = torch.randn(rows, n, generator=g), torch.randn(rows, n, generator=g) * 3, torch.randn(n, generator=g) * 0.1
    x0 = x.cpu().double()
    ops.postnorm_residual(y1.to(DEV), w.to(DEV), eps, x, h, y2=y2.to(DEV), s1=1.2, s2=0.9)
    want = x0 + ref.offset_norm(1.2 * y1.double() + 0.9 * y2.double(), w.double(), eps)
    assert (x.cpu().double() - want).abs().max().item() < 1e-5
    assert torch.equal(h.cpu(), x.cpu().to(dt))
    ops.postnorm_residual(y1.to(DEV), w.to(DEV), eps, x, h)
    want = want + ref.offset_norm(y1.double(), w.double(), eps)
    assert (x.cpu().double() - want).abs().max().item() < 2e-5
    idx = torch.tensor([4, 0, 2], dtype=torch.int32)
    out = torch.empty(3, n, dtype=dt, device=DEV)
    ops.offset_rmsnorm_gather(x, idx.to(DEV), w.to(DEV), eps, out)
    wn = ref.offset_norm(x.cpu().double()[idx.long()], w.double(), eps)
    assert (out.cpu().double() - wn).abs().max().item() < (1e-5 if f32 else 0.04)
    r = torch.empty(rows, n, dtype=dt, device=DEV)
    ops.relu_squared(y1.to(DEV), r)
    assert (r.cpu().double() - torch.relu(y1.double()) ** 2).abs().max().item() < (1e-6 if f32 else 0.05)
    lg = (torch.randn(4, 77, generator=g) * 40).to(DEV)
    want = 30.0 * torch.tanh(lg.cpu().double() / 30.0)
    assert (ops.softcap_(lg, 30.0).cpu().double() - want).abs().max().item() < 1e-5


@pytest.mark.parametrize("taps", [1, 2, 4])
def test_conv_whole_and_in_portions(ops, taps):
    g = torch.Generator().manual_seed(taps)
    C, T = 70, 23
    x, w, b = torch.randn(T, C + 6, generator=g), torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    want = ref.causal_conv_silu(x[:, 3:3 + C].double(), w.double(), b.double())
    for portions in ([T], [1] * T, [2, 1, 3, 2, 15], [5, 18]):
        cache = make_cache(state={0: {"conv": (taps - 1, C)}})
        cache.admit("other")                       # the request under test does not sit in slot 0
        cache.states[0]["conv"].fill_(7.0)         # what an earlier owner of the slot left behind
        out, pos = [], 0
        for n in portions:
            st = step_of(cache, [("s", [0] * n)])
            o = torch.empty(n, C, device=DEV)
            ops.conv_silu(x[pos:pos + n].to(DEV)[:, 3:3 + C], cache.states[0]["conv"], w.to(DEV), b.to(DEV), o, st)
            out.append(o.cpu())
            pos += n
        assert (torch.cat(out).double() - want).abs().max().item() < 1e-5, portions


def test_softplus_decay(ops):
    g = torch.Generator().manual_seed(5)
    raw = torch.randn(9, 11, generator=g) * 30         # far into both tails: no clamp anywhere
    bias, a_log = torch.randn(5, generator=g), torch.randn(5, generator=g)
    gain, decay, logd = torch.empty(9, 5, device=DEV), torch.empty(9, 5, device=DEV), torch.empty(9, 5, device=DEV)
    ops.softplus_decay(raw.to(DEV)[:, 4:9], bias.to(DEV), a_log.to(DEV), gain, decay, logd)
    v = raw[:, 4:9].double() + bias.double()
    dt = torch.where(v > 30, v, torch.log1p(torch.exp(v)))
    assert ((gain.cpu().double() - dt).abs() / dt.abs().clamp_min(1e-30)).max().item() < 1e-5
    assert (decay.cpu().double() - torch.exp(-torch.exp(a_log.double()) * dt)).abs().max().item() < 1e-6
    want = -torch.exp(a_log.double()) * dt
    assert ((logd.cpu().double() - want).abs() / want.abs().clamp_min(1e-30)).max().item() < 1e-5


@pytest.mark.parametrize("H,G,n,p", [(4, 2, 40, 24), (3, 3, 48, 20), (2, 1, 128, 64), (1, 1, 8, 128), (6, 1, 48, 48)])
def test_scan_whole_portions_and_rows(ops, H, G, n, p):
    g = torch.Generator().manual_seed(H * 100 + n)
    T = 19
    q, k = torch.randn(T, G * n, generator=g), torch.randn(T, G * n, generator=g)
    v = torch.randn(T, H * p, generator=g)
    decay, gain = torch.rand(T, H, generator=g), torch.rand(T, H, generator=g) + 0.1
    skip = torch.randn(H, generator=g)
    rep = H // G
    want, _ = ref.decayed_outer_product_scan(
        q.double().view(T, G, n).repeat_interleave(rep, 1), k.double().view(T, G, n).repeat_interleave(rep, 1),
        v.double().view(T, H, p), decay.double(), gain.double())
    want = (want + skip.double()[None, :, None] * v.double().view(T, H, p)).reshape(T, H * p)
    dv = lambda t: t.to(DEV)
    for portions in ([T], [1] * T, [2, 3, 2, 12]):
        cache = make_cache(state={0: {"s": (H, n, p)}})
        cache.admit("other")
        cache.states[0]["s"].fill_(3.0)
        out, pos = [], 0
        for m in portions:
            st = step_of(cache, [("a", [0] * m)])
            o = torch.empty(m, H * p, device=DEV)
            sl = slice(pos, pos + m)
            ops.scan_outer(dv(q[sl]), dv(k[sl]), dv(v[sl]), dv(decay[sl]), dv(gain[sl]), dv(skip), cache.states[0]["s"], o,
                           st, H, n, p, q_div=rep, k_div=rep)
            out.append(o.cpu())
            pos += m
        assert (torch.cat(out).double() - want).abs().max().item() < 2e-4, portions
    # two rows of unequal length in one launch, fixed decay per head, no gain, no skip
    cache = make_cache(state={0: {"s": (H, n, p)}})
    st = step_of(cache, [("a", [0] * 7), ("b", [0] * 12)])
    qq, kk = q.view(T, G, n).repeat_interleave(rep, 1).reshape(T, H * n), k.view(T, G, n).repeat_interleave(rep, 1).reshape(T, H * n)
    o = torch.empty(T, H * p, device=DEV)
    ops.scan_outer(dv(qq), dv(kk), dv(v), dv(decay[0].contiguous()), None, None, cache.states[0]["s"], o, st, H, n, p)
    for lo, hi in ((0, 7), (7, 19)):
        w2, _ = ref.decayed_outer_product_scan(qq[lo:hi].double().view(-1, H, n), kk[lo:hi].double().view(-1, H, n),
                                               v[lo:hi].double().view(-1, H, p), decay[0].double().repeat(hi - lo, 1),
                                               torch.ones(hi - lo, H, dtype=torch.float64))
        assert (o[lo:hi].cpu().double() - w2.reshape(hi - lo, H * p)).abs().max().item() < 2e-4


@pytest.mark.parametrize("H,G,n,p", [(4, 2, 40, 24), (2, 1, 128, 64), (1, 1, 8, 130), (3, 3, 64, 32)])
def test_scan_in_chunks_equals_token_by_token(ops, H, G, n, p):
    """Long rows: the chunked form against the restatement and against the token-by-token kernel, whole
    and cut at places that are no multiple of the chunk, beside a short row in the same launch; decays
    from nearly one down to values whose products underflow."""
    g = torch.Generator().manual_seed(H * 7 + p)
    T, rep = 333, H // G
    q, k = torch.randn(T, G * n, generator=g), torch.randn(T, G * n, generator=g)
    v = torch.randn(T, H * p, generator=g)
    logd = -torch.exp(torch.randn(T, H, generator=g) * 3.0 - 3.0)
    logd[100:110] = -120.0                       # a stretch that forgets everything
    decay, gain = torch.exp(logd), torch.rand(T, H, generator=g) + 0.1
    skip = torch.randn(H, generator=g)
    want, _ = ref.decayed_outer_product_scan(
        q.double().view(T, G, n).repeat_interleave(rep, 1), k.double().view(T, G, n).repeat_interleave(rep, 1),
        v.double().view(T, H, p), torch.exp(logd.double()), gain.double())
    want = (want + skip.double()[None, :, None] * v.double().view(T, H, p)).reshape(T, H * p)
    dv = lambda t: t.to(DEV)
    outs = {}
    for chunked in (True, False):
        for portions in ([T], [70, 3, 129, 17, 64, 50], [200] + [1] * 133):
            cache = make_cache(state={0: {"s": (H, n, p)}})
            cache.admit("other")
            cache.states[0]["s"].fill_(3.0)
            out, pos = [], 0
            for m in portions:
                rows = [("a", [0] * m)] + ([("b", [0] * 5)] if pos == 0 else [])     # a short row rides along once
                st = step_of(cache, rows)
                if chunked:
                    assert st.n_chunks == (m + 63) // 64 * (m > 16)
                tot = st.tokens
                o = torch.empty(tot, H * p, device=DEV)
                pad = lambda t: torch.cat([t[pos:pos + m], t[:tot - m]]).to(DEV)
                ops.scan_outer(pad(q), pad(k), pad(v), pad(decay), pad(gain), dv(skip), cache.states[0]["s"], o, st,
                               H, n, p, q_div=rep, k_div=rep, log_decay=pad(logd), chunked=chunked)
                out.append(o[:m].cpu())
                if pos == 0:
                    assert (o[m:].cpu().double() - want[:5]).abs().max().item() < 2e-4
                pos += m
            got = torch.cat(out).double()
            assert (got - want).abs().max().item() < 5e-4 * max(1.0, want.abs().max().item()), (chunked, portions)
            outs[(chunked, len(portions))] = got
    assert (outs[(True, 1)] - outs[(False, 1)]).abs().max().item() < 5e-4 * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("dim,rot", [(48, 32), (64, 64), (40, 0), (6, 2)])
def test_rotary_pairs(ops, dim, rot):
    g = torch.Generator().manual_seed(dim)
    T, H, base = 6, 3, 1e6
    x = torch.randn(T, H * dim + 5, generator=g)
    pos = torch.tensor([0, 1, 63, 64, 1000, 70001], dtype=torch.int32)
    inv = base ** (-2.0 * torch.arange(rot // 2, dtype=torch.float64) / max(rot, 1))
    xd = x.to(DEV)
    ops.rotary_pairs_(xd[:, :H * dim], inv.to(DEV), pos.to(DEV), H, dim, rot, dim ** -0.5)
    want = ref.rotate_half_pairs(x[:, :H * dim].double().view(T, H, dim), pos, rot, base) * dim ** -0.5
    assert (xd[:, :H * dim].cpu().double() - want.reshape(T, H * dim)).abs().max().item() < 2e-6
    assert torch.equal(xd[:, H * dim:].cpu(), x[:, H * dim:])


@pytest.mark.parametrize("f32", [False, True])
def test_gated_group_norm_both_orders(ops, f32):
    g = torch.Generator().manual_seed(8)
    rows, n, eps = 7, 120, 1e-5
    y, z, w = torch.randn(rows, n, generator=g) * 4, torch.randn(rows, n, generator=g), torch.randn(n, generator=g)
    dt = torch.float32 if f32 else torch.bfloat16
    tol = 1e-5 if f32 else 0.05
    for groups in (1, 3, 120):
        out = torch.empty(rows, n, dtype=dt, device=DEV)
        ops.gated_group_norm(y.to(DEV), z.to(DEV), w.to(DEV), out, groups, True, eps)
        u = y.double() * z.double() * torch.sigmoid(z.double())
        want = ref.unit_rms(u.view(rows, groups, -1), eps).reshape(rows, n) * w.double()
        assert (out.cpu().double() - want).abs().max().item() < tol * max(1.0, want.abs().max().item())
        ops.gated_group_norm(y.to(DEV), z.to(DEV), None, out, groups, False, eps)
        want = ref.unit_rms(y.double().view(rows, groups, -1), eps).reshape(rows, n) * z.double() * torch.sigmoid(z.double())
        assert (out.cpu().double() - want).abs().max().item() < tol * max(1.0, want.abs().max().item())


def _attend(ops, q, k, v, H, G, d, dv, scale, window, slopes, portions, f32=True, pages=16, shuffle=True, tiled=True):
    """Feed q|k|v rows in portions through qk_unitnorm_store + window_attn; returns [T, H*dv]."""
    dt = torch.float32 if f32 else torch.bfloat16
    cache = make_cache(kv={0: (G, d, dv)}, pages=pages, dtype=dt, max_tokens=pages * 64)
    if shuffle:   # pages in no particular order, none of them page 0 for the first tokens
        order = list(cache._free_pages)
        order = order[1::2] + order[0::2]
        cache._free_pages.clear()
        cache._free_pages.extend(order)
    cache.k_caches[0].fill_(9.0)
    cache.v_caches[0].fill_(-9.0)
    T = q.shape[0]
    qkv = torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1)], 1).float()
    out, pos = [], 0
    for n in portions:
        st = step_of(cache, [("s", [0] * n)])
        rows = qkv[pos:pos + n].to(DEV).contiguous()
        ops.qk_unitnorm_store(rows, cache.k_caches[0], cache.v_caches[0], st, H, G, d, dv, 1e-6)
        o = torch.empty(n, H * dv, dtype=dt, device=DEV)
        ops.window_attn(rows, cache.k_caches[0], cache.v_caches[0], o, st, torch.tensor(slopes).float().to(DEV), H, G, d,
                        dv, scale, window, tiled=tiled)
        out.append(o.float().cpu())
        pos += n
    return torch.cat(out)


@pytest.mark.parametrize("H,G,d,dv,window", [(6, 2, 40, 56, 37), (2, 2, 64, 64, 5), (4, 1, 96, 130, 200), (3, 3, 8, 8, 1),
                                             (2, 1, 64, 64, 300)])
def test_window_attention_random(ops, H, G, d, dv, window):
    g = torch.Generator().manual_seed(d + window)
    T, scale = 150, 0.3
    q, k, v = torch.randn(T, H, d, generator=g), torch.randn(T, G, d, generator=g), torch.randn(T, G, dv, generator=g)
    slopes = [2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]
    want = ref.windowed_softmax_attention(ref.unit_rms(q.double(), 1e-6), ref.unit_rms(k.double(), 1e-6), v.double(),
                                          scale, window, slopes).reshape(T, H * dv)
    for portions in ([T], [64, 64, 22], [3, 61, 2, 63, 1, 20], [100] + [1] * 50):
        got = _attend(ops, q, k, v, H, G, d, dv, scale, window, slopes, portions)
        assert (got.double() - want).abs().max().item() < 1e-4, portions
    got = _attend(ops, q, k, v, H, G, d, dv, scale, window, slopes, [T], f32=False, tiled=False)
    assert (got.double() - want).abs().max().item() < 0.05


@pytest.mark.parametrize("H,G,d,dv,window", [(2, 2, 64, 64, 5), (4, 2, 128, 64, 100), (3, 1, 96, 96, 72), (2, 1, 32, 32, 40),
                                             (8, 2, 128, 128, 64), (2, 2, 64, 128, 300)])
def test_window_attention_on_the_matrix_cores(ops, H, G, d, dv, window):
    """Long rows in bf16: the tiled kernel against the restatement and against the plain kernel, whole and
    in portions that start in the middle of a page, a short row riding along on the plain kernel."""
    g = torch.Generator().manual_seed(d * 3 + window)
    T, scale = 333, 0.3
    q, k, v = torch.randn(T, H, d, generator=g), torch.randn(T, G, d, generator=g), torch.randn(T, G, dv, generator=g)
    slopes = [2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]
    want = ref.windowed_softmax_attention(ref.unit_rms(q.double(), 1e-6), ref.unit_rms(k.double(), 1e-6), v.double(),
                                          scale, window, slopes).reshape(T, H * dv)
    plain = _attend(ops, q, k, v, H, G, d, dv, scale, window, slopes, [T], f32=False, tiled=False)
    for portions in ([T], [70, 3, 129, 17, 64, 50], [200] + [1] * 133):
        got = _attend(ops, q, k, v, H, G, d, dv, scale, window, slopes, portions, f32=False)
        assert (got.double() - want).abs().max().item() < 0.06, portions
        assert (got - plain).abs().max().item() < 0.06, portions
    assert (got.double() - want).abs().mean().item() < 0.006


@pytest.mark.parametrize("window", [72, 64, 65, 130, 260])
@pytest.mark.parametrize("decode,f32", [(False, True), (True, True), (False, False)])
def test_window_edge_shows_in_the_output(ops, window, decode, f32):
    """One key carries a value of its own and is made to win the softmax whenever it is visible: the
    query that still sees it (distance window - 1) returns that value, the next one does not."""
    H = G = 1
    d = dv = 32              # a head shape the tiled bf16 kernel takes, so the bf16 prompt run goes through it
    T = 2 * window + 70
    g = torch.Generator().manual_seed(window)
    q, k, v = torch.randn(T, H, d, generator=g) * 0.01, torch.randn(T, G, d, generator=g) * 0.01, torch.zeros(T, G, dv)
    marks = (0, 5, 63, 64, window + 3)                    # first tokens, a page border, past one window
    for n, mark in enumerate(marks):
        k[mark, 0] = 0
        k[mark, 0, n] = 1.0                               # a direction of its own
        v[mark, 0, 0] = 100.0 + mark
    portions = [T] if not decode else [window // 2, 2] + [1] * (T - window // 2 - 2)
    seen = {}
    for n, mark in enumerate(marks):
        qq = q.clone()
        for i in (mark + window - 1, mark + window):     # just inside, just outside
            qq[i, 0] = 0
            qq[i, 0, n] = 1.0
        out = _attend(ops, qq, k, v, H, G, d, dv, 40.0, window, [0.0], portions, f32=f32)
        seen[mark] = (out[mark + window - 1, 0].item(), out[mark + window, 0].item())
        assert abs(seen[mark][0] - (100.0 + mark)) < (1.0 if f32 else 2.5), (mark, seen)
        assert abs(seen[mark][1]) < 60.0 and abs(seen[mark][1] - (100.0 + mark)) > 40.0, (mark, seen)


def test_distance_penalty_is_per_head_and_in_distance(ops):
    """Equal keys everywhere: the weights are softmax(-slope * distance), a different one per head."""
    H, G, d, dv, T, window = 4, 2, 8, 4, 40, 16
    q, k = torch.ones(T, H, d), torch.ones(T, G, d)
    v = torch.arange(T).float()[:, None, None].repeat(1, G, dv)      # value = position
    slopes = [2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]
    out = _attend(ops, q, k, v, H, G, d, dv, 1.0, window, slopes, [7, 33]).view(T, H, dv)
    for h in range(H):
        for i in (0, 3, 15, 16, 39):
            js = torch.arange(max(0, i - window + 1), i + 1).double()
            p = torch.softmax(-slopes[h] * (i - js), 0)
            assert abs(out[i, h, 0].item() - (p * js).sum().item()) < 1e-3


@pytest.mark.parametrize("H,G,n,p", [(16, 16, 128, 64), (32, 2, 64, 48), (17, 1, 64, 16), (128, 1, 64, 64), (128, 2, 128, 64)])
def test_scan_of_whole_rows_equals_token_by_token(ops, H, G, n, p):
    """The two-launch form (n of 64 or 128, sixteen heads and more): both state heights, column slices of 16 and of 32."""
    test_scan_in_chunks_equals_token_by_token(ops, H, G, n, p)


@pytest.mark.parametrize("H,G,n,p", [(16, 1, 64, 16), (16, 1, 128, 32), (128, 1, 128, 64)])
def test_scan_of_whole_rows_rounds_the_state_once_a_chunk(ops, H, G, n, p):
    """States that hardly decay, eight chunks: what a chunk adds is summed apart, so the state is rounded once a chunk, each
    time by at most 2^-24 of itself and independently: sqrt(8) 2^-24 of it in the 2-norm.  (Added to the state product by
    product it is rounded sixteen times a chunk.)  The outputs read such states over n products of random sign in n / 4
    instructions, and a chunk's own 64 terms are rounded like those: as much again as n / 4 roundings of partial sums that grow to the whole."""
    g = torch.Generator().manual_seed(n + p)
    T, rep = 8 * 64, H // G
    q, k, v = torch.randn(T, G * n, generator=g), torch.randn(T, G * n, generator=g), torch.randn(T, H * p, generator=g)
    logd = -torch.rand(T, H, generator=g) * 4e-4
    cache = make_cache(state={0: {"s": (H, n, p)}})
    st = step_of(cache, [("a", [0] * T)])
    o = torch.empty(T, H * p, device=DEV)
    ops.scan_outer(q.to(DEV), k.to(DEV), v.to(DEV), torch.exp(logd).to(DEV), None, None, cache.states[0]["s"], o, st, H, n, p,
                   q_div=rep, k_div=rep, log_decay=logd.to(DEV))
    # chunk by chunk in 64 bits: S = exp(L_end) S + k^T (w v), o = exp(L) (q S + ...)
    qd, kd, vd = (x.double().to(DEV).view(T, -1, w).transpose(0, 1) for x, w in ((q, n), (k, n), (v, p)))
    qd, kd = qd.repeat_interleave(rep, 0), kd.repeat_interleave(rep, 0)
    L = logd.double().to(DEV).T
    S, want = torch.zeros(H, n, p, dtype=torch.float64, device=DEV), []
    for c in range(0, T, 64):
        s = slice(c, c + 64)
        l = L[:, s].cumsum(1)
        P = torch.tril(qd[:, s] @ kd[:, s].transpose(1, 2).contiguous() * torch.exp(l[:, :, None] - l[:, None, :]))
        want.append(P @ vd[:, s] + torch.exp(l)[:, :, None] * (qd[:, s] @ S))
        w = torch.exp(l[:, -1:] - l)[:, :, None]
        S = torch.exp(l[:, -1])[:, None, None] * S + kd[:, s].transpose(1, 2).contiguous() @ (w * vd[:, s])
    want = torch.cat(want, 1).transpose(0, 1).reshape(T, H * p)
    state = cache.states[0]["s"][int(st.row_slot[0])].double()
    assert ((state - S).norm() / S.norm()).item() < 8 ** 0.5 * 2.0 ** -24
    assert ((o.double() - want).norm() / want.norm()).item() < (8 ** 0.5 + (n / 4) ** 0.5) * 2.0 ** -24


@pytest.mark.parametrize("H,n,p", [(16, 64, 16), (16, 128, 64), (4, 64, 32)])
def test_scan_in_chunks_with_an_infinite_key_at_the_end(ops, H, n, p):
    """An infinite element of the last token's key: its state row becomes infinite in every column (v has no zero), as in the
    recurrence itself, and every other state row stays what it is.  Both chunked forms; rows that end inside a chunk."""
    g = torch.Generator().manual_seed(H + p)
    T = 70
    q, k, v = torch.randn(T, n, generator=g), torch.randn(T, n, generator=g), torch.randn(T, H * p, generator=g)
    v[T - 1] = v[T - 1].abs() + 0.1
    k[T - 1, 5] = float("inf")
    logd = -torch.rand(T, H, generator=g)
    cache = make_cache(state={0: {"s": (H, n, p)}})
    st = step_of(cache, [("a", [0] * T)])
    o = torch.empty(T, H * p, device=DEV)
    ops.scan_outer(q.to(DEV), k.to(DEV), v.to(DEV), torch.exp(logd).to(DEV), None, None, cache.states[0]["s"], o, st, H, n, p,
                   q_div=H, k_div=H, log_decay=logd.to(DEV))
    state = cache.states[0]["s"][int(st.row_slot[0])].cpu()
    assert bool((state[:, 5] == float("inf")).all())
    assert bool(torch.isfinite(state[:, torch.arange(n) != 5]).all()) and bool(torch.isfinite(o[:T - 1]).all())


@pytest.mark.parametrize("C,taps", [(4, 4), (1028, 4), (8448, 4), (260, 3), (64, 2), (24, 5), (30, 4), (14336, 4),
                                    (14336, 3), (14336, 2)])
def test_conv_silu_forms(ops, C, taps):
    """Runs of eight tokens over several rows in one step (14336 channels; row starts inside a run, rows shorter than the
    taps) or a thread per output (fewer), then one token a row, then both again: the same sums in the same order, so every
    output is the plain form's to its last bits (1e-5 covers the exponential against 64 bits)."""
    g = torch.Generator().manual_seed(C)
    lens = {"a": 21, "b": 2, "c": 9, "d": 64}
    x = {k: torch.randn(2 * n + 4, C, generator=g) for k, n in lens.items()}
    w, b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    want = {k: ref.causal_conv_silu(v.double(), w.double(), b.double()) for k, v in x.items()}
    cache = make_cache(state={0: {"conv": (taps - 1, C)}}, slots=6)
    cache.admit("other")
    cache.states[0]["conv"].fill_(7.0)
    pos = {k: 0 for k in lens}
    for step_lens in (lens, {k: 1 for k in lens}, {k: 1 for k in lens}, {"c": 3, "a": 1}, {"b": 1}, {"a": 19, "b": 2, "c": 4, "d": 63}):
        st = step_of(cache, [(k, [0] * n) for k, n in step_lens.items()])
        inp = torch.cat([x[k][pos[k]:pos[k] + n] for k, n in step_lens.items()])
        o = torch.full(inp.shape, float("nan"), device=DEV)
        ops.conv_silu(inp.to(DEV), cache.states[0]["conv"], w.to(DEV), b.to(DEV), o, st)
        at = 0
        for k, n in step_lens.items():
            assert (o[at:at + n].cpu().double() - want[k][pos[k]:pos[k] + n]).abs().max().item() < 1e-5, (k, pos[k], n)
            at, pos[k] = at + n, pos[k] + n


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("rows,n,groups", [(1, 8192, 1), (300, 8192, 1), (3, 1024, 1), (2, 4104, 2), (260, 2052, 2), (1, 33000, 1),
                                           (300, 9000, 1), (5, 1026, 1)])
def test_gated_group_norm_of_wide_groups(ops, rows, n, groups, f32):
    """Values in registers (1024 and 256 threads, one to eight pieces each, the last partly past the end) and the looped form
    (groups too wide or not in fours), for the three modes, with a weight of a group and of a row."""
    g = torch.Generator().manual_seed(n + rows)
    y, z = torch.randn(rows, n, generator=g) * 4, torch.randn(rows, n + 4, generator=g)
    dt, eps = torch.float32 if f32 else torch.bfloat16, 1e-5
    for mode, wn in ((0, n), (1, n), (2, n // groups), (0, 0)):
        w = torch.randn(wn, generator=g) if wn else None
        out = torch.empty(rows, n, dtype=dt, device=DEV)
        ops.gated_group_norm(y.to(DEV), z.to(DEV)[:, :n], None if w is None else w.to(DEV), out, groups, mode == 1, eps,
                             sigmoid=mode == 2)
        zd = z[:, :n].double()
        gate = torch.sigmoid(zd) if mode == 2 else zd * torch.sigmoid(zd)
        u = y.double() * gate if mode == 1 else y.double()
        want = ref.unit_rms(u.view(rows, groups, -1), eps).reshape(rows, n)
        if mode != 1:
            want = want * gate
        if w is not None:
            want = want * (w.double() if wn == n else w.double().repeat(groups))
        tol = (1e-5 if f32 else 2 ** -8) * want.abs() + 1e-6       # fp32 products, a rounding to the output's type
        assert ((out.cpu().double() - want).abs() <= tol).all(), mode


@pytest.mark.parametrize("H,G,n,p", [(4, 2, 64, 64), (3, 1, 128, 128), (3, 3, 256, 64), (2, 1, 64, 192)])
def test_scan_token_by_token_in_whole_pieces(ops, H, G, n, p):
    """The form that reads state, q, k and v in 16-byte pieces: its three state heights, one to three column tiles."""
    test_scan_whole_portions_and_rows(ops, H, G, n, p)


@pytest.mark.parametrize("taps,C,H", [(4, 8448, 128), (3, 260, 300), (2, 64, 1), (4, 70, 5), (1, 64, 8)])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1], [5, 1, 9]])
def test_convolution_and_step_decays_in_one_call(ops, taps, C, H, lens):
    """What conv_silu and softplus_decay give one after the other, bit for bit: one launch where every row brings one token and
    the channels allow it (heads past one workgroup, one head), two elsewhere."""
    g = torch.Generator().manual_seed(C + H)
    T = sum(lens)
    x = torch.randn(T, C + 4 + H, generator=g).to(DEV)
    w, b, dt, al = (torch.randn(*s, generator=g).to(DEV) for s in ((C, taps), (C,), (H,), (H,)))
    start = torch.randn(6, max(taps - 1, 0), C, generator=g).to(DEV)
    res = []
    for joint in (True, False):
        cache = make_cache(state={0: {"conv": (max(taps - 1, 1), C)}}, slots=6)
        names = [f"r{i}" for i in range(len(lens))]
        state = start.clone()
        out = []
        for _ in range(2):      # the second step carries the first one's inputs
            st = step_of(cache, [(k, [0] * n) for k, n in zip(names, lens)])
            o, gain, dec, lg = (torch.full((T, n), float("nan"), device=DEV) for n in (C, H, H, H))
            d = (x[:, C + 4:], dt, al, gain, dec, lg)
            ops.conv_silu(x[:, :C], state, w, b, o, st, decay=d if joint else None)
            if not joint:
                ops.softplus_decay(*d)
            out += [o, gain, dec, lg, state.clone()]
        res.append(out)
    for a, c in zip(*res):
        assert torch.equal(a, c)
