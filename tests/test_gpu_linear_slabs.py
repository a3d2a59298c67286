"""Projections left in k-slices (mv_linear_slabs) and the residual norms that add them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _take(rows, cols):
    return torch.full((rows, cols), float("nan"), dtype=torch.float32, device=DEV)


# up to four rows strips that leave compute units idle are cut (1, 2, 4 and 8 ways and a k too short for it), 5 to 64 as the
# batched projections, more as the prompts' (cut, and whole in tiles whose left-overs are cut inside the launch)
@pytest.mark.parametrize("m,n,k", [(1, 1024, 5120), (1, 1024, 1024), (2, 512, 8192), (3, 2048, 8192), (4, 16, 8192), (4, 4096, 512),
                                   (5, 2048, 8192), (16, 1040, 2048), (33, 2048, 8192), (64, 1024, 4096), (65, 1024, 4096),
                                   (300, 2048, 8192), (700, 2048, 8192), (3072, 6144, 4096)])
def test_slices_add_up_to_the_product(mv, m, n, k):
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(DEV)
    lin = AnyLinear(w)
    got = lin.slabs(x, _take)
    assert got.shape == (nv.lib().mv_linear_slab_count(m, n, k), m, n)
    want = x.double() @ w.double().t()
    # fp32 sums of k products of order 1 / sqrt(k): their error stays below sqrt(k) * 2^-24 of the largest partial sum
    tol = k ** 0.5 * 2 ** -24 * 8
    assert (got.double().sum(0) - want).abs().max().item() <= tol
    again = lin.slabs(x, _take)
    assert torch.equal(got, again)


@pytest.mark.parametrize("rows,n", [(1, 64), (1, 1024), (3, 2048), (5, 4096), (2, 8192), (513, 1024), (600, 4096), (7, 100), (3, 33)])
@pytest.mark.parametrize("ks", [1, 2, 3, 4, 5, 8, 16])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32])
def test_norms_add_the_slices_in_order(mv, rows, n, ks, act):
    """The residual steps over slices give what they give over the slices' sum taken in order, bit for bit (every width of
    the register forms and, with n not a multiple of four, the plain one)."""
    from micro_vllm_amd.kernel import ragged_ops as ops

    g = torch.Generator().manual_seed(rows * n + ks)
    mk = lambda *s: torch.randn(*s, generator=g).to(DEV)   # noqa: E731
    y1, y2, x, w, nxt, bias = mk(ks, rows, n), mk(2, rows, n), mk(rows, n), mk(n), mk(n), mk(n)
    total = y1[0].clone()
    for i in range(1, ks):
        total += y1[i]
    total2 = y2[0] + y2[1]
    for second in (False, True):
        res = []
        for a, b in ((y1, y2), (total, total2)):
            xs, h = x.clone(), torch.empty(rows, n, dtype=act, device=DEV)
            ops.postnorm_residual(a, w, 1e-5, xs, h, y2=b if second else None, s1=0.5, s2=2.0, bias=bias, mult=0.7, next_w=nxt)
            res += [xs, h]
        assert torch.equal(res[0], res[2]) and torch.equal(res[1], res[3])
        res = []
        for a in (y1, total):
            xs, h = x.clone(), torch.empty(rows, n, dtype=act, device=DEV)
            ops.add_rmsnorm(xs, a, total2 if second else None, w=w, eps=1e-5, h=h)
            res += [xs, h]
        assert torch.equal(res[0], res[2]) and torch.equal(res[1], res[3])
        want = x.double() + total.double() + (total2.double() if second else 0.0)
        normed = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5) * w.double()
        # the square sum's error grows with the chain of additions, far below one bf16 unit; fp32 results lie within 2^-20
        tol = 2 ** -8 if act == torch.bfloat16 else 2 ** -18
        assert ((res[1].double() - normed).abs() <= tol * normed.abs() + 1e-6).all()


# streamed slices of fp32 weights: whole, two, four, eight; k that is no multiple of a slice's share and one that ends inside a
# step; rows up to the limit of the streamed form and past it
@pytest.mark.parametrize("m,n,k", [(1, 1024, 5120), (3, 1024, 1024), (8, 1024, 2048), (16, 512, 4096), (16, 2048, 4100), (2, 40, 8192),
                                   (1, 16, 12), (3, 1030, 5132), (17, 1024, 5120), (4, 9472, 2048)])
def test_streamed_fp32_slices_add_up_to_the_product(mv, m, n, k):
    from micro_vllm_amd import _native as nv
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(DEV)
    lin = AnyLinear((torch.randn(n, k, generator=g) / k ** 0.5).to(DEV))
    got = lin.slabs(x, _take)
    ks = nv.lib().mv_linear_any_slab_count(m, n, k)
    assert got.shape == (ks, m, n) and (ks > 1) == ((m, n, k) in ((1, 1024, 5120), (8, 1024, 2048), (16, 512, 4096), (16, 2048, 4100),
                                                                 (2, 40, 8192), (3, 1030, 5132)))
    want = x.double() @ lin.w.double().t()
    tol = k ** 0.5 * 2 ** -24 * 8      # as above: fp32 sums of products of order 1 / sqrt(k)
    assert (got.double().sum(0) - want).abs().max().item() <= tol
    # an operand that is not aligned goes whole, as it did
    wide = torch.randn(m, k + 1, generator=g).to(DEV)[:, 1:]
    assert lin.slabs(wide, _take).shape == (1, m, n)


# streamed fp32 weights: one piece of 128 k a quarter, a piece and a step, three pieces, four and a part; four, eight and sixteen rows of
# x and one past each; wide outputs from k = 512 on and tiles short of it.  A row by itself has the same bits
@pytest.mark.parametrize("m,n,k", [(4, 33, 512), (5, 40, 516), (8, 1030, 1100), (9, 17, 2052), (16, 16, 4), (3, 8200, 1668), (9, 8208, 512),
                                   (16, 8208, 508), (16, 9001, 1024)])
def test_streamed_fp32_pieces(mv, m, n, k):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.full((m, k + 4), float("nan"), device=DEV), torch.full((n, k + 4), float("nan"), device=DEV)
    x[:, :k] = torch.randn(m, k, generator=g).to(DEV)
    w[:, :k] = (torch.randn(n, k, generator=g) / k ** 0.5).to(DEV)
    lin = AnyLinear(w[:, :k].contiguous())
    got = lin(x[:, :k], torch.full((m, n), float("nan"), device=DEV))
    assert (got.double() - x[:, :k].double() @ lin.w.double().t()).abs().max().item() <= k ** 0.5 * 2 ** -24 * 8
    assert torch.equal(lin(x[m - 1:, :k].contiguous()), got[m - 1:])


# 64 x 64 tiles in four groups: up to one for every compute unit, k from 18 steps of 32 on and one short of it, k that ends
# inside a step and inside a group of four, rows and columns that end inside a tile
@pytest.mark.parametrize("m,n,k", [(567, 1024, 5120), (1000, 1024, 576), (1000, 1024, 544), (641, 1601, 1030), (1000, 1000, 1092),
                                   (70, 9480, 1024), (1024, 1024, 4099)])
def test_fp32_tiles_by_themselves_on_a_unit(mv, m, n, k):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(DEV)
    lin = AnyLinear((torch.randn(n, k, generator=g) / k ** 0.5).to(DEV))
    got = lin(x, torch.full((m, n), float("nan"), device=DEV))
    want = x.double() @ lin.w.double().t()
    assert (got.double() - want).abs().max().item() <= k ** 0.5 * 2 ** -24 * 8


# every kernel that has such an epilogue: dot form, matrix form, slices behind a reduction (few rows and many), 64-row tiles of one,
# two and four strips, 128-row tiles, both wide tiles; columns that end inside a workgroup's
@pytest.mark.parametrize("m", [1, 4, 5, 40, 64, 65, 300, 700, 2048])
@pytest.mark.parametrize("n,k", [(1024, 512), (1040, 2048), (8192, 1024), (16384, 2048)])
@pytest.mark.parametrize("kind", [1, 2])
def test_activations_in_the_product(mv, m, n, k, kind):
    from micro_vllm_amd.kernel import ragged_ops as ops

    g = torch.Generator().manual_seed(m + n + k + kind)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (2.0 * torch.randn(n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(DEV)
    v = x.double() @ w.double().t()
    none = lambda *a: pytest.fail("not in the epilogue")   # noqa: E731
    err = k ** 0.5 * 2 ** -24 * 8      # of the product, as above
    if kind == 1:
        got = ops.linear_relu_squared(x, ops.AnyLinear(w), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), none)
        want, slope = v.clamp(min=0) ** 2, 2 * v.abs()
    else:
        gate, up = w[:n // 2].contiguous(), w[n // 2:].contiguous()
        got = ops.GatedLinear(gate, up)(x, torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV), none, 2.5, 1.702)
        a, b = v[:, :n // 2].clamp(max=2.5), v[:, n // 2:].clamp(-2.5, 2.5)
        want, slope = a * torch.sigmoid(1.702 * a) * (b + 1), 1.5 * (b + 1).abs() + a.abs()
    # half a bf16 unit, the product's error through the function's slope, and 2^-20 for the function itself
    tol = 2.0 ** -8 * want.abs() + 2 * err * slope + err + 2.0 ** -20 * want.abs()
    assert ((got.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("rows,n", [(1, 64), (2, 1024), (3, 2048), (5, 4096), (2, 8192), (1, 16384), (513, 1024), (600, 4096), (2, 16388), (3, 33)])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32])
def test_gathered_norms_of_every_width(mv, rows, n, act):
    from micro_vllm_amd.kernel import ragged_ops as ops

    g = torch.Generator().manual_seed(rows + n)
    x, w = (torch.randn(rows + 2, n, generator=g) * 3).to(DEV), torch.randn(n, generator=g).to(DEV)
    idx = torch.randint(0, rows + 2, (rows,), generator=g).to(torch.int32).to(DEV)
    for offset in (0.0, 1.0):
        out = torch.empty(rows, n, dtype=act, device=DEV)
        ops.rmsnorm_gather(x, idx, w, 1e-5, out, offset)
        v = x.double()[idx.long()]
        want = v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5) * (offset + w.double())
        # one bf16 rounding; in fp32 the square sum's n additions and the four operations behind it
        tol = 2 ** -8 if act == torch.bfloat16 else 2 ** -18
        assert ((out.double() - want).abs() <= tol * want.abs() + 1e-6).all()


# both sides of 64 rows and every form of the product; gates far below zero, where the exponential's argument is large
@pytest.mark.parametrize("m", [1, 5, 64, 65, 130, 700, 2048])
@pytest.mark.parametrize("n,k", [(1040, 512), (8192, 1024), (16384, 2048)])
@pytest.mark.parametrize("kind", [1, 2])
def test_activations_in_the_product_are_those_behind_it(mv, m, n, k, kind):
    """The epilogue's functions are the activation kernels' own: bit for bit what they make of the same product's fp32 sums,
    whatever form the number of rows takes."""
    from micro_vllm_amd.kernel import ragged_ops as ops

    g = torch.Generator().manual_seed(m + n + k + kind)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (8.0 * torch.randn(n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(DEV)
    none = lambda *a: pytest.fail("not in the epilogue")   # noqa: E731
    sums = ops.AnyLinear(w)(x)
    if kind == 1:
        got = ops.linear_relu_squared(x, ops.AnyLinear(w), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), none)
        want = torch.empty_like(got)
        ops.relu_squared(sums, want)
    else:
        # w as the product holds it: eight rows of up, their eight gates
        rows = w.view(n // 16, 2, 8, k)
        up, gate = rows[:, 0].reshape(n // 2, k), rows[:, 1].reshape(n // 2, k)
        got = ops.GatedLinear(gate, up)(x, torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV), none, 7.0, 1.702)
        v = sums.view(m, n // 16, 2, 8)
        want = torch.empty_like(got)
        ops.gated_act(torch.cat([v[:, :, 1].reshape(m, n // 2), v[:, :, 0].reshape(m, n // 2)], 1), want, ops.GATE_CLAMPED, 7.0, 1.702)
    assert torch.equal(got, want)


@pytest.mark.parametrize("m,n,k", [(1, 1024, 5120), (16, 2048, 4100), (3, 1030, 5132), (1, 16, 12)])
@pytest.mark.parametrize("x_off,w_off", [(0, 1), (0, 2), (1, 0), (3, 3)])
def test_unaligned_fp32_operands_go_whole(mv, m, n, k, x_off, w_off):
    """Weights and rows that are views at any offset of a larger buffer, at shapes that are cut where both are aligned: the whole
    product, as mv_linear_any gives it."""
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    flat_w = (torch.randn(n * k + w_off, generator=g) / k ** 0.5).to(DEV)
    flat_x = torch.randn(m * k + x_off, generator=g).to(DEV)
    x, lin = flat_x[x_off:].view(m, k), AnyLinear(flat_w[w_off:].view(n, k))
    assert lin.w.data_ptr() % 16 == 4 * w_off
    got = lin.slabs(x, _take)
    assert got.shape == (1, m, n) and torch.equal(got[0], lin(x))
    want = x.double() @ lin.w.double().t()
    assert (got[0].double() - want).abs().max().item() <= k ** 0.5 * 2 ** -24 * 8      # as above


# x of two to four rows that just fits the dot form's LDS, that fits with half the waves only (256 strips), and that does not
@pytest.mark.parametrize("m,k", [(4, 20096), (4, 20160), (4, 20480), (3, 26944), (3, 28672), (2, 40512), (2, 40576)])
@pytest.mark.parametrize("n", [64, 4096])
def test_few_rows_of_a_long_k(mv, m, n, k):
    from micro_vllm_amd.kernel import ragged_ops as ops
    from micro_vllm_amd.kernel.linear import StreamedWeight, wgemm, wgemm_postnorm

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(DEV)
    res, ln = torch.randn(m, n, generator=g).to(torch.bfloat16).to(DEV), torch.ones(n, dtype=torch.bfloat16, device=DEV)
    want = x.double() @ w.double().t()
    tol = k ** 0.5 * 2 ** -24 * 8      # as above
    lin = ops.AnyLinear(w)
    assert (lin(x).double() - want).abs().max().item() <= tol
    assert (lin.slabs(x, _take).double().sum(0) - want).abs().max().item() <= tol
    act = ops.linear_relu_squared(x, lin, torch.empty(m, n, dtype=torch.bfloat16, device=DEV), None)
    sq = want.clamp(min=0) ** 2
    assert ((act.double() - sq).abs() <= 2 ** -8 * sq + 2 * tol * want.abs() + tol).all()
    sw = StreamedWeight.from_linear(w)
    out, out2, normed = (torch.empty(m, n, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    wgemm(x, sw, out, residual=res)
    # two roundings to bf16, of the product and of the sum
    assert ((out.double() - want - res.double()).abs() <= 2 ** -8 * (want.abs() + (want + res.double()).abs()) + 2 * tol).all()
    wgemm_postnorm(x, sw, out2, ln, 1e-5, normed, residual=res, var_from_rounded=True)
    ref = out2.double() / torch.sqrt((out2.double() ** 2).mean(-1, keepdim=True) + 1e-5)
    assert ((out2.double() - want - res.double()).abs() <= 2 ** -8 * (want.abs() + (want + res.double()).abs()) + 2 * tol).all()
    # the norm's factor and the result round to bf16 once each, the weight is one
    assert ((normed.double() - ref).abs() <= 2 ** -7 * ref.abs() + 1e-6).all()


# one and two rows up to the k whose tiles fill one stage, and a tile past it: the sums of the three-row kernel, bit for bit, plain,
# with a norm in front, with a bias and with a gate; strips that end inside a round of workgroups
@pytest.mark.parametrize("n,k", [(48, 32), (528, 256), (9472, 992), (1040, 1024), (9472, 1024), (16400, 1024), (1040, 1056)])
def test_short_k_of_one_and_two_rows(mv, n, k):
    from micro_vllm_amd.kernel.linear import StreamedWeight, wgemm, wgemm_norm

    g = torch.Generator().manual_seed(n + k)
    x = torch.randn(3, k, generator=g).bfloat16().to(DEV)
    wt = (torch.randn(n, k, generator=g) / k ** 0.5).bfloat16().to(DEV)
    ln, bias = torch.rand(k, generator=g).bfloat16().to(DEV), torch.randn(n, generator=g).bfloat16().to(DEV)
    w, gu = StreamedWeight.from_linear(wt), StreamedWeight.from_up_gate(wt[:n // 2].contiguous(), wt[n // 2:].contiguous())

    def forms(rows):
        r, out = x[:rows], lambda c, dt=torch.bfloat16: torch.empty(rows, c, dtype=dt, device=DEV)
        return (wgemm(r, w, out(n, torch.float32)), wgemm(r, w, out(n), bias=bias), wgemm(r, gu, out(n // 2), swiglu=True),
                wgemm_norm(r, ln, 1e-5, w, out(n)), wgemm_norm(r, ln, 1e-5, w, out(n), add_r=r, sum_out=out(k)))

    want = forms(3)
    assert (want[0].double() - x.double() @ wt.double().t()).abs().max().item() <= k ** 0.5 * 2 ** -24 * 64
    for rows in (1, 2):
        for a, b in zip(forms(rows), want):
            assert torch.equal(a, b[:rows])


# fp32 factors in three bf16 parts: what those cannot hold (infinities, NaN, values that round to an infinite bf16, sums in the
# range of the smallest numbers) has the value of fp32 arithmetic, and only it: neighbours keep their bits.  Every form has a shape
# (test_fp32_forms_of_the_shapes_here): streamed, six tiles, a k that ends inside a step
_BEYOND = [(3, 1024, 1024), (1100, 4112, 1000), (16, 50, 516), (20, 1000, 1022), (33, 9472, 256), (200, 4000, 128), (567, 1024, 640), (333, 9472, 68),
           (2048, 4096, 64), (4, 1024, 2048), (8, 528, 516), (1000, 5000, 516), (700, 5001, 514), (567, 9472, 1024), (2050, 9472, 1028)]


@pytest.mark.parametrize("m,n,k", _BEYOND)
def test_fp32_values_beyond_the_parts(mv, m, n, k):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(DEV)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).bfloat16().float().to(DEV)
    w[n // 2:] += 2.0 ** -12 * torch.randn(n - n // 2, k, generator=g).to(DEV)     # rows of bf16 values, and rows of more
    plain = AnyLinear(w)(x)
    err = (plain.double() - x.double() @ w.double().t()).abs()
    assert bool((err <= k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())).all())
    big, odd = torch.finfo(torch.float32).max, x.clone()
    odd[0, 1], odd[1, 2], odd[2, :] = float("inf"), float("nan"), x[2] * 2.0 ** -116
    wo = w.clone()
    wo[3, 0], wo[5, :] = -float("inf"), 0.0
    wo[7, :] = 0.0
    wo[7, 4] = 1.0
    if m > 3:
        odd[3, :] = 0.0
        odd[3, 4] = big          # its bf16 is infinite
    got = AnyLinear(wo)(odd)
    want = odd.double() @ wo.double().t()
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got[inf].double(), want[inf])
    fine = [i for i in range(m) if i > 3]
    cols = [j for j in range(n) if j not in (3, 5, 7)]
    if fine:
        assert torch.equal(got[fine][:, cols], plain[fine][:, cols])
    tiny = (got[2].double() - want[2]).abs() <= k * 2.0 ** -24 * (odd[2].double().abs() @ wo.double().abs().t()) + k * 2.0 ** -149
    assert bool(tiny[torch.tensor([j for j in range(n) if j != 3])].all())
    assert bool((got[:, 5][torch.isfinite(odd).all(1)] == 0).all())
    if m > 3:
        assert got[3, 7].item() == big


# fp32 factors far apart in size, whose sum is an ordinary number: of a small factor the parts lose bits, and a sum of zeros may be
# parts that are all lost.  The shapes go to each form: streamed with 4, 8, 16 rows, whole and in slices, the six tiles (the last
# four by scalar loads)
_FAR_APART = [(3, 1024, 1024), (1100, 4112, 1002), (33, 5000, 516), (3, 1024, 5120), (8, 528, 516), (16, 50, 516), (33, 9472, 256), (333, 9472, 68), (1000, 5000, 516),
              (567, 9472, 1024), (2050, 9472, 1028), (20, 1000, 1022), (200, 16390, 514), (700, 5001, 514), (2050, 9001, 1022)]


@pytest.mark.parametrize("m,n,k", _FAR_APART)
def test_fp32_factors_of_any_size(mv, m, n, k):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(DEV), (torch.randn(n, k, generator=g) / k ** 0.5).to(DEV)
    plain = AnyLinear(w)(x)
    odd, wo = x.clone(), w.clone()
    odd[0] *= 2.0 ** -120                    # against row 1: 2^-50
    wo[1] *= 2.0 ** 70
    odd[1] *= 2.0 ** 66                      # against row 2: 2^-54
    wo[2] = (wo[2] * 2.0 ** -120).bfloat16().float()
    odd[2] = 0.0
    odd[2, 5] = 2.0 ** -140                  # no part of it is a bf16 number
    wo[3, 5], wo[4, 5] = 2.0 ** 100, 1.0     # 2^-40, 2^-140
    wo[5, 0::2], wo[5, 1::2] = 2.0 ** 100, 0.0
    odd[min(3, m - 1), 0::2] *= 2.0 ** -118   # beside ordinary factors
    got = AnyLinear(wo)(odd)
    want, size = odd.double() @ wo.double().t(), odd.double().abs() @ wo.double().abs().t()
    held = size < 2.0 ** 127
    # a fp32 rounding of each product and each sum, and the smallest fp32 number for each
    off = lambda y: (y - want).abs() > k * 2.0 ** -24 * size + k * 2.0 ** -149   # noqa: E731
    assert not bool((off(got.double()) & held).any())
    assert not bool((off(AnyLinear(wo).slabs(odd, _take).double().sum(0)) & held).any())
    assert got[2, 3].item() == 2.0 ** -40 and got[2, 4].item() == 2.0 ** -140
    assert torch.equal(AnyLinear(wo)(odd[:3].contiguous())[held[:3]], got[:3][held[:3]])
    assert torch.equal(got[4:, 6:], plain[4:, 6:])


# the sums of a row are those of four quarters of k in ascending order in every form: streamed, and the six tiles
_AMONG_MANY = [(20, 1000, 1022), (33, 9472, 256), (567, 1024, 640), (333, 9472, 68), (700, 3000, 250), (1100, 4112, 1000),
               (1000, 5000, 516), (567, 9472, 1024), (2050, 9472, 1028)]


@pytest.mark.parametrize("many,n,k", _AMONG_MANY)
def test_fp32_rows_do_not_depend_on_the_others(mv, many, n, k):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(many + n + k)
    x, lin = torch.randn(many, k, generator=g).to(DEV), AnyLinear((torch.randn(n, k, generator=g) / k ** 0.5).to(DEV))
    want = lin(x)
    for rows in (1, 5, 9, 17, 40, 130):
        assert torch.equal(lin(x[:rows]), want[:rows])


# fp32 weights that are bf16 values but in single steps of 32 k: which rows take six products and which three changes from step to
# step, from one block of sixteen rows to the next, and with how many steps a form looks at together.  A row alone (streamed, a step
# or four at a time), 5, 8, 9 and 16 rows (streamed, and tiles where k is short and n wide) and many (tiles of every
# size that goes with k) are the same bits
@pytest.mark.parametrize("n,k,many", [(48, 1024, 40), (1040, 1028, 300), (1040, 1030, 300), (8208, 256, 70), (8208, 260, 600), (16400, 256, 70), (9472, 544, 600),
                                      (4112, 1000, 1100), (528, 2052, 300)])
def test_low_bits_in_some_steps_only(mv, n, k, many):
    from micro_vllm_amd.kernel.ragged_ops import AnyLinear

    g = torch.Generator().manual_seed(n + k)
    x = torch.randn(many, k, generator=g).to(DEV)
    full = (torch.randn(n, k, generator=g) / k ** 0.5).to(DEV)
    w, step, block = full.bfloat16().float(), torch.arange(k, device=DEV) // 32, torch.arange(n, device=DEV) // 16
    last = (k - 1) // 32
    odd = ((block[:, None] % 5 == 1) & (step % 2 == 1)) | ((block[:, None] % 5 == 2) & (step == 0)) | \
          ((block[:, None] % 5 == 3) & (step == last)) | ((block[:, None] % 5 == 4) & (step % 7 == 3))
    odd &= torch.arange(n, device=DEV)[:, None] % 16 == 11       # one row of a block
    w = torch.where(odd, full, w)
    lin = AnyLinear(w)
    want = lin(x)
    err = (want.double() - x.double() @ w.double().t()).abs()
    # a rounding of each product and each sum
    assert bool((err <= k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())).all())
    for rows in (1, 4, 5, 8, 9, 16, 33):
        assert torch.equal(lin(x[:rows]), want[:rows])


def test_fp32_forms_of_the_shapes_here(mv):
    """The lists above reach what they say they do: all streamed forms and all six tiles."""
    from micro_vllm_amd import _native as nv

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("laid out for 256 compute units")
    forms = lambda shapes: {nv.lib().mv_linear_any_form(*s) for s in shapes}   # noqa: E731
    assert forms(_BEYOND) == forms(_FAR_APART) == set(range(10))
    assert forms(_AMONG_MANY) == set(range(4, 10))
    assert [nv.lib().mv_linear_any_form(rows, 1024, 2048) for rows in (1, 5, 9, 17)] == [1, 2, 3, 4]
