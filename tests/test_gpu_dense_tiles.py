"""The tile sizes of the dense product: each chosen by size, all with the same bits for a row whatever the rows around it."""
import numpy as np
import pytest

from tests import dimesun_fixture as dx
from tests import takosun_fixture as tx

pytestmark = pytest.mark.gpu


FORMS = ["256 x 256", "128 x 256", "128 x 128", "64 x 128", "64 x 64, four stages", "64 x 64, two stages", "64 x 32", "64-bit offsets"]


def form_of(pkg, M, N, K, dtype="bfloat16"):
    """The kernel of a product whose rows are as long as K, padded."""
    step = 64 if dtype == "bfloat16" else 32
    ld = -(-K // step) * step
    return FORMS[pkg.capi.dense().a81w41_dense_form_selfcheck(M, N, K, ld, ld, dtype == "bfloat16")]


# Ragged rows and columns, by 64 x 64 tiles with two stages but for 256 x 256 (1793 rows) and 128 x 128 (1921), against few rows of them
@pytest.mark.parametrize("M,N,K", [(2047, 6136, 64), (1793, 6400, 192), (2300, 2050, 128), (2045, 2000, 64), (2045, 1990, 192),
                                   (1921, 2048, 320), (1025, 1990, 64), (1030, 2048, 192), (700, 3070, 320)])
def test_rows_of_a_product(pkg, M, N, K):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    got = pkg.ops.dense_gemm(a, w, K)
    want = a.double() @ w.double().t()
    # K exact products of size about 1, K sums rounded to 24 bits
    assert (got.double() - want).abs().max().item() <= K * 2.0 ** -24 * 4 * K ** 0.5
    assert form_of(pkg, M, N, K) == {1793: FORMS[0], 1921: FORMS[2]}.get(M, FORMS[5])
    for m in (1, 32, 33, 64, 65, 100):   # the kernel for few rows and, where the product is wide, 64 x 64 tiles
        assert torch.equal(pkg.ops.dense_gemm(a[M - m:], w, K), got[M - m:]), m


# In float: 64 x 64 tiles with two stages, against few rows of them.
@pytest.mark.parametrize("M,N,K", [(2300, 2050, 32), (2047, 4100, 96), (2045, 1990, 160), (1025, 1990, 64)])
def test_rows_of_a_float_product(pkg, M, N, K):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    a, w = torch.randn(M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g)
    got = pkg.ops.dense_gemm(a, w, K)
    # K products and K sums of size about 1, each rounded to 24 bits
    assert (got.double() - a.double() @ w.double().t()).abs().max().item() <= 2 * K * 2.0 ** -24 * 4 * K ** 0.5
    for m in (33, 100):
        assert torch.equal(pkg.ops.dense_gemm(a[M - m:], w, K), got[M - m:]), m


# Steps of 128 bytes of K around the ring lengths of the kernel for few rows, 10 stages of rows and 20 of weights, and past them; one and
# two row tiles, ragged columns.  The same rows among many more go through 64 x 128 and 128 x 128 tiles, in float 64 x 64.
@pytest.mark.parametrize("steps", [9, 10, 11, 19, 20, 21, 22, 97])
@pytest.mark.parametrize("M,N", [(33, 784), (65, 1990)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_few_rows_around_the_ring(pkg, steps, M, N, dtype):
    import torch
    g = torch.Generator(device="cuda").manual_seed(steps)
    bf16 = dtype == "bfloat16"
    K = steps * (64 if bf16 else 32)
    a = torch.randn(2047, K, device="cuda", generator=g).to(getattr(torch, dtype))
    w = torch.randn(N, K, device="cuda", generator=g).to(getattr(torch, dtype))
    got = pkg.ops.dense_gemm(a[:M], w, K)
    assert form_of(pkg, M, N, K, dtype) == FORMS[6] and form_of(pkg, 2047, N, K, dtype) in FORMS[2:6]
    # K products (exact in bfloat16) and K sums, rounded to 24 bits
    bound = (1 if bf16 else 2) * K * 2.0 ** -24 * 4 * K ** 0.5
    assert (got.double() - a[:M].double() @ w.double().t()).abs().max().item() <= bound
    assert torch.equal(pkg.ops.dense_gemm(a, w, K)[:M], got)


def _same_in_portions(pkg, cfg, n, cuts):
    """One pass over n tokens on large tiles, and the same in portions on small ones, attention by the kernel that goes row by row."""
    ids = np.random.default_rng(5).integers(0, cfg["vocab"], n).astype(np.int32)
    want = list(range(0, n, 97)) + [n - 1]
    model = pkg.Model.random(cfg, n, "bfloat16", seed=3)
    model.set_option("attention", 1)
    whole = model.forward(ids, want)
    model.reset()
    parts, at = [], 0
    while at < n:
        m = min(cuts, n - at)
        parts.append(model.forward(ids[at:at + m], [w - at for w in want if at <= w < at + m]))
        at += m
    assert np.isfinite(whole).all() and np.array_equal(whole, np.concatenate(parts))


# one step of K, which goes by 64 x 64 tiles, and four and eleven, by 256 x 256
@pytest.mark.parametrize("width", [64, 256, 704])
def test_gated_pairs_on_large_tiles(pkg, width):
    assert form_of(pkg, 2100, 12224, width) == FORMS[5 if width == 64 else 0]
    cfg = tx.config(64, width, 1, [tx.layer(tx.mixer(2, 8, 8, 8, 16, 24, 0.3), tx.dense(6100))])
    _same_in_portions(pkg, cfg, 2100, 100)


def test_experts_on_many_small_tiles(pkg):
    cfg = tx.config(64, 64, 1, [tx.layer(tx.mixer(2, 8, 8, 8, 16, 24, 0.3), tx.moe(8, 2, 250))])
    _same_in_portions(pkg, cfg, 2100, 100)


# one step of K, which goes by 64 x 64 tiles, and three and four, by 256 x 256; columns behind the heads, five of them, are no whole fours
@pytest.mark.parametrize("width,experts", [(64, 0), (192, 0), (256, 5)])
def test_head_columns_on_large_tiles(pkg, width, experts):
    assert form_of(pkg, 2100, 6144 + experts, width) == FORMS[5 if width == 64 else 0]
    mlp = dx.moe(experts, 2, 16) if experts else None
    cfg = dx.config(64, width, [dx.attention(32, 8, 128, 128, 70, 0.09, rot_dims=64, mlp=mlp)], (0, 1, 1))
    _same_in_portions(pkg, cfg, 2100, 100)


# ---- attention over a prompt ------------------------------------------------------------------
# Many turns of both key groups, ends inside a tile of 64 keys, of 128 rows and of a share; a scale below zero and of zero;
# value widths and output strides that are no multiple of four.  97 tokens of three heads go to the kernel of short prompts.
@pytest.mark.parametrize("M,pos,chunk,splits", [(97, 0, 0, 1), (700, 5, 0, 1), (641, 64, 0, 3), (520, 130, 192, 1), (333, 3, 500, 2)])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (128, 125), (104, 61), (256, 254)])
@pytest.mark.parametrize("scale", [0.09, -0.11, 0.0])
def test_attention_over_a_prompt(pkg, M, pos, chunk, splits, dim, vdim, scale):
    import torch
    heads, kv_heads, seq = 6, 2, pos + M + 9
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    value = (vdim + 7) // 8 * 8
    q = torch.randn(M, heads, dim, device="cuda", generator=g).bfloat16()
    rows = torch.randn(seq, kv_heads * (dim + value), device="cuda", generator=g).bfloat16()
    rows[pos + M:] *= 1e4
    got = pkg.ops.grouped_attention(q, rows, pos, kv_heads, dim, vdim, scale, chunk, False, 1, splits).double()
    t, s = torch.arange(pos, pos + M, device="cuda")[:, None], torch.arange(seq, device="cuda")[None]
    sees = (s <= t) & (s // chunk == t // chunk) if chunk else s <= t
    parts = rows.double().view(seq, kv_heads, dim + value)
    for h in range(heads):
        part = parts[:, h // 3]
        p = (q[:, h].double() @ part[:, value:].t() * scale).masked_fill(~sees, -1e300).softmax(1)
        want = p @ part[:, :vdim]
        # weights and the result are rounded to 8 significant bits: off by at most 2^-8 of each term and of the sum
        bound = 2.0 ** -8 * (p @ part[:, :vdim].abs() + want.abs()) + 1e-5
        assert ((got[:, h] - want).abs() <= bound).all(), (h, ((got[:, h] - want).abs() / bound).max().item())


# A sink as the models have it, in all the shares there can be (most of them empty) and in one; more than 512 rows of a key head.
@pytest.mark.parametrize("M,pos,chunk,splits", [(700, 5, 0, 1), (200, 0, 0, 64), (641, 64, 192, 5)])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (256, 254)])
def test_attention_over_a_prompt_with_a_sink(pkg, M, pos, chunk, splits, dim, vdim):
    import torch
    heads, kv_heads, seq = 6, 2, pos + M
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    value = (vdim + 7) // 8 * 8
    q = torch.randn(M, heads, dim, device="cuda", generator=g).bfloat16()
    rows = torch.randn(seq, kv_heads * (dim + value), device="cuda", generator=g).bfloat16()
    got = pkg.ops.grouped_attention(q, rows, pos, kv_heads, dim, vdim, 0.09, chunk, True, 1, splits).double()
    t, s = torch.arange(pos, pos + M, device="cuda")[:, None], torch.arange(seq, device="cuda")[None]
    sees = (s <= t) & (s // chunk == t // chunk) if chunk else s <= t
    parts = rows.double().view(seq, kv_heads, dim + value)
    for h in range(heads):
        part = parts[:, h // 3]
        _assert_attended(got[:, h], _weights_of(q[:, h].double() @ part[:, value:].t() * 0.09, sees, True), part[:, :vdim])


@pytest.mark.parametrize("M,pos", [(1100, 0), (515, 333)])
@pytest.mark.parametrize("dim,rot,vdim", [(64, 32, 64), (128, 64, 128), (192, 64, 256)])
def test_formed_attention_over_a_prompt(pkg, M, pos, dim, rot, vdim):
    import torch
    heads, seq = 3, pos + M
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    q = torch.randn(M, heads, dim + rot, device="cuda", generator=g).bfloat16()
    k = torch.randn(seq, heads * dim, device="cuda", generator=g).bfloat16()
    k_rot = torch.randn(seq, rot, device="cuda", generator=g).bfloat16()
    v = torch.randn(heads * vdim, (seq + 63) // 64 * 64, device="cuda", generator=g).bfloat16()
    gates = torch.randn(M, heads, device="cuda", generator=g)
    got = pkg.ops.formed_attention(q, k, k_rot, v, gates, pos, vdim, 0.07).double().view(M, heads, vdim)
    sees = torch.arange(seq, device="cuda")[None] <= torch.arange(pos, seq, device="cuda")[:, None]
    for h in range(heads):
        keys = torch.cat([k[:, h * dim:(h + 1) * dim], k_rot], 1).double()
        p = _weights_of(q[:, h].double() @ keys.t() * 0.07, sees, False)
        _assert_attended(got[:, h], p, v[h * vdim:(h + 1) * vdim, :seq].double().t(), gates[:, h:h + 1].double().sigmoid())


def _weights_of(scores, sees, sink):
    """Softmax over the keys that are seen, in 64 bits; a score that is no number takes its key away."""
    import torch
    s = torch.where(sees & ~scores.isnan(), scores, -float("inf"))
    if sink:
        s = torch.cat([s, torch.zeros_like(s[:, :1])], 1)
    return s.softmax(1)[:, :sees.shape[1]]


def _assert_attended(got, p, v, gate=1.0):
    want = p @ v * gate
    bad = want.isnan()
    assert (got.isnan() == bad).all()
    bound = 2.0 ** -8 * ((p @ v.abs()) * gate + want.abs()) + 1e-5
    assert ((got - want).abs() <= bound)[~bad].all(), ((got - want).abs() / bound)[~bad].max().item()


# Keys that give no number, minus infinity and, late in the sequence, infinity, as the first key of all and among others; by the kernel
# of short prompts (150 tokens of three heads on one) and that of long ones.
@pytest.mark.parametrize("M,splits", [(150, 1), (700, 1), (700, 3)])
@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("scale", [0.09, 0.0])
@pytest.mark.parametrize("sink", [False, True])
def test_keys_without_a_score(pkg, M, splits, dim, scale, sink):
    import torch
    heads, kv_heads = 6, 2
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    q = torch.randn(M, heads, dim, device="cuda", generator=g).bfloat16()
    q[..., 11] = q[..., 11].abs() + 0.5
    rows = torch.randn(M, kv_heads * 2 * dim, device="cuda", generator=g).bfloat16()
    rows[0, dim + 5] = rows[77, dim] = rows[64, 3 * dim + 9] = float("nan")
    rows[40, dim + 11] = rows[130, 3 * dim + 11] = -float("inf")
    rows[M - 40, dim + 11] = float("inf")
    got = pkg.ops.grouped_attention(q, rows, 0, kv_heads, dim, dim, scale, 0, sink, 1, splits).double()
    sees = torch.ones(M, M, dtype=torch.bool, device="cuda").tril()
    parts = rows.double().view(M, kv_heads, 2 * dim)
    for h in range(heads):
        part = parts[:, h // 3]
        scores = (q[:, h, None].double() * part[None, :, dim:]).sum(2) * scale
        _assert_attended(got[:, h], _weights_of(scores, sees, sink), part[:, :dim])


@pytest.mark.parametrize("dim,rot,vdim", [(64, 32, 64), (128, 64, 128), (256, 64, 256)])
@pytest.mark.parametrize("scale", [0.09, 0.0])
def test_formed_keys_without_a_score(pkg, dim, rot, vdim, scale):
    import torch
    M, heads = 300, 3
    g = torch.Generator(device="cuda").manual_seed(dim)
    q = torch.randn(M, heads, dim + rot, device="cuda", generator=g).bfloat16()
    q[..., 11] = q[..., 11].abs() + 0.5
    k = torch.randn(M, heads * dim, device="cuda", generator=g).bfloat16()
    k_rot = torch.randn(M, rot, device="cuda", generator=g).bfloat16()
    v = torch.randn(heads * vdim, (M + 63) // 64 * 64, device="cuda", generator=g).bfloat16()
    gates = torch.randn(M, heads, device="cuda", generator=g)
    k[0, 5] = k[77, 2 * dim + 1] = k_rot[64, 2] = float("nan")
    k[40, 11] = -float("inf")
    k[M - 40, dim + 11] = float("inf")
    got = pkg.ops.formed_attention(q, k, k_rot, v, gates, 0, vdim, scale).double().view(M, heads, vdim)
    sees = torch.ones(M, M, dtype=torch.bool, device="cuda").tril()
    for h in range(heads):
        keys = torch.cat([k[:, h * dim:(h + 1) * dim], k_rot], 1).double()
        scores = (q[:, h, None].double() * keys[None]).sum(2) * scale
        p = _weights_of(scores, sees, False)
        _assert_attended(got[:, h], p, v[h * vdim:(h + 1) * vdim, :M].double().t(), gates[:, h:h + 1].double().sigmoid())


def test_logits_that_do_not_fit_the_staging(pkg):
    """Nine rows of 32768 logits are copied, eight and fewer go out through pinned memory."""
    cfg = tx.config(32768, 64, 1, [tx.layer(tx.mixer(2, 8, 8, 8, 16, 24, 0.3), tx.dense(64))])
    ids = np.arange(5, 35, dtype=np.int32)
    model = pkg.Model.random(cfg, 64, "bfloat16", seed=3)
    nine = model.forward(ids, range(3, 30, 3))
    model.reset()
    eight = model.forward(ids, range(3, 27, 3))
    model.reset()
    assert nine.shape == (9, 32768) and np.array_equal(nine[:8], eight) and np.array_equal(nine[8], model.forward(ids[:28])[0])


# a residual row in two float4s a thread at most, in three or four, and past what a thread holds
@pytest.mark.parametrize("width", [2048, 2052, 4096, 4100])
def test_one_token_rows(pkg, width):
    cfg = tx.config(50, width, 1, [tx.layer(tx.mixer(1, 8, 8, 8, 16, 24, 0.4), tx.dense(40)),
                                   tx.layer(tx.mixer(1, 8, 8, 8, 16, 24, 0.4, kv_from=0), tx.moe(2, 1, 16, shared=24))])
    model = pkg.Model.random(cfg, 8, "float32", seed=3)
    got = [model.forward([t]) for t in (7, 7, 49, 3)]
    model.reset()
    model.set_option("unfused", 1)
    for i, t in enumerate((7, 7, 49, 3)):   # the same sums in 32 bits in another order, two layers deep
        want = model.forward([t])
        assert np.linalg.norm(got[i] - want) <= 3e-5 * np.linalg.norm(want), i


# Ragged rows and columns over K on both sides of the lines between 64 x 64 and larger tiles: 128 x 256 from two steps on (2045 rows); 64 x 64 with
# two stages, four and 64 x 128 (1000); 64 x 64 with two stages for all of them (300, and all in float)
@pytest.mark.parametrize("K", [64, 128, 192, 256, 448])
@pytest.mark.parametrize("M,N", [(2045, 3100), (300, 12280), (1000, 2000)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_one_round_of_tiles(pkg, M, N, K, dtype):
    import torch
    g = torch.Generator(device="cuda").manual_seed(K)
    bf16 = dtype == "bfloat16"
    K = K if bf16 else K // 2
    a = torch.randn(M, K, device="cuda", generator=g).to(getattr(torch, dtype))
    w = torch.randn(N, K, device="cuda", generator=g).to(getattr(torch, dtype))
    got = pkg.ops.dense_gemm(a, w, K)
    # K products (exact in bfloat16) and K sums, rounded to 24 bits
    bound = (1 if bf16 else 2) * K * 2.0 ** -24 * 4 * K ** 0.5
    assert (got.double() - a.double() @ w.double().t()).abs().max().item() <= bound
    assert torch.equal(pkg.ops.dense_gemm(a[M - 33:], w, K), got[M - 33:])


# 256 x 256 tiles, whose rings of A and W have two and three stages: fewer steps than stages of W, as many, more (one step goes by 64 x 64 tiles);
# rows of C that take four columns at a time and rows that do not.
@pytest.mark.parametrize("N", [4096, 4094, 4093])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 9])
def test_rings_of_two_lengths(pkg, N, steps):
    import torch
    g, K, M = torch.Generator(device="cuda").manual_seed(steps), 64 * steps, 4090
    assert form_of(pkg, M, N, K) == FORMS[0 if steps > 1 else 5]
    a = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    got = pkg.ops.dense_gemm(a, w, K)
    # K products, exact, and K sums, rounded to 24 bits
    assert (got.double() - a.double() @ w.double().t()).abs().max().item() <= K * 2.0 ** -24 * 4 * K ** 0.5
    assert torch.equal(pkg.ops.dense_gemm(a[M - 33:], w, K), got[M - 33:])


# The tile that the estimate of times takes, in each of its forms, the one in bfloat16 beside the sizes: as few steps as lead to it and one more, ragged
# rows and columns; of 128 x 128 tiles as many steps as they have stages.  In float 64 x 64 with two stages, and with four.
@pytest.mark.parametrize("M,N,steps,form", [
    (4090, 4093, 2, 0), (4090, 4093, 3, 0), (4090, 4093, 4, 0), (2045, 8000, 3, 0), (1921, 4093, 1, 1), (1921, 4093, 2, 1), (2045, 4093, 3, 1), (3000, 6136, 8, 1),
    (1000, 3100, 4, 2), (1000, 3100, 5, 2), (1000, 3100, 8, 2), (1025, 3100, 9, 2), (500, 4093, 5, 3), (500, 4093, 6, 3), (65, 12280, 5, 3), (65, 6136, 3, 4),
    (65, 6136, 4, 4), (500, 4093, 4, 4), (300, 12280, 2, 5), (129, 6136, 3, 5), (65, 6136, 1, 5), (129, 12280, 1, 5), (1025, 1990, 2, 5), (65, 6136, 8, 4),
    (65, 6136, 12, 4)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_each_form_of_tile(pkg, M, N, steps, form, dtype):
    import torch
    bf16 = dtype == "bfloat16"
    K = steps * (64 if bf16 else 32)
    assert form_of(pkg, M, N, K, dtype) == FORMS[form if bf16 else 4 if steps >= 8 and M == 65 else 5]
    g = torch.Generator(device="cuda").manual_seed(M + steps)
    a = torch.randn(M, K, device="cuda", generator=g).to(getattr(torch, dtype))
    w = torch.randn(N, K, device="cuda", generator=g).to(getattr(torch, dtype))
    got = pkg.ops.dense_gemm(a, w, K)
    # K products (exact in bfloat16) and K sums, rounded to 24 bits
    bound = (1 if bf16 else 2) * K * 2.0 ** -24 * 4 * K ** 0.5
    assert (got.double() - a.double() @ w.double().t()).abs().max().item() <= bound
    assert torch.equal(pkg.ops.dense_gemm(a[M - 33:], w, K), got[M - 33:])


# Rows so far apart that a tile's reach past 4 GB: of A, of W, of W with gated units.
@pytest.mark.parametrize("dtype,M,N,lda,ldw", [("float32", 65, 6136, 17_100_000, 64), ("bfloat16", 130, 300, 128, 8_400_000),
                                               ("bfloat16", 257, 288, 8_388_608, 64)])
def test_rows_far_apart(pkg, dtype, M, N, lda, ldw):
    import torch
    bf16 = dtype == "bfloat16"
    K, g = 64, torch.Generator(device="cuda").manual_seed(M)
    assert pkg.capi.dense().a81w41_dense_form_selfcheck(M, N, K, lda, ldw, bf16) == 7
    near = [torch.randn(n, K, device="cuda", generator=g).to(getattr(torch, dtype)) for n in (M, N)]
    a, w = far = [torch.empty(n, ld, device="cuda", dtype=near[0].dtype) for n, ld in ((M, lda), (N, ldw))]
    for x, y in zip(far, near):
        x[:, :K] = y
    got = pkg.ops.dense_gemm(a, w, K)
    # K products (exact in bfloat16) and K sums, rounded to 24 bits
    assert (got.double() - near[0].double() @ near[1].double().t()).abs().max().item() <= 2 * K * 2.0 ** -24 * 4 * K ** 0.5
    assert torch.equal(pkg.ops.dense_gemm(near[0], near[1], K), got)
    if N % 32 == 0:
        assert torch.equal(pkg.ops.dense_gated(near[0], near[1], K), pkg.ops.dense_gated(a, w, K))


# Step by step of K: the same bits for a row in a call of 33 rows, which goes through another kernel.  128 x 256 tiles and 64 x 64 with two stages and
# four; in float 64 x 64 with two.
@pytest.mark.parametrize("M,N,dtype,steps", [(2045, 3100, "bfloat16", (10, 11, 12, 13)), (2045, 3100, "float32", (5, 6, 7)),
                                             (1000, 2000, "bfloat16", (2, 3, 4)), (1000, 2000, "float32", (2, 3))])
def test_one_round_from_some_steps_on(pkg, M, N, dtype, steps):
    import torch
    bf16 = dtype == "bfloat16"
    for n in steps:
        g, K = torch.Generator(device="cuda").manual_seed(n), n * (64 if bf16 else 32)
        a = torch.randn(M, K, device="cuda", generator=g).to(getattr(torch, dtype))
        w = torch.randn(N, K, device="cuda", generator=g).to(getattr(torch, dtype))
        got = pkg.ops.dense_gemm(a, w, K)
        # K products (exact in bfloat16) and K sums, rounded to 24 bits
        bound = (1 if bf16 else 2) * K * 2.0 ** -24 * 4 * K ** 0.5
        assert (got.double() - a.double() @ w.double().t()).abs().max().item() <= bound, n
        assert torch.equal(pkg.ops.dense_gemm(a[M - 33:], w, K), got[M - 33:]), n


# 128 x 256 tiles over eleven steps, with the epilogues of a prompt: queries turned and stored, gated units, columns of
# heads with what is no head's behind them; the same rows in portions go through small tiles.
def test_epilogues_on_one_round_of_tiles(pkg):
    assert form_of(pkg, 2045, 3072, 704) == form_of(pkg, 2045, 3104, 704) == FORMS[1]
    _same_in_portions(pkg, tx.config(64, 704, 1, [tx.layer(tx.mixer(16, 128, 64, 8, 704, 24, 0.1), tx.dense(1552))]), 2045, 100)
    _same_in_portions(pkg, dx.config(64, 704, [dx.attention(16, 4, 128, 128, 70, 0.09, rot_dims=64, mlp=None)], (0, 1, 1)), 2045, 100)


# Experts' rows in tiles of 128 (one pass) and of 64 (portions): 128 x 256 and 128 x 128 tiles, 64 x 128 with two and three stages, 64 x 64;
# experts with few rows or none, tables of few ids against many
@pytest.mark.parametrize("n,experts,top,ff,width", [(2100, 8, 2, 600, 1088), (1100, 4, 1, 2048, 64), (700, 5, 3, 96, 2048), (1400, 16, 2, 520, 320)])
def test_experts_in_tiles_of_two_heights(pkg, n, experts, top, ff, width):
    cfg = tx.config(40, width, 1, [tx.layer(tx.mixer(2, 8, 8, 8, 16, 24, 0.3), tx.moe(experts, top, ff, shared=40))])
    _same_in_portions(pkg, cfg, n, 100)


# a gated unit at the limits of its gate: exponentials past the range of a float, in both types
def test_gated_units_of_large_gates(pkg, tmp_path):
    from oracle import takosun_forward as tf
    cfg = tx.config(64, 64, 1, [tx.layer(tx.mixer(2, 8, 8, 8, 16, 24, 0.3), tx.dense(96))])
    w = tf.random_weights(cfg, 12)
    w["l0.mlp.gate"] = tf.round_bf16(w["l0.mlp.gate"] * 150)   # gates of some hundreds, both signs
    tx.write_model(str(tmp_path), cfg, w)
    ids = np.arange(40) % 64
    want = tf.TakosunOracle(cfg, w).forward(ids)
    for dtype, tol in (("float32", 3e-5), ("bfloat16", 0.06)):
        got = pkg.Model.load(str(tmp_path), 64, dtype).forward(ids, range(40))
        err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() <= tol, (dtype, err.max())


# queries turned and stored by the product: heads of an odd and of an even width, on 256 x 256 tiles and on small ones
@pytest.mark.parametrize("heads,dim,rot,rank,form", [(41, 95, 62, 70, 0), (40, 96, 64, 70, 5), (9, 33, 2, 70, 5), (41, 95, 62, 200, 0), (40, 96, 64, 200, 0),
                                                     (9, 33, 2, 200, 4)])
def test_query_columns_on_large_tiles(pkg, heads, dim, rot, rank, form):
    assert form_of(pkg, 2100, heads * (dim + rot), rank) == FORMS[form]
    cfg = tx.config(64, 64, 1, [tx.layer(tx.mixer(heads, dim, rot, 8, rank, 24, 0.1), None)])
    _same_in_portions(pkg, cfg, 2100, 100)


# The unit is formed in 32 bits ahead of its rounding to bfloat16: only a unit that lies within the error of that arithmetic of the middle
# between two bfloat16 may be rounded the other way.  A product of three columns by ones puts any float of 24 bits together, exactly.
# Relative errors in 2^-24: the exponential 2 (one unit in the last place) and 2 |slope g| of its rounded argument, one each of the sum,
# the division and, with an up that is no constant, of u + shift and the product.  Gates end where 1.702 g is -85: from -88.7 on the exponential
# is no float and the unit zero.
@pytest.mark.parametrize("limit,slope,shift", [(float("inf"), 1.0, 0.0), (7.0, 1.702, 1.0)])
@pytest.mark.parametrize("low,high", [(-4.0, 4.0), (-20.0, -4.0), (-50.0, -20.0)])
@pytest.mark.parametrize("M", [320, 40])
def test_gated_units_are_formed_in_32_bits(pkg, limit, slope, shift, low, high, M):
    import torch
    units, groups = 2048, 64
    g = torch.Generator(device="cuda").manual_seed(M)
    gate = torch.rand(groups, units, device="cuda", generator=g) * (high - low) + low
    up = torch.rand(groups, units, device="cuda", generator=g) * 2 - 1 if shift else torch.ones(groups, units, device="cuda")

    def columns(x):   # [groups][units] floats -> [units][3 groups], whose sums over a group's three columns are x
        parts, rest = [], x
        for _ in range(3):
            parts.append(rest.bfloat16())
            rest = rest - parts[-1].float()
        assert not rest.any()
        return torch.stack(parts, 1).permute(2, 0, 1).reshape(units, 3 * groups)

    w = torch.stack([columns(gate).view(units // 16, 16, -1), columns(up).view(units // 16, 16, -1)], 1).reshape(2 * units, -1).contiguous()
    rows = torch.arange(M, device="cuda") % groups
    a = torch.zeros(M, groups, 3, device="cuda", dtype=torch.bfloat16)
    a[torch.arange(M, device="cuda"), rows] = 1
    got = pkg.ops.dense_gated(a.view(M, -1), w, 3 * groups, limit, slope, shift)
    x, u = gate.double().clamp(max=limit), up.double().clamp(-limit, limit)
    want = (x / (1 + (-float(np.float32(slope)) * x).exp()) * (u + shift))[rows]
    units_off = 4 + 2 + (2 * slope * x[rows].abs() if slope != 1 else 0)
    near = (want.abs() * 2.0 ** -24 * units_off + 2.0 ** -149)
    ok = (got == (want - near).bfloat16()) | (got == (want + near).bfloat16())
    assert ok.all(), ((~ok).sum().item(), gate[rows][~ok][:4].tolist(), got[~ok][:4].tolist(), want[~ok][:4].tolist())
