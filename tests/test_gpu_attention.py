"""The attention step on its own (a81w41_qwen3_attention) against a float64 numpy statement of
QK^T * scale, causal mask, softmax, PV with grouped heads (QwenAttention.cc:150-195) over the
same fp16-rounded cache: the vector kernel and the matrix-core kernel, every head grouping the
latter is built for, prompts that start on a cached context, ragged tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-5   # output rows relative to their norm: fp32 products and sums, exp to a few ulp


@pytest.fixture(scope="module")
def torch():
    import torch as t

    assert t.cuda.is_available()
    return t


def reference(q, k, v, pos, n_q, n_kv, scale):
    """q [M][n_q][128] fp32, k / v [n_kv][T][128] (fp16 values) -> [M][n_q*128] float64."""
    M = q.shape[0]
    out = np.zeros((M, n_q, 128))
    grp = n_q // n_kv
    for h in range(n_q):
        s = (q[:, h].astype(np.float64) @ k[h // grp].astype(np.float64).T) * float(scale)     # [M][T]
        for m in range(M):
            row = s[m, :pos + m + 1]
            e = np.exp(row - row.max())
            out[m, h] = (e / e.sum()) @ v[h // grp, :pos + m + 1].astype(np.float64)
    return out.reshape(M, n_q * 128)


def make(synth, M, pos, n_q, n_kv, max_seq, seed):
    q = (synth.standard_normal(M * n_q * 128, seed).reshape(M, n_q, 128) * np.float32(1.5)).astype(np.float32)
    k = synth.standard_normal(n_kv * max_seq * 128, seed + 1).reshape(n_kv, max_seq, 128).astype(np.float16)
    v = synth.standard_normal(n_kv * max_seq * 128, seed + 2).reshape(n_kv, max_seq, 128).astype(np.float16)
    return q, k, v


def run(pkg, torch, q, k, v, pos, n_q, n_kv, scale, variant, row_pad=0):
    M = q.shape[0]
    qd = torch.zeros((M, n_q * 128 + row_pad), dtype=torch.float32, device="cuda")
    qd[:, :n_q * 128] = torch.from_numpy(q.reshape(M, -1)).cuda()
    return pkg.ops.attention(qd, torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), pos, n_q, n_kv, scale,
                             variant).cpu().numpy()


def row_err(got, want):
    return float(np.max(np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)))


@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("M,pos,n_q,n_kv,max_seq", [
    (9, 0, 4, 1, 64),        # one ragged query tile, one key tile
    (32, 0, 2, 1, 64),       # exactly one tile
    (33, 0, 2, 2, 64),       # second query tile with a single token; one head per KV head
    (100, 0, 8, 1, 128),     # eight heads per KV head
    (45, 150, 4, 2, 200),    # prompt chunk on top of 150 cached tokens: ragged last key tile
    (322, 0, 8, 2, 384),     # the benchmark's prompt length
    (64, 31, 4, 4, 96),      # context ends one short of a tile boundary
])
def test_against_float64(pkg, synth, torch, variant, M, pos, n_q, n_kv, max_seq):
    scale = 1.0 / np.sqrt(128.0)
    q, k, v = make(synth, M, pos, n_q, n_kv, max_seq, 700 + M)
    got = run(pkg, torch, q, k, v, pos, n_q, n_kv, scale, variant, row_pad=256)   # rows wider than the heads, like the fused qkv row
    want = reference(q, k.astype(np.float32), v.astype(np.float32), pos, n_q, n_kv, scale)
    assert np.isfinite(got).all()
    assert row_err(got, want) < TOL


@pytest.mark.parametrize("M,pos,n_q,n_kv,max_seq", [(100, 0, 8, 1, 128), (45, 150, 8, 2, 200), (322, 0, 8, 2, 384)])
def test_every_split_of_a_head_group(pkg, synth, torch, M, pos, n_q, n_kv, max_seq):
    """The matrix-core kernel with 1, 2, 4 and 8 query heads of a KV group per workgroup (variants 3..6;
    left alone it picks by the number of query tiles): each against float64, and too many heads refused."""
    scale = 1.0 / np.sqrt(128.0)
    q, k, v = make(synth, M, pos, n_q, n_kv, max_seq, 720 + M)
    want = reference(q, k.astype(np.float32), v.astype(np.float32), pos, n_q, n_kv, scale)
    for variant in (3, 4, 5, 6):
        if (1 << (variant - 3)) > n_q // n_kv:
            with pytest.raises(pkg.capi.A81W41Error):
                run(pkg, torch, q, k, v, pos, n_q, n_kv, scale, variant)
            continue
        got = run(pkg, torch, q, k, v, pos, n_q, n_kv, scale, variant, row_pad=128)
        assert row_err(got, want) < TOL, variant


@pytest.mark.parametrize("M,pos", [(31, 0), (33, 64), (64, 33), (65, 127), (97, 96)])
@pytest.mark.parametrize("n_q,n_kv", [(8, 1), (2, 2)])
def test_edges_of_tiles_and_rounds(pkg, synth, torch, n_q, n_kv, M, pos):
    """One query more and less than a tile, contexts that end in the middle of a round of the key splits, for every number of
    heads a workgroup takes; keys behind the context hold what no token may see."""
    scale = 1.0 / np.sqrt(128.0)
    q, k, v = make(synth, M, pos, n_q, n_kv, M + pos + 40, 900 + M)
    want = reference(q, k[:, :M + pos].astype(np.float32), v[:, :M + pos].astype(np.float32), pos, n_q, n_kv, scale)
    k[:, M + pos:], v[:, M + pos:] = 60000.0, np.nan
    for variant in (2, 3, 4, 5, 6):
        if variant > 2 and (1 << (variant - 3)) > n_q // n_kv:
            continue
        got = run(pkg, torch, q, k, v, pos, n_q, n_kv, scale, variant, row_pad=4)
        assert row_err(got, want) < TOL, variant


@pytest.mark.parametrize("M", [128, 129, 256, 257])
def test_heads_a_workgroup_of_many_heads(pkg, synth, torch, M):
    """64 heads on 16: what the number of workgroups chooses, one head, two and all four of a group, to the last row that each takes."""
    scale = 1.0 / np.sqrt(128.0)
    q, k, v = make(synth, M, 3, 64, 16, M + 3, 940 + M)
    want = reference(q, k.astype(np.float32), v.astype(np.float32), 3, 64, 16, scale)
    got = run(pkg, torch, q, k, v, 3, 64, 16, scale, 2)
    heads = {128: 1, 129: 2, 256: 2, 257: 4}[M]   # 256 workgroups of one head at 128 tokens, 256 of two at 256
    assert row_err(got, want) < TOL
    assert np.array_equal(got, run(pkg, torch, q, k, v, 3, 64, 16, scale, {1: 3, 2: 4, 4: 5}[heads]))


def test_sharp_and_flat_rows(pkg, synth, torch):
    """Scores far apart (one key dominates) and all equal (uniform weights): the running-maximum
    bookkeeping across tiles and the masked entries of partial tiles."""
    M, n_q, n_kv, max_seq = 70, 4, 1, 96
    q, k, v = make(synth, M, 0, n_q, n_kv, max_seq, 750)
    q[:, 0] *= np.float32(12.0)          # head 0: very peaked
    q[:, 1] = 0.0                        # head 1: all scores 0 -> plain mean of the visible values
    scale = 1.0 / np.sqrt(128.0)
    want = reference(q, k.astype(np.float32), v.astype(np.float32), 0, n_q, n_kv, scale)
    for variant in (1, 2):
        got = run(pkg, torch, q, k, v, 0, n_q, n_kv, scale, variant)
        assert row_err(got, want) < TOL, variant
    mean0 = v[0, :1].astype(np.float64).mean(axis=0)
    assert np.allclose(got[0, 128:256], mean0, rtol=1e-6, atol=1e-7)      # token 0 sees only key 0


def test_default_picks_by_length_and_errors(pkg, synth, torch):
    q, k, v = make(synth, 40, 0, 4, 1, 64, 760)
    scale = 1.0 / np.sqrt(128.0)
    assert np.array_equal(run(pkg, torch, q, k, v, 0, 4, 1, scale, 0), run(pkg, torch, q, k, v, 0, 4, 1, scale, 2))
    assert np.array_equal(run(pkg, torch, q[:5], k, v, 0, 4, 1, scale, 0), run(pkg, torch, q[:5], k, v, 0, 4, 1, scale, 1))
    with pytest.raises(pkg.capi.A81W41Error):
        run(pkg, torch, q[:5], k, v, 0, 4, 1, scale, 2)          # too few tokens for the matrix-core kernel
    with pytest.raises(pkg.capi.A81W41Error):
        run(pkg, torch, q[:, :3], k, v, 0, 3, 2, scale, 0)       # heads not a multiple of KV heads



@pytest.mark.parametrize("pos,n_q,n_kv,splits", [(0, 4, 1, 1), (1, 2, 2, 1), (63, 8, 2, 1), (300, 32, 8, 1), (511, 4, 4, 1),
                                                 (700, 8, 2, 1), (37, 4, 1, 4), (700, 8, 2, 3), (1500, 32, 8, 4),
                                                 (5, 4, 2, 16)])
def test_one_token_step_against_float64(pkg, synth, torch, pos, n_q, n_kv, splits):
    """The decode step's kernel on its own (q/k RMSNorm, RoPE, cache append, attention over pos + 1 keys),
    one workgroup per head and with the key range cut into shares (more shares than keys included),
    against float64 numpy over the same fp16 cache; the appended cache rows must be the fp16 roundings."""
    from oracle import qwen3_forward as qf

    max_seq, eps = pos + 9, 1e-6
    scale = 1.0 / np.sqrt(128.0)
    q, k, v = make(synth, 1, pos, n_q, n_kv, max_seq, 800 + pos)          # cache rows 0 .. pos-1 (row pos is overwritten)
    qkv = synth.standard_normal((n_q + 2 * n_kv) * 128, 801 + pos).astype(np.float32)
    q_w = (1.0 + 0.1 * synth.standard_normal(128, 802)).astype(np.float32)
    k_w = (1.0 + 0.1 * synth.standard_normal(128, 803)).astype(np.float32)
    cos, sin = qf.rope_tables(max_seq, 1e6)
    kd, vd = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda()
    got = pkg.ops.attention_one_token(torch.from_numpy(qkv).cuda(), torch.from_numpy(q_w).cuda(), torch.from_numpy(k_w).cuda(),
                                      torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda(), kd, vd, pos, n_q, n_kv,
                                      eps, scale, splits).cpu().numpy()
    # float64 reference over what the kernel defines: fp32 norm and rotation as the oracle does them, fp16 cache
    qh = qf.rotate_half_apply(qf.rmsnorm(qkv[:n_q * 128].reshape(n_q, 128), q_w, eps), cos[pos], sin[pos])
    kh = qf.rotate_half_apply(qf.rmsnorm(qkv[n_q * 128:(n_q + n_kv) * 128].reshape(n_kv, 128), k_w, eps), cos[pos], sin[pos])
    vh = qkv[(n_q + n_kv) * 128:].reshape(n_kv, 128)
    k_ref, v_ref = k.copy(), v.copy()
    k_ref[:, pos], v_ref[:, pos] = kh.astype(np.float16), vh.astype(np.float16)
    assert np.array_equal(vd.cpu().numpy()[:, pos], v_ref[:, pos])
    k_got = kd.cpu().numpy()[:, pos].astype(np.float32)
    assert np.max(np.abs(k_got - k_ref[:, pos].astype(np.float32))) <= 2e-3 * np.max(np.abs(kh))   # an fp16 ulp where the fp32 norms differ in the last bit
    want = np.zeros((n_q, 128))
    group = n_q // n_kv
    for h in range(n_q):
        K = kd.cpu().numpy()[h // group, :pos + 1].astype(np.float64)       # the rows the kernel itself cached
        V = v_ref[h // group, :pos + 1].astype(np.float64)
        s_ = (qh[h].astype(np.float64) @ K.T) * scale
        p_ = np.exp(s_ - s_.max())
        want[h] = (p_ / p_.sum()) @ V
    err = np.max(np.linalg.norm(got.reshape(n_q, 128) - want, axis=1) / np.linalg.norm(want, axis=1))
    assert np.isfinite(got).all() and err < TOL, err

