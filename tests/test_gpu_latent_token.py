"""One token's latent attention with its value product in one launch: edges of its tiles, the line to the longer form, stale rows."""
import numpy as np
import pytest

from oracle import takosun_forward as tf
from tests.takosun_fixture import config, dense, layer, mixer, write_model

pytestmark = pytest.mark.gpu
TOL = 0.06  # of logits in bfloat16 against the fp32 oracle, as for the other forms of this attention
# a latent of one chunk and of all 64 lanes' chunks, rotated parts with a partial chunk, value rows that end inside a workgroup's 32
SIZES = {"least": (1, 8, 2, 1, 8), "partial": (3, 24, 10, 33, 56), "full": (5, 32, 64, 96, 512)}


def _model(pkg, tmp_path, name, vocab=67, nan_row=None):
    heads, dim, rot, vdim, rank = SIZES[name]
    cfg = config(vocab, 64, 2, [layer(mixer(heads, dim, rot, vdim, 48, rank, dim ** -0.5), None),
                                layer(mixer(heads, dim, rot, vdim, 48, rank, dim ** -0.5, kv_from=0), dense(40))])
    w = tf.random_weights(cfg, 41)
    oracle = tf.TakosunOracle(cfg, w)
    if nan_row is not None:
        w = dict(w, embed=w["embed"].copy())
        w["embed"][nan_row] = np.nan
    write_model(str(tmp_path), cfg, w)
    return pkg.Model.load(str(tmp_path), 640, "bfloat16"), oracle


def _close(got, want, what):
    err = np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)
    assert err.max() <= TOL, (what, int(err.argmax()), float(err.max()))


@pytest.mark.parametrize("name", SIZES)
@pytest.mark.parametrize("start", [0, 6, 125, 509])  # whole passes there and past the last context of this form; each key by itself below
def test_contexts(pkg, tmp_path, name, start):
    model, oracle = _model(pkg, tmp_path, name)
    ids = np.random.default_rng(start).integers(0, 67, start + 6).astype(np.int32)
    want = oracle.forward(ids)[start:]
    if start:
        model.forward(ids[:start])
    _close(np.concatenate([model.forward(ids[i:i + 1]) for i in range(start, start + 6)]), want, (name, start))


def test_rows_behind_the_token_do_not_count(pkg, tmp_path):
    model, oracle = _model(pkg, tmp_path, "partial", nan_row=66)
    ids = np.random.default_rng(3).integers(0, 66, 20).astype(np.int32)
    model.forward(np.full(30, 66, np.int32))  # leaves rows that are no numbers
    model.reset()
    _close(np.concatenate([model.forward(ids[i:i + 1]) for i in range(20)]), oracle.forward(ids), "stale rows")


@pytest.mark.parametrize("q_rank", [4, 30, 2048, 2052])  # held by the threads: least, no whole float4s, most, one more
@pytest.mark.parametrize("heads,rank,rot", [(2, 24, 6), (1, 30, 2)])
def test_latents_held_and_not(pkg, tmp_path, q_rank, heads, rank, rot):
    cfg = config(67, 64, 2, [layer(mixer(heads, 16, rot, 8, q_rank, rank, 0.25), dense(40)) for _ in range(3)])
    w = tf.random_weights(cfg, 43)
    write_model(str(tmp_path), cfg, w)
    model, oracle = pkg.Model.load(str(tmp_path), 64, "bfloat16"), tf.TakosunOracle(cfg, w)
    ids = np.random.default_rng(q_rank).integers(0, 67, 9).astype(np.int32)
    _close(np.concatenate([model.forward(ids[:3])] + [model.forward(ids[i:i + 1]) for i in range(3, 9)]), oracle.forward(ids)[2:], q_rank)


# Every key counts: key j has a latent of one 1 at j % rank, so that each output is a sum over few keys with small whole factors, and weights
# are all alike or powers of two by the rotated part.  The sums are exact in 32 bits; what is not is the scale (log2 e rounded, so weights
# of exponents up to 6 are off by 6 x 2^-23), a division and the gate's sigmoid: 1e-5 holds all of it, and a key left out moves an output by
# more than ten times that.  Tiles of eight keys, sixteen waves of them, the second and later turns of a wave; rows behind the token are
# no numbers.
KEYS = [0, 6, 7, 8, 9, 62, 63, 64, 126, 127, 128, 129, 134, 135, 136, 254, 255, 256, 383, 384, 504, 510, 511, 512, 640]


@pytest.mark.parametrize("rank,rot,vdim", [(8, 2, 8), (24, 64, 40), (56, 10, 33), (512, 64, 512)])
@pytest.mark.parametrize("alike", [True, False])
def test_every_key_counts(pkg, rank, rot, vdim, alike):
    import torch
    heads, seq, scale = 3, 700, float(np.log(2.0))
    ld = (rank + rot + 63) // 64 * 64
    q = torch.zeros(heads, ld, dtype=torch.bfloat16)
    rows = torch.zeros(seq, ld, dtype=torch.bfloat16)
    j = torch.arange(seq)
    rows[j, j % rank] = 1
    if not alike:
        for h in range(heads):   # each head by another column
            q[h, rank + (h + 1) % rot] = 1
            rows[:, rank + (h + 1) % rot] = -((j * (2 * h + 5)) % 7).to(torch.bfloat16)
    uv = torch.zeros(heads, vdim, (rank + 7) // 8 * 8, dtype=torch.bfloat16)
    c = torch.arange(rank)
    for v in range(vdim):
        uv[:, v, :rank] = torch.where(c % vdim == v % rank, 1 + c % 128, 0).to(torch.bfloat16)
    gates = torch.tensor([0.3, -1.2, 2.5])
    for pos in KEYS:
        def attended(left_out=None):
            s = q.double() @ rows[:pos + 1].double().t() * scale
            if left_out is not None:
                s[:, left_out] = -float("inf")
            o = s.softmax(1) @ rows[:pos + 1, :rank].double()
            return (uv[..., :rank].double() @ o[..., None])[..., 0] * gates.double().sigmoid()[:, None]
        cache = rows.clone()
        cache[pos + 1:] = float("nan")
        got = pkg.ops.latent_token(q.cuda(), cache.cuda(), pos, rank, rot, scale, uv.cuda(), gates.cuda()).cpu().double()
        want = attended()
        bound = 1e-5 * want.abs()
        assert ((got - want).abs() <= bound).all(), (pos, ((got - want).abs() - bound).max().item())
        if pos in (6, 8, 128, 512):   # the bound sees each key left out of the oracle
            for left_out in range(pos + 1):
                assert ((attended(left_out) - want).abs() > 10 * bound).any(1).all(), (pos, left_out)
