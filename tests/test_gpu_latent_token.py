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
@pytest.mark.parametrize("start", [0, 6, 125, 509])  # tiles of eight keys, sixteen waves of them, the last context of this form
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
