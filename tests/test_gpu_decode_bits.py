"""Orders of sums in the decoder step that are fixed bit for bit, against the same sums taken one fp32 operation at a
time in numpy.

The engines here have one decoder layer whose weights are zero but for what a test reads through: an identity
out-projection puts an attention's fp16 output into the residual.
"""
import numpy as np
import pytest

from mimizuku_amd import _lib as L
from mimizuku_amd import model, synth

pytestmark = pytest.mark.gpu

f32 = np.float32
DEC = "model.decoder.layers.0."


@pytest.fixture(scope="module")
def ctx():
    c = model.Context(0)
    yield c
    c.close()


def engine(ctx, d, rows, weights, vocab=1536, max_t=448):
    g = synth.Geometry(d=d, ff=4 * d, nh=d // 64, enc_layers=1, dec_layers=1, n_mels=80, vocab=vocab, max_t=max_t)
    dims = model.Dims(g.d, g.ff, g.nh, 1, 1, g.n_mels, g.vocab, g.max_t)
    gc = model.GenCfg(sot=3, eos=2, no_timestamps=6, langs=[("en", 4)], tasks=[("transcribe", 5)], suppress=[],
                      begin_suppress=[], align_heads=[(0, 1)])
    e = model.Engine(ctx, dims, gc, rows, 1)
    W = {k: np.zeros(s, np.float16) for k, s in synth.tensor_shapes(g).items()}
    for k in W:
        if k.endswith("layer_norm.weight"):
            W[k][:] = 1.0
    W.update(weights)
    e.load(W)
    return e


# ---------------------------------------------------------------- attention: the merge of the key groups

def values(rng, n):
    """[n][64] fp16 values over many binades whose sum cancels to a few units: what is left shows every rounding of the
    sums that lead there."""
    r = rng.standard_normal((n // 2 - 1, 64)) * 2.0 ** rng.integers(-12, 14, (n // 2 - 1, 64))
    r = np.clip(r, -60000, 60000).astype(np.float16)
    v = np.concatenate([r, -r, rng.standard_normal((n - 2 * len(r), 64)).astype(np.float16)])
    return v[rng.permutation(n)]


def group_sums(v):
    """The 32 groups' sums of the values (group g: keys g, g + 32, ... in order), every weight being exp2(0) = 1."""
    acc = np.zeros((32, 64), f32)
    for j in range(len(v)):
        acc[j % 32] += v[j].astype(f32)
    return acc


def chain(a):
    t = np.zeros(a.shape[1:], f32)
    for x in a:
        t = t + x
    return t


def merged(v):
    """One query's attention output where every score is equal: the groups' sums added one after the other."""
    return (chain(group_sums(v)) / f32(len(v))).astype(np.float16)


def merged_by_waves(v):
    """Another order, eight groups at a time: the values above are drawn so that it shows."""
    return (chain(np.stack([chain(a) for a in group_sums(v).reshape(4, 8, 64)])) / f32(len(v))).astype(np.float16)


@pytest.mark.parametrize("rows", [1, 12, 32, 40, 130])
def test_cross_attention_merges_groups_in_order(ctx, rows):
    """The forms of the cross-attention (four workgroups per (row, head) up to 12 rows, one per CU up to 256, the
    general kernel above) give the 32 groups' states merged one after the other."""
    rng = np.random.default_rng(rows)
    e = engine(ctx, 128, rows, {DEC + "encoder_attn.out_proj.weight": np.eye(128, dtype=np.float16)})
    base, nbytes = e.buffer(L.BUF_XKV)
    assert nbytes == rows * 2 * 2 * 1536 * 64 * 2
    want, other = {}, {}
    for b in sorted({0, rows // 2, rows - 1}):
        v = np.zeros((2, 1536, 64), np.float16)
        for h in range(2):
            v[h, :1500] = values(rng, 1500)
        ctx.upload(base + (2 * b + 1) * v.nbytes, v)  # [row][k | v][head]
        want[b] = np.concatenate([merged(v[h, :1500]) for h in range(2)])
        other[b] = np.concatenate([merged_by_waves(v[h, :1500]) for h in range(2)])
    e.reset([[3, 4, 5, 6]] * rows)
    e.step(rows, False, 4)
    x = e.dec_x()
    for b in want:
        np.testing.assert_array_equal(x[b], want[b].astype(f32), err_msg=f"row {b}")
        assert (want[b] != other[b]).mean() > 0.5
    e.close()


def test_self_attention_merges_groups_in_order(ctx):
    """The same for the self-attention over caches of fewer keys than groups, of some keys per group, and of more than
    one batch of keys; the step's own value is zero."""
    rng = np.random.default_rng(9)
    e = engine(ctx, 128, 2, {DEC + "self_attn.out_proj.weight": np.eye(128, dtype=np.float16)})
    base, nbytes = e.buffer(L.BUF_SELF_V)
    assert nbytes == 2 * 2 * 448 * 64 * 2
    e.reset([[3, 4, 5, 6]] * 2)
    done = 0
    for pos in (20, 100, 300):
        while done < pos:
            e.step(2, False, 4)
            done += 1
        v = np.zeros((2, 2, 448, 64), np.float16)
        for b in range(2):
            for h in range(2):
                v[b, h, :pos] = values(rng, pos)
        ctx.upload(base, v)
        e.step(2, False, 4)
        done += 1
        x = e.dec_x()
        for b in range(2):
            want = np.concatenate([merged(v[b, h, :pos + 1]) for h in range(2)])
            np.testing.assert_array_equal(x[b], want.astype(f32), err_msg=f"position {pos}, row {b}")
            if pos > 32:
                other = np.concatenate([merged_by_waves(v[b, h, :pos + 1]) for h in range(2)])
                assert (want != other).mean() > 0.3
    e.close()


# ---------------------------------------------------------------- layer norms: one row, whichever kernel takes it

@pytest.mark.parametrize("d", [384, 512, 768, 1024])
def test_layer_norms_of_one_row_agree(ctx, d):
    """The first layer norm of a step (in the embedding's kernel, one workgroup per row) and the last one (after the
    residual add, one wave per row at these widths) of the same row with the same weights are the same bits: the first
    comes back through an identity k_proj as the position's key, the last through the identity part of the tied embedding
    as logits. The weights cancel most of each result, so that fp16 shows the statistics' last places."""
    rng = np.random.default_rng(d)
    emb = np.zeros((1536, d), np.float16)
    emb[:d] = np.eye(d)
    rows = emb[d:d + 32]  # alike to 2^-10, so that one set of weights cancels all of them
    rows[:] = (rng.standard_normal(d) * 1.5 + 0.3 + rng.standard_normal((32, d)) * 2.0 ** -10).astype(np.float16)
    gamma = np.full(d, 4096.0, np.float16)
    x = rows[0].astype(np.float64)
    beta = (-4096.0 * (x - x.mean()) / np.sqrt(x.var() + 1e-5)).astype(np.float16)
    ln = {DEC + "self_attn_layer_norm.", "model.decoder.layer_norm."}
    w = {p + "weight": gamma for p in ln} | {p + "bias": beta for p in ln}
    w |= {DEC + "self_attn.k_proj.weight": np.eye(d, dtype=np.float16), "model.decoder.embed_tokens.weight": emb}
    e = engine(ctx, d, 32, w, max_t=16)
    e.reset([[d + b, d] for b in range(32)])
    e.step(32, False, 2)
    np.testing.assert_array_equal(e.dec_x(), rows.astype(f32))
    keys = e.self_kv()[0][0, :, :, 0].reshape(32, d)
    got = e.logits()[:, :d]
    assert np.abs(got).max() <= 64 and np.ptp(got[0]) > 1
    np.testing.assert_array_equal(got, keys.astype(f32))
    e.close()
