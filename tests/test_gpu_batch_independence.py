"""Batch independence at turbo widths (the batch API, src/transcribe.rs:104-167).

Every kernel on the path computes a clip (encoder, cross keys / values, timestamps) or a decoder row on its own, and
accumulates in an order that does not depend on the clips beside it (the products sum K in the same 64-wide steps
whatever tile shape the batch size selects). So a clip's language, tokens and token timestamps are the same bits
whether it is transcribed alone or in a batch: a property that holds at any batch size, checked here on six clips
(two encoder groups on two lanes) against three of them alone (one group, smaller product tiles), in both timestamp
modes, for graph replay against eager steps, and for encoder groups of 2 and of 6 against groups of 4. Turbo widths (d 1280, 20 heads, 4 decoder layers, 128 mels, the
51866-token vocabulary) with 2 encoder layers; random weights with non-zero biases and LayerNorm parameters.
"""
import numpy as np
import pytest

from mimizuku_amd import model, synth, transcribe

pytestmark = pytest.mark.gpu

G = synth.Geometry(d=1280, ff=5120, nh=20, enc_layers=2, dec_layers=4, n_mels=128, vocab=51866)
N, EG, MAX_NEW = 6, 4, 24


@pytest.fixture(scope="module")
def parts():
    W = synth.random_weights(G, seed=3, bias_std=0.02, ln_std=0.05)
    heads = synth.generation_config(synth.LARGE_V3_TURBO)["alignment_heads"]
    gen = synth.generation_config(G, align_heads=heads)
    dims = model.Dims(G.d, G.ff, G.nh, G.enc_layers, G.dec_layers, G.n_mels, G.vocab, G.max_t)
    gc = model.GenCfg.from_dict(gen, dims)
    ctx = model.Context(0)

    def engine(eg: int) -> model.Engine:
        e = model.Engine(ctx, dims, gc, N, eg)
        e.load(W)
        return e
    mel = synth.synthetic_mel(N, G.n_mels, seed=5)
    prompt = transcribe.Prompt(gc, "auto", "transcribe")
    yield engine, mel, prompt


@pytest.fixture(scope="module")
def setup(parts):
    engine, mel, prompt = parts
    e = engine(EG)
    yield e, mel, prompt
    e.close()


def same(a: transcribe.Decoded, b: transcribe.Decoded, what: str):
    assert a.lang == b.lang, what
    assert a.seq == b.seq, what
    np.testing.assert_array_equal(np.array(a.ts, np.float32), np.array(b.ts, np.float32), err_msg=what)


@pytest.mark.parametrize("half", [True, False])
def test_clip_alone_equals_clip_in_batch(setup, half):
    e, mel, prompt = setup
    batch, tm = transcribe.transcribe(e, mel, prompt, max_new=MAX_NEW, half_align=half)
    assert tm.steps > MAX_NEW // 2
    for c in (0, 3, 5):
        alone, _ = transcribe.transcribe(e, mel[c:c + 1], prompt, max_new=MAX_NEW, half_align=half)
        same(alone[0], batch[c], f"clip {c} half {half}")


def test_graph_replay_equals_eager_steps(setup):
    e, mel, prompt = setup
    graph, _ = transcribe.transcribe(e, mel, prompt, max_new=MAX_NEW, graph=True)
    eager, _ = transcribe.transcribe(e, mel, prompt, max_new=MAX_NEW, graph=False)
    for c in range(N):
        same(graph[c], eager[c], f"clip {c}")


def test_encoder_group_size_does_not_change_results(setup, parts):
    """The six clips encoded in groups of 2 (three groups over the two lanes) and in one group of 6 (one lane, larger
    products) give the same bits as in groups of 4."""
    e, mel, prompt = setup
    engine = parts[0]
    ref, _ = transcribe.transcribe(e, mel, prompt, max_new=MAX_NEW)
    for eg in (2, N):
        other = engine(eg)
        try:
            got, _ = transcribe.transcribe(other, mel, prompt, max_new=MAX_NEW)
        finally:
            other.close()
        for c in range(N):
            same(got[c], ref[c], f"clip {c}, groups of {eg}")


@pytest.mark.parametrize("d,clips", [(384, 5), (384, 8), (640, 3), (640, 6)])
def test_encoder_of_odd_widths_in_one_group(d, clips):
    """Widths whose QKV product ends in a partial column tile: a group of clips encodes to the bits of each clip alone."""
    g = synth.Geometry(d=d, ff=4 * d, nh=d // 64, enc_layers=1, dec_layers=1, n_mels=80, vocab=51865, max_t=16)
    dims = model.Dims(g.d, g.ff, g.nh, g.enc_layers, g.dec_layers, g.n_mels, g.vocab, g.max_t)
    gc = model.GenCfg(sot=3, eos=2, no_timestamps=6, langs=[("en", 4)], tasks=[("transcribe", 5)], suppress=[],
                      begin_suppress=[], align_heads=[(0, 1)])
    ctx = model.Context(0)
    e = model.Engine(ctx, dims, gc, clips, clips)
    e.load(synth.random_weights(g, seed=d, bias_std=0.02, ln_std=0.05))
    mel = synth.synthetic_mel(clips, g.n_mels, seed=4)
    e.encode(mel, 0)
    group = e.enc_out(clips).copy(), e.xkv()
    assert np.isfinite(group[0]).all()
    for c in range(clips):
        e.encode(mel[c:c + 1], c)
        np.testing.assert_array_equal(e.enc_out(1)[0], group[0][c], err_msg=f"clip {c}")
    np.testing.assert_array_equal(e.xkv(), group[1])
    e.close()
    ctx.close()


@pytest.mark.parametrize("d,nh,rows", [(128, 2, (33, 32, 5)), (128, 2, (13, 12, 5)), (384, 6, (11, 10, 1)), (1024, 16, (5, 4, 3))])
def test_decoder_rows_alone_and_split(d, nh, rows):
    """Batches on both sides of the borders at which a row's cross-attention goes over four workgroups (64 (row, head)
    pairs, 12 rows):
    the same logits, residual and alignment rows (fp32 and fp16) bit for bit, for the rows they share, over a prompt and
    some generated positions."""
    from mimizuku_amd import _lib as L
    g = synth.Geometry(d=d, ff=4 * d, nh=nh, enc_layers=1, dec_layers=2, n_mels=80, vocab=51865, max_t=32)
    W = synth.random_weights(g, seed=nh, bias_std=0.02, ln_std=0.05)
    heads = [[0, 1], [1, 0], [1, nh - 1]]
    dims = model.Dims(g.d, g.ff, g.nh, g.enc_layers, g.dec_layers, g.n_mels, g.vocab, g.max_t)
    gc = model.GenCfg.from_dict(synth.generation_config(g, align_heads=heads), dims)
    ctx = model.Context(0)
    e = model.Engine(ctx, dims, gc, max(rows), 1)
    e.load(W)
    mel = synth.synthetic_mel(max(rows), g.n_mels, seed=2)
    for c in range(max(rows)):
        e.encode(mel[c:c + 1], c)
    steps, out = 9, []
    for b in rows:
        e.reset([[gc.sot, 50259 + i % 8, 50359, gc.no_timestamps] for i in range(b)])
        for p in range(steps):
            e.step(b, False, 4)
        out.append((e.logits()[:b], e.dec_x()[:b], e.align()[:b, :steps], e.tokens()[:b, :steps + 1],
                    e.read(L.BUF_ALIGN_H, np.float16, (max(rows), g.max_t, 3, 1500))[:b, :steps]))
    assert np.isfinite(out[0][0]).all()
    np.testing.assert_allclose(out[0][2].sum(-1), 1.0, atol=1e-4)
    for o in out:
        np.testing.assert_array_equal(o[4], o[2].astype(np.float16))
    for b, o in zip(rows[1:], out[1:]):
        k = min(b, rows[0])
        for x, y in zip(o, out[0]):
            np.testing.assert_array_equal(x[:k], y[:k], err_msg=f"{b} rows against {rows[0]}")
    e.close()
    ctx.close()


@pytest.mark.parametrize("d,nh,rows", [(128, 2, (12, 13)), (384, 6, (10, 11)), (1280, 20, (3, 4))])
def test_finished_rows_alone_and_split(d, nh, rows):
    """Rows that are finished, one before an engine's first step and one between steps, on both sides of that border: every
    value stays finite and the rows that both batches have, the finished ones among them, are the same bits."""
    from mimizuku_amd import _lib as L
    g = synth.Geometry(d=d, ff=4 * d, nh=nh, enc_layers=1, dec_layers=2, n_mels=80, vocab=51865, max_t=32)
    W = synth.random_weights(g, seed=nh, bias_std=0.02, ln_std=0.05)
    dims = model.Dims(g.d, g.ff, g.nh, g.enc_layers, g.dec_layers, g.n_mels, g.vocab, g.max_t)
    gc = model.GenCfg.from_dict(synth.generation_config(g, align_heads=[[0, 1], [1, 0], [1, nh - 1]]), dims)
    mel = synth.synthetic_mel(1, g.n_mels, seed=2)
    ctx, out = model.Context(0), []
    for b in rows:
        e = model.Engine(ctx, dims, gc, b, 1)
        e.load(W)
        for c in range(b):
            e.encode(mel, c)
        e.reset([[gc.sot, 50259 + i % 8, 50359, gc.no_timestamps] for i in range(b)])
        for p in range(6):
            for step, row in ((0, 0), (3, 2)):
                if p == step:
                    ctx.upload(e.buffer(L.BUF_DONE)[0] + 4 * row, np.ones(1, np.int32))
            e.step(b, False, 4)
            k = min(rows)
            out.append([a[:k] for a in (e.logits(), e.dec_x(), e.align(), e.tokens(), e.done())])
        e.close()
    ctx.close()
    assert out[5][4][0] == 1 and out[5][4][2] == 1
    for p in range(6):
        for x, y in zip(out[p], out[6 + p]):
            assert np.isfinite(x).all() and np.isfinite(y).all(), f"step {p}"
            np.testing.assert_array_equal(x, y, err_msg=f"step {p}")
