"""GPU parity of the individual kernels through the C ABI, against float64 closed forms on the same fp16 inputs (or
the oracle's functions), at small shapes and at the full large-v3 shapes with subsampled checks.

Tolerances: an fp16 output is the exact result rounded to fp16 within one ulp (assert_f16); an fp32 output within
max-abs error <= 2e-3 x RMS of the reference; the attention output (whose P operand the kernel rounds to fp16) within
the larger of that and 1.5 x the error of the same attention computed exactly but with fp16 probabilities.
"""
import numpy as np
import pytest

from mimizuku_amd import _lib as L
from mimizuku_amd import model
from oracle import whisper_ref as R

pytestmark = pytest.mark.gpu

TOL = 2e-3
TPAD = 1536


@pytest.fixture(scope="module")
def ctx():
    c = model.Context(0)
    yield c
    c.close()


def rel_err(got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    return np.abs(got - ref).max() / np.sqrt((ref ** 2).mean())


def assert_f16(got, ref, ulps=1.0):
    """An fp16 output must be the exact value rounded to fp16, within `ulps` units in the last place of that value
    (correct rounding is half an ulp; fp32 accumulation order may flip a rounding), plus 1e-5 x RMS for results that
    cancel to near zero."""
    ref = np.asarray(ref, np.float64)
    got = np.asarray(got, np.float64)
    ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64)
    bound = ulps * ulp + 1e-5 * np.sqrt((ref ** 2).mean())
    bad = np.abs(got - ref) > bound
    assert not bad.any(), f"{bad.sum()} of {bad.size} outside {ulps} ulp: worst at {np.argwhere(bad)[:3].tolist()}"


def f16(rng, shape, scale=1.0):
    return (rng.standard_normal(shape, dtype=np.float32) * scale).astype(np.float16)


# ---------------------------------------------------------------- encoder attention

def pack_qkvh(q, k, v):
    """q, k, v [G][nh][1500][64] fp16 -> [G][3][nh][1536 * 64] with v transposed, zero padded."""
    G, nh = q.shape[:2]
    out = np.zeros((G, 3, nh, TPAD * 64), np.float16)
    for a, x in enumerate((q, k)):
        t = np.zeros((G, nh, TPAD, 64), np.float16)
        t[:, :, :1500] = x
        out[:, a] = t.reshape(G, nh, -1)
    t = np.zeros((G, nh, 64, TPAD), np.float16)
    t[:, :, :, :1500] = v.transpose(0, 1, 3, 2)
    out[:, 2] = t.reshape(G, nh, -1)
    return out


QSCALE = 0.125 * np.log2(np.e)  # the QKV product stores q multiplied by the attention's exponent scale


def prescaled(q):
    """(q as the QKV product stores it: fp16(q x log2(e) / 8), the query that stored value stands for) - the kernel's
    input and the reference's."""
    qs = (q.astype(np.float64) * QSCALE).astype(np.float16)
    return qs, qs.astype(np.float64) / QSCALE


def run_attention(ctx, qs, k, v):
    """qs: prescaled(q)[0]"""
    G, nh = qs.shape[:2]
    dq = ctx.upload_new(pack_qkvh(qs, k, v))
    do = ctx.alloc(G * 1500 * nh * 64 * 2)
    L.check(L.lib().mz_enc_attention(ctx.h, dq, do, G, nh))
    out = ctx.download(do, (G, 1500, nh, 64), np.float16)
    ctx.free(dq)
    ctx.free(do)
    return out.transpose(0, 2, 1, 3)  # [G][nh][1500][64]


def attention64(q, k, v):
    return R.attention(q, k, v, 0.125, dtype=np.float64)


def attention_p16(q, k, v):
    """The fp16-probability arithmetic the kernel (and the reference's fused attention) uses, otherwise exact:
    P = fp16(exp(s - max)), O = fp16(P v / sum P)."""
    s = (q.astype(np.float64) * 0.125) @ np.swapaxes(k.astype(np.float64), -1, -2)
    p = np.exp(s - s.max(-1, keepdims=True)).astype(np.float16).astype(np.float64)
    return ((p @ v.astype(np.float64)) / p.sum(-1, keepdims=True)).astype(np.float16)


def attention_bar(q, k, v, ref):
    """Error bar of an fp16-probability attention: the larger of TOL and 1.5 x the error of attention_p16, whose fp16
    rounding of P and of the output alone reaches about 2e-3 x RMS on near-uniform softmaxes. The max-abs metric
    moves by about +-25% with where the running max stands when each P is rounded (blockwise vs exact max)."""
    return max(TOL, 1.5 * rel_err(attention_p16(q, k, v), ref))


def test_enc_attention_small(ctx):
    rng = np.random.default_rng(10)
    q, k, v = (f16(rng, (1, 2, 1500, 64)) for _ in range(3))
    qs, q = prescaled(q)
    out = run_attention(ctx, qs, k, v)
    ref = attention64(q, k, v)
    assert rel_err(out, ref) < attention_bar(q, k, v, ref)
    # a transposed V (a plausible layout mistake) is far outside the bar
    assert rel_err(out, attention64(q, k, v[..., ::-1])) > 0.1


def test_enc_attention_peaked_scores(ctx):
    """Large logits (scale 4 x N(0,1) inputs): the online max/rescale path dominates."""
    rng = np.random.default_rng(11)
    q, k = f16(rng, (1, 1, 1500, 64), 4.0), f16(rng, (1, 1, 1500, 64), 4.0)
    v = f16(rng, (1, 1, 1500, 64))
    qs, q = prescaled(q)
    out = run_attention(ctx, qs, k, v)
    ref = attention64(q, k, v)
    assert rel_err(out, ref) < attention_bar(q, k, v, ref)


def test_enc_attention_late_peak(ctx):
    """Every query's largest scores far past the running max in late blocks: a peak at key 700 and a dominant one at
    key 1490 (the padded last tile, whose keys past 1500 are masked), so each of those blocks is recomputed against
    a raised max with O rescaled (its probabilities would sum far past 2^12, or overflow fp16, otherwise)."""
    rng = np.random.default_rng(13)
    q, k, v = (f16(rng, (1, 2, 1500, 64)) for _ in range(3))
    c = np.full(64, 1.0, np.float32)
    q = (q.astype(np.float32) + c).astype(np.float16)
    k = k.astype(np.float32)
    k[:, :, 700] += 3.0 * c
    k[:, :, 1490] += 6.0 * c
    k = k.astype(np.float16)
    qs, q = prescaled(q)
    out = run_attention(ctx, qs, k, v)
    ref = attention64(q, k, v)
    assert rel_err(out, ref) < attention_bar(q, k, v, ref)
    # the output is dominated by v[1490] (a kernel that missed the late peak would not be)
    assert rel_err(out, np.broadcast_to(v[:, :, 1490:1491].astype(np.float64), out.shape)) < 0.05


@pytest.mark.parametrize("shape", [(1, 21), (2, 11), (3, 14), (7, 10), (5, 18), (6, 20)])
def test_enc_attention_block_sizes(ctx, shape):
    """Pair counts on both sides of every border between blocks of 128 and of 256 queries (one block per CU and more):
    the same bits as each pair alone, peaks past the running max among them (so the recomputed blocks too), and the
    float64 attention on some rows."""
    rng = np.random.default_rng(sum(shape))
    q, k, v = (f16(rng, (*shape, 1500, 64), s) for s in (2.0, 2.0, 1.0))
    qs, q = prescaled(q)
    out = run_attention(ctx, qs, k, v)
    rows = np.r_[np.arange(0, 1500, 131), 1408, 1499]
    for g, h in ((0, 0), (shape[0] // 2, shape[1] // 3), (shape[0] - 1, shape[1] - 1)):
        one = np.s_[g:g + 1, h:h + 1]
        np.testing.assert_array_equal(run_attention(ctx, qs[one], k[one], v[one]), out[one])
        ref = attention64(q[one][:, :, rows], k[one], v[one])
        assert rel_err(out[one][:, :, rows], ref) < attention_bar(q[one][:, :, rows], k[one], v[one], ref)


def test_enc_attention_large_v3_shape(ctx):
    """8 clips x 20 heads x 1500 x 1500, head 64 (the encoder group's attention); every (clip, head) checked on 48
    query rows spread over the window, including the last ones of the padded tile."""
    rng = np.random.default_rng(12)
    shape = (8, 20, 1500, 64)
    q, k, v = (f16(rng, shape) for _ in range(3))
    qs, q = prescaled(q)
    out = run_attention(ctx, qs, k, v)
    rows = np.r_[np.arange(0, 1500, 37), 1496, 1497, 1498, 1499]
    ref = attention64(q[:, :, rows], k, v)
    assert rel_err(out[:, :, rows], ref) < attention_bar(q[:, :, rows], k, v, ref)
    assert np.isfinite(out).all()


# ---------------------------------------------------------------- GEMMs

def linear_args(**kw):
    a = L.LinearArgs()
    for k_, v_ in kw.items():
        setattr(a, k_, v_)
    return a


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (7, 100, 384), (32, 1280, 1280), (33, 96, 128), (3000, 768, 384),
                                   (1500, 1284, 448)])
def test_gemm_f16(ctx, m, n, k):
    rng = np.random.default_rng(m * 7 + n)
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.05), f16(rng, (n,), 0.1)
    dx, dw, db = ctx.upload_new(x), ctx.upload_new(w), ctx.upload_new(b)
    dy = ctx.alloc(m * n * 2)
    L.check(L.lib().mz_gemm(ctx.h, dx, k, dw, dy, n, m, n, k, db))
    y = ctx.download(dy, (m, n), np.float16)
    ref = x.astype(np.float64) @ w.astype(np.float64).T + b
    assert_f16(y, ref)
    for p in (dx, dw, db, dy):
        ctx.free(p)


def test_gemm_epilogues(ctx):
    rng = np.random.default_rng(3)
    m, n, k = 3000, 512, 640
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.05), f16(rng, (n,), 0.1)
    res = rng.standard_normal((m, n)).astype(np.float32)
    pos = f16(rng, (1500, n))
    acc = x.astype(np.float64) @ w.astype(np.float64).T + b
    dx, dw, db, dpos = (ctx.upload_new(a) for a in (x, w, b, pos))
    # GELU -> fp16
    dy = ctx.alloc(m * n * 2)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_F16, a=dx, lda=k, w=dw, bias=db, m=m, n=n, k=k,
                                                 out=dy, ldo=n)))
    assert_f16(ctx.download(dy, (m, n), np.float16), R.gelu(acc.astype(np.float32)))
    # residual add into fp32
    dr = ctx.upload_new(res)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_RESID_F32, a=dx, lda=k, w=dw, bias=db, m=m, n=n, k=k,
                                                 out=dr, ldo=n)))
    got = ctx.download(dr, (m, n), np.float32)
    ref = res + acc
    assert rel_err(got, ref) < 1e-5
    # GELU + positions (the conv2 epilogue) exists only on the implicit-conv load: refused on a plain product
    with pytest.raises(L.MzError):
        L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_POS, a=dx, lda=k, w=dw, bias=db, m=m, n=n,
                                                     k=k, out=dr, ldo=n, pos=dpos)))
    for p in (dx, dw, db, dpos, dy, dr):
        ctx.free(p)


def test_gemm_gelu_every_fp16_value(ctx):
    """The GELU epilogue on every finite fp16 input: row m of x holds value m in column 0 and w is 1 there, so each
    accumulator is exactly that value; no bias (a missing bias reads zeros). Against 0.5 v erfc(-v / sqrt 2) in float64:
    within 0.6 fp16 ulp everywhere (0.505 measured, at v = 0.0036; an emulation of the fp32 arithmetic on the host
    gives the same, with exp2 correctly rounded or one ulp off) and correctly rounded for all but a few hundred values
    (164 measured; 157-171 in the emulation). Every column of a row is the same value, and the 64 columns cover both
    the whole-block and the column-checked stores."""
    from scipy.special import erfc
    v = np.arange(65536, dtype=np.uint32).astype(np.uint16).view(np.float16)
    v = v[np.isfinite(v)]
    m, n, k = v.size, 64, 64
    x = np.zeros((m, k), np.float16)
    x[:, 0] = v
    w = np.zeros((n, k), np.float16)
    w[:, 0] = 1
    dx, dw = ctx.upload_new(x), ctx.upload_new(w)
    dy = ctx.alloc(m * n * 2)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_F16, a=dx, lda=k, w=dw, m=m, n=n, k=k, out=dy,
                                                 ldo=n)))
    y = ctx.download(dy, (m, n), np.float16)
    for p in (dx, dw, dy):
        ctx.free(p)
    bits = y.view(np.uint16)
    assert (bits == bits[:, :1]).all()
    vd = v.astype(np.float64)
    ref = 0.5 * vd * erfc(-vd / np.sqrt(2))
    got = y[:, 0].astype(np.float64)
    ulp = 2.0 ** (np.maximum(np.floor(np.log2(np.maximum(np.abs(ref), 1e-300))), -14) - 10)
    err = np.abs(got - ref) / ulp
    sub = np.abs(vd) < 2.0 ** -14  # fp16 subnormal inputs (and zeros)
    worst = int(np.argmax(err))
    print("GELU over %d fp16 values: max %.3f ulp at v = %g; %d not correctly rounded" %
          (v.size, err[worst], vd[worst], int((y[:, 0] != ref.astype(np.float16)).sum())))
    assert err[~sub].max() <= 0.6, ("normal inputs", vd[~sub][np.argmax(err[~sub])])
    assert err[sub].max() <= 0.6, ("subnormal inputs", vd[sub][np.argmax(err[sub])])
    assert (y[:, 0] != ref.astype(np.float16)).sum() < 300


@pytest.mark.parametrize("kind", [3, 2])
def test_gemm_head_scatter(ctx, kind):
    """kind 3: [q|k|v][head] tiles of the encoder self-attention (v tiles transposed, q tiles multiplied by
    log2(e) / 8); kind 2: [layer][k|v][head] of the cross k/v (all tiles row-major); both into clip slots (slot0
    offset)."""
    rng = np.random.default_rng(kind)
    nh, clips, slot0 = 2, 2, 1
    groups = 3 if kind == 3 else 2 * 2  # kind 2: two decoder layers
    n, k, m = groups * nh * 64, 128, clips * 1500
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.1), f16(rng, (n,), 0.1)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    bpc = groups * nh
    nslots = slot0 + clips + 1  # one slot past the call's clips, which must stay untouched
    dh = ctx.alloc(nslots * bpc * TPAD * 64 * 2)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_HEADS, a=dx, lda=k, w=dw, bias=db, m=m, n=n, k=k,
                                                 heads=dh, blocks_per_clip=bpc, nh=nh, kind=kind, slot0=slot0)))
    got = ctx.download(dh, (nslots, bpc, TPAD * 64), np.float16)
    ref = (x.astype(np.float64) @ w.astype(np.float64).T + b).reshape(clips, 1500, bpc, 64)
    if kind == 3:
        ref[:, :, :nh] *= QSCALE
    assert not got[:slot0].any(), "a slot before slot0 was written"
    assert not got[slot0 + clips:].any(), "a slot after the last clip was written"
    for c in range(clips):
        for blk in range(bpc):
            tile = got[slot0 + c, blk]
            if kind == 3 and blk // nh == 2:  # encoder v: [64][1536]
                t = tile.reshape(64, TPAD)
                assert not t[:, 1500:].any()
                assert_f16(t[:, :1500].T, ref[c, :, blk])
            else:
                t = tile.reshape(TPAD, 64)
                assert not t[1500:].any()
                assert_f16(t[:1500], ref[c, :, blk])
    for p in (dx, dw, db, dh):
        ctx.free(p)


@pytest.mark.parametrize("kind,nh,clips,blocks", [(3, 6, 5, 18), (2, 1, 6, 7), (3, 1, 7, 3)])
def test_gemm_head_scatter_partial_columns(ctx, kind, nh, clips, blocks):
    """Head counts that leave the last column tile partial (1152 columns in 256 x 256 tiles, 448 in 256 x 128, 192 in
    128 x 128): the columns past the last head write nothing. Each clip has two more tiles than the product has heads, which
    must stay as they were, as must every tile's padding."""
    rng = np.random.default_rng(blocks)
    n, k, m, bpc = blocks * 64, 128, clips * 1500, blocks + 2
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.1), f16(rng, (n,), 0.1)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    dh = ctx.upload_new(np.full((clips, bpc, TPAD * 64), 7, np.float16))
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_HEADS, a=dx, lda=k, w=dw, bias=db, m=m, n=n, k=k,
                                                 heads=dh, blocks_per_clip=bpc, nh=nh, kind=kind, slot0=0)))
    got = ctx.download(dh, (clips, bpc, TPAD * 64), np.float16)
    assert (got[:, blocks:] == 7).all(), "a tile past the last head was written"
    ref = (x.astype(np.float64) @ w.astype(np.float64).T + b).reshape(clips, 1500, blocks, 64)
    if kind == 3:
        ref[:, :, :nh] *= QSCALE
    for c in range(clips):
        for blk in range(blocks):
            v = kind == 3 and blk // nh == 2
            tile = got[c, blk].reshape(64, TPAD).T if v else got[c, blk].reshape(TPAD, 64)
            assert (tile[1500:] == 7).all()
            assert_f16(tile[:1500], ref[c, :, blk])
    for p in (dx, dw, db, dh):
        ctx.free(p)


@pytest.mark.parametrize("kind,nh,clips,blocks", [(3, 16, 7, 48), (2, 24, 3, 96)])
def test_gemm_head_scatter_several_tiles_per_workgroup(ctx, kind, nh, clips, blocks):
    """10500 x 3072 and 4500 x 6144: 504 and 432 tiles of 256 x 256 in equal shares of 63 and 54 per XCD, so that each
    workgroup scatters a tile while the next one's operands come in. Bit for bit what each clip alone (one tile per
    workgroup) gives; test_gemm_head_scatter compares that with float64."""
    rng = np.random.default_rng(blocks)
    n, k, m = blocks * 64, 192, clips * 1500
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.1), f16(rng, (n,), 0.1)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    out = []
    for step in (clips, 1):
        dh = ctx.upload_new(np.full((clips, blocks, TPAD * 64), 7, np.float16))
        for c in range(0, clips, step):
            L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_HEADS, a=dx + c * 1500 * k * 2, lda=k, w=dw, bias=db,
                                                         m=step * 1500, n=n, k=k, heads=dh, blocks_per_clip=blocks, nh=nh,
                                                         kind=kind, slot0=c)))
        out.append(ctx.download(dh, (clips, blocks, TPAD * 64), np.float16))
        ctx.free(dh)
    np.testing.assert_array_equal(out[0], out[1])
    assert (out[0][0, 0].reshape(TPAD, 64)[:1500] != 7).any()
    for p in (dx, dw, db):
        ctx.free(p)


def test_gemm_large_qkv_shape(ctx):
    """The encoder group's fused QKV product, M = 12000, N = 3840, K = 1280, 256 rows checked."""
    rng = np.random.default_rng(5)
    m, n, k = 12000, 3840, 1280
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.02), f16(rng, (n,), 0.02)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    dy = ctx.alloc(m * n * 2)
    L.check(L.lib().mz_gemm(ctx.h, dx, k, dw, dy, n, m, n, k, db))
    y = ctx.download(dy, (m, n), np.float16)
    rows = np.r_[rng.choice(m, 250, replace=False), m - 6:m]
    ref = x[rows].astype(np.float64) @ w.astype(np.float64).T + b
    assert_f16(y[rows], ref)
    for p in (dx, dw, db, dy):
        ctx.free(p)


@pytest.mark.parametrize("m,n,k", [(9000, 2304, 320), (12000, 768, 448), (6000, 1000, 192), (10500, 3072, 320),
                                   (9000, 5116, 192), (6000, 2688, 192), (24988, 640, 128)])
def test_gemm_persistent_shapes(ctx, m, n, k):
    """Products of 256 x 256 and 256 x 128 tiles, whose workgroups walk several tiles where there are more than CUs
    (requesting the next tile's first K tile before each epilogue):
      9000 x 2304   256 x 256, 324 tiles, whole bands per XCD; partial last block row, odd count of 64-wide K tiles
      10500 x 3072  256 x 256, 504 tiles, equal shares of 63 per XCD
      9000 x 5116   256 x 256, 720 tiles, equal shares of 90, a last band of one block row and a partial last column
      6000 x 2688   256 x 128, 504 tiles, whole bands (256 x 256 would take as many rounds)
      24988 x 640   256 x 128, 490 tiles, equal shares of 62
      12000 x 768   256 x 256, 141 tiles: one per workgroup
      6000 x 1000   256 x 128, 192 tiles: one per workgroup, partial last row and column
    fp16 output against float64 on sampled rows and bit for bit against the last 1500 rows alone (other tiles); the
    GELU and fp32 residual epilogues too where a workgroup has several tiles."""
    rng = np.random.default_rng(m + n + k)
    x, w, b = f16(rng, (m, k)), f16(rng, (n, k), 0.05), f16(rng, (n,), 0.1)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    rows = np.r_[rng.choice(m, 300, replace=False), m - 40:m]
    acc = x[rows].astype(np.float64) @ w.astype(np.float64).T + b
    dy = ctx.alloc(m * n * 2)
    L.check(L.lib().mz_gemm(ctx.h, dx, k, dw, dy, n, m, n, k, db))
    y = ctx.download(dy, (m, n), np.float16)
    assert_f16(y[rows], acc)
    L.check(L.lib().mz_gemm(ctx.h, dx + (m - 1500) * k * 2, k, dw, dy, n, 1500, n, k, db))
    np.testing.assert_array_equal(ctx.download(dy, (1500, n), np.float16), y[-1500:])
    if m * n >= 6000 * 2304:
        L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_F16, a=dx, lda=k, w=dw, bias=db, m=m, n=n,
                                                     k=k, out=dy, ldo=n)))
        assert_f16(ctx.download(dy, (m, n), np.float16)[rows], R.gelu(acc.astype(np.float32)))
        res = rng.standard_normal((m, n)).astype(np.float32)
        dr = ctx.upload_new(res)
        L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_RESID_F32, a=dx, lda=k, w=dw, bias=db, m=m, n=n,
                                                     k=k, out=dr, ldo=n)))
        got = ctx.download(dr, (m, n), np.float32)
        assert rel_err(got[rows], res[rows] + acc) < 1e-5
        ctx.free(dr)
    for p in (dx, dw, db, dy):
        ctx.free(p)


@pytest.mark.parametrize("m,n,k", [(33, 4, 64), (64, 64, 256), (65, 132, 128), (1500, 384, 192), (1500, 516, 1280),
                                   (1500, 1284, 320), (1500, 1280, 5120), (1499, 2308, 448), (3000, 768, 384)])
def test_gemm_small_grids(ctx, m, n, k):
    """Products of few tiles: 64 x 64, 128 x 64 and 128 x 128 tiles with partial last rows and columns, and K tile counts
    on both sides of the ring's four slots (1, 2, 3, 4, 5, 7 and whole rounds). The same bits as the same rows within a
    product large enough for tiles of 256 rows, and the float64 product."""
    rng = np.random.default_rng(m + 3 * n + k)
    big = 256 * (132 // ((n + 255) // 256) + 1)
    x, w, b = f16(rng, (max(m, big), k)), f16(rng, (n, k), 0.05), f16(rng, (n,), 0.1)
    dx, dw, db = (ctx.upload_new(a) for a in (x, w, b))
    dy = ctx.alloc(x.shape[0] * n * 2)
    out = []
    for rows in (m, x.shape[0]):
        L.check(L.lib().mz_gemm(ctx.h, dx, k, dw, dy, n, rows, n, k, db))
        out.append(ctx.download(dy, (rows, n), np.float16))
    np.testing.assert_array_equal(out[0], out[1][:m])
    assert_f16(out[0], x[:m].astype(np.float64) @ w.astype(np.float64).T + b)
    for p in (dx, dw, db, dy):
        ctx.free(p)


@pytest.mark.parametrize("clips,cin,n,stride", [(1, 80, 384, 1), (1, 384, 384, 2), (3, 128, 512, 1), (1, 512, 1280, 2),
                                                (1, 1280, 1280, 2), (2, 1024, 1024, 2), (8, 896, 896, 2)])
def test_conv_small_grids(ctx, clips, cin, n, stride):
    """The convolution's padding (both ends of each clip, K past the taps) in each of its tile shapes (64 x 64 for the
    first two and the fourth, two buffers of 128 x 128 for the third, then 128 x 64, the ring of 128 x 128, and 256 x 256):
    the same bits as the plain product of the unrolled rows."""
    rng = np.random.default_rng(clips + cin + n)
    src, b = f16(rng, (clips, 3000, cin)), f16(rng, (n,), 0.1)
    k, t = (3 * cin + 63) // 64 * 64, 3000 // stride
    w = f16(rng, (n, k), 0.05)  # non-zero past the taps too: those columns of the rows read as zero
    rows = np.zeros((clips, t, k), np.float16)
    pad = np.pad(src, ((0, 0), (1, 1), (0, 0)))
    for tap in range(3):
        rows[:, :, tap * cin:(tap + 1) * cin] = pad[:, tap:tap + stride * (t - 1) + 1:stride]
    ds, dr, dw, db = (ctx.upload_new(a) for a in (src, rows, w, b))
    dy = ctx.alloc(clips * t * n * 2)
    out = []
    for conv in (dict(a=ds, conv_cin=cin, conv_tin=3000, conv_tout=t, conv_stride=stride), dict(a=dr, lda=k)):
        L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_F16, w=dw, bias=db, m=clips * t, n=n, k=k,
                                                     out=dy, ldo=n, **conv)))
        out.append(ctx.download(dy, (clips * t, n), np.float16))
    np.testing.assert_array_equal(out[0], out[1])
    for p in (ds, dr, dw, db, dy):
        ctx.free(p)


def test_conv_stem_implicit_gemm(ctx):
    """mel transpose + conv1 (k 3, pad 1) + GELU, conv2 (stride 2) + GELU + positions, against the oracle's conv1d."""
    rng = np.random.default_rng(6)
    nm, d, clips = 80, 384, 2
    mel = np.clip(rng.normal(-0.3, 0.4, (clips, nm, 3000)), -1.5, 1.5).astype(np.float32)
    w1, b1 = f16(rng, (d, nm, 3), 0.05), f16(rng, (d,), 0.05)
    w2, b2 = f16(rng, (d, d, 3), 0.02), f16(rng, (d,), 0.05)
    pos = f16(rng, (1500, d), 0.5)
    k1 = ((3 * nm + 63) // 64) * 64
    w1t = np.zeros((d, k1), np.float16)
    w1t[:, :3 * nm] = w1.transpose(0, 2, 1).reshape(d, 3 * nm)
    w2t = np.ascontiguousarray(w2.transpose(0, 2, 1).reshape(d, 3 * d))
    dmel = ctx.upload_new(mel)
    dmt = ctx.alloc(clips * 3000 * nm * 2)
    L.check(L.lib().mz_mel_transpose(ctx.h, dmel, dmt, clips, nm))
    mt = ctx.download(dmt, (clips, 3000, nm), np.float16)
    np.testing.assert_array_equal(mt, mel.transpose(0, 2, 1).astype(np.float16))
    dw1, db1, dw2, db2, dpos = (ctx.upload_new(a) for a in (w1t, b1, w2t, b2, pos))
    dh1 = ctx.alloc(clips * 3000 * d * 2)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_F16, a=dmt, w=dw1, bias=db1, m=clips * 3000, n=d,
                                                 k=k1, out=dh1, ldo=d, conv_cin=nm, conv_tin=3000, conv_tout=3000,
                                                 conv_stride=1)))
    h1 = ctx.download(dh1, (clips, 3000, d), np.float16)
    dx = ctx.alloc(clips * 1500 * d * 4)
    L.check(L.lib().mz_linear(ctx.h, linear_args(epilogue=L.EPI_GELU_POS, a=dh1, w=dw2, bias=db2, m=clips * 1500, n=d,
                                                 k=3 * d, out=dx, ldo=d, pos=dpos, conv_cin=d, conv_tin=3000,
                                                 conv_tout=1500, conv_stride=2)))
    x = ctx.download(dx, (clips, 1500, d), np.float32)
    for c in range(clips):
        m16 = mel[c].astype(np.float16).astype(np.float64)
        r1 = R.gelu(R.conv1d(m16, w1.astype(np.float64), b1.astype(np.float64), 1, 1).astype(np.float32))
        assert_f16(h1[c].T, r1)
        # conv2 on the kernel's own fp16 conv1 output (layer-local)
        r2 = R.gelu(R.conv1d(h1[c].T.astype(np.float64), w2.astype(np.float64), b2.astype(np.float64), 2, 1)
                    .astype(np.float32)).T + pos.astype(np.float32)
        assert rel_err(x[c], r2) < 1e-4
    for p in (dmel, dmt, dw1, db1, dw2, db2, dpos, dh1, dx):
        ctx.free(p)


# ---------------------------------------------------------------- LayerNorm

@pytest.mark.parametrize("dim", [384, 1280, 2048])
def test_layernorm_and_add_layernorm(ctx, dim):
    rng = np.random.default_rng(dim)
    rows = 301
    x = (rng.standard_normal((rows, dim)) * 3 + 1).astype(np.float32)
    dlt = f16(rng, (rows, dim))
    w, b = f16(rng, (dim,), 0.1) + np.float16(1), f16(rng, (dim,), 0.1)
    dxx, dd, dw, db = (ctx.upload_new(a) for a in (x, dlt, w, b))
    dy = ctx.alloc(rows * dim * 2)
    L.check(L.lib().mz_layernorm(ctx.h, dxx, dim, dw, db, dy, dim, rows, dim, 1e-5))
    y = ctx.download(dy, (rows, dim), np.float16)
    assert_f16(y, R.layer_norm(x.astype(np.float64), w, b))
    L.check(L.lib().mz_add_layernorm(ctx.h, dxx, dd, dw, db, dy, rows, dim, 1e-5))
    xs = ctx.download(dxx, (rows, dim), np.float32)
    np.testing.assert_allclose(xs, x + dlt.astype(np.float32), rtol=0, atol=0)
    y = ctx.download(dy, (rows, dim), np.float16)
    assert_f16(y, R.layer_norm((x + dlt.astype(np.float32)).astype(np.float64), w, b))
    for p in (dxx, dd, dw, db, dy):
        ctx.free(p)


# ---------------------------------------------------------------- token timestamps (median filter + DTW)

def softmax_rows(rng, shape, peak=3.0):
    s = rng.standard_normal(shape) * peak
    w = np.exp(s - s.max(-1, keepdims=True))
    return (w / w.sum(-1, keepdims=True)).astype(np.float16).astype(np.float32)


@pytest.mark.parametrize("half", [False, True])
def test_timestamps_device_match_host_bits(ctx, half):
    """k_align.hip against the host routine mz_jump_times (itself pinned to the oracle and to the golden vectors):
    identical floats for every clip, with ragged row and column counts, clips without rows or columns, fewer
    columns than the filter's half width, constant columns (zero deviation) and a diagonal alignment."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(11 + half)
    heads, full = 6, 1500
    rows = [40, 1, 0, 223, 17, 5, 60, 33]
    cols = [1500, 700, 300, 1500, 3, 0, 911, 64]
    rmax = max(rows)
    w = softmax_rows(rng, (len(rows), rmax, heads, full))
    w[4, :, 2, :] = 0.25                       # constant columns in one head
    for i in range(rows[6]):                   # a clean diagonal in clip 6
        w[6, i, :, 15 * i:15 * i + 15] += 0.5
    dw = ctx.upload_new(w)
    got = transcribe.jump_times_device(ctx, dw, rmax * heads * full, rows, cols, heads, full, 7, half)
    for c in range(len(rows)):
        ref = transcribe.jump_times(w[c, :rows[c]], cols[c], 7, half)
        np.testing.assert_array_equal(got[c], ref, err_msg=f"clip {c}")
        if 0 < rows[c] <= 40 and cols[c] <= 64:
            np.testing.assert_array_equal(got[c], R.jump_times(w[c, :rows[c]], cols[c], 7, half))


@pytest.mark.parametrize("rows,cols", [([255, 3, 128], [1500, 1500, 1]),      # one wave per clip, its largest table
                                       ([300, 256, 9], [1500, 1499, 77])])   # more rows than a wave holds
def test_timestamps_device_row_limits(ctx, rows, cols):
    """Tables at and past 256 rows, where the one-wave DTW hands over to the workgroup DTW: identical floats."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(sum(rows))
    heads, full, rmax = 2, 1500, max(rows)
    w = softmax_rows(rng, (len(rows), rmax, heads, full))
    dw = ctx.upload_new(w)
    got = transcribe.jump_times_device(ctx, dw, rmax * heads * full, rows, cols, heads, full, 7, True)
    for c in range(len(rows)):
        np.testing.assert_array_equal(got[c], transcribe.jump_times(w[c, :rows[c]], cols[c], 7, True),
                                      err_msg=f"clip {c}")


@pytest.mark.parametrize("rows,cols,heads", [([64, 63, 1], [1500, 1, 130], 1), ([65, 64, 2], [1500, 63, 65], 3),
                                             ([129, 128, 65], [1500, 1500, 1499], 2), ([256, 193, 192], [1500, 64, 1500], 2)])
def test_timestamps_device_wave_borders(ctx, rows, cols, heads):
    """Rows at the borders of the DTW's waves (64 rows each, one to four of them), tables of less than one chunk of
    diagonals and of a whole number of them, a NaN in one column of one clip: identical floats to the host routine."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(sum(rows) + sum(cols))
    full, rmax = 1500, max(rows)
    for half in (True, False):
        w = softmax_rows(rng, (len(rows), rmax, heads, full))
        if half:
            w[2, 0::2, :, 40] = 0.0
            w[2, 1::2, :, 40] = 2e5
        dw = ctx.upload_new(w)
        got = transcribe.jump_times_device(ctx, dw, rmax * heads * full, rows, cols, heads, full, 7, half)
        for c in range(len(rows)):
            np.testing.assert_array_equal(got[c], transcribe.jump_times(w[c, :rows[c]], cols[c], 7, half),
                                          err_msg=f"clip {c} ({rows[c]} x {cols[c]}, half {half})")
        ctx.free(dw)


def test_timestamps_device_nan_costs(ctx):
    """A column whose values overflow fp16 (0 and 2e5 alternating: mean and deviation round to inf, z = inf / inf)
    gives NaN DTW costs in half mode. The DTW must then choose its moves with the reference's comparisons as written
    (a NaN neighbour loses every comparison, align.rs:77-83), in the one-wave kernel (<= 255 rows) as in the
    workgroup kernel and the host routine: identical floats."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(29)
    heads, full = 6, 1500
    rows, cols = [40, 255, 7, 300], [1500, 1500, 900, 1500]
    rmax = max(rows)
    w = softmax_rows(rng, (len(rows), rmax, heads, full))
    for c, col in enumerate((700, 1201, 450, 333)):
        w[c, 0::2, :, col] = 0.0
        w[c, 1::2, :, col] = 2e5
    for c in range(len(rows)):
        assert np.isnan(transcribe.align_cost(w[c, :rows[c]], cols[c], 7, True)).any(), f"clip {c}: no NaN cost"
    dw = ctx.upload_new(w)
    got = transcribe.jump_times_device(ctx, dw, rmax * heads * full, rows, cols, heads, full, 7, True)
    for c in range(len(rows)):
        np.testing.assert_array_equal(got[c], transcribe.jump_times(w[c, :rows[c]], cols[c], 7, True),
                                      err_msg=f"clip {c} ({rows[c]} rows)")


@pytest.mark.parametrize("full", [1500, 203])
def test_timestamps_device_column_layouts(ctx, full):
    """Rows of 1500 columns (four columns per thread in the column statistics) and of an odd count (one per thread):
    identical floats in both modes."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(full)
    heads, rows, cols = 3, [12, 30, 7], [full, full - 1, full // 2]
    w = softmax_rows(rng, (3, 30, heads, full))
    dw = ctx.upload_new(w)
    for half in (False, True):
        got = transcribe.jump_times_device(ctx, dw, 30 * heads * full, rows, cols, heads, full, 7, half)
        for c in range(3):
            np.testing.assert_array_equal(got[c], transcribe.jump_times(w[c, :rows[c]], cols[c], 7, half),
                                          err_msg=f"clip {c} half {half}")


def test_timestamps_device_other_widths(ctx):
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(5)
    heads, full, rows, cols = 3, 200, [12, 30], [200, 150]
    w = softmax_rows(rng, (2, 30, heads, full))
    dw = ctx.upload_new(w)
    for width in (1, 5, 9, 15):
        got = transcribe.jump_times_device(ctx, dw, 30 * heads * full, rows, cols, heads, full, width, True)
        for c in range(2):
            np.testing.assert_array_equal(got[c], transcribe.jump_times(w[c, :rows[c]], cols[c], width, True))
