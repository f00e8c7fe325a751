"""The work that programs built on this framework have it do, as cases that can be timed.

Four kinds of call, each through the package's own entry points:

  mel     log-mel features of a batch of clips on the device (mz_log_mel): what the command line does for every file
  encode  the encoder of a group of clips (Engine.encode_device): conv stem, layers, every decoder layer's cross
          keys and values
  decode  a run of decoder steps over a prompt (Engine.reset, then the captured step replayed once per token)
  times   token timestamps of a batch of clips from alignment-head weights (jump_times_device and its variant that
          allocates nothing)

The widths are the Whisper family's (384 to 1280, 64-wide heads, four times as wide inside); the encoder cases run
two to four layers and the decoder cases two to four, which is what a layer costs in a deep model too.
"""
import ctypes as C
import math

import numpy as np
import torch

from mimizuku_amd import _lib as L
from mimizuku_amd import model, transcribe
from mimizuku_amd.synth import Geometry, sinusoids, tensor_shapes

TENC, TPAD, NFR, NSAMP, HD = 1500, 1536, 3000, 480000, 64
WIDTHS = (384, 512, 768, 1024, 1280)
MAX_T = 448


def listed():
    return [
        # one short recording on an 80-band model: the smallest call of the front end, waited for by a user
        {"name": "mel_1x7s", "kind": "mel", "clips": 1, "mels": 80, "seconds": 7.3},
        # a batch of the command line's default size over full windows
        {"name": "mel_32x30s", "kind": "mel", "clips": 32, "mels": 128, "seconds": 30.0},
        # one clip through the smallest model's encoder (its four layers): latency of an interactive call
        {"name": "encode_384_c1", "kind": "encode", "d": 384, "mels": 80, "clips": 1, "layers": 4, "xlayers": 4},
        # the last, partial group of a batch on a middle-sized model
        {"name": "encode_768_c3", "kind": "encode", "d": 768, "mels": 80, "clips": 3, "layers": 2, "xlayers": 2},
        # one clip through the widest encoder: latency of a single request to the large models
        {"name": "encode_1280_c1", "kind": "encode", "d": 1280, "mels": 128, "clips": 1, "layers": 2, "xlayers": 2},
        # the encoder group that the benchmark and the command line use
        {"name": "encode_1280_c8", "kind": "encode", "d": 1280, "mels": 128, "clips": 8, "layers": 2, "xlayers": 2},
        # the smallest decoder, one row: launches and latency
        {"name": "decode_384_b1", "kind": "decode", "d": 384, "rows": 1, "layers": 4, "vocab": 51865, "steps": 48},
        # a handful of rows on a middle-sized model
        {"name": "decode_1024_b6", "kind": "decode", "d": 1024, "rows": 6, "layers": 4, "vocab": 51865, "steps": 40},
        # the four-layer wide decoder for a single request, and for the benchmark's batch
        {"name": "decode_1280_b1", "kind": "decode", "d": 1280, "rows": 1, "layers": 4, "vocab": 51866, "steps": 48},
        {"name": "decode_1280_b32", "kind": "decode", "d": 1280, "rows": 32, "layers": 4, "vocab": 51866, "steps": 48},
        # timestamps of one clip's sentence, and of a whole batch of full transcripts
        {"name": "times_1x41", "kind": "times", "clips": 1, "rows": 41, "heads": 6, "half": True, "scratch": "static"},
        {"name": "times_32x220", "kind": "times", "clips": 32, "rows": 220, "heads": 10, "half": True,
         "scratch": "call"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mel", "encode", "encode", "decode", "decode", "times"])
    if kind == "mel":
        return {"kind": kind, "clips": _log_int(rng, 1, 32), "mels": rng.choice([80, 128]),
                "seconds": round(rng.uniform(1.0, 30.0), 3)}
    if kind == "encode":
        return {"kind": kind, "d": rng.choice(WIDTHS), "mels": rng.choice([80, 128]), "clips": _log_int(rng, 1, 8),
                "layers": 2, "xlayers": rng.randint(1, 2)}
    if kind == "decode":
        return {"kind": kind, "d": rng.choice(WIDTHS), "rows": _log_int(rng, 1, 32), "layers": rng.randint(2, 4),
                "vocab": rng.choice([51864, 51865, 51866]), "steps": rng.randint(16, 48)}
    return {"kind": kind, "clips": _log_int(rng, 1, 32), "rows": _log_int(rng, 5, 224), "heads": rng.randint(4, 10),
            "half": rng.random() < 0.7, "scratch": rng.choice(["static", "call"])}


# ---------------------------------------------------------------- inputs


_ctx = []


def _context():
    if not _ctx:
        _ctx.append(model.Context(0))
    return _ctx[0]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, std=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _ragged(n, top, low):
    """Lengths of the clips of a batch, the first one the longest: transcripts and recordings differ in length."""
    return [max(low, int(top * (1.0 - 0.45 * ((5 * i) % 11) / 11.0))) for i in range(n)]


def _audio(case, seed):
    """Speech-like 16 kHz audio: three slowly wandering tones and noise under a syllable-rate envelope."""
    g, n = _gen(seed), case["clips"]
    t = torch.arange(NSAMP, device="cuda", dtype=torch.float32) / 16000.0
    r = torch.rand((n, 8), generator=g, device="cuda")
    y = torch.empty((n, NSAMP), device="cuda")
    for i in range(n):
        env = 0.55 + 0.45 * torch.sin(2 * math.pi * (3.0 + 2.0 * r[i, 0]) * t)
        y[i] = _randn(g, (NSAMP,), 0.02)
        for k, f in enumerate((180.0, 900.0, 2600.0)):
            y[i] += env * (0.2 / (k + 1)) * torch.sin(2 * math.pi * f * (0.8 + 0.4 * r[i, 1 + k]) * t + 6.0 * r[i, 4 + k])
    ns = _ragged(n, min(NSAMP, int(16000 * case["seconds"])), 400)
    for i in range(n):
        y[i, ns[i]:] = 0.0
    return y, ns


def _geometry(case):
    d = case["d"]
    if case["kind"] == "encode":
        # the token embedding takes no part in the encoder: a short vocabulary keeps the engine small
        return Geometry(d, 4 * d, d // HD, case["layers"], case["xlayers"], case["mels"], 1024, MAX_T)
    return Geometry(d, 4 * d, d // HD, 1, case["layers"], 80, case["vocab"], MAX_T)


def _weights(g, seed):
    """fp16 weights N(0, 0.02) with biases and LayerNorm parameters that are not trivial, on the GPU."""
    gen, out = _gen(seed), {}
    for name, shape in tensor_shapes(g).items():
        if name == "model.encoder.embed_positions.weight":
            w = torch.from_numpy(sinusoids(TENC, g.d)).cuda().half()
        elif "layer_norm" in name:
            w = (_randn(gen, shape, 0.1) + (1.0 if name.endswith("weight") else 0.0)).half()
        else:
            w = _randn(gen, shape, 0.02, torch.float16)
        out[name] = w
    return out


def _align_heads(g):
    """Six alignment heads in the last two layers, as the published configurations of the small decoders have."""
    a, b = max(0, g.dec_layers - 2), g.dec_layers - 1
    heads = [(a, 1), (b, 0), (b, 2), (b, 3), (b, 5)]
    return [(a, 4)] + heads if a != b else [(b, 4), (b, 1)] + heads[1:]


def _engine(g, weights, bmax, eg):
    dims = model.Dims(g.d, g.ff, g.nh, g.enc_layers, g.dec_layers, g.n_mels, g.vocab, g.max_t)
    sot = min(50258, g.vocab - 4)
    gc = model.GenCfg(sot=sot, eos=sot - 1, no_timestamps=sot + 3, langs=[("en", sot + 1)],
                      tasks=[("transcribe", sot + 2)], suppress=[1, 2, 7, 8, 9], begin_suppress=[220, sot - 1],
                      align_heads=_align_heads(g))
    e = model.Engine(_context(), dims, gc, bmax, eg)
    e.load({k: v.cpu().numpy() for k, v in weights.items()})
    return e


class _Device:
    """An engine buffer as torch sees it; it keeps the engine, whose memory it is."""

    def __init__(self, e, which, shape, typestr):
        p, nbytes = e.buffer(which)
        assert nbytes == int(np.prod(shape)) * int(typestr[2:])
        self.engine = e
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (p, False), "version": 2}


def _view(e, which, shape, typestr):
    return torch.as_tensor(_Device(e, which, tuple(shape), typestr), device="cuda")


def _mel_input(case, seed):
    return _randn(_gen(seed + 1), (case["clips"], case["mels"], NFR), 0.4).sub_(0.3).clamp_(-1.5, 1.5)


def _cross_kv(case, g, seed):
    """Cross keys and values as the encoder leaves them: a projection of a normalised row, about N(0, 0.7)."""
    kv = torch.zeros((case["rows"], g.dec_layers, 2, g.nh, TPAD, HD), device="cuda", dtype=torch.float16)
    gen = _gen(seed + 2)
    for b in range(case["rows"]):
        kv[b, :, :, :, :TENC] = _randn(gen, (g.dec_layers, 2, g.nh, TENC, HD), 0.7, torch.float16)
    return kv


def _prompt(case, seed):
    """A prompt of previous text, another one for each row: one token per step."""
    r = np.random.RandomState(seed % (1 << 31))
    p = r.randint(300, 50000, size=(case["rows"], case["steps"]))
    p[:, 0] = 50258
    return p


def _alignment(case, seed):
    """Alignment-head weights: softmax rows whose peak moves through the clip with the tokens."""
    n, rows, heads = case["clips"], case["rows"], case["heads"]
    rc = _ragged(n, rows, 1)
    cols = _ragged(n, TENC, 50)
    g = _gen(seed)
    t = torch.arange(TENC, device="cuda", dtype=torch.float32)
    w = torch.empty((n, rows, heads, TENC), device="cuda")
    for c in range(n):
        step = torch.rand((rows,), generator=g, device="cuda") + 0.3
        at = torch.cumsum(step, 0) / step[:rc[c]].sum() * (cols[c] - 10)
        s = _randn(g, (rows, heads, TENC), 1.0)
        s += 7.0 * torch.exp(-0.5 * ((t[None, None] - at[:, None, None]) / 9.0) ** 2)
        w[c] = torch.softmax(s, -1)
    return w, rc, cols


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = {"case": case, "ctx": ctx}
    if kind == "mel":
        s["audio"], ns = _audio(case, seed)
        s["ns"] = np.array(ns, np.int32)
        s["frames"] = np.zeros(case["clips"], np.int32)
        s["mel"] = torch.empty((case["clips"], case["mels"], NFR), device="cuda")
    elif kind == "encode":
        g = _geometry(case)
        n = case["clips"]
        s["engine"] = e = _engine(g, _weights(g, seed), n, n)
        s["mel"] = _mel_input(case, seed)
        s["out"] = {"encoded": _view(e, L.BUF_ENC_OUT, (n, TENC, g.d), "<f2"),
                    "residual": _view(e, L.BUF_ENC_X, (n, TENC, g.d), "<f4"),
                    "cross": _view(e, L.BUF_XKV, (n, g.dec_layers, 2, g.nh, TPAD, HD), "<f2")}
    elif kind == "decode":
        g = _geometry(case)
        b, t, na = case["rows"], case["steps"], len(_align_heads(g))
        s["engine"] = e = _engine(g, _weights(g, seed), b, 1)
        _view(e, L.BUF_XKV, (b, g.dec_layers, 2, g.nh, TPAD, HD), "<f2").copy_(_cross_kv(case, g, seed))
        s["prompt"] = _prompt(case, seed)
        e.capture(b, t)
        # positions past the last step hold nothing
        cache = (g.dec_layers, b, g.nh, MAX_T, HD)
        s["out"] = {"logits": _view(e, L.BUF_LOGITS, (b, g.vocab), "<f4"),
                    "residual": _view(e, L.BUF_DEC_X, (b, g.d), "<f4"),
                    "keys": _view(e, L.BUF_SELF_K, cache, "<f2")[:, :, :, :t],
                    "values": _view(e, L.BUF_SELF_V, cache, "<f2")[:, :, :, :t],
                    "align": _view(e, L.BUF_ALIGN, (b, MAX_T, na, TENC), "<f4")[:, :t]}
    else:
        s["w"], rc, cols = _alignment(case, seed)
        s["rows"], s["cols"] = np.array(rc, np.int32), np.array(cols, np.int32)
    torch.cuda.synchronize()  # the library works on its own stream
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "mel":
        L.check(L.lib().mz_log_mel(s["ctx"].h, s["audio"].data_ptr(), s["ns"].ctypes.data_as(C.c_void_p),
                                   case["clips"], case["mels"], s["mel"].data_ptr(),
                                   s["frames"].ctypes.data_as(C.c_void_p)))
        return {"mel": s["mel"], "frames": s["frames"]}
    if kind == "encode":
        s["engine"].encode_device(s["mel"].data_ptr(), case["clips"])
        return s["out"]
    if kind == "decode":
        e = s["engine"]
        e.reset(s["prompt"])
        for _ in range(case["steps"]):
            e.replay()
        return s["out"]
    fn = transcribe.jump_times_device_noalloc if case["scratch"] == "static" else transcribe.jump_times_device
    return fn(s["ctx"], s["w"].data_ptr(), case["rows"] * case["heads"] * TENC, s["rows"], s["cols"], case["heads"],
              TENC, 7, case["half"])


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "mel":
        ns = _ragged(case["clips"], min(NSAMP, int(16000 * case["seconds"])), 400)
        frames = sum(min(NFR, -(-(k + 200) // 160)) for k in ns)
        # a real transform of 400 points by the fast algorithm, the power, the (sparse) filters
        return {"bytes": 4 * sum(ns) + 4 * case["clips"] * case["mels"] * NFR,
                "flops": frames * (2.5 * 400 * math.log2(400) + 3 * 201 + 2 * 2 * 201)}
    if kind == "times":
        rc = _ragged(case["clips"], case["rows"], 1)
        cols = _ragged(case["clips"], TENC, 50)
        cells = sum(r * c for r, c in zip(rc, cols))
        return {"bytes": 4 * (cells * case["heads"] + sum(rc)), "flops": cells * (case["heads"] * (5 + 13) + 4)}
    g = _geometry(case)
    d, ff = g.d, g.ff
    if kind == "encode":
        n, m = case["clips"], case["clips"] * TENC
        layer = 2.0 * m * (3 * d * d + d * d + 2 * d * ff) + 4.0 * n * g.nh * TENC * TENC * HD
        flops = 2.0 * 2 * m * d * 3 * g.n_mels + 2.0 * m * d * 3 * d + g.enc_layers * layer + 2.0 * m * g.dec_layers * 2 * d * d
        weights = d * 3 * g.n_mels + 3 * d * d + g.enc_layers * (4 * d * d + 2 * d * ff) + g.dec_layers * 2 * d * d
        out = m * d * (2 + 4) + m * g.dec_layers * 2 * d * 2
        return {"bytes": 2 * weights + 4 * n * g.n_mels * NFR + TENC * d * 2 + out, "flops": flops}
    b, t, nl = case["rows"], case["steps"], g.dec_layers
    weights = nl * (6 * d * d + 2 * d * ff) + g.vocab * d
    step = 2 * weights + 2 * b * nl * 2 * TENC * d + 4 * b * g.vocab + 6 * b * len(_align_heads(g)) * TENC
    cache = 2 * b * nl * 2 * d * (t * (t + 1) // 2)
    return {"bytes": t * step + cache, "flops": t * 2.0 * b * (weights + nl * 2 * TENC * d)}


def tolerance(case):
    if case["kind"] == "mel":
        return {"rel": 4e-7}  # fp32 sums and log10: about four times 9e-8, the distance from 64 bits
    if case["kind"] == "times":
        return "exact"  # the path through the table is a choice, made from values defined bit for bit
    if case["kind"] == "encode":
        return {"rel": 2e-3}  # fp16 operands and outputs through two to four layers: 4.4e-4 from 64 bits
    return {"rel": 2e-3}  # fp16 operands through up to four layers and the head: 5.2e-4 from 64 bits


# ---------------------------------------------------------------- the same in 64 bits, in plain torch


def _slaney(n_mels):
    def to_hz(m):
        return np.where(m >= 15.0, 1000.0 * np.exp(math.log(6.4) / 27.0 * (m - 15.0)), 200.0 * m / 3.0)
    top = 15.0 + math.log(8000.0 / 1000.0) * 27.0 / math.log(6.4)
    edge = to_hz(np.linspace(0.0, top, n_mels + 2))
    f = np.linspace(0.0, 8000.0, 201)
    up = (f[:, None] - edge[None, :-2]) / (edge[1:-1] - edge[:-2])
    down = (edge[None, 2:] - f[:, None]) / (edge[2:] - edge[1:-1])
    return torch.from_numpy(np.maximum(0.0, np.minimum(up, down)) * 2.0 / (edge[2:] - edge[:-2])).cuda()


def _exact_mel(case, seed):
    y, ns = _audio(case, seed)
    filt = _slaney(case["mels"])
    k = torch.arange(201, device="cuda", dtype=torch.float64)
    j = torch.arange(400, device="cuda", dtype=torch.float64)
    win = 0.5 - 0.5 * torch.cos(2 * math.pi * j / 400)
    arg = 2 * math.pi * torch.remainder(j[:, None] * k[None, :], 400.0) / 400
    cb, sb = win[:, None] * torch.cos(arg), win[:, None] * torch.sin(arg)
    out = torch.empty((case["clips"], case["mels"], NFR), device="cuda", dtype=torch.float64)
    for i in range(case["clips"]):
        p = y[i].double()
        p = torch.cat([p[1:201].flip(0), p, p[-201:-1].flip(0)])
        f = p.unfold(0, 400, 160)[:NFR].contiguous()
        power = (f @ cb) ** 2 + (f @ sb) ** 2
        v = torch.log10(torch.clamp((power @ filt).T, min=1e-10))
        out[i] = (torch.maximum(v, v.max() - 8.0) + 4.0) / 4.0
    return {"mel": out, "frames": np.array([min(NFR, -(-k // 160)) for k in ns], np.int32)}


def _norm(x, w, p):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w[p + ".weight"], w[p + ".bias"], 1e-5)


def _lin(x, w, p, bias=True):
    y = x @ w[p + ".weight"].T
    return y + w[p + ".bias"] if bias else y


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _heads(x, nh):
    return x.reshape(*x.shape[:-1], nh, HD).transpose(-2, -3).contiguous()


def _exact_encode(case, seed):
    g = _geometry(case)
    w = {k: v.double() for k, v in _weights(g, seed).items()}
    mel = _mel_input(case, seed).double()
    n, nh = case["clips"], g.nh
    enc = torch.empty((n, TENC, g.d), device="cuda", dtype=torch.float64)
    res = torch.empty_like(enc)
    cross = torch.zeros((n, g.dec_layers, 2, nh, TPAD, HD), device="cuda", dtype=torch.float64)

    def conv(x, p, stride):  # x [time][channels], kernel 3, padding 1
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1)).unfold(0, 3, stride)  # [t][ci][3]
        wt = w[p + ".weight"]
        return _gelu(xp.reshape(xp.shape[0], -1) @ wt.reshape(wt.shape[0], -1).T + w[p + ".bias"])

    for i in range(n):
        x = conv(conv(mel[i].T.contiguous(), "model.encoder.conv1", 1), "model.encoder.conv2", 2)
        x = x + w["model.encoder.embed_positions.weight"]
        for l in range(g.enc_layers):
            p = "model.encoder.layers.%d" % l
            h = _norm(x, w, p + ".self_attn_layer_norm")
            q = _heads(_lin(h, w, p + ".self_attn.q_proj"), nh) / 8.0
            k = _heads(_lin(h, w, p + ".self_attn.k_proj", False), nh)
            v = _heads(_lin(h, w, p + ".self_attn.v_proj"), nh)
            a = torch.softmax(q @ k.transpose(-1, -2).contiguous(), -1) @ v
            x = x + _lin(a.transpose(0, 1).reshape(TENC, g.d), w, p + ".self_attn.out_proj")
            h = _norm(x, w, p + ".final_layer_norm")
            x = x + _lin(_gelu(_lin(h, w, p + ".fc1")), w, p + ".fc2")
        res[i] = x
        enc[i] = h = _norm(x, w, "model.encoder.layer_norm")
        for l in range(g.dec_layers):
            p = "model.decoder.layers.%d.encoder_attn" % l
            cross[i, l, 0, :, :TENC] = _heads(_lin(h, w, p + ".k_proj", False), nh)
            cross[i, l, 1, :, :TENC] = _heads(_lin(h, w, p + ".v_proj"), nh)
    return {"encoded": enc, "residual": res, "cross": cross}


def _exact_decode(case, seed):
    g = _geometry(case)
    w = {k: v.double() for k, v in _weights(g, seed).items() if k.startswith("model.decoder")}
    kv = _cross_kv(case, g, seed)
    b, t, nh, nl = case["rows"], case["steps"], g.nh, g.dec_layers
    tok = torch.from_numpy(_prompt(case, seed)).cuda()
    x = w["model.decoder.embed_tokens.weight"][tok] + w["model.decoder.embed_positions.weight"][:t]
    heads = _align_heads(g)
    keys = torch.empty((nl, b, nh, t, HD), device="cuda", dtype=torch.float64)
    values, align = torch.empty_like(keys), torch.empty((b, t, len(heads), TENC), device="cuda", dtype=torch.float64)
    causal = torch.full((t, t), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    for l in range(nl):
        p = "model.decoder.layers.%d" % l
        h = _norm(x, w, p + ".self_attn_layer_norm")
        q = _heads(_lin(h, w, p + ".self_attn.q_proj"), nh) / 8.0
        k = keys[l] = _heads(_lin(h, w, p + ".self_attn.k_proj", False), nh)
        v = values[l] = _heads(_lin(h, w, p + ".self_attn.v_proj"), nh)
        a = torch.softmax(q @ k.transpose(-1, -2).contiguous() + causal, -1) @ v
        x = x + _lin(a.transpose(1, 2).reshape(b, t, g.d), w, p + ".self_attn.out_proj")
        h = _norm(x, w, p + ".encoder_attn_layer_norm")
        q = _heads(_lin(h, w, p + ".encoder_attn.q_proj"), nh) / 8.0
        a = torch.empty_like(q)
        for i in range(b):
            pr = torch.softmax(q[i] @ kv[i, l, 0, :, :TENC].double().transpose(-1, -2).contiguous(), -1)
            a[i] = pr @ kv[i, l, 1, :, :TENC].double()
            for s, (la, ha) in enumerate(heads):
                if la == l:
                    align[i, :, s] = pr[ha]
        x = x + _lin(a.transpose(1, 2).reshape(b, t, g.d), w, p + ".encoder_attn.out_proj")
        h = _norm(x, w, p + ".final_layer_norm")
        x = x + _lin(_gelu(_lin(h, w, p + ".fc1")), w, p + ".fc2")
    x = x[:, -1]
    logits = _norm(x, w, "model.decoder.layer_norm") @ w["model.decoder.embed_tokens.weight"].T
    return {"logits": logits, "residual": x, "keys": keys, "values": values, "align": align}


def _warp(m):
    """First column of each row on the cheapest path through -m (a step goes diagonally, down or right)."""
    R, Q = m.shape
    cost = np.full((R + 1, Q + 1), np.inf)
    move = np.zeros((R + 1, Q + 1), np.int8)
    cost[0, 0] = 0.0
    for d in range(2, R + Q + 1):
        i = np.arange(max(1, d - Q), min(R, d - 1) + 1)
        j = d - i
        c0, c1, c2 = cost[i - 1, j - 1], cost[i - 1, j], cost[i, j - 1]
        a, u = (c0 < c1) & (c0 < c2), (c1 < c0) & (c1 < c2)
        move[i, j] = np.where(a, 0, np.where(u, 1, 2))
        cost[i, j] = np.where(a, c0, np.where(u, c1, c2)) - m[i - 1, j - 1]
    first, i, j = np.zeros(R), R, Q
    while i > 0 and j > 0:
        first[i - 1] = j - 1
        k = move[i, j]
        i, j = i - (k != 2), j - (k != 1)
    return first * 0.02


def _exact_times(case, seed):
    w, rc, cols = _alignment(case, seed)
    out = []
    for c in range(case["clips"]):
        x = w[c, :rc[c], :, :cols[c]].double()
        z = (x - x.mean(0)) / x.std(0, unbiased=False)
        z = torch.where(torch.isfinite(z), z, torch.zeros_like(z))
        z = torch.nn.functional.pad(z, (3, 3), mode="reflect").unfold(-1, 7, 1).median(-1).values
        out.append(_warp(z.mean(1).cpu().numpy()))
    return out


def exact(case, seed):
    return {"mel": _exact_mel, "encode": _exact_encode, "decode": _exact_decode, "times": _exact_times}[case["kind"]](
        case, seed)
