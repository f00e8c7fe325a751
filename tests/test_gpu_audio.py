"""GPU parity of the log-mel features (mz_log_mel, k_mel.hip) against the oracle's restatement of the reference's
Mel::features (oracle/audio_ref.py) and transformers' feature extractor (tests/golden/mel_*.npz)."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

from mimizuku_amd import _lib as L
from mimizuku_amd import model
from oracle import audio_ref as A

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
sys.path.insert(0, GOLDEN)
from waves import waveform  # noqa: E402

NS = 480000


@pytest.fixture(scope="module")
def ctx():
    c = model.Context(0)
    yield c
    c.close()


def log_mel(ctx, clips, n_mels, junk_tail=False):
    """Runs mz_log_mel on clips (host float32 arrays); returns features [n][n_mels][3000] and frame counts."""
    n = len(clips)
    buf = np.zeros((n, NS), np.float32)
    rng = np.random.default_rng(9)
    for i, y in enumerate(clips):
        k = min(len(y), NS)
        buf[i, :k] = y[:k]
        if junk_tail and k < NS:
            buf[i, k:] = rng.standard_normal(NS - k)  # past n_samples: must read as zero
    ns = np.array([len(y) for y in clips], np.int32)
    d_audio = ctx.upload_new(buf)
    d_mel = ctx.alloc(n * n_mels * 3000 * 4)
    frames = np.zeros(n, np.int32)
    print(f"mz_log_mel n={n} n_mels={n_mels} lengths={ns.tolist()}", flush=True)
    L.check(L.lib().mz_log_mel(ctx.h, d_audio, ns.ctypes.data_as(C.c_void_p), n, n_mels, d_mel,
                               frames.ctypes.data_as(C.c_void_p)))
    out = ctx.download(d_mel, (n, n_mels, 3000), np.float32)
    ctx.free(d_audio)
    ctx.free(d_mel)
    return out, frames


@pytest.mark.parametrize("n_mels", [80, 128])
def test_log_mel_matches_the_oracle(ctx, n_mels):
    rng = np.random.default_rng(n_mels)
    lengths = [0, 1, 159, 16000 * 7 + 123, NS, NS + 40000]
    clips = [(0.3 * rng.standard_normal(k)).astype(np.float32) for k in lengths]
    got, frames = log_mel(ctx, clips, n_mels, junk_tail=True)
    tables = A.mel_tables(n_mels)
    for i, y in enumerate(clips):
        ref, fr = A.features(y, n_mels, tables)
        assert frames[i] == fr, (i, frames[i], fr)
        err = np.abs(got[i] - ref).max()
        assert err <= 1e-6, (i, lengths[i], err)


def test_log_mel_of_silence_and_a_tone(ctx):
    """features_of_silence_and_frames (src/audio.rs:336-348) on the device."""
    t = np.sin(2 * np.pi * 1000.0 * np.arange(16000) / 16000).astype(np.float32)
    got, frames = log_mel(ctx, [np.zeros(16000, np.float32), t], 80)
    assert frames.tolist() == [100, 100]
    assert np.all(np.abs(got[0] - (-10.0 + 4.0) / 4.0) < 1e-6)
    assert 20 <= int(np.argmax(got[1][:, 50])) < 40


def test_log_mel_matches_transformers(ctx):
    for name in ("mel80_7s", "mel128_30s", "mel128_short"):
        fx = np.load(os.path.join(GOLDEN, f"{name}.npz"))
        y = waveform(int(fx["seed"]), float(fx["seconds"]))
        got, frames = log_mel(ctx, [y], int(fx["n_mels"]))
        assert frames[0] == int(fx["frames"])
        assert np.abs(got[0][:, fx["cols"]] - fx["features"]).max() < 2e-5, name


@pytest.mark.parametrize("n_mels,lengths", [(1, [400, 161]), (40, [16000 * 12 + 77, 2401, 2400]), (256, [NS, 16 * 160, 41 * 160]),
                                            (80, [NS] * 6)])
def test_log_mel_tiles_and_widths(ctx, n_mels, lengths):
    """Frame counts at the borders of the 16- and 32-frame tiles (six full clips take the larger), the fewest and the
    most filters the entry point takes."""
    rng = np.random.default_rng(n_mels + len(lengths))
    clips = [(0.2 * rng.standard_normal(k)).astype(np.float32) for k in lengths]
    got, frames = log_mel(ctx, clips, n_mels)
    tables = A.mel_tables(n_mels)
    for i in sorted({0, len(clips) // 2, len(clips) - 1}):
        ref, fr = A.features(clips[i], n_mels, tables)
        assert frames[i] == fr
        assert np.abs(got[i] - ref).max() <= 1e-6, (i, lengths[i])


def test_log_mel_unaligned_output_and_a_nan_sample(ctx):
    """An output address that is only 4-byte aligned; and a NaN sample, whose frames have no finite power: every filter's
    sum is NaN there, which the floor turns into -10 (before the clamp), and no other frame changes."""
    rng = np.random.default_rng(3)
    y = (0.2 * rng.standard_normal(NS)).astype(np.float32)
    ref, _ = log_mel(ctx, [y], 80)
    z = y.copy()
    z[100000] = np.nan
    d_audio = ctx.upload_new(z[None])
    d_mel = ctx.alloc(80 * 3000 * 4 + 16)
    ns = np.array([NS], np.int32)
    L.check(L.lib().mz_log_mel(ctx.h, d_audio, ns.ctypes.data_as(C.c_void_p), 1, 80, d_mel + 4, None))
    got = ctx.download(d_mel + 4, (80, 3000), np.float32)
    t = np.arange(3000)
    hit = (160 * t - 200 < 100000) & (100000 < 160 * t + 200)  # (the first sample of a frame has weight 0)
    assert np.ptp(got[:, hit]) == 0 and got[0, hit][0] <= ref[0].min()
    edge = (160 * t - 200 <= 100000) & (100000 < 160 * t + 200)
    np.testing.assert_array_equal(got[:, ~edge], ref[0][:, ~edge])
    ctx.free(d_audio)
    ctx.free(d_mel)


def test_scratch_kept_between_calls():
    """Features and timestamps take turns on one context's scratch, in sizes that grow and shrink it, and from two threads
    at once: the same values as on a context of their own."""
    import threading

    from mimizuku_amd import transcribe
    rng = np.random.default_rng(12)
    own = model.Context(0)
    jobs = []
    for n, rows, seconds in ((1, 9, 0.5), (3, 130, 7.0), (2, 300, 2.0), (1, 40, 30.0)):
        w = rng.random((n, rows, 4, 1500), dtype=np.float32)
        clips = [(0.1 * rng.standard_normal(int(16000 * seconds))).astype(np.float32) for _ in range(n)]
        jobs.append((w, clips))

    def do(ctx, job):
        w, clips = job
        n, rows = w.shape[:2]
        dw = ctx.upload_new(w)
        t = transcribe.jump_times_device(ctx, dw, rows * 4 * 1500, [rows - i for i in range(n)], [1500] * n, 4, 1500)
        ctx.free(dw)
        return t, log_mel(ctx, clips, 80)[0]

    ref = []
    for job in jobs:
        c = model.Context(0)
        ref.append(do(c, job))
        c.close()

    def same(a, b):
        for x, y in zip(a[0], b[0]):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a[1], b[1])

    for i in (0, 1, 2, 3, 1, 0):
        same(do(own, jobs[i]), ref[i])
    # two threads, each with a context's timestamps of its own weights at once on one shared context
    dws = [own.upload_new(jobs[i][0]) for i in (1, 2)]
    got = [[], []]

    def times(k):
        w = jobs[k + 1][0]
        n, rows = w.shape[:2]
        for _ in range(5):
            got[k].append(transcribe.jump_times_device(own, dws[k], rows * 4 * 1500, [rows - i for i in range(n)],
                                                       [1500] * n, 4, 1500))

    threads = [threading.Thread(target=times, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in (0, 1):
        assert len(got[k]) == 5
        for g in got[k]:
            for x, y in zip(g, ref[k + 1][0]):
                np.testing.assert_array_equal(x, y)
    own.close()


def test_scratch_beyond_what_is_kept():
    """Calls whose device scratch alone (120 clips: 220 MiB), or whose device and pinned scratch (60000 short clips: 200 MiB
    and 5 MiB), are beyond what a context keeps, with small calls in between: the values of the entry point whose scratch
    is static."""
    from mimizuku_amd import transcribe
    rng = np.random.default_rng(13)
    ctx = model.Context(0)
    for n, rows, full in ((3, 40, 1500), (120, 220, 1500), (3, 40, 1500), (60000, 20, 8), (3, 40, 1500)):
        dw = ctx.upload_new(rng.random((n + rows, full), dtype=np.float32))  # clip c: rows c .. c + rows - 1
        args = (ctx, dw, full, [rows - i % 7 for i in range(n)], [full] * n, 1, full)
        got, ref = transcribe.jump_times_device(*args), transcribe.jump_times_device_noalloc(*args)
        np.testing.assert_array_equal(np.concatenate(got), np.concatenate(ref))
        ctx.free(dw)
    ctx.close()


def test_scratch_of_a_call_within_another():
    """A call that runs while another thread's (8000 clips, about 20 ms) holds the context's scratch: it began
    after that one and before its end, and both give the values they give alone."""
    import threading
    import time

    from mimizuku_amd import transcribe
    rng = np.random.default_rng(14)
    ctx = model.Context(0)
    big, small, full = 8000, 4, 1500
    dw = ctx.upload_new(rng.random((big + 220, full), dtype=np.float32))
    long_args = (ctx, dw, full, [220] * big, [full] * big, 1, full)
    short_args = (ctx, dw, full, [50 + i for i in range(small)], [full] * small, 1, full)
    want = [np.concatenate(transcribe.jump_times_device_noalloc(*a)) for a in (long_args, short_args)]
    within = 0
    for _ in range(5):
        span, got = {}, {}
        gate = threading.Barrier(2)

        def call(name, args, wait):
            gate.wait()
            time.sleep(wait)
            t0 = time.perf_counter()
            got[name] = np.concatenate(transcribe.jump_times_device(*args))
            span[name] = t0, time.perf_counter()

        threads = [threading.Thread(target=call, args=a) for a in (("long", long_args, 0.0), ("short", short_args, 0.008))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        np.testing.assert_array_equal(got["long"], want[0])
        np.testing.assert_array_equal(got["short"], want[1])
        within += span["long"][0] + 0.004 < span["short"][0] < span["long"][1] - 0.004
        print("long %.1f ms, the short one began %.1f ms into it" % (1e3 * (span["long"][1] - span["long"][0]),
                                                                     1e3 * (span["short"][0] - span["long"][0])))
    assert within > 0
    ctx.close()
