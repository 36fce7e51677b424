"""shp_log_mel against the restatement of the Qwen3-TTS speaker encoder's
compute_log_mel (qwen3-tts/mel.cpp:174-299), which equals the reference's
own compiled code bit for bit: one-second and ten-second clips of noise and
tones at the production parameters (n_fft 1024, hop 256, 128 Slaney bins to
12 kHz), hop 512, a shorter zero-padded window with fewer bins, the
shortest clip the reflect pad allows; the upstream frame counts (93, 46).
The FFT is the host code's, stage for stage, with f32 results; the device's
double cos/sin/log move a twiddle or a log in its last bit, so the log
energies are held within 1e-5 and > 99 % identical."""
import numpy as np
import pytest

import ggml_ref as R
from test_gpu_parity import _np, _t
from test_oracle_goldens import MEL, oracle_log_mel

pytestmark = pytest.mark.gpu

SEED = 20261218


def _gpu_mel(gpu, pcm, p):
    fb = gpu.mel_filterbank(p["sample_rate"], p["n_fft"], p["mel_bins"], p["fmin"], p["fmax"])
    return _np(gpu.log_mel(_t(gpu, pcm), _t(gpu, fb), p["n_fft"], p["hop"], p["win_length"]))


def _close(got, ref):
    assert got.shape == ref.shape
    assert np.abs(got - ref).max() <= 1e-5
    assert (got == ref).mean() > 0.99


@pytest.mark.parametrize("kind,seconds,p", [("noise", 1, MEL), ("tone", 1, MEL), ("noise", 10, MEL),
                                            ("tone", 1, dict(MEL, hop=512)),
                                            ("noise", 1, dict(MEL, n_fft=512, win_length=400, hop=160, mel_bins=80)),
                                            ("noise", 1, dict(MEL, n_fft=2048, win_length=2048, hop=512))])
def test_log_mel_matches_restatement(gpu, kind, seconds, p):
    ns = 24000 * seconds
    rng = np.random.default_rng([SEED, ns, p["n_fft"], p["hop"]])
    pcm = (rng.standard_normal(ns) * 0.2).astype(np.float32) if kind == "noise" else \
        (0.4 * np.sin(2 * np.pi * 440 * np.arange(ns) / 24000)).astype(np.float32)
    _close(_gpu_mel(gpu, pcm, p), oracle_log_mel(pcm, p))


def test_log_mel_frame_counts_and_short_clips(gpu):
    """93 frames at hop 256 and 46 at hop 512 for one second (the upstream
    counts); 385 samples are the fewest the reflect pad takes, 384 refused."""
    pcm = np.full(24000, 0.5, np.float32)
    assert _gpu_mel(gpu, pcm, MEL).shape == (93, 128)
    assert _gpu_mel(gpu, pcm, dict(MEL, hop=512)).shape == (46, 128)
    short = (np.random.default_rng(SEED).standard_normal(385) * 0.3).astype(np.float32)
    _close(_gpu_mel(gpu, short, MEL), oracle_log_mel(short, MEL))
    with pytest.raises(gpu.ShpError):
        _gpu_mel(gpu, short[:384], MEL)


def test_log_mel_refusals(gpu):
    import torch
    fb = _t(gpu, gpu.mel_filterbank(24000, 1024, 128, 0.0, 12000.0))
    pcm = torch.zeros(24000, device="cuda")
    with pytest.raises(gpu.ShpError):       # not a power of two
        gpu.log_mel(pcm, _t(gpu, gpu.mel_filterbank(24000, 1000, 128, 0.0, 12000.0)), 1000, 250, 1000)
    with pytest.raises(gpu.ShpError):       # window wider than the transform
        gpu.log_mel(pcm, fb, 1024, 256, 1100)
    with pytest.raises(gpu.ShpError):       # a filterbank of another transform
        gpu.log_mel(pcm, fb, 512, 128, 512)


@pytest.mark.parametrize("n_fft,hop,win,bins,dense", [(2, 1, 2, 3, True), (4, 2, 3, 5, True), (8, 3, 8, 4, True),
                                                      (16, 16, 16, 7, True), (32, 5, 20, 6, True), (64, 16, 64, 513, True),
                                                      (128, 31, 100, 20, False), (256, 64, 256, 1025, True),
                                                      (512, 512, 512, 512, False), (1024, 300, 1000, 40, True),
                                                      (2048, 700, 1500, 128, False)])
def test_log_mel_transform_sizes_and_filterbanks(gpu, n_fft, hop, win, bins, dense):
    """Every pass length of the transform, windows of any width, more bins than
    one span table holds, frame counts that leave a block part empty; filter
    rows of any weights, and rows with zeros inside, at the ends or throughout.
    (Held by the energies, as the production cases: 1e-5 absolute on the log.)"""
    rng = np.random.default_rng([SEED, n_fft, bins])
    nf = n_fft // 2 + 1
    pcm = (rng.standard_normal(5 * n_fft + 3 * hop + 7) * 0.3).astype(np.float32)
    fb = rng.uniform(0.1, 1.0, (bins, nf)).astype(np.float32)
    if not dense:
        fb[rng.random((bins, nf)) < 0.7] = 0.0
        fb[1] = 0.0
        fb[2] = -0.0
        fb[0, -1] = 0.5
    got = _np(gpu.log_mel(_t(gpu, pcm), _t(gpu, fb), n_fft, hop, win))
    ref = R.run(lambda g: g.log_mel(pcm, fb, n_fft, hop, win))
    _close(got, ref)


def test_log_mel_one_sample_frames(gpu):
    """n_fft 1: the periodic window's only value is 0, so every bin is the floor of sqrt(1e-9) times its weight."""
    fb = np.float32([[1.0], [3.0]])
    got = _np(gpu.log_mel(_t(gpu, np.ones(5, np.float32)), _t(gpu, fb), 1, 1, 1))
    amp = np.float32(np.sqrt(1e-9))
    assert np.abs(got - np.log(fb.T.astype(np.float64) * amp)).max() <= 1e-6


@pytest.mark.parametrize("value", [np.inf, np.nan, 3e38])
def test_log_mel_infinite_amplitudes(gpu, value):
    """A sample that is not finite, or whose transform overflows: its frames'
    zero weights multiply an infinity, which the host code's dense sum turns
    into NaN; the other frames are untouched."""
    rng = np.random.default_rng(SEED + 9)
    pcm = (rng.standard_normal(24000) * 0.2).astype(np.float32)
    pcm[9000:9003] = value
    ref, got = oracle_log_mel(pcm, MEL), _gpu_mel(gpu, pcm, MEL)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.isnan(ref).any()
    assert np.array_equal(np.isinf(got), np.isinf(ref))
    ok = np.isfinite(ref)
    _close(got[ok], ref[ok])


@pytest.mark.parametrize("n_fft,hop,bins", [(2, 1, 5), (16, 4, 30), (32, 8, 80), (64, 16, 80), (256, 64, 128), (512, 128, 80),
                                            (1024, 256, 128)])
def test_log_mel_frames_do_not_depend_on_the_clip(gpu, n_fft, hop, bins):
    """A frame's bits are the same alone, in a short clip and in one of thousands
    of frames: a block per frame, one to four waves, one to eight frames each."""
    rng = np.random.default_rng([SEED, n_fft, 3])
    pad = (n_fft - hop) // 2
    pcm = _t(gpu, (rng.standard_normal(hop * 8500 if n_fft <= 64 else 400000) * 0.2).astype(np.float32))
    fb = _t(gpu, gpu.mel_filterbank(24000, n_fft, bins, 0.0, 12000.0))
    long = _np(gpu.log_mel(pcm, fb, n_fft, hop, n_fft))
    for frames in (3, 20, 150, 300, 600, 1200, 2049, 3000):
        ns = frames * hop + n_fft
        if ns > pcm.numel():
            break
        got = _np(gpu.log_mel(pcm[:ns], fb, n_fft, hop, n_fft))
        inside = frames - pad // hop - 1            # frames that the end's reflection does not reach
        assert np.array_equal(got[:inside].view(np.uint32), long[:inside].view(np.uint32)), frames
    ref = R.run(lambda g: g.log_mel(_np(pcm)[:50 * hop + n_fft], _np(fb), n_fft, hop, n_fft))
    _close(long[:49 - pad // hop], ref[:49 - pad // hop])
