"""The calls a synthesis makes into this library, as cases to time and compare.

Nine kinds, each one pass of the stage a TTS program runs on the GPU between
its matrix products, called through the Python binding (synth_hip):

  decode     one token of one stream through 28 talker layers with the
             KV-cache write and the attention softmax, as the captured HIP
             graph a serving loop replays token after token
  layer      layer_nongemm_step: a Qwen3 layer's norms, QK-norm + rope, SwiGLU
             and adds; up to 64 positions (concurrent decode streams) as a
             captured graph of 28 chained layers, a prefill as one call
  probs      the attention softmax of a prefill, over a mask tensor (talker)
             or with the causal mask built in (codec encoder)
  embed      a prefill's input: the text rows from the vocabulary table, the
             codebook rows of every frame summed, the run added into the text
             stream at a position
  vits       a time-major vocoder stage: the transposed convolution's
             scatter-back and bias, then a resblock step (leaky, im2col, and
             the convolution's transposing tail with bias, residual and leaky)
  codec      the neural codec's decoder: a ConvNeXt norm/affine/GELU on the
             latent frames, then a channel-major convolution block (SnakeBeta,
             im2col from the transposed view, transposing tail)
  generator  Kokoro's last generator stage: AdaIN over time, Snake and the
             inverse short-time transform to the waveform
  source     Kokoro's harmonic source and its short-time spectrum
  speaker    the speaker encoder's two ends: log-mel of the reference clip and
             the attentive statistics pooling over its frames
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "synthesize.cpp_amd"))

import synth_hip as S  # noqa: E402

EPS, THETA, HD, HEADS, KV = 1e-6, 1e6, 128, 16, 8
LAYERS = 28          # talker layers
RATE = 24000         # samples per second, everywhere
VARIANCE_FLOOR = 1e-12


def listed():
    return [
        # the serving loop's latency: one stream, one token at position 37
        dict(name="decode_1", kind="decode", keys=38),
        # 64 concurrent decode streams, batched into each layer's step
        dict(name="layers_64_streams", kind="layer", tokens=64, hidden=1024, gain="bf16"),
        # an ordinary prompt of the 0.6B talker, of no round length
        dict(name="layer_prefill_509", kind="layer", tokens=509, hidden=1024, gain="bf16"),
        # the longest prompt, 1.7B talker
        dict(name="layer_prefill_8192", kind="layer", tokens=8192, hidden=2048, gain="bf16"),
        # the scores of a 1021-position prompt: rows of odd length
        dict(name="softmax_prefill_1021", kind="probs", tokens=1021, past=0, heads=16, mask="tensor"),
        # 4096 frames of 16 codebooks at Q8_0
        dict(name="embed_q8_0_4096", kind="embed", frames=4096, groups=16, table="q8_0", hidden=1024, text=512),
        # the first vocoder stage of a short sentence: small and ragged
        dict(name="vits_stage_small", kind="vits", channels=256, columns=517, up=8, kernel=3, dilation=1),
        # the last stage of a long one
        dict(name="vits_stage_large", kind="vits", channels=128, columns=65536, up=2, kernel=3, dilation=1),
        # a codec block of an ordinary sentence
        dict(name="codec_block", kind="codec", channels=256, length=31999, latent=1000, kernel=7, dilation=3),
        # five seconds of speech out of Kokoro's generator
        dict(name="kokoro_generator_5s", kind="generator", frames=24001, channels=128),
        # ... and its harmonic source, 400 f0 frames
        dict(name="kokoro_source_5s", kind="source", f0_frames=400),
        # a ten-second reference clip
        dict(name="speaker_10s", kind="speaker", samples=240000, channels=1536),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "layer", "probs", "embed", "vits", "codec", "generator", "source", "speaker"])
    if kind == "decode":
        return dict(kind=kind, keys=_log(rng, 2, 4096))
    if kind == "layer":
        tokens = _log(rng, 1, 8000)
        return dict(kind=kind, tokens=tokens, hidden=rng.choice([1024, 2048]) if tokens > 64 else 1024,
                    gain=rng.choice(["bf16", "bf16", "f32", "f16"]))
    if kind == "probs":
        tokens = _log(rng, 16, 2000)
        return dict(kind=kind, tokens=tokens, past=rng.choice([0, 0, rng.randrange(1, 600)]), heads=rng.choice([8, 16]),
                    mask=rng.choice(["tensor", "causal"]))
    if kind == "embed":
        return dict(kind=kind, frames=_log(rng, 1, 4096), groups=rng.choice([15, 16]),
                    table=rng.choice(["q8_0", "q5_k", "bf16", "f16"]), hidden=rng.choice([1024, 2048]),
                    text=_log(rng, 4, 1024))
    if kind in ("vits", "codec"):
        channels = rng.choice([64, 96, 128, 192, 256, 512])
        kernel, dilation = rng.choice([3, 3, 7, 11]), rng.choice([1, 3, 5])
        length = _log(rng, 600, (3 << 24) // (kernel * channels))
        if kind == "codec":
            return dict(kind=kind, channels=channels, length=length, latent=_log(rng, 16, 4000), kernel=kernel,
                        dilation=dilation)
        up = rng.choice([2, 4, 8])
        return dict(kind=kind, channels=channels, columns=max(length // up, 16), up=up, kernel=kernel, dilation=dilation)
    if kind == "generator":
        return dict(kind=kind, frames=_log(rng, 1200, 24000), channels=rng.choice([64, 128, 256]))
    if kind == "source":
        return dict(kind=kind, f0_frames=_log(rng, 20, 1600))
    return dict(kind=kind, samples=_log(rng, 12000, 240000), channels=rng.choice([512, 1536]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def randn(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)

    def rand(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda", dtype=torch.float32) * (hi - lo) + lo

    def ids(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def gain(self, n, kind="bf16"):
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
        return (1.0 + 0.1 * self.randn(n)).to(dt)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)


def _empty(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _captured(step):
    """`step` as a HIP graph (run once before the capture, as a program's warm-up does)."""
    step()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            step()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    return graph


def _decode_inputs(c, d):
    n, keys = LAYERS, c["keys"]
    return dict(x=d.randn(1, 1024), q=d.randn(n, 1, HEADS, HD), k=d.randn(n, 1, KV, HD), v=d.randn(n, 1, KV, HD),
                scores=d.randn(n, HEADS, 1, keys) * 8, attn=d.randn(n, 1, 1024), gate=d.randn(n, 1, 3072),
                up=d.randn(n, 1, 3072), mlp=d.randn(n, 1, 1024), w_in=[d.gain(1024) for _ in range(n)],
                w_post=[d.gain(1024) for _ in range(n)], wq=[d.gain(HD) for _ in range(n)],
                wk=[d.gain(HD) for _ in range(n)], kcache=d.randn(n, keys, KV, HD), vcache=d.randn(n, keys, KV, HD),
                pos=torch.full((1,), keys - 1, dtype=torch.int32, device="cuda"),
                slot=torch.full((1,), keys - 1, dtype=torch.int32, device="cuda"))


def _decode(c, d):
    i, n = _decode_inputs(c, d), LAYERS
    o = dict(resid_in=_empty(n, 1, 1024), normed=_empty(n, 1, 1024), q=_empty(n, 1, HEADS, HD),
             probs=_empty(n, HEADS, 1, c["keys"]), resid=_empty(n, 1, 1024), mlp_in=_empty(n, 1, 1024),
             act=_empty(n, 1, 3072), kcache=i["kcache"], vcache=i["vcache"], status=torch.zeros(1, dtype=torch.int32,
                                                                                              device="cuda"))

    def step():
        x, y = i["x"], i["x"]
        for l in range(n):
            # the layer below's output add and this layer's input norm
            S.add_rms_norm_mul(x, y, i["w_in"][l], EPS, out=o["normed"][l], sum_out=o["resid_in"][l])
            S.qk_norm_rope_kv_at(i["q"][l], i["k"][l], i["v"][l], i["wq"][l], i["wk"][l], EPS, i["pos"], HD, THETA,
                                 i["kcache"][l], i["vcache"][l], i["slot"], o["status"], q_out=o["q"][l])
            S.soft_max_ext(i["scores"][l], None, HD ** -0.5, out=o["probs"][l])
            S.add_rms_norm_mul(o["resid_in"][l], i["attn"][l], i["w_post"][l], EPS, out=o["mlp_in"][l],
                               sum_out=o["resid"][l])
            S.swiglu(i["gate"][l], i["up"][l], out=o["act"][l])
            x, y = o["resid"][l], i["mlp"][l]
    return dict(graph=_captured(step), outputs=o, inputs=i)


def _layer_inputs(c, d):
    t, h, ffn = c["tokens"], c["hidden"], 3 * c["hidden"]
    n = LAYERS if t <= 64 else 1
    # decode streams stand at unlike positions, a prefill at consecutive ones
    pos = d.ids(8192, t) if n > 1 else torch.arange(t, dtype=torch.int32, device="cuda")
    return dict(x=d.randn(t, h), pos=pos, layers=[dict(
        w_in=d.gain(h, c["gain"]), q=d.randn(t, HEADS, HD), k=d.randn(t, KV, HD), wq=d.gain(HD, c["gain"]),
        wk=d.gain(HD, c["gain"]), attn_out=d.randn(t, h), w_post=d.gain(h, c["gain"]), gate=d.randn(t, ffn),
        up=d.randn(t, ffn), mlp_out=d.randn(t, h)) for _ in range(n)])


def _layer(c, d):
    i = _layer_inputs(c, d)
    t, h, n = c["tokens"], c["hidden"], len(i["layers"])
    o = dict(normed=_empty(n, t, h), q_out=_empty(n, t, HEADS, HD), k_out=_empty(n, t, KV, HD), resid=_empty(n, t, h),
             mlp_in=_empty(n, t, h), act=_empty(n, t, 3 * h), out=_empty(n, t, h))
    outs = [{k: v[l] for k, v in o.items()} for l in range(n)]

    def step():
        x = i["x"]
        for a, out in zip(i["layers"], outs):
            S.layer_nongemm_step(x, pos=i["pos"], eps=EPS, n_dims=HD, freq_base=THETA, outs=out, **a)
            x = out["out"]
    return dict(graph=_captured(step) if n > 1 else None, step=step, outputs=o, inputs=i)


def _probs(c, d):
    keys = c["tokens"] + c["past"]
    s = dict(scores=d.randn(c["heads"], c["tokens"], keys) * 8, past=c["past"], mask=None,
             out=_empty(c["heads"], c["tokens"], keys))
    if c["mask"] == "tensor":
        hidden = torch.ones(c["tokens"], keys, dtype=torch.bool, device="cuda").triu(c["past"] + 1)
        s["mask"] = torch.zeros(c["tokens"], keys, device="cuda").masked_fill_(hidden, -math.inf)
    return s


TABLE_ROWS, VOCAB, TEXT_HIDDEN = 2048, 151936, 2048


def _table(c, d):
    h, n = c["hidden"], c["groups"] * TABLE_ROWS
    if c["table"] == "q8_0":
        raw = d.bytes(n, h // 32, 34)
        raw[:, :, 0:2] = d.rand(1e-3, 1e-2, n, h // 32).to(torch.float16).view(torch.uint8).view(n, h // 32, 2)
        return raw.view(c["groups"], TABLE_ROWS, -1)
    if c["table"] == "q5_k":
        raw = d.bytes(n, h // 256, 176)
        raw[:, :, 0:4] = d.rand(1e-4, 1e-3, n, h // 256, 2).to(torch.float16).view(torch.uint8).view(n, h // 256, 4)
        return raw.view(c["groups"], TABLE_ROWS, -1)
    return (0.02 * d.randn(c["groups"], TABLE_ROWS, h)).to(torch.bfloat16 if c["table"] == "bf16" else torch.float16)


def _embed(c, d):
    wrap = {"q8_0": lambda r: S.Q8Tensor(r, c["hidden"]), "q5_k": lambda r: S.Q5KTensor(r, c["hidden"])}
    raw = _table(c, d)
    vocab = torch.empty(VOCAB, TEXT_HIDDEN, dtype=torch.bfloat16, device="cuda").normal_(0, 0.02, generator=d.g)
    return dict(raw=raw, tables=[wrap.get(c["table"], lambda r: r)(raw[g]) for g in range(c["groups"])], vocab=vocab,
                text_ids=d.ids(VOCAB, c["text"]), codes=d.ids(TABLE_ROWS, c["groups"], c["frames"]),
                stream=d.randn(c["frames"] + 16, c["hidden"]))


def _vits(c, d):
    ch, l, s = c["channels"], c["columns"], c["up"]
    t = l * s
    return dict(cols=d.randn(l, 2 * s * ch), up=s, ch=ch, up_bias=d.randn(ch, 1), kernel=c["kernel"],
                dilation=c["dilation"], conv=d.randn(t, ch), conv_bias=d.randn(ch, 1))


def _codec(c, d):
    ch, t, latent = c["channels"], c["length"], c["latent"]
    return dict(latent=d.randn(latent, 1024), ln_w=1 + 0.1 * d.randn(1024), ln_b=0.1 * d.randn(1024),
                x=d.randn(t, ch), la=d.rand(-1.0, 1.0, ch), lb=d.rand(-1.0, 1.0, ch), kernel=c["kernel"],
                dilation=c["dilation"], conv=d.randn(ch, t), bias=d.randn(ch))


def _generator(c, d):
    ch, t = c["channels"], c["frames"]
    return dict(x=d.randn(t, ch) * 2 + 0.5, gamma=1 + 0.3 * d.randn(ch, 1), beta=0.3 * d.randn(ch, 1),
                alpha=torch.exp(d.rand(math.log(0.1), math.log(10.0), ch)), spectrum=d.rand(-3.0, 2.0, t, 22))


SOURCE = dict(rate=RATE, scale=300, sine_amp=0.1, noise_std=0.003, voiced_threshold=10.0, n_fft=20, hop=5)


def _source(c, d):
    n, h = c["f0_frames"], 9
    f0 = d.rand(60.0, 360.0, n)
    f0[d.rand(0.0, 1.0, n) < 0.2] = 0.0  # unvoiced frames
    return dict(f0=f0, weight=d.randn(h) * 0.5, bias=0.1, initial=d.rand(0.0, 1.0, h), noise=d.randn(n * 300, h))


def _speaker(c, d):
    frames = 1 + (c["samples"] + 768 - 1024) // 256
    bank = torch.from_numpy(S.mel_filterbank(RATE, 1024, 128, 0.0, 12000.0)).cuda()
    return dict(pcm=0.2 * d.randn(c["samples"]), bank=bank, features=d.randn(frames, c["channels"]),
                logits=3 * d.randn(frames, c["channels"]))


_PREPARE = dict(decode=_decode, layer=_layer, probs=_probs, embed=_embed, vits=_vits, codec=_codec,
                generator=_generator, source=_source, speaker=_speaker)


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, _Draws(seed))
    s["kind"] = case["kind"]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _run_embed(s):
    total = S.get_rows_sum(s["tables"], s["codes"])
    n, row = s["stream"].shape[0], s["stream"].shape[1] * 4
    return dict(text=S.get_rows(s["vocab"], s["text_ids"]), first=S.get_rows(s["tables"][0], s["codes"][0]),
                input=S.acc(s["stream"], total, row, row * n, row * n, 16 * row), total=total)


def _run_vits(s):
    x = S.col2im_1d(s["cols"], s["up"], s["ch"], padding=s["up"] // 2)
    x = S.add(x, s["up_bias"])
    d, k = s["dilation"], s["kernel"]
    columns = S.im2col(S.leaky_relu(x, 0.1), k, 1, d * (k - 1) // 2, d)
    total = torch.empty_like(x)
    y = S.cont_add_leaky_relu(s["conv"].t(), s["conv_bias"], x, 0.1, sum_out=total)
    return dict(x=x, columns=columns, sum=total, y=y)


def _run_codec(s):
    z = S.gelu_erf(S.add(S.mul(S.norm(s["latent"], EPS), s["ln_w"]), s["ln_b"]))
    a = S.snake_beta(s["x"], s["la"], s["lb"])
    d, k = s["dilation"], s["kernel"]
    columns = S.im2col(a.t(), k, 1, d * (k - 1), d)  # left padding; the causal crop follows the product
    return dict(z=z, columns=columns, y=S.cont_add_leaky_relu(s["conv"].t(), s["bias"]))


def _run_generator(s):
    n = S.norm(S.cpy(s["x"].t()), 1e-5)
    a = S.add(S.mul(n, s["gamma"]), s["beta"])
    return dict(y=S.snake(S.cpy(a.t()), s["alpha"]), audio=S.inverse_stft(s["spectrum"], 20, 5))


def _run_source(s):
    exc, har = S.harmonic_source(s["f0"], s["weight"], s["bias"], s["initial"], s["noise"], **SOURCE)
    return dict(excitation=exc, spectrum=har)


def _deviation(x, mean, attention):
    v = S.sqr(S.sub(x, mean))
    v = S.mean(v) if attention is None else S.mul_sum_rows(v, attention)
    return S.sqrt(S.clamp(v, VARIANCE_FLOOR, math.inf))


def _run_speaker(s):
    mel = S.log_mel(s["pcm"], s["bank"], 1024, 256, 1024)
    x = S.cpy(s["features"].t())
    mean = S.mean(x)
    attention = S.soft_max_ext(S.cpy(s["logits"].t()), None, 1.0)
    wmean = S.mul_sum_rows(x, attention)
    return dict(mel=mel, mean=mean, deviation=_deviation(x, mean, None), wmean=wmean,
                wdeviation=_deviation(x, wmean, attention))


def run(s):
    kind = s["kind"]
    if kind in ("decode", "layer"):
        if s["graph"] is not None:
            s["graph"].replay()
        else:
            s["step"]()
        return s["outputs"]
    if kind == "probs":
        if s["mask"] is not None:
            return S.soft_max_ext(s["scores"], s["mask"], HD ** -0.5, out=s["out"])
        return S.soft_max_causal(s["scores"], s["past"], HD ** -0.5, out=s["out"])
    return dict(embed=_run_embed, vits=_run_vits, codec=_run_codec, generator=_run_generator, source=_run_source,
                speaker=_run_speaker)[kind](s)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Every input read once and every output written once; the flops are the
    transforms' and reductions' f64/f32 operations, nowhere the bound at the
    rates of a product."""
    c, f = case, 4
    kind = c["kind"]
    flops = 0.0
    if kind == "decode":
        # x, q, k, v, scores, attn, gate, up, mlp in; six activations, the cache rows and the probabilities out
        n = LAYERS * (1024 * 2 + 4 * KV * HD + 2 * HEADS * HD + 2 * HEADS * c["keys"] + 3 * 3072 + 4 * 1024)
        b = n * f + LAYERS * 2 * (2 * 1024 + 2 * HD)
    elif kind == "layer":
        t, h = c["tokens"], c["hidden"]
        layers = LAYERS if t <= 64 else 1
        g = 4 if c["gain"] == "f32" else 2
        b = layers * (t * f * (2 * (HEADS + KV) * HD + 3 * 3 * h + 6 * h) + g * (2 * h + 2 * HD)) + t * f * (h + 1)
    elif kind == "probs":
        keys = c["tokens"] + c["past"]
        n = c["heads"] * c["tokens"] * keys
        b = f * (2 * n + (c["tokens"] * keys if c["mask"] == "tensor" else 0))
        flops = 8.0 * n
    elif kind == "embed":
        h, t = c["hidden"], c["frames"]
        row = {"q8_0": h // 32 * 34, "q5_k": h // 256 * 176}.get(c["table"], 2 * h)
        # no table row needs reading twice
        rows = min(t, TABLE_ROWS) * c["groups"]
        b = rows * row + t * (c["groups"] + 1) * f + c["text"] * (f + TEXT_HIDDEN * 6) + 2 * t * h * f + \
            2 * (t + 16) * h * f
    elif kind == "vits":
        t = c["columns"] * c["up"]
        # the columns, the product in; x, the column matrix, the sum and y out
        b = f * c["channels"] * t * (2 + 1 + 1 + c["kernel"] + 2)
    elif kind == "codec":
        n, t = c["channels"], c["length"]
        b = f * (2 * c["latent"] * 1024 + n * (t + (t + c["dilation"] * (c["kernel"] - 1)) * c["kernel"] + 2 * t))
    elif kind == "generator":
        t = c["frames"]
        b = f * (2 * t * c["channels"] + t * 22 + (t - 1) * 5)
        flops = t * 5 * 4 * (4.0 * 11)
    elif kind == "source":
        u = c["f0_frames"] * 300
        b = f * (c["f0_frames"] + u * 9 + u + (u // 5 + 1) * 22)
        flops = (u // 5 + 1) * 11 * 20 * 4.0 + u * 9 * 10.0
    else:
        frames = 1 + (c["samples"] + 768 - 1024) // 256
        b = f * (c["samples"] + frames * 128 + 2 * frames * c["channels"] + 4 * c["channels"])
        flops = frames * (512 * 10 * 10.0 + 2 * 513 * 2) + 12.0 * frames * c["channels"]
    return {"bytes": float(b), "flops": float(flops)}


def tolerance(case):
    """Four times the largest distance from exact() seen over the ranges of draw()."""
    kind = case["kind"]
    if kind == "embed":
        return "exact"  # conversions, and f32 sums in group order
    if kind == "source":
        # 2e-5 without them; the first and the last frame are their own mirror image, so their bins' imaginary parts
        # are rounding noise, and a negative real part's phase is +pi or -pi by its sign: two such turns
        values = (case["f0_frames"] * 300 // 5 + 1) * 22
        return {"rel": 2e-5 + 2 * 4.6 / math.sqrt(values)}
    return {"rel": {"decode": 5e-7, "layer": 5e-7, "probs": 3e-7, "vits": 2e-7, "codec": 4e-7, "generator": 4e-7,
                    "speaker": 2e-7}[kind]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _rms(x, w):
    x = x.double()
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    """NEOX rope of x (T, heads, 128). The angles are f32 by definition: the
    position times powers of theta_scale, multiplied up in f32."""
    libm = ctypes.CDLL("libm.so.6")
    libm.powf.restype, libm.powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    scale = np.float32(libm.powf(THETA, -2.0 / HD))
    th = np.empty((pos.numel(), HD // 2), np.float32)
    th[:, 0] = pos.cpu().numpy().astype(np.float32)
    for k in range(1, HD // 2):
        th[:, k] = th[:, k - 1] * scale
    th = torch.from_numpy(th).cuda().double()[:, None, :]
    lo, hi = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([lo * th.cos() - hi * th.sin(), lo * th.sin() + hi * th.cos()], -1)


def _exact_decode(c, d):
    i, o = _decode_inputs(c, d), {k: [] for k in ("resid_in", "normed", "q", "probs", "resid", "mlp_in", "act")}
    kc, vc = i["kcache"].double(), i["vcache"].double()
    x = i["x"].double() + i["x"].double()
    for l in range(LAYERS):
        o["resid_in"].append(x)
        o["normed"].append(_rms(x, i["w_in"][l]))
        o["q"].append(_rope(_rms(i["q"][l], i["wq"][l]), i["pos"]))
        kc[l, -1] = _rope(_rms(i["k"][l], i["wk"][l]), i["pos"])[0]
        vc[l, -1] = i["v"][l, 0].double()
        o["probs"].append(torch.softmax(i["scores"][l].double() * HD ** -0.5, -1))
        r = x + i["attn"][l].double()
        o["resid"].append(r)
        o["mlp_in"].append(_rms(r, i["w_post"][l]))
        o["act"].append(F.silu(i["gate"][l].double()) * i["up"][l].double())
        x = r + i["mlp"][l].double()
    return dict({k: torch.stack(v) for k, v in o.items()}, kcache=kc, vcache=vc,
                status=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _exact_layer(c, d):
    i, o = _layer_inputs(c, d), {}
    x = i["x"].double()
    for a in i["layers"]:
        r = x + a["attn_out"].double()
        step = dict(normed=_rms(x, a["w_in"]), q_out=_rope(_rms(a["q"], a["wq"]), i["pos"]),
                    k_out=_rope(_rms(a["k"], a["wk"]), i["pos"]), resid=r, mlp_in=_rms(r, a["w_post"]),
                    act=F.silu(a["gate"].double()) * a["up"].double(), out=r + a["mlp_out"].double())
        for k, v in step.items():
            o.setdefault(k, []).append(v)
        x = step["out"]
    return {k: torch.stack(v) for k, v in o.items()}


def _exact_probs(c, d):
    s = _probs(c, d)
    w = s["scores"].double() * HD ** -0.5
    hidden = torch.ones(w.shape[1:], dtype=torch.bool, device="cuda").triu(c["past"] + 1)
    return torch.softmax(w.masked_fill_(hidden, -math.inf), -1)


def _values(c, raw):
    """A table's rows in 64 bits: (groups * rows, hidden)."""
    h = c["hidden"]
    if c["table"] == "q8_0":
        blk = raw.reshape(-1, h // 32, 34)
        scale = blk[:, :, 0:2].contiguous().view(torch.float16).double()
        return (blk[:, :, 2:].contiguous().view(torch.int8).double() * scale).reshape(-1, h)
    if c["table"] == "q5_k":
        blk = raw.reshape(-1, h // 256, 176)
        scales = blk[:, :, 0:4].contiguous().view(torch.float16).double()
        s, qh, qs = blk[:, :, 4:16].int(), blk[:, :, 16:48].int(), blk[:, :, 48:].reshape(-1, h // 256, 4, 32).int()
        sc = torch.cat([s[:, :, 0:4] & 63, (s[:, :, 8:12] & 15) | (s[:, :, 0:4] >> 6 << 4)], -1)
        m = torch.cat([s[:, :, 4:8] & 63, (s[:, :, 8:12] >> 4) | (s[:, :, 4:8] >> 6 << 4)], -1)
        low = torch.stack([qs & 15, qs >> 4], 3).reshape(-1, h // 256, 8, 32)
        bit = torch.arange(8, device="cuda", dtype=torch.int32)[None, None, :, None]
        q = low + ((qh[:, :, None, :] >> bit & 1) << 4)
        v = (scales[:, :, 0:1] * sc)[..., None] * q - (scales[:, :, 1:2] * m)[..., None]
        return v.reshape(-1, h)
    return raw.reshape(-1, h).double()


def _exact_embed(c, d):
    s = _embed(c, d)
    v = _values(c, s["raw"]).view(c["groups"], TABLE_ROWS, -1)
    first = v[0][s["codes"][0].long()]
    total = torch.zeros_like(first)
    for g in range(c["groups"]):
        total += v[g][s["codes"][g].long()]
    y = s["stream"].double()
    y[16:] += total
    return dict(text=s["vocab"][s["text_ids"].long()].double(), first=first, input=y, total=total)


def _columns(x, k, p, d):
    """x (C, T) -> (T + 2p - d(k-1), C*k)."""
    x = F.pad(x, (p, p))
    n = x.shape[1] - d * (k - 1)
    return torch.stack([x[:, j * d:j * d + n] for j in range(k)], -1).permute(1, 0, 2).reshape(n, -1)


def _exact_vits(c, d):
    s = _vits(c, d)
    ch, l, up, k = s["ch"], c["columns"], s["up"], 2 * s["up"]
    taps = s["cols"].view(l, ch, k).double()
    x = torch.zeros(ch, (l - 1) * up + k, dtype=torch.float64, device="cuda")
    for j in range(k):
        x[:, j:j + (l - 1) * up + 1:up] += taps[:, :, j].t()
    x = x[:, up // 2:up // 2 + l * up] + s["up_bias"].double()
    columns = _columns(F.leaky_relu(x, 0.1), s["kernel"], s["dilation"] * (s["kernel"] - 1) // 2, s["dilation"])
    total = s["conv"].t().double() + s["conv_bias"].double() + x
    return dict(x=x, columns=columns, sum=total, y=F.leaky_relu(total, 0.1))


def _exact_codec(c, d):
    s = _codec(c, d)
    z = s["latent"].double()
    z = z - z.mean(-1, keepdim=True)
    z = z / torch.sqrt(z.square().mean(-1, keepdim=True) + EPS) * s["ln_w"].double() + s["ln_b"].double()
    x = s["x"].double()
    a = x + torch.sin(x * s["la"].double().exp()).square() / (s["lb"].double().exp() + 1e-9)
    columns = _columns(a.t(), s["kernel"], s["dilation"] * (s["kernel"] - 1), s["dilation"])
    return dict(z=F.gelu(z), columns=columns, y=s["conv"].t().double() + s["bias"].double())


def _hann(n):
    return (0.5 * (1.0 - torch.cos(2.0 * math.pi * torch.arange(n, dtype=torch.float64) / n))).float().double().cuda()


def _exact_generator(c, d):
    s = _generator(c, d)
    x = s["x"].double()
    x = x - x.mean(0, keepdim=True)
    x = x / torch.sqrt(x.square().mean(0, keepdim=True) + 1e-5) * s["gamma"].double().t() + s["beta"].double().t()
    al = s["alpha"].double()
    sp = s["spectrum"].double()
    z = torch.polar(sp[:, :11].exp(), sp[:, 11:].sin())
    w, n = _hann(20), c["frames"]
    seg = torch.fft.irfft(z, 20) * w
    audio, env = (torch.zeros((n - 1) * 5 + 20, dtype=torch.float64, device="cuda") for _ in range(2))
    for k in range(0, 20, 5):
        at = slice(k, k + 5 * n)
        audio[at] += seg[:, k:k + 5].reshape(-1)
        env[at] += w.square()[k:k + 5].repeat(n)
    keep = slice(10, 10 + (n - 1) * 5)
    return dict(y=x + torch.sin(al * x).square() / al, audio=audio[keep] / env[keep])


def _resample(out_len, in_len):
    p = np.maximum((np.arange(out_len) + 0.5) * (in_len / out_len) - 0.5, 0.0)
    lo = p.astype(np.int64)
    return lo, np.minimum(lo + 1, in_len - 1), (p - lo).astype(np.float32)[:, None]


def _exact_source(c, d):
    """The phase is f32 by definition up to the sine's argument (a running f32
    sum, some 1e5 radians); the sines, the merge and the transform in 64 bits."""
    s = _source(c, d)
    f0, ri, nz, mw = (s[k].cpu().numpy() for k in ("f0", "initial", "noise", "weight"))
    h, scale, n = mw.size, SOURCE["scale"], f0.size
    u, one = n * scale, np.float32(1)
    up = np.repeat(f0, scale)
    v = up[:, None] * np.arange(1, h + 1, dtype=np.float32) / np.float32(RATE)
    v = v - np.floor(v)
    v[0] += ri
    lo, hi, w = _resample(n, u)
    run = np.cumsum(v[lo] * (one - w) + v[hi] * w, axis=0, dtype=np.float32)
    phase = (run.astype(np.float64) * 2.0 * math.pi * scale).astype(np.float32)
    lo, hi, w = _resample(u, n)
    fine = phase[lo] * (one - w) + phase[hi] * w
    voiced = (up > SOURCE["voiced_threshold"]).astype(np.float64)[:, None]
    amp, std = np.float64(np.float32(SOURCE["sine_amp"])), np.float64(np.float32(SOURCE["noise_std"]))
    value = np.sin(fine.astype(np.float64)) * amp * voiced + (voiced * std + (1 - voiced) * amp / 3) * nz
    exc = np.tanh(np.float64(np.float32(s["bias"])) + value @ mw.astype(np.float64))
    nf, hop = SOURCE["n_fft"], SOURCE["hop"]
    pad = np.pad(exc, nf // 2, mode="reflect")
    seg = np.lib.stride_tricks.sliding_window_view(pad, nf)[::hop] * _hann(nf).cpu().numpy()
    angle = -2.0 * math.pi * np.arange(nf // 2 + 1)[:, None] * np.arange(nf) / nf
    re, im = seg @ np.cos(angle).T, seg @ np.sin(angle).T + 0.0
    return dict(excitation=exc, spectrum=np.concatenate([np.hypot(re, im), np.arctan2(im, re)], -1))


def _slaney(bins, n_fft):
    """librosa's Slaney filterbank from 0 to 12000 Hz, in 64 bits."""
    step, knee = math.log(6.4) / 27.0, 15.0
    top = knee + math.log(12.0) / step
    mel = np.linspace(0.0, top, bins + 2)
    edge = np.where(mel >= knee, 1000.0 * np.exp(step * (mel - knee)), mel * (200.0 / 3.0))[:, None]
    hz = np.arange(n_fft // 2 + 1) * (RATE / n_fft)
    up = (hz - edge[:-2]) / (edge[1:-1] - edge[:-2])
    down = (edge[2:] - hz) / (edge[2:] - edge[1:-1])
    return np.maximum(0.0, np.minimum(up, down)) * 2.0 / (edge[2:] - edge[:-2])


def _exact_speaker(c, d):
    s = _speaker(c, d)
    pcm = F.pad(s["pcm"].double()[None], (384, 384), mode="reflect")[0]
    spec = torch.fft.rfft(pcm.unfold(0, 1024, 256) * _hann(1024))
    mag = torch.sqrt(spec.real.square() + spec.imag.square() + 1e-9)
    mel = torch.log(torch.clamp(mag @ torch.from_numpy(_slaney(128, 1024)).cuda().t(), min=1e-5))
    x = s["features"].double().t()
    att = torch.softmax(s["logits"].double().t(), -1)
    mean, wmean = x.mean(-1, keepdim=True), (x * att).sum(-1, keepdim=True)
    return dict(mel=mel, mean=mean, deviation=(x - mean).square().mean(-1, keepdim=True).clamp(min=VARIANCE_FLOOR).sqrt(),
                wmean=wmean,
                wdeviation=((x - wmean).square() * att).sum(-1, keepdim=True).clamp(min=VARIANCE_FLOOR).sqrt())


def exact(case, seed):
    return dict(decode=_exact_decode, layer=_exact_layer, probs=_exact_probs, embed=_exact_embed, vits=_exact_vits,
                codec=_exact_codec, generator=_exact_generator, source=_exact_source,
                speaker=_exact_speaker)[case["kind"]](case, _Draws(seed))
