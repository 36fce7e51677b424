"""shp_layer_nongemm_step's one launch at the edges of its blocks: one position
to past the decode form's 64, hidden sizes of one to four float4 a lane, head
counts that end inside a block and past what the launch takes (the five
launches then), every gain type, strided rows, and outputs laid over inputs,
where the step keeps the five launches' order. Every output equals the single
entry points' bit for bit (the row sums are double: their order may show only
on an f32 rounding boundary, which these fixed inputs do not meet)."""
import numpy as np
import pytest

from test_gpu_parity import _np, assert_bitexact

pytestmark = pytest.mark.gpu
EPS, THETA = 1e-6, 1e6


def _inputs(T, H, ffn, heads, kv, dtype, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")
    w = lambda n: (1 + 0.1 * r(n)).to(dtype)
    return dict(x=r(T, H), w_in=w(H), q=r(T, heads, 128), k=r(T, kv, 128), wq=w(128), wk=w(128),
                pos=torch.randint(0, 9000, (T,), generator=g, device="cuda", dtype=torch.int32), attn_out=r(T, H),
                w_post=w(H), gate=4 * r(T, ffn), up=r(T, ffn), mlp_out=r(T, H))


def _step(gpu, a, outs=None):
    return gpu.layer_nongemm_step(eps=EPS, n_dims=128, freq_base=THETA, outs=outs, **a)


def _singles(gpu, a):
    q, k = gpu.qk_norm_rope(a["q"], a["k"], a["wq"], a["wk"], EPS, a["pos"], 128, THETA)
    resid, mlp_in = gpu.add_rms_norm_mul(a["x"], a["attn_out"], a["w_post"], EPS)
    return dict(normed=gpu.rms_norm_mul(a["x"], a["w_in"], EPS), q_out=q, k_out=k, resid=resid, mlp_in=mlp_in,
                act=gpu.swiglu(a["gate"], a["up"]), out=gpu.add(resid, a["mlp_out"]))


@pytest.mark.parametrize("T,H,ffn,heads,kv,gain", [
    (1, 4, 4, 1, 1, "float32"), (1, 1024, 3072, 16, 8, "bfloat16"), (3, 1020, 12, 11, 1, "float16"),
    (64, 1024, 1028, 16, 8, "bfloat16"), (65, 1028, 3072, 16, 8, "float32"), (66, 2048, 516, 24, 8, "bfloat16"),
    (130, 2052, 1024, 31, 1, "float16"), (5, 4096, 2048, 16, 16, "bfloat16"), (300, 4096, 8, 5, 3, "float32"),
    (2, 4100, 64, 16, 8, "bfloat16"), (70, 256, 64, 25, 8, "bfloat16")])   # the last two: five launches
def test_one_launch_equals_the_entry_points(gpu, T, H, ffn, heads, kv, gain):
    import torch
    a = _inputs(T, H, ffn, heads, kv, getattr(torch, gain), T + H)
    got, ref = _step(gpu, a), _singles(gpu, a)
    for n in ref:
        assert_bitexact(_np(got[n]), _np(ref[n]))


@pytest.mark.parametrize("T", [7, 90])
def test_strided_rows_and_untouched_surroundings(gpu, T):
    import torch
    a = _inputs(T, 1024, 256, 16, 8, torch.bfloat16, T)
    wide = {n: torch.full((T, 1032), 7.0, device="cuda") for n in ("x", "attn_out", "mlp_out", "normed", "resid", "out")}
    for n in ("x", "attn_out", "mlp_out"):
        wide[n][:, 4:1028] = a[n]
        a[n] = wide[n][:, 4:1028]
    outs = {n: wide[n][:, 4:1028] for n in ("normed", "resid", "out")}
    got, ref = _step(gpu, a, outs), _singles(gpu, a)
    for n in ref:
        assert_bitexact(_np(got[n]), _np(ref[n]))
    for n in outs:
        assert (_np(wide[n])[:, :4] == 7).all() and (_np(wide[n])[:, 1028:] == 7).all()


@pytest.mark.parametrize("over", [dict(resid="x"), dict(act="gate"), dict(q_out="q", k_out="k"), dict(out="mlp_out"),
                                  dict(mlp_in="attn_out"), dict(out="resid"), dict(mlp_in="normed")])
def test_outputs_over_inputs_keep_the_launch_order(gpu, over):
    """An output in the memory of an input the later runs no longer need, or of
    an earlier output: what is left is what the runs in order leave."""
    import torch
    a = _inputs(33, 1024, 512, 16, 8, torch.bfloat16, 5)
    ref = {n: _np(t) for n, t in _singles(gpu, a).items()}
    outs = {n: torch.empty_like(dict(a, normed=a["x"], resid=a["x"])[m]) for n, m in over.items()}
    outs.update({n: a[m] for n, m in over.items() if m in a})
    if over == dict(out="resid") or over == dict(mlp_in="normed"):
        (n, m), = over.items()
        outs[m] = outs[n] = torch.empty_like(a["x"])
    got = _step(gpu, a, outs)
    for n in ref:
        if n in over.values():
            continue        # overwritten by the later output
        assert_bitexact(_np(got[n]), ref[n])
