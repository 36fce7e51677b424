"""shp_layer_nongemm_step's one launch at the edges of its blocks: one position
to past the decode form's 64, hidden sizes of one to four float4 a lane, head
counts that end inside a block and past what the launch takes (the five
launches then), every gain type, strided rows, and outputs laid over inputs,
where the step keeps the five launches' order. Every output equals the single
entry points' bit for bit, also where the single norms share a row among fewer
lanes and rows lie on an f32 rounding boundary of their sum of squares."""
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


def _boundary_rows(H):
    """Rows whose sum of squares is halfway between two f32, and moves off it only
    if the two smallest squares (0.3 ulp of the double sum each) meet before they
    meet the largest: at float4 64 and 192 if 128 lanes share the row, not if 64 or
    256 do; at 65 and 193 if 64 or 128 do. 1.25^2 has an even f32 mantissa, and at
    eps 1e-6 (512 float4: other leading values too) the scale shows the step."""
    rows = []
    for big in (1.0, 1.25, 1.375, 1.125):
        for p, q in ((64, 192), (65, 193), (64, 128), (65, 129), (128, 192), (3, 67)):
            x = np.zeros(H, np.float32)
            x[0], x[1] = big, np.sqrt(np.spacing(np.float32(big) * np.float32(big)) / 2)
            x[4 * p], x[4 * q] = (np.sqrt(0.3 * 2.0 ** -52),) * 2
            rows.append(x)
    return np.stack(rows)


@pytest.mark.parametrize("H,T", [(1024, t) for t in (1023, 1024, 2048, 2049, 4095, 4096, 6143, 6144, 16383, 16384)] +
                         [(2048, t) for t in (2047, 2048, 2049, 4095, 4096)] + [(512, 2100), (256, 1025), (1020, 3000)])
def test_many_positions_add_their_rows_as_the_single_norms_do(gpu, H, T):
    import torch
    a = _inputs(T, H, 4, 1, 1, torch.float32, T)
    rows = torch.from_numpy(_boundary_rows(H)).cuda() if H >= 1020 else a["x"][:8].clone()
    n = rows.shape[0]
    a["w_in"].fill_(1.0)
    a["w_post"].fill_(1.0)
    for at in (0, T // 2, T - n):
        a["x"][at:at + n] = rows
        a["attn_out"][at:at + n] = 0.0
    got, ref = _step(gpu, a), _singles(gpu, a)
    for name in ref:
        assert_bitexact(_np(got[name]), _np(ref[name]))
