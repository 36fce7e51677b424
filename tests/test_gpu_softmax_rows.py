"""The softmax at the edges of its row forms: one score to past what registers
hold, every remainder of a float4, few rows (16 waves each) and many (one wave
each), rows on any 4-byte boundary, in place, with a mask and causal, against
the restatement, > 99 % identical and within 3 ulp: glibc's expf and the
kernel's exp differ by at most one ulp of v, 2^-23 relative at the bottom of a
binade, which is two ulp of y = v*inv when y lies at the top of one, and the two
products' roundings may part by one more (5.5 million values a case meet it; the
double sum's order moves the reciprocal only on a rounding boundary)."""
import numpy as np
import pytest

import ggml_ref as R
from test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu
SEED = 20261232


def _close(got, ref):
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    ulp = np.abs(got - ref)[ok] / np.spacing(np.abs(ref[ok]).astype(np.float32)).astype(np.float64)
    assert ulp.size == 0 or ulp.max() <= 3, ulp.max()
    assert ulp.size < 200 or (ulp == 0).mean() > 0.99


WIDTHS = [1, 2, 3, 4, 5, 6, 7, 255, 257, 511, 514, 1021, 1027, 2049, 4099, 8191, 16383, 16384, 16385, 20003]


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("heads,rows", [(3, 1), (5, 67)])
def test_mask_and_none(gpu, n, heads, rows):
    rng = np.random.default_rng([SEED, n, rows])
    x = (rng.standard_normal((heads, rows, n)) * 6).astype(np.float32)
    m = np.where(rng.random((rows, n)) < 0.3, -np.inf, rng.standard_normal((rows, n))).astype(np.float32)
    m[:, n // 2] = 0.0
    scale = np.float32(0.3)
    t = _t(gpu, x)
    _close(_np(gpu.soft_max_ext(t, None, scale)), R.run(lambda g: g.soft_max_ext(x, None, scale)))
    ref = R.run(lambda g: g.soft_max_ext(x, m, scale))
    got = _np(gpu.soft_max_ext(t, _t(gpu, m), scale))
    _close(got, ref)
    gpu.soft_max_ext(t, _t(gpu, m), scale, out=t)       # in place
    assert np.array_equal(_np(t).view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("rows,n", [(2100, 1021), (2049, 2050), (2048, 5), (2050, 4101), (2051, 300)])
def test_many_rows(gpu, rows, n):
    x = (np.random.default_rng([SEED, rows, n]).standard_normal((1, rows, n)) * 4).astype(np.float32)
    _close(_np(gpu.soft_max_ext(_t(gpu, x), None, 0.5)), R.run(lambda g: g.soft_max_ext(x, None, np.float32(0.5))))


@pytest.mark.parametrize("n", [5, 255, 1022, 4097, 17001])
def test_strided_rows(gpu, n):
    import torch
    x = (np.random.default_rng([SEED, n]).standard_normal((2, 9, n + 3)) * 4).astype(np.float32)
    buf = torch.full((2, 9, n + 2), 7.0, device="cuda")
    gpu.soft_max_ext(_t(gpu, x)[:, :, 3:], None, 0.7, out=buf[:, :, 1:1 + n])
    got = _np(buf)
    _close(got[:, :, 1:1 + n], R.run(lambda g: g.soft_max_ext(np.ascontiguousarray(x[:, :, 3:]), None, np.float32(0.7))))
    assert (got[:, :, 0] == 7).all() and (got[:, :, -1] == 7).all()


@pytest.mark.parametrize("heads,rows,n,past", [(2, 5, 5, 0), (3, 37, 41, 4), (2, 255, 257, 2), (1, 1021, 1021, 0),
                                               (2, 9, 2051, 2042), (1, 3, 17003, 9000), (1, 700, 2500, 0)])
def test_causal_with_hidden_infinities(gpu, heads, rows, n, past):
    """Scores past the diagonal are never read: infinities and NaN there change nothing."""
    x = (np.random.default_rng([SEED, rows, n]).standard_normal((heads, rows, n)) * 4).astype(np.float32)
    clean = _np(gpu.soft_max_causal(_t(gpu, x), past, 0.25))
    masked = np.where(np.arange(n)[None, :] > past + np.arange(rows)[:, None], np.float32(-np.inf), np.float32(0))
    _close(clean, R.run(lambda g: g.soft_max_ext(np.where(np.isinf(masked), np.float32(-np.inf), x).astype(np.float32),
                                                 None, np.float32(0.25))))
    hidden = np.broadcast_to(np.isinf(masked), x.shape)
    x[hidden] = np.resize(np.float32([np.nan, np.inf, 3e38]), int(hidden.sum()))
    assert np.array_equal(_np(gpu.soft_max_causal(_t(gpu, x), past, 0.25)).view(np.uint32), clean.view(np.uint32))


@pytest.mark.parametrize("n", [129, 191, 193, 301, 321, 383, 385, 509, 511])
@pytest.mark.parametrize("rows", [1, 2048, 4096, 4097])
def test_short_odd_rows(gpu, n, rows):
    """Either side of the row counts from which they go by float4."""
    x = (np.random.default_rng([SEED, rows, n]).standard_normal((1, rows, n)) * 4).astype(np.float32)
    _close(_np(gpu.soft_max_ext(_t(gpu, x), None, 0.5)), R.run(lambda g: g.soft_max_ext(x, None, np.float32(0.5))))
