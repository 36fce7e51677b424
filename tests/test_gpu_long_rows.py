"""ggml_norm and the row sums at the edges of their register and block forms:
rows of one value to past what a block holds, remainders of one to three
values, few rows and many, rows on any 4-byte boundary, and in place, against
the restatement. The sums are double sums in another order, so a row sum
rounds to the restatement's f32 (bit for bit) and a norm's mean and variance
to its f32 statistics unless a double sum lies within its own rounding error
(~1e-16 * ne0) of a rounding boundary; one ulp of the mean or of the scale
moves a result by at most 2^-23 of |x| + |mean| times the scale, under 1e-5
for these inputs (|x| < 16, scale ~0.5)."""
import numpy as np
import pytest

import ggml_ref as R
from test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu
SEED = 20261230

SHAPES = [(3, 1), (5, 3), (9, 255), (2, 256), (7, 257), (300, 259), (4, 510), (3, 1024), (260, 1030), (257, 2049),
          (258, 4099), (300, 8192), (2, 4097), (3, 8191), (130, 16385), (2, 32771), (1, 65536), (2, 65537), (3, 140001)]


def _x(rng, shape):
    return (rng.standard_normal(shape) * 2 + 3).astype(np.float32)


@pytest.mark.parametrize("rows,ne0", SHAPES)
def test_norm(gpu, rows, ne0):
    x = _x(np.random.default_rng(SEED + rows + ne0), (rows, ne0))
    x[0] = 5.0
    ref = R.run(lambda g: g.norm(x, 1e-6))
    t = _t(gpu, x)
    got = _np(gpu.norm(t, 1e-6))
    assert (got[0] == 0).all()
    assert np.abs(got - ref).max() <= 1e-5
    gpu.norm(t, 1e-6, out=t)
    assert np.array_equal(_np(t).view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("rows,ne0", [(5, 257), (3, 1023), (2, 4099), (2, 65540)])
def test_norm_strided_and_special(gpu, rows, ne0):
    import torch
    rng = np.random.default_rng(SEED + ne0)
    x = _x(rng, (rows, ne0 + 5))
    x[1, 7] = np.nan
    buf = torch.full((rows, ne0 + 3), 7.0, device="cuda")
    gpu.norm(_t(gpu, x)[:, 3:3 + ne0], 1e-5, out=buf[:, 1:1 + ne0])
    got = _np(buf)
    assert (got[:, 0] == 7).all() and (got[:, -2:] == 7).all()     # nothing past the rows
    ref = R.run(lambda g: g.norm(np.ascontiguousarray(x[:, 3:3 + ne0]), 1e-5))
    assert np.isnan(got[1, 1:1 + ne0]).all()
    keep = [r for r in range(rows) if r != 1]
    assert np.abs(got[keep, 1:1 + ne0] - ref[keep]).max() <= 1e-5


@pytest.mark.parametrize("rows,ne0", SHAPES)
def test_row_sums(gpu, rows, ne0):
    rng = np.random.default_rng(SEED + 2 * rows + ne0)
    x, w = _x(rng, (rows, ne0)), rng.standard_normal((rows, ne0)).astype(np.float32)
    for name, args in (("sum_rows", (x,)), ("mean", (x,))):
        ref = R.run(lambda g: getattr(g, name)(*args))
        assert np.array_equal(_np(getattr(gpu, name)(_t(gpu, x))).view(np.uint32), ref.view(np.uint32)), name
    ref = R.run(lambda g: g.sum_rows(x * w))
    assert np.array_equal(_np(gpu.mul_sum_rows(_t(gpu, x), _t(gpu, w))).view(np.uint32), ref.view(np.uint32))
