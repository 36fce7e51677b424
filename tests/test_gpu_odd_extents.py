"""The elementwise kernels on extents that are no multiple of four values, from
any 4-byte boundary, and on few long rows: bit for bit against numpy's f32
operations (one rounding per operation), and for the ops with a sine or an
exponential against the same op on an aligned copy padded to whole float4s."""
import numpy as np
import pytest

from test_gpu_parity import _np, _t, assert_bitexact

pytestmark = pytest.mark.gpu
SEED = 20261231
LEAKY = np.float32(0.1)

# totals around one lane's, one block's and the mid-size kernel's bounds; rows of 1 to 3 values; one long odd row
SHAPES = [(1, 1), (1, 3), (3, 3), (5, 5), (7, 37), (2, 511), (1, 1021), (3, 1025), (128, 2401), (9, 24001),
          (1, 1048577), (2, 2097151), (1, 4194307)]


def _pair(shape):
    rng = np.random.default_rng(SEED + sum(shape))
    return rng.standard_normal(shape).astype(np.float32), rng.standard_normal(shape).astype(np.float32)


def _shifted(gpu, x, shift):
    """x on the device, `shift` values past a 16-byte boundary, the rest of the buffer 7."""
    import torch
    buf = torch.full((x.size + 8,), 7.0, device="cuda")
    v = buf[shift:shift + x.size].view(x.shape)
    v.copy_(_t(gpu, x))
    return buf, v


@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("shape", SHAPES)
def test_same_shape(gpu, shape, shift):
    x, b = _pair(shape)
    (_, tx), (_, tb), (ybuf, y) = _shifted(gpu, x, shift), _shifted(gpu, b, (shift + 2) % 4), _shifted(gpu, x, 3 - shift)
    gpu.add(tx, tb, out=y)
    assert_bitexact(_np(y), x + b)
    edge = _np(ybuf)
    assert (edge[:3 - shift] == 7).all() and (edge[3 - shift + x.size:] == 7).all()
    sum_out, y = gpu.add_leaky_relu(tx, tb, 0.1, want_sum=True)
    s = x + b
    assert_bitexact(_np(sum_out), s)
    assert_bitexact(_np(y), np.maximum(s, 0) + LEAKY * np.minimum(s, 0))
    assert_bitexact(_np(gpu.sqr(tx)), x * x)
    gpu.mul(tx, tb, out=tx)     # in place
    assert_bitexact(_np(tx), x * b)


@pytest.mark.parametrize("shape", SHAPES)
def test_one_value_per_row_and_one_row(gpu, shape):
    x, b = _pair(shape)
    col, row = b[:, :1], b[0]
    tx = _t(gpu, x)
    assert_bitexact(_np(gpu.add(tx, _t(gpu, col))), x + col)
    assert_bitexact(_np(gpu.sub(tx, _t(gpu, row))), x - row)
    if shape[0] % 3 == 0:       # b's rows repeat over a's, one value each
        b3 = np.ascontiguousarray(col[:3])
        assert_bitexact(_np(gpu.mul(tx, _t(gpu, b3))), x * np.tile(b3, (shape[0] // 3, 1)))
    _, ts = _shifted(gpu, x, 1)
    gpu.mul(ts, _t(gpu, col), out=ts)
    assert_bitexact(_np(ts), x * col)


@pytest.mark.parametrize("shape", [(3, 5), (2, 1023), (5, 1025), (3, 9001)])
def test_strided_rows(gpu, shape):
    """Rows cut out of wider ones: a view's add of one value per row, of a row, and of its own shape."""
    import torch
    x, b = _pair((shape[0], shape[1] + 3))
    n = shape[1]
    xv, bv = x[:, 1:1 + n], b[:, 2:2 + n]
    tx, tb = _t(gpu, x)[:, 1:1 + n], _t(gpu, b)[:, 2:2 + n]
    out = torch.full((shape[0], n + 2), 7.0, device="cuda")
    for rhs, ref in ((tb, xv + bv), (_t(gpu, bv[:, :1]), xv + bv[:, :1]), (_t(gpu, bv[0]), xv + bv[0])):
        gpu.add(tx, rhs, out=out[:, 1:1 + n])
        got = _np(out)
        assert_bitexact(np.ascontiguousarray(got[:, 1:1 + n]), ref)
        assert (got[:, 0] == 7).all() and (got[:, -1] == 7).all()


@pytest.mark.parametrize("op", ["exp", "sin", "gelu_erf", "tanh", "sigmoid"])
def test_same_values_as_aligned(gpu, op):
    x, _ = _pair((3, 4099))
    _, tx = _shifted(gpu, x, 1)
    pad = np.zeros(x.size + 4 - x.size % 4, np.float32)
    pad[:x.size] = x.reshape(-1)
    ref = _np(getattr(gpu, op)(_t(gpu, pad)))[:x.size].reshape(x.shape)
    assert_bitexact(_np(getattr(gpu, op)(tx)), ref)
