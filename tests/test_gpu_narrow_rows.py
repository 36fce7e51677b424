"""The row kernels where a row is a wave's float4 or less and where few short
rows go by elements: widths either side of 64, 256, 512 and 513 elements, few
rows and more than the grid holds, strided, in place, with a value per row and a
repeated row. Sums and products are bit-exact; what lies between the rows stays."""
import numpy as np
import pytest

from test_gpu_parity import _np, _t, assert_bitexact

pytestmark = pytest.mark.gpu
SEED = 20261204


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 67, 128, 255, 256, 257, 259, 260, 263, 511, 512, 513, 515, 516, 1023])
@pytest.mark.parametrize("rows", [1, 37, 1025, 66000])
def test_strided_rows(gpu, n, rows):
    import torch
    if rows * n > 20e6:
        rows = 2100
    rng = np.random.default_rng([SEED, rows, n])
    x = rng.standard_normal((rows, n + 3)).astype(np.float32)
    b = rng.standard_normal((rows, 1)).astype(np.float32)
    w = rng.standard_normal((1, n)).astype(np.float32)
    tx, core = _t(gpu, x), x[:, 1:1 + n]
    buf = torch.full((rows, n + 2), 7.0, device="cuda")
    out = buf[:, 1:1 + n]
    for call, ref in ((lambda: gpu.sqr(tx[:, 1:1 + n], out=out), core * core),
                      (lambda: gpu.add(tx[:, 1:1 + n], _t(gpu, b), out=out), core + b),
                      (lambda: gpu.mul(tx[:, 1:1 + n], _t(gpu, w), out=out), core * w),
                      (lambda: gpu.add(tx[:, 1:1 + n], tx[:, 1:1 + n], out=out), core + core)):
        buf.fill_(7.0)
        call()
        got = _np(buf)
        assert_bitexact(got[:, 1:1 + n], ref)
        assert (got[:, 0] == 7).all() and (got[:, -1] == 7).all()
    gpu.sqr(tx[:, 1:1 + n], out=tx[:, 1:1 + n])         # in place
    got = _np(tx)
    assert_bitexact(got[:, 1:1 + n], core * core)
    assert_bitexact(got[:, :1], x[:, :1])


@pytest.mark.parametrize("n", [2, 65, 257, 512, 516])
@pytest.mark.parametrize("rows", [9, 1500])
def test_sum_kept_and_two_inputs(gpu, n, rows):
    """add_leaky_relu with its sum, residual in place, on strided rows."""
    rng = np.random.default_rng([SEED, rows, n, 1])
    a, b = (rng.standard_normal((rows, n + 1)).astype(np.float32) for _ in range(2))
    ta, tb = _t(gpu, a), _t(gpu, b)
    s, y = gpu.add_leaky_relu(ta[:, 1:], tb[:, 1:], 0.1, sum_out=ta[:, 1:])
    ref = a[:, 1:] + b[:, 1:]
    assert_bitexact(_np(s), ref)
    assert_bitexact(_np(y), np.where(ref > 0, ref, np.float32(0)) + np.float32(0.1) * np.where(ref < 0, ref, np.float32(0)))
