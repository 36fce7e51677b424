"""The transposing copy and the convolution tails on extents of every remainder
of four, rows that share cache lines with their neighbours' tiles, and views off
a 16-byte boundary; tiles one value wide, ragged in both directions, and enough
of them that every XCD has its run; one case past the size from which stores
are kept in L2. Bit for bit against numpy: copies, f32 adds in the nodes' order."""
import numpy as np
import pytest

from test_gpu_parity import _np, _t, assert_bitexact

pytestmark = pytest.mark.gpu
SEED = 20261233
LEAKY = np.float32(0.1)
SHAPES = [(1, 2), (3, 2), (5, 7), (64, 129), (65, 128), (66, 131), (127, 257), (130, 1021), (1021, 130), (37, 4099), (4098, 33)]


def _inside(gpu, x, shift):
    """x inside a wider buffer of sevens, its rows `shift` values in."""
    import torch
    buf = torch.full((x.shape[0], x.shape[1] + 5), 7.0, device="cuda")
    v = buf[:, shift:shift + x.shape[1]]
    v.copy_(_t(gpu, x))
    return buf, v


@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("T,C", SHAPES)
def test_copy(gpu, T, C, shift):
    x = np.random.default_rng([SEED, T, C]).standard_normal((T, C)).astype(np.float32)
    _, v = _inside(gpu, x, shift)
    buf, out = _inside(gpu, np.zeros((C, T), np.float32), (shift + 2) % 4)
    gpu.cpy(v.t(), out=out)
    assert_bitexact(_np(out), np.ascontiguousarray(x.T))
    b = _np(buf)
    s = (shift + 2) % 4
    assert (b[:, :s] == 7).all() and (b[:, s + T:] == 7).all()


@pytest.mark.parametrize("T,C", SHAPES + [(30001, 141)])
def test_tails(gpu, T, C):
    rng = np.random.default_rng([SEED, C, T])
    x, r = rng.standard_normal((T, C)).astype(np.float32), rng.standard_normal((C, T)).astype(np.float32)
    col, row = rng.standard_normal((C, 1)).astype(np.float32), rng.standard_normal(T).astype(np.float32)
    tx, tr = _t(gpu, x).t(), _t(gpu, r)
    s = (x.T + col) + r
    y = np.maximum(s, 0) + LEAKY * np.minimum(s, 0)
    total = tr.clone()
    got = gpu.cont_add_leaky_relu(tx, _t(gpu, col), total, 0.1, sum_out=total)     # the sum over its residual
    assert_bitexact(_np(total), s)
    assert_bitexact(_np(got), y)
    assert_bitexact(_np(gpu.cont_add_leaky_relu(tx, _t(gpu, col))), x.T + col)
    assert_bitexact(_np(gpu.cont_add_leaky_relu(tx, _t(gpu, col), tr)), s)
    if T > 1:      # one value per column ([T] against C rows)
        import torch
        off = torch.zeros(T + 1, device="cuda")
        off[1:] = _t(gpu, row)
        assert_bitexact(_np(gpu.cont_add_leaky_relu(tx, off[1:])), x.T + row)


def test_large_copy(gpu):
    import torch
    x = torch.randn(30011, 143, device="cuda")
    assert torch.equal(gpu.cpy(x.t()), x.t().contiguous())


@pytest.mark.parametrize("T,C", [(1027, 1024), (513, 4096), (8192, 771), (8192, 1025), (16384, 769)])
def test_whole_rows_a_power_of_two_apart(gpu, T, C):
    """One side's rows start 4 KB or 32 KB apart and the other's share lines:
    tiles in order."""
    import torch
    x, r = torch.randn(T, C, device="cuda"), torch.randn(C, T, device="cuda")
    assert torch.equal(gpu.cpy(x.t()), x.t().contiguous())
    col = torch.randn(C, 1, device="cuda")
    assert torch.equal(gpu.cont_add_leaky_relu(x.t(), col, r), (x.t() + col) + r)
