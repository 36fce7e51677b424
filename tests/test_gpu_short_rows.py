"""ggml_norm and the row sums where a row is one or two elements or a few float4
per lane: widths either side of 64, 128, 256, 512 and 1024 elements, few rows and
enough for one wave each, on any 4-byte boundary. Bounds as test_gpu_long_rows.py
derives them: row sums bit for bit, norms within 1e-5."""
import numpy as np
import pytest

import ggml_ref as R
from test_gpu_parity import _np, _t

pytestmark = pytest.mark.gpu
SEED = 20261205


@pytest.mark.parametrize("ne0", [1, 2, 5, 63, 64, 65, 67, 127, 128, 129, 255, 256, 259, 260, 511, 513, 1023, 1024, 1027])
@pytest.mark.parametrize("rows", [1, 6, 2049])
def test_rows(gpu, rows, ne0):
    rng = np.random.default_rng([SEED, rows, ne0])
    x = (rng.standard_normal((rows, ne0 + 3)) * 2 + 3).astype(np.float32)
    w = rng.standard_normal((rows, ne0 + 2)).astype(np.float32)
    tx, tw = _t(gpu, x)[:, 1:1 + ne0], _t(gpu, w)[:, 2:]
    x, w = np.ascontiguousarray(x[:, 1:1 + ne0]), np.ascontiguousarray(w[:, 2:])
    bits = lambda a: np.ascontiguousarray(a).view(np.uint32)
    for name in ("sum_rows", "mean"):
        assert np.array_equal(bits(_np(getattr(gpu, name)(tx))), bits(R.run(lambda g: getattr(g, name)(x)))), name
    assert np.array_equal(bits(_np(gpu.mul_sum_rows(tx, tw))), bits(R.run(lambda g: g.sum_rows(x * w))))
    assert np.abs(_np(gpu.norm(tx, 1e-5)) - R.run(lambda g: g.norm(x, 1e-5))).max() <= 1e-5


@pytest.mark.parametrize("ne0", [3, 64, 128, 515])
def test_special_values(gpu, ne0):
    """NaN and infinities stay in their row."""
    x = np.random.default_rng([SEED, ne0]).standard_normal((9, ne0)).astype(np.float32)
    x[1, ne0 - 1], x[3, 0], x[5, ne0 // 2] = np.nan, np.inf, -np.inf
    s = _np(gpu.sum_rows(_t(gpu, x)))[:, 0]
    ref = R.run(lambda g: g.sum_rows(x))[:, 0]
    assert np.isnan(s[1]) and s[3] == np.inf and s[5] == -np.inf
    clean = [0, 2, 4, 6, 7, 8]
    assert np.array_equal(s[clean], ref[clean])
    y = _np(gpu.norm(_t(gpu, x), 1e-5))
    assert np.isnan(y[[1, 3, 5]]).any(axis=1).all() and np.isfinite(y[clean]).all()
