"""The binding's native half (csrc/shp_bind.cpp) on host tensors: descriptors
of every type, rank and stride against the rule written out here, what it
refuses, and the conversion of call arguments through entry points that refuse
their arguments before touching a device."""
import ctypes

import numpy as np
import pytest
import torch

import synth_hip as S


def _rule(t):
    """ne, nb of a tensor: its extents and byte strides innermost first, a
    scalar one element, then extents of 1 at the stride of all below."""
    item = t.element_size()
    ne, nb = list(t.shape[::-1]) or [1], [s * item for s in t.stride()[::-1]] or [item]
    while len(ne) < 4:
        nb.append(nb[-1] * ne[-1])
        ne.append(1)
    return ne, nb


@pytest.mark.parametrize("dtype,type_", [(torch.float32, S.TYPE_F32), (torch.float16, S.TYPE_F16),
                                         (torch.bfloat16, S.TYPE_BF16), (torch.int32, S.TYPE_I32)])
def test_descriptors(dtype, type_):
    base = torch.zeros(2, 3, 5, 8).to(dtype)
    for t in (base, base[0], base[1, 2], base[1, 2, 3], base[1, 2, 3, 4], base.transpose(1, 3), base[:, :, 1:4, 2:7],
              base[0].t() if base[0].dim() == 2 else base[0].permute(2, 0, 1), base[:, :1], base.expand(2, 3, 5, 8)[:, :, :, ::2]):
        d = S.desc(t)
        ne, nb = _rule(t)
        assert (d.type, d.reserved, d.data) == (type_, 0, t.data_ptr())
        assert list(d.ne) == ne and list(d.nb) == nb


@pytest.mark.parametrize("cls", [S.Q8Tensor, S.Q5KTensor])
def test_block_descriptors(cls):
    raw = torch.zeros(4, 7, 3 * cls.BYTES, dtype=torch.uint8)
    for r in (raw, raw[1], raw[:, 2:5], raw[0, :, :cls.BYTES]):
        n = r.shape[-1] // cls.BYTES * cls.ELEMS
        d = S.desc(cls(r, n))
        ne, nb = _rule(r)
        ne[0], nb[0] = n, cls.BYTES
        assert d.type == cls.TYPE and d.data == r.data_ptr()
        assert list(d.ne) == ne and list(d.nb)[:r.dim()] == nb[:r.dim()]


def test_refused_tensors():
    assert S.desc(None) is None
    with pytest.raises(KeyError):
        S.desc(torch.zeros(3, dtype=torch.float64))
    with pytest.raises(KeyError):
        S.desc(torch.zeros(3, dtype=torch.uint8))       # raw blocks come in a BlockTensor
    with pytest.raises(ValueError):
        S.desc(torch.zeros(1, 1, 1, 1, 2))
    with pytest.raises((AttributeError, TypeError)):
        S.desc(3.0)


def test_calls():
    a, b = torch.zeros(2, 8), torch.zeros(2, 4)
    f = S._fn("shp_swiglu")
    assert f(a, None, b, 0) == S.ERR_INVALID_ARG        # shapes differ
    assert f(None, a, a, None) == S.ERR_INVALID_ARG
    with pytest.raises(TypeError):
        f(a, a, a)                                      # no stream
    with pytest.raises(TypeError):
        S._fn("shp_norm")(a, "eps", a, 0)
    with pytest.raises(AttributeError):
        S._binding().bind(S.load()._handle, "shp_no_such_entry")
    assert S._fn("shp_get_rows_sum")([a, a], 2, b, a, 0) == S.ERR_INVALID_ARG      # ids are not I32
    assert S._fn("shp_pad")(a, [0, 0, 0, 0], b, 0) == S.ERR_INVALID_ARG
    with pytest.raises(TypeError):
        S._fn("shp_pad")(a, [0, 0], b, 0)
    d = S.kernel_shape(3, 2)                            # a ctypes descriptor without data
    assert S._fn("shp_im2col")(d, a, 1, 0, 1, b, 0) != S.OK
    assert ctypes.sizeof(S.ShpTensor) == len(S._binding().describe(a))


@pytest.mark.parametrize("name,args", [
    ("shp_soft_max_ext", lambda a, bad: (a, bad, 1.0, 0.0, a, 0)),
    ("shp_swiglu", lambda a, bad: (a, bad, a, 0)),
    ("shp_swiglu", lambda a, bad: (bad, a, a, 0)),
    ("shp_add", lambda a, bad: (a, bad, a, 0)),
    ("shp_add", lambda a, bad: (a, a, bad, 0)),
    ("shp_sum_rows", lambda a, bad: (bad, a, 0)),
    ("shp_get_rows_sum", lambda a, bad: ([a, bad], 2, a, a, 0)),
    ("shp_im2col", lambda a, bad: (bad if not isinstance(bad, S.ShpTensor) else [bad], a, 1, 0, 1, a, 0)),
    ("shp_im2col", lambda a, bad: (S.kernel_shape(3, 2), bad, 1, 0, 1, a, 0)),
    ("shp_layer_nongemm_step", lambda a, bad: (a,) * 18 + (bad, 1e-6, 1e6, 128, 0)),
])
def test_a_tensor_parameter_takes_nothing_but_a_tensor(name, args):
    """A list or tuple (also of one tensor, or empty: no mask by mistake), a
    descriptor, or any object with as many bytes as one, raises."""
    a = torch.zeros(2, 8)
    size = ctypes.sizeof(S.ShpTensor)
    class Alike:
        data, ne0, TYPE, BYTES = torch.zeros(2, 34, dtype=torch.uint8), 32, S.TYPE_Q8_0, 34
    for bad in ([], (), [a], (a, a), [None], S.kernel_shape(8, 2), bytes(size), bytearray(size), np.zeros(size, np.uint8),
                np.zeros((2, 8), np.float32), memoryview(bytes(size)), 3, "x", Alike()):
        with pytest.raises(TypeError):
            S._fn(name)(*args(a, bad))


@pytest.mark.parametrize("name,rest", [("shp_get_rows_sum", lambda a: (a, a, 0)),
                                       ("shp_sum_scale_leaky_relu", lambda a: (1.0, 0.1, None, a, 0))])
def test_an_array_is_a_list_of_the_count_beside_it(name, rest):
    a, f = torch.zeros(2, 8), S._fn(name)
    for tables, n, exc in (([a], 2, ValueError), ([a, a], 1, ValueError), ([], 1, ValueError), ((a,), -1, ValueError),
                           ([a], 2 ** 32 + 1, ValueError), ([a], "1", TypeError), ([a], None, TypeError),
                           (a, 1, TypeError), (None, 1, TypeError), (iter([a]), 1, TypeError)):
        with pytest.raises(exc):
            f(tables, n, *rest(a))
    b = torch.zeros(2, 8, dtype=torch.float16)              # refused for its type, after the conversion
    assert f((b, b), 2, *rest(b)) not in (S.OK, S.ERR_BACKEND)


def test_public_calls_refuse_what_is_no_tensor(monkeypatch):
    monkeypatch.setattr(S, "_stream", lambda: 0)
    a = torch.zeros(2, 8)
    for call in (lambda: S.soft_max_ext(a, [], 1.0), lambda: S.soft_max_ext(a, [a, a], 1.0), lambda: S.swiglu(a, []),
                 lambda: S.add(a, [a]), lambda: S.rms_norm_mul(a, (), 1e-6), lambda: S.qk_norm_rope(
                     a, a, [], a, 1e-6, a, 8, 1e6), lambda: S.im2col(a, 3.0, out=a), lambda: S.get_rows_sum([a, [a]], a, out=a)):
        with pytest.raises(TypeError):
            call()


def test_tensors_of_another_load_of_the_binding():
    """A reload, or a second copy of the module, has classes of its own; tensors
    made with either go through both, in any order of loading."""
    import importlib.util
    spec = importlib.util.spec_from_file_location("synth_hip_again", S.__file__)
    again = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(again)
    raw, a = torch.zeros(3, 68, dtype=torch.uint8), torch.zeros(2, 8)
    for first, second in ((S, again), (again, S)):
        want = bytes(first.desc(first.Q8Tensor(raw, 64)))
        assert bytes(second.desc(second.Q8Tensor(raw, 64))) == want
        assert bytes(first.desc(second.Q8Tensor(raw, 64))) == want and bytes(second.desc(first.Q8Tensor(raw, 64))) == want
        for shape in (first.kernel_shape(3, 2), second.kernel_shape(3, 2)):
            assert first._fn("shp_im2col")(shape, a, 1, 0, 1, a, 0) != S.OK
