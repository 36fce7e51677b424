"""The launches that entry points make, without a GPU: record() runs calls of
libsynth_hip.so in a process of its own in which tests/host/launch_record.cpp
stands in for the kernel launch. Tensors are descriptors of addresses that
nothing reads."""
import ctypes
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "synthesize.cpp_amd")
_at = [1 << 44]


def t(*ne, nb=None, type_=0, at=None):
    """A descriptor of ggml extents ne (F32; byte strides nb, contiguous unless
    given) at an address of its own, 256-byte aligned, or `at`."""
    ne = list(ne) + [1] * (4 - len(ne))
    size = {0: 4, 1: 2, 26: 4, 30: 2}[type_]
    if nb is None:
        nb = [size]
        for k in range(1, 4):
            nb.append(nb[-1] * ne[k - 1])
    nb = list(nb) + [nb[-1] * ne[len(nb) - 1]] * (4 - len(nb))
    if at is None:
        at = _at[0]
        _at[0] += (max(nb[k] * ne[k] for k in range(4)) + 4096) // 256 * 256
    return dict(ne=ne, nb=nb, type=type_, data=at)


def layer(x, w_in, normed, q, k, wq, wk, pos, q_out, k_out, attn_out, w_post, resid, mlp_in, gate, up, act, mlp_out, out,
          eps=1e-6, freq_base=1e6, n_dims=128):
    """shp_layer_step as an argument."""
    return dict(layer=[x, w_in, normed, q, k, wq, wk, pos, q_out, k_out, attn_out, w_post, resid, mlp_in, gate, up, act,
                       mlp_out, out], eps=eps, freq_base=freq_base, n_dims=n_dims)


def record(calls):
    """[(name, args...)] -> [(status, [(kernel, grid, block, lds)])]; the stream
    is added."""
    with tempfile.TemporaryDirectory() as tmp:
        shim = os.path.join(tmp, "launch_record.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", shim,
                        os.path.join(HERE, "host", "launch_record.cpp")], check=True)
        r = subprocess.run([sys.executable, os.path.abspath(__file__), shim], input=json.dumps(calls), capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        out = json.loads(r.stdout)
    return [(st, [(n, tuple(g), tuple(b), s) for n, g, b, s in ls]) for st, ls in out]


def _run(shim_path, calls):
    sys.path.insert(0, PKG)
    import synth_hip as S

    shim = ctypes.CDLL(shim_path, mode=ctypes.RTLD_GLOBAL)      # ahead of the HIP runtime
    lib = ctypes.CDLL(S.LIB_PATH)

    class Launch(ctypes.Structure):
        _fields_ = [("name", ctypes.c_char_p), ("grid", ctypes.c_uint32 * 3), ("block", ctypes.c_uint32 * 3),
                    ("lds", ctypes.c_uint64)]

    shim.launch_at.restype = ctypes.POINTER(Launch)
    keep = []

    def tensor(a):
        d = S.ShpTensor()
        d.type, d.reserved, d.data = a["type"], 0, a["data"]
        for k in range(4):
            d.ne[k], d.nb[k] = a["ne"][k], a["nb"][k]
        keep.append(d)
        return ctypes.pointer(d)

    def arg(a):
        if a is None:
            return ctypes.c_void_p(None)
        if isinstance(a, float):
            return ctypes.c_float(a)
        if isinstance(a, int):
            return ctypes.c_int32(a)
        if "layer" in a:
            s = S.ShpLayerStep()
            for (name, _), v in zip(s._fields_, a["layer"]):
                setattr(s, name, tensor(v))
            s.eps, s.freq_base, s.n_dims, s.reserved = a["eps"], a["freq_base"], a["n_dims"], 0
            keep.append(s)
            return ctypes.byref(s)
        return tensor(a)

    out = []
    for name, *args in calls:
        shim.launch_clear()
        st = getattr(lib, name)(*[arg(a) for a in args], ctypes.c_void_p(None))
        ls = [shim.launch_at(i).contents for i in range(shim.launch_count())]
        out.append((st, [(l.name.decode(), list(l.grid), list(l.block), l.lds) for l in ls]))
    return out


if __name__ == "__main__":
    json.dump(_run(sys.argv[1], json.load(sys.stdin)), sys.stdout)
