"""The native host side of a call (csrc/pyhost.cpp) against the ctypes one beside it: the same descriptors, the same
results, the same errors, and what it does not take goes the ctypes way unchanged."""
import ctypes as C
import gc
import glob
import os
import shutil
import subprocess
import sys
import sysconfig
import weakref

import numpy as np
import pytest

import zenu_amd
from zenu_amd import Matrix, ZenuHipError, _lib, _pyhost
from zenu_amd.matrix import _DESC

DTYPES = [np.float32, np.float64]
IDS = ["f32", "f64"]


class Memory:
    def __init__(self, ptr):
        self.ptr = ptr


class Derived(Matrix):
    pass


def ctypes_bytes(m):
    return _DESC[len(m.shape)](m.as_ptr(), len(m.shape), *m.shape, *m.stride)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", [(), (1,), (0,), (7,), (3, 5), (2, 0, 4), (2, 3, 4, 5), (1, 2, 3, 4, 5, 6)], ids=str)
def test_descriptors(dtype, shape):
    for ptr in (4096, (1 << 63) + 256):
        for offset in (0, 3):
            m = Matrix(Memory(ptr), offset, shape, zenu_amd.default_stride(shape), dtype)
            views = [m]
            if len(shape) >= 2:
                views += [m.transpose(), m.transpose_by_index(list(range(len(shape)))[::-1])]
            if shape and shape[0] > 1:
                views += [m.slice(slice(1, None, 2))]
            for v in views:
                assert _pyhost.pack(v) == ctypes_bytes(v)
                d = v.desc()
                assert (d.ptr, d.ndim, tuple(d.shape[:d.ndim]), tuple(d.stride[:d.ndim])) == (v.as_ptr(), v.ndim, v.shape, v.stride)


def test_transposed_view():
    m = Matrix(Memory(4096), 5, (2, 3, 4), (12, 4, 1), np.float32)
    t = m.transpose()
    assert type(t) is Matrix and vars(t) == {"buf": m.buf, "offset": 5, "shape": (2, 4, 3), "stride": (12, 1, 4), "dtype": m.dtype}
    assert vars(m)["shape"] == (2, 3, 4)
    with pytest.raises(ValueError):
        Matrix(Memory(4096), 0, (4,), (1,), np.float32).transpose()
    assert _pyhost.transpose(Derived(Memory(4096), 0, (2, 3), (3, 1), np.float32)) is None
    u = Derived(Memory(4096), 0, (2, 3), (3, 1), np.float32).transpose()
    assert (u.shape, u.stride) == ((3, 2), (1, 3))


def test_module_is_built_for_this_interpreter_alone(tmp_path):
    """its name carries the interpreter's tag, and an interpreter that there is none for imports the package all the same"""
    package = os.path.dirname(zenu_amd.__file__)
    assert _pyhost.__file__ == os.path.join(package, "_pyhost" + sysconfig.get_config_var("EXT_SUFFIX")) and zenu_amd.matrix._pyhost is _pyhost
    assert not os.path.exists(os.path.join(package, "_pyhost.so"))
    copy = tmp_path / "zenu_amd"
    copy.mkdir()
    for f in glob.glob(os.path.join(package, "*.py")):
        shutil.copy(f, copy)
    os.symlink(os.path.join(package, "lib"), copy / "lib")
    program = """
import numpy as np, zenu_amd as z
class Memory: ptr = 4096
m = z.Matrix(Memory(), 0, (2, 3), (3, 1), np.float32)
t = m.transpose()
assert (t.shape, t.stride) == ((3, 2), (1, 3)) and t.desc().ptr == 4096
z.lib()
try:
    m.add_array(z.Matrix(Memory(), 0, (4, 5), (5, 1), np.float32), m)
except z.ZenuHipError:
    print("refused")
"""
    done = subprocess.run([sys.executable, "-c", program], cwd=tmp_path, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout == "refused\n", done.stderr


def test_a_module_without_a_tag_is_taken_away(tmp_path):
    """such as builds left before modules were named after their interpreter: any interpreter would load it"""
    package = os.path.dirname(zenu_amd.__file__)
    (tmp_path / "zenu_amd" / "csrc").mkdir(parents=True)
    for f in ("Makefile", "pyhost.cpp"):
        shutil.copy(os.path.join(package, "csrc", f), tmp_path / "zenu_amd" / "csrc")
    os.symlink(os.path.join(os.path.dirname(package), "include"), tmp_path / "include")
    (tmp_path / "zenu_amd" / "_pyhost.so").write_bytes(b"")
    module = "_pyhost" + sysconfig.get_config_var("EXT_SUFFIX")
    subprocess.run(["make", "-C", str(tmp_path / "zenu_amd" / "csrc"), "../" + module, "PYTHON=" + sys.executable], check=True, capture_output=True, timeout=100)
    assert [f for f in os.listdir(tmp_path / "zenu_amd") if f.endswith(".so")] == [module]


def test_optimizer_operands_are_held_while_they_are_read():
    """reading a buffer's address can run code that takes the entry, its moments and its name away"""
    zenu_amd.lib()

    def matrix(memory, stride=(3, 1)):
        return Matrix(memory, 0, (2, 3), stride, np.float32)

    for kinds in (2, 4):
        alive = []

        class Taking:
            @property
            def ptr(self):
                for d in (params, m, v, weights):
                    d.clear()
                gc.collect()
                alive.append([r() is not None for r in refs])
                return 4096

        # the last matrix that is read has another stride: the call is declined after all of them
        last = (1, 2)
        g, first, second = matrix(Memory(4096), last if kinds == 2 else (3, 1)), matrix(Memory(4096)), matrix(Memory(4096), last)
        refs = [weakref.ref(x) for x in (g, first, second)[:kinds - 1]]
        name = "".join(["layer", ".", "weight"])
        params, m, v, weights = {name: (matrix(Taking()), g)}, {name: first}, {name: second}, {name}
        del g, first, second, name
        if kinds == 2:
            assert _pyhost.sgd_step_multi(params, 1e-3, None) is False
        else:
            assert _pyhost.adam_step_multi(params, m, v, weights, 1e-3, 0.9, 0.999, 1e-8, 0.0, 1, None) is False
        assert alive == [[True] * (kinds - 1)]
        assert not params and all(r() is None for r in refs)      # and let go afterwards


def test_transposed_view_holds_what_it_copies():
    """an allocation can start the collector, and a finalizer can replace the attributes that the view takes"""
    m = Matrix(Memory(4096), 0, (2, 3), (3, 1), np.float32)
    ref, old = weakref.ref(m.buf), gc.get_threshold()

    def replace(phase, info):
        m.buf, m.shape, m.stride = Memory(0), (9, 9), (9, 1)

    gc.collect()
    gc.callbacks.append(replace)
    gc.set_threshold(1)
    try:
        t = _pyhost.transpose(m)
    finally:
        gc.set_threshold(*old)
        gc.callbacks.remove(replace)
    assert (t.shape, t.stride) in (((3, 2), (1, 3)), ((9, 9), (1, 9)))     # one state or the other, whole
    assert t.buf is ref() if t.shape == (3, 2) else t.buf is m.buf


def test_other_forms_are_left_to_ctypes():
    m = Matrix(Memory(4096), 0, (2, 3), (3, 1), np.float32)
    odd = [Derived(Memory(4096), 0, (2, 3), (3, 1), np.float32), Matrix(Memory(4096), 0, (2, 3), (3, 1), np.int64),
           Matrix(Memory(4096), 0, (2, 3), (3, 1), ">f4"), Matrix(Memory(None), 0, (2, 3), (3, 1), np.float32)]
    for name, value in (("offset", -1), ("offset", np.int64(0)), ("shape", [2, 3]), ("shape", (2,)), ("shape", (1 << 64, 3)),
                        ("stride", (np.int64(3), 1)), ("shape", (1,) * 7), ("dtype", "float32")):
        o = Matrix(Memory(4096), 0, (2, 3), (3, 1), np.float32)
        setattr(o, name, value)
        odd.append(o)
    o = Matrix(Memory(4096), 0, (2, 3), (3, 1), np.float32)
    del o.stride
    odd.append(o)
    for o in odd + [None, 3, "m"]:
        assert _pyhost.pack(o) is None
        zenu_amd.lib()
        assert _pyhost.copy(o, m, None) is False and _pyhost.copy(m, o, None) is False
    for stream in ("0", 1.0, -1, C.c_int(0)):
        assert _pyhost.copy(m, m, stream) is False
    assert _pyhost.binary(np.int64(0), m, m, m, None) is False and _pyhost.binary(1 << 40, m, m, m, None) is False
    assert _pyhost.relu(m, m, np.float32(0), None) is False and _pyhost.relu(m, m, "0", None) is False
    assert _pyhost.softmax(m, m, True, None) is False
    p = {"w": (m, m)}
    for args in (([("w", (m, m))], {}, {}), (p, {}, {}), ({"w": [m, m]}, p, p), ({1: (m, m)}, p, p),
                 ({"w": (m.transpose(), m)}, {"w": m}, {"w": m}), ({"w": (m, odd[1])}, {"w": m}, {"w": m})):
        assert _pyhost.adam_step_multi(*args, None, 1e-3, 0.9, 0.999, 1e-8, 0.0, 1, None) is False
    assert _pyhost.adam_step_multi(p, {"w": m}, {"w": m}, ["w"], 1e-3, 0.9, 0.999, 1e-8, 0.0, 1, None) is False
    assert _pyhost.adam_step_multi({"w": (m, None)}, {}, {}, None, 1e-3, 0.9, 0.999, 1e-8, 0.0, 1, None) is True    # no gradient


class General:
    """the package with every native call declined"""
    def __init__(self, monkeypatch):
        self.patch = monkeypatch

    def __enter__(self):
        for module in (zenu_amd.matrix, zenu_amd.optim):
            self.patch.setattr(module, "_pyhost", type("Declined", (), {
                "__getattr__": lambda _, name: (lambda *a: None if name in ("pack", "transpose") else False)})())

    def __exit__(self, *_):
        self.patch.undo()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_calls_give_what_ctypes_gives(hip, dtype, monkeypatch):
    r = np.random.default_rng(3)
    a, b, row = (r.standard_normal(s).astype(dtype) for s in ((6, 5), (6, 5), (5,)))
    A, B, Row = map(Matrix.from_numpy, (a, b, row))

    def all_calls():
        out = []

        def do(fn):
            m, extra = Matrix.from_numpy(np.full((6, 5), 9, dtype)), Matrix.from_numpy(np.full((5,), 9, dtype))
            fn(m, extra)
            out.extend((m.to_numpy(), extra.to_numpy()))
        do(lambda m, e: m.add_array(A, Row))
        do(lambda m, e: m.sub_assign(B))
        do(lambda m, e: m.mul_scalar(A, 3))
        do(lambda m, e: m.div_scalar_assign(0.3))
        do(lambda m, e: m.tanh_array(A))
        do(lambda m, e: m.copy_from(Matrix.from_numpy(np.ascontiguousarray(a.T)).transpose()))
        do(lambda m, e: m.broadcast(Row))
        do(lambda m, e: m.relu(A, 0.1))
        do(lambda m, e: m.relu_backward(B, A, 0.1))
        do(lambda m, e: m.tanh_backward(B, A))
        do(lambda m, e: m.sigmoid_backward(B, A))
        do(lambda m, e: m.relu_backward_bias_grad(e, B, A, 0.1))
        do(lambda m, e: m.softmax_assign(A, 1))
        do(lambda m, e: m.bias_add_relu(A, Row, 0.1))
        pre = Matrix.from_numpy(np.zeros((6, 5), dtype))
        do(lambda m, e: m.bias_add_relu(A, Row, 0.1, pre=pre))
        out.append(pre.to_numpy())
        do(lambda m, e: hip.sum_to(A, e))
        params = {k: (Matrix.from_numpy(x.copy()), g) for k, x, g in (("l.weight", a, B), ("l.bias", row, Row), ("frozen", b, None))}
        for opt in (hip.SGD(0.1), hip.Adam(0.1, 0.9, 0.99, 1e-8, params), hip.AdamW(0.1, 0.9, 0.99, 1e-8, 0.05, params, ["l.weight"])):
            opt.update(params)
            opt.update(params)
            out.extend(p.to_numpy() for p, _ in params.values())
            for k in ("l.weight", "l.bias"):
                if hasattr(opt, "m"):
                    out.extend((opt.m[k].to_numpy(), opt.v[k].to_numpy()))
        return out

    stream = C.c_void_p()
    _lib.check(hip.lib().zenu_hip_stream_create(C.byref(stream)), "stream_create")
    old = hip.get_stream()
    try:
        with General(monkeypatch):
            expect = all_calls()
        for s in (None, stream, stream.value):
            hip.set_stream(s)
            got = all_calls()
            hip.synchronize()
            assert len(got) == len(expect)
            for i, (x, y) in enumerate(zip(got, expect)):
                assert np.array_equal(x, y), (s, i)
    finally:
        hip.set_stream(old)
        _lib.check(hip.lib().zenu_hip_stream_destroy(stream), "stream_destroy")


@pytest.mark.gpu
def test_errors_are_the_same(hip, monkeypatch):
    A, B = (Matrix.from_numpy(np.zeros(s, np.float32)) for s in ((6, 5), (4, 3)))

    def errors():
        seen = []
        for fn in (lambda: A.add_array(A, B), lambda: A.copy_from(B), lambda: A.relu(B, 0.0), lambda: A.softmax_assign(B, 1),
                   lambda: hip.sum_to(B, A), lambda: A.softmax_assign(A, 2), lambda: A.copy_from(A.transpose()), lambda: A._unary_array(99, A),
                   lambda: A.add_array(A, 3), lambda: A.relu(A, "x"), lambda: A.mul_scalar(A, None)):
            try:
                fn()
                seen.append(None)
            except Exception as e:
                seen.append((type(e), getattr(e, "status", None), str(e)))
        return seen
    with General(monkeypatch):
        expect = errors()
    assert sum(isinstance(e, tuple) and e[0] is ZenuHipError for e in expect) >= 6
    assert errors() == expect
