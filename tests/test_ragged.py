"""Sizes and alignments that are nobody's choice: rows of odd length, views that start in the middle of a
vector, edge tiles one element wide.  The elementwise results are IEEE operations on the same operands, so
numpy gives the same bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64]
IDS = ["f32", "f64"]


def same(got, exp, what):
    assert got.shape == exp.shape and np.array_equal(got, exp), what


def offset_matrix(hip, a, off):
    """`a` in device memory `off` elements behind a 256-byte boundary"""
    flat = np.concatenate([np.zeros(off, a.dtype), a.reshape(-1)])
    m = hip.Matrix.from_numpy(flat)
    return hip.Matrix(m.buf, off, a.shape, hip.default_stride(a.shape), a.dtype)


# one element, around one vector, around the 32 / 64 tile edges and one row piece, a last tile of 1, 3, 4 and 63
EDGES = [(1, 1), (1, 5), (3, 2), (4, 4), (5, 3), (31, 33), (33, 31), (63, 65), (64, 64), (65, 129), (127, 68), (196, 130), (67, 1025)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", EDGES, ids=str)
def test_broadcast_and_transposed_operands(hip, dtype, shape):
    r = np.random.default_rng(shape[0] * 7 + shape[1])
    rows, cols = shape
    for off in (0, 1, 3):
        a, b = r.standard_normal(shape).astype(dtype), r.standard_normal((cols, rows)).astype(dtype)
        row, col = r.standard_normal(cols).astype(dtype), r.standard_normal((rows, 1)).astype(dtype)
        A, B, Row, Col = (offset_matrix(hip, t, o) for t, o in ((a, off), (b, 3 - off), (row, off // 2), (col, 1)))
        out = offset_matrix(hip, np.zeros(shape, dtype), 2 if off else 0)
        what = (shape, off)
        out.add_array(A, Row)
        same(out.to_numpy(), a + row, ("row", what))
        out.sub_array(Row, A)
        same(out.to_numpy(), row - a, ("row first", what))
        out.mul_array(A, Col)
        same(out.to_numpy(), a * col, ("column", what))
        out.add_array(A, B.transpose())
        same(out.to_numpy(), a + b.T, ("transposed", what))
        out.copy_from(B.transpose())
        same(out.to_numpy(), b.T, ("transposed copy", what))
        out.mul_scalar(A, 0.5)
        same(out.to_numpy(), a * dtype(0.5), ("scalar", what))
        A.add_assign(B.transpose())                        # in place: every element is added to once
        same(A.to_numpy(), a + b.T, ("transposed, in place", what))


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("cols", [1, 3, 4, 5, 15, 16, 17, 255, 1027])
def test_rows_of_a_wider_matrix(hip, dtype, cols):
    """row slices: neither the row starts nor the row length are multiples of a vector, and nothing outside is written"""
    r = np.random.default_rng(cols)
    wide = r.standard_normal((37, cols + 6)).astype(dtype)
    row = r.standard_normal(cols).astype(dtype)
    W, D, Row = hip.Matrix.from_numpy(wide), hip.Matrix.from_numpy(wide), hip.Matrix.from_numpy(row)
    at = (slice(None), slice(3, 3 + cols))
    D.slice(*at).add_array(W.slice(*at), Row)
    exp = wide.copy()
    exp[at] = wide[at] + row
    same(D.to_numpy(), exp, "slice + row")
    D.slice(*at).copy_from(W.slice(slice(None), slice(1, 1 + cols)))
    exp[at] = wide[:, 1:1 + cols]
    same(D.to_numpy(), exp, "slice copy")


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 7])
def test_short_rows_repeated(hip, dtype, cols):
    """a row shorter than a vector, as long, and longer, over many rows"""
    row = np.arange(1, cols + 1).astype(dtype)
    for rows in (1, 37, 3001):
        out = offset_matrix(hip, np.zeros((rows, cols), dtype), 1)
        out.broadcast(offset_matrix(hip, row, 3))
        same(out.to_numpy(), np.broadcast_to(row, (rows, cols)), rows)


def test_streaming_sizes(hip):
    """beyond the caches (streaming accesses), every operand starting in the middle of a vector"""
    r = np.random.default_rng(3)
    rows, cols = 2051, 2047
    a, b = r.standard_normal((rows, cols), dtype=np.float32), r.standard_normal((cols, rows), dtype=np.float32)
    row = r.standard_normal(cols, dtype=np.float32)
    A, B, Row = offset_matrix(hip, a, 1), offset_matrix(hip, b, 2), offset_matrix(hip, row, 3)
    out = offset_matrix(hip, np.zeros((rows, cols), np.float32), 1)
    out.add_array(A, Row)
    same(out.to_numpy(), a + row, "row")
    out.add_array(A, B.transpose())
    same(out.to_numpy(), a + b.T, "transposed")
    out.copy_from(B.transpose())
    same(out.to_numpy(), b.T, "transposed copy")
    out.relu(A, 0.0)
    same(out.to_numpy(), np.maximum(a, 0), "relu")


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("fn", ["sigmoid", "exp", "sin", "tanh_backward", "add"])
def test_small_tensors_give_the_bits_of_large_ones(hip, dtype, fn):
    """Transcendental functions over small tensors go one element per lane, over larger ones by vectors: both sides of
    either limit (2^17 and 2^20 elements on 256 CUs), single elements and every remainder of a vector, at two
    alignments, against the same elements inside a tensor beyond both limits; nothing else is written"""
    lim, r = 4096 * 256, np.random.default_rng(5)
    n_all = lim + 4099
    x, gy = (r.standard_normal(n_all) * 3).astype(dtype), r.standard_normal(n_all).astype(dtype)

    def run(n, off):
        whole = hip.Matrix.from_numpy(np.full(off + n + 4, 7, dtype))
        out = hip.Matrix(whole.buf, off, (n,), (1,), dtype)
        X, G = offset_matrix(hip, x[:n], off), offset_matrix(hip, gy[:n], 3)
        if fn == "sigmoid":
            code = hip._lib.F32 if dtype == np.float32 else hip._lib.F64
            hip._lib.check(hip.lib().zenu_hip_unary(hip._lib.SIGMOID, code, C.byref(out.desc()), C.byref(X.desc()), None), fn)
        elif fn == "tanh_backward":
            out.tanh_backward(G, X)
        elif fn == "add":
            out.add_array(X, G)
        else:
            getattr(out, fn + "_array")(X)
        got = whole.to_numpy()
        assert np.all(got[:off] == 7) and np.all(got[off + n:] == 7), (n, off)
        return got[off:off + n]

    expect = run(n_all, 0)
    for n in (1, 2, 3, 63, 65, 257, 511, 512, 514, 2047, 10007, 512 * 256, 512 * 256 + 1, lim - 1, lim, lim + 1, lim + 2, lim + 3):
        for off in (0, 1):
            assert np.array_equal(run(n, off), expect[:n]), (n, off)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("largest", [4099, 1 << 20], ids=["cached", "streamed"])
def test_optimizer_tensors_of_any_size_and_alignment(hip, dtype, largest):
    """More tensors than one launch holds, around a vector and a tile long, each at another alignment: the
    operations of the update are single IEEE operations, so the CPU gives the same bits; nothing else is written"""
    import zenu_oracle as zo
    r = np.random.default_rng(3)
    sizes = [1, 2, 3, 4, 5, 511, 512, 513, 1021, 1023, 1024, 1025, 1027, 2049, largest] * 5
    params, state, expect = {}, {"m": {}, "v": {}}, {}
    keep = []
    for i, n in enumerate(sizes):
        host = [r.standard_normal(n).astype(dtype) * s for s in (1, 0.1, 0.01)] + [np.square(r.standard_normal(n)).astype(dtype)]
        host = [np.ascontiguousarray(h, dtype) for h in host]
        dev = []
        for j, h in enumerate(host):
            m = hip.Matrix.from_numpy(np.concatenate([np.full(i % 4 if j else (i + 1) % 4, 7, dtype), h, np.full(3, 7, dtype)]))
            dev.append(hip.Matrix(m.buf, m.shape[0] - n - 3, (n,), (1,), dtype))
            keep.append((m, dev[-1]))
        name = f"t{i}.weight" if i % 2 else f"t{i}.bias"
        params[name] = (dev[0], dev[1])
        state["m"][name], state["v"][name] = dev[2], dev[3]
        p, g, m, v = (h.copy() for h in host)
        zo.adamw_update(p, g, m, v, 1e-2, 0.9, 0.999, 1e-8, 0.01, i % 2, 4)
        expect[name] = (p, m, v)
    opt = hip.AdamW(1e-2, 0.9, 0.999, 1e-8, 0.01, {}, [k for k in params if k.endswith("weight")])
    opt.m, opt.v, opt.step = state["m"], state["v"], 3
    opt.update(params)
    for name, (p, m, v) in expect.items():
        same(params[name][0].to_numpy(), p, (name, p.size, "parameter"))
        same(state["m"][name].to_numpy(), m, (name, p.size, "first moment"))
        same(state["v"][name].to_numpy(), v, (name, p.size, "second moment"))
    for whole, part in keep:
        around = np.delete(whole.to_numpy(), np.arange(part.offset, part.offset + part.shape[0]))
        assert np.all(around == 7)
    before = {k: p.to_numpy() for k, (p, _) in params.items()}
    hip.SGD(0.3).update(params)
    for name, (p, g) in params.items():
        same(p.to_numpy(), before[name] - g.to_numpy() * dtype(0.3), (name, "sgd"))


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", [(5, 1), (9, 3), (3, 16), (70, 17), (33, 31), (600, 129), (40, 1003), (2049, 127), (3, 8195),
                                   (1, 300001), (9000, 1021)], ids=str)
def test_reductions_at_any_alignment(hip, dtype, shape):
    """Sums, magnitudes, maxima and their first positions along both axes, rows starting anywhere in a vector, the
    source a whole tensor and a column slice of a wider one.  n terms added in any order are off by less than
    (n - 1) eps of the sum of their magnitudes."""
    rows, cols = shape
    r = np.random.default_rng(cols)
    eps = np.finfo(dtype).eps
    wide = r.standard_normal((rows, cols + 3)).astype(dtype)
    for a in (wide[:, :cols], wide[:, 2:cols + 2]):
        a = np.ascontiguousarray(a)
        if cols > 2:
            a[::3, cols - 1] = a[::3].max(axis=1)          # the maximum twice, the second time at the end
            a[1::4, 1] = np.nan                            # not in position 0: the scan passes over it
        clean = np.nan_to_num(a, nan=0.0)
        whole = offset_matrix(hip, a, 1)
        big = hip.Matrix.from_numpy(np.concatenate([np.full((rows, 3), 9, dtype), a, np.full((rows, 2), 9, dtype)], axis=1))
        part = big.slice(slice(None), slice(3, 3 + cols))
        for name, m in (("whole", whole), ("slice", part)):
            what = (shape, name)
            for axis, n in ((0, rows), (1, cols)):
                at = hip.Matrix.alloc((a.size // n,), np.float64)
                top = offset_matrix(hip, np.zeros(a.size // n, dtype), 1)
                code = hip._lib.F32 if dtype == np.float32 else hip._lib.F64
                hip._lib.check(hip.lib().zenu_hip_max_axis_idx(code, at.as_ptr(), C.byref(m.desc()), axis, None), "max_axis_idx")
                hip._lib.check(hip.lib().zenu_hip_max_axis(code, C.byref(top.desc()), C.byref(m.desc()), axis, None), "max_axis")
                # a NaN in position 0 stays; elsewhere it never replaces
                scan = np.where(np.isnan(a), -np.inf, a)
                first = np.isnan(np.take(a, 0, axis=axis))
                want = np.where(first, 0, np.argmax(scan, axis=axis))
                assert np.array_equal(at.to_numpy().view(np.int64), want), what
                picked = np.take_along_axis(a, np.expand_dims(want, axis), axis).reshape(-1)
                assert np.array_equal(top.to_numpy(), picked, equal_nan=True), what
        for name, m in (("whole", offset_matrix(hip, clean, 3)),):
            for axis, n in ((0, rows), (1, cols)):
                kept = (1, cols) if axis == 0 else (rows, 1)
                out = offset_matrix(hip, np.zeros(kept, dtype), 1)
                hip.sum_to(m, out)
                exact = clean.sum(axis=axis, keepdims=True, dtype=np.longdouble)
                bound = n * eps * np.abs(clean).sum(axis=axis, keepdims=True, dtype=np.longdouble)
                assert np.all(np.abs(out.to_numpy() - exact) <= bound), (shape, axis)
            total = hip.Matrix.alloc((1,), dtype)
            hip._lib.check(hip.lib().zenu_hip_asum(hip._lib.F32 if dtype == np.float32 else hip._lib.F64, total.as_ptr(),
                                                   C.byref(m.desc()), None), "asum")
            exact = np.abs(clean).sum(dtype=np.longdouble)
            assert abs(total.to_numpy()[0] - exact) <= clean.size * eps * exact, shape


# rows of a wavefront's lanes and one around them; columns: one per lane, narrow and wide vector tiles, each with and
# without splits, around the limits of rows (512, 1024, 4096) and columns (64, 128, 256, 512)
EXACT = [(70, 63), (70, 64), (70, 65), (64, 17), (513, 65), (600, 127), (1024, 129), (1025, 127), (1025, 131), (2048, 255), (3000, 257),
         (4097, 33), (5000, 67), (10007, 127), (30001, 65), (3000, 513), (1000, 1001)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", EXACT, ids=str)
def test_reductions_of_small_integers_are_exact(hip, dtype, shape):
    """Integers of -15 .. 15 without 0: every partial sum stays below 2^24, so any order of the additions gives the exact
    result in f32, and an element that is lost, added twice or taken from beside the source changes it.  The same source
    gives the first positions of the maxima, of which every row and column holds several."""
    rows, cols = shape
    r = np.random.default_rng(rows + cols)
    a = (r.integers(1, 16, shape) * r.choice([-1, 1], shape)).astype(dtype)
    whole = offset_matrix(hip, a, 1)
    big = hip.Matrix.from_numpy(np.concatenate([np.full((rows, 3), 1e6, dtype), a, np.full((rows, 2), 1e6, dtype)], axis=1))
    code = hip._lib.F32 if dtype == np.float32 else hip._lib.F64
    for m in (hip.Matrix.from_numpy(a), whole, big.slice(slice(None), slice(3, 3 + cols))):
        for axis in (0, 1):
            kept = (1, cols) if axis == 0 else (rows, 1)
            out = offset_matrix(hip, np.full(kept, 7, dtype), 1)
            hip.sum_to(m, out)
            same(out.to_numpy(), a.sum(axis=axis, keepdims=True), ("sum", shape, axis))
            at = hip.Matrix.alloc((a.size // a.shape[axis],), np.float64)
            hip._lib.check(hip.lib().zenu_hip_max_axis_idx(code, at.as_ptr(), C.byref(m.desc()), axis, None), "max_axis_idx")
            same(at.to_numpy().view(np.int64), np.argmax(a, axis=axis), ("arg-max", shape, axis))
    total = hip.Matrix.alloc((1,), dtype)
    few = offset_matrix(hip, np.clip(a, -1, 1), 3)
    hip._lib.check(hip.lib().zenu_hip_asum(code, total.as_ptr(), C.byref(few.desc()), None), "asum")
    assert total.to_numpy()[0] == a.size


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", [(3, 1), (5, 3), (4, 256), (7, 1500), (33, 1027), (9000, 999), (8200, 1024)], ids=str)
@pytest.mark.parametrize("with_pre", [True, False])
def test_bias_relu_at_any_alignment(hip, dtype, shape, with_pre):
    r = np.random.default_rng(shape[1])
    z, bias = r.standard_normal(shape).astype(dtype), r.standard_normal(shape[1]).astype(dtype)
    act, pre = offset_matrix(hip, np.zeros(shape, dtype), 3), offset_matrix(hip, np.zeros(shape, dtype), 2)
    act.bias_add_relu(offset_matrix(hip, z, 1), offset_matrix(hip, bias, 1), 0.25, pre=pre if with_pre else None)
    a = z + bias
    if with_pre:
        same(pre.to_numpy(), a, ("pre", shape))
    same(act.to_numpy(), np.where(a > 0, a, dtype(0.25) * a), ("act", shape))


# the kept run in front, in the middle and at the end; pieces shorter than a vector, of one vector, longer than a
# workgroup; more channels than workgroups wanted, fewer, and so few that the axes go one after the other
SUMS = [((2, 3, 5, 7), (1, 3, 1, 1)), ((64, 5, 2, 1), (1, 5, 1, 1)), ((6, 4, 3, 1), (1, 4, 1, 1)), ((9, 16, 2, 2), (1, 16, 1, 1)),
        ((64, 33, 14, 14), (1, 33, 1, 1)), ((130, 3, 65, 67), (1, 3, 1, 1)), ((2, 2, 80, 81), (1, 2, 1, 1)), ((1, 40, 9, 11), (1, 40, 1, 1)),
        ((3, 600, 7, 7), (1, 600, 1, 1)), ((20, 70, 90, 91), (1, 70, 1, 1)), ((4, 5, 6, 37), (37,)), ((4, 5, 6, 37), (6, 37)), ((7, 3, 5), ()),
        ((3, 4, 5, 6), (1, 4, 1, 6)), ((3, 4, 5, 6), (3, 1, 1, 6))]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape,kept", SUMS, ids=str)
def test_sums_over_several_axes(hip, dtype, shape, kept):
    """n terms added in any order are off by less than (n - 1) eps of the sum of their magnitudes"""
    x = np.random.default_rng(len(kept)).standard_normal(shape).astype(dtype)
    out = offset_matrix(hip, np.full(kept, 5, dtype), 1)
    hip.sum_to(offset_matrix(hip, x, 1), out)
    axes = tuple(i for i in range(len(shape)) if i < len(shape) - len(kept) or (len(kept) == len(shape) and kept[i] != shape[i]))
    wide = x.astype(np.longdouble)
    exact, scale = wide.sum(axis=axes).reshape(kept), np.abs(wide).sum(axis=axes).reshape(kept)
    n = x.size // max(exact.size, 1)
    assert np.all(np.abs(out.to_numpy() - exact) <= n * np.finfo(dtype).eps * scale)


# channels fewer and more than compute units (one and several workgroups per channel), pieces of part of a cache line, of
# whole ones and of one and a part, and a million pieces, whose axes go one after the other
PIECES = [(5, 3, 7), (2, 256, 4), (37, 257, 9), (130, 300, 25), (600, 31, 32), (9, 520, 64), (70, 513, 16), (2100, 500, 4), (3, 40, 3001)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", PIECES, ids=str)
def test_sums_over_images_and_pixels_are_exact(hip, dtype, shape):
    """integers whose sums are exact in any order, the source starting at three alignments; one element counted twice or
    left out changes a channel's sum"""
    n, c, i = shape
    r = np.random.default_rng(sum(shape))
    x = (r.integers(1, 16, shape) * r.choice([-1, 1], shape)).astype(dtype)
    exp = x.sum(axis=(0, 2), keepdims=True)
    for off in (0, 1, 32):
        out = offset_matrix(hip, np.full((1, c, 1), 7, dtype), 1)
        hip.sum_to(offset_matrix(hip, x, off), out)
        same(out.to_numpy(), exp, (shape, off))


# rows that don't start at cache lines, in column tiles that are dealt to the XCDs in bands: one tile, fewer tiles than
# XCDs, a number of them that 8 does not divide; one workgroup per tile and several; the gradient on the loads
BANDS = [(1, 40, 36), (1, 300, 1404), (1, 1000, 1500), (1, 2100, 1004), (5, 33, 1004), (3, 1100, 716), (1, 9, 4100)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", BANDS, ids=str)
def test_column_tiles_that_share_cache_lines_are_exact(hip, dtype, shape):
    """small integers: every order of the sums gives the same value"""
    outer, rows, cols = shape
    r = np.random.default_rng(cols)
    a = r.integers(-8, 9, shape).astype(dtype)
    for off in (0, 1, 4):
        m = offset_matrix(hip, a, off)
        same(m.sum(1).to_numpy().reshape(outer, cols), a.sum(axis=1), (shape, off, "sum"))
        same(np.array(m.max_axis_idx_ravel(1)).reshape(outer, cols), a.argmax(axis=1), (shape, off, "position"))
    if outer == 1:
        x = r.integers(-3, 4, (rows, cols)).astype(dtype)
        gy, gx, gb = (hip.Matrix.from_numpy(t) for t in (a[0], np.zeros((rows, cols), dtype), np.zeros(cols, dtype)))
        gx.relu_backward_bias_grad(gb, gy, hip.Matrix.from_numpy(x), 0.0)
        grad = a[0] * np.where(x > 0, dtype(1), dtype(0) * dtype(-1))
        same(gx.to_numpy(), grad, (shape, "gradient"))
        same(gb.to_numpy(), grad.sum(axis=0), (shape, "bias gradient"))
        gy.relu_backward_bias_grad(gb, gy, hip.Matrix.from_numpy(x), 0.0)      # in place
        same(gy.to_numpy(), grad, (shape, "gradient in place"))
        same(gb.to_numpy(), grad.sum(axis=0), (shape, "bias gradient in place"))


# runs of one element less than a vector to one more than the kernel for a short side takes, last workgroups of 1 .. 64 positions,
# sizes on both sides of the line below which square tiles take the copy
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", [(130, 1, 64), (129, 2, 65), (17, 3, 1023), (3, 3, 4097), (9, 4, 1024), (33, 5, 259), (1, 7, 9001), (140, 16, 67),
                                   (86, 23, 96), (2, 24, 4161), (2, 24, 4096), (40, 25, 300), (300, 3, 49)], ids=str)
def test_copies_with_one_short_side(hip, dtype, shape):
    r = np.random.default_rng(shape[2])
    n, short, long = shape
    for off in (0, 1):
        a = r.standard_normal(shape).astype(dtype)
        A = offset_matrix(hip, a, off)
        out = offset_matrix(hip, np.full((n, long, short), 7, dtype), 3 - off)
        out.copy_from(A.transpose())
        same(out.to_numpy(), a.transpose(0, 2, 1), ("into the short side", shape, off))
        back = offset_matrix(hip, np.full(shape, 7, dtype), off)
        back.copy_from(out.transpose())
        same(back.to_numpy(), a, ("out of it", shape, off))
        # runs that are part of longer ones, on either side; nothing else is written
        wide = hip.Matrix.from_numpy(np.full((n, short, long + 5), 7, dtype))
        wide.slice(slice(0, n), slice(0, short), slice(2, long + 2)).copy_from(out.transpose())
        exp = np.full((n, short, long + 5), 7, dtype)
        exp[:, :, 2:long + 2] = a
        same(wide.to_numpy(), exp, ("into part of longer runs", shape, off))
        out.copy_from(wide.slice(slice(0, n), slice(0, short), slice(1, long + 1)).transpose())
        same(out.to_numpy(), exp[:, :, 1:long + 1].transpose(0, 2, 1), ("from part of longer runs", shape, off))


# column sums whose splits are folded by a launch of their own: 8 to 64 row lanes, two splits to a hundred, outputs that are no
# whole number of its workgroups, sources just below and above the size from which it is used.  Small whole numbers: every sum is exact
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", [(16383, 64), (16384, 64), (70001, 16), (65536, 33), (30000, 65), (4097, 257), (3000, 400), (1001, 1500), (517, 4100)],
                         ids=str)
def test_column_sums_folded_by_a_second_launch(hip, dtype, shape):
    r = np.random.default_rng(shape[0])
    a = r.integers(-3, 4, shape).astype(dtype)
    x = r.integers(-1, 2, shape).astype(dtype)
    rows, cols = shape
    for off in (0, 1):
        A, X = offset_matrix(hip, a, off), offset_matrix(hip, x, off)
        out = hip.Matrix.from_numpy(np.full(cols + 2, 7, dtype))
        hip.sum_to(A, hip.Matrix(out.buf, 1, (cols,), (1,), dtype))
        exp = np.full(cols + 2, 7, dtype)
        exp[1:-1] = a.sum(0, dtype=np.float64)
        same(out.to_numpy(), exp, ("column sums", shape, off))
        gx, gb = offset_matrix(hip, np.zeros(shape, dtype), off), hip.Matrix.from_numpy(np.zeros(cols, dtype))
        gx.relu_backward_bias_grad(gb, A, X, 0.0)
        g = np.where(x > 0, a, 0).astype(dtype)
        same(np.abs(gx.to_numpy()), np.abs(g), ("ReLU gradient", shape, off))
        same(gb.to_numpy(), g.sum(0, dtype=np.float64).astype(dtype), ("bias gradient", shape, off))


# How many accumulators a lane has where workgroups share a row, on both sides of the 32 MB from which there are eight and of
# the 128 MB from which the loads stream.  A value so large that single ones added to it are lost stands first; two ones
# stand where the first lane meets them as well, one by one, if it has four accumulators, and another workgroup adds them
# up first if it has eight.
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("mbytes,accumulators", [(31, 4), (32, 8), (100, 8), (127, 8), (128, 8), (160, 8)])
def test_accumulators_of_shared_rows(hip, dtype, mbytes, accumulators):
    size = np.dtype(dtype).itemsize
    vec, large = 16 // size, dtype(2) ** (24 if size == 4 else 53)
    splits = 512                                           # two workgroups on each of 256 CUs
    for rows in (1, 4):
        a = np.zeros((rows, mbytes * (1 << 20) // size // rows), dtype)
        second = 4 * 256 * vec * (splits // rows)          # the first workgroup's second chunk with four accumulators
        a[:, 0] = large
        a[:, second:second + 2] = 1
        assert second + 2 <= a.shape[1]
        exp = np.full(rows, large + 2 if accumulators == 8 else large, dtype)
        m = hip.Matrix.from_numpy(a)
        same((m.sum(1) if rows > 1 else m.sum_all()).to_numpy().reshape(rows), exp, ("sum", rows))
        if rows == 1:
            assert m.asum() == exp[0]


# sources on both sides of the sizes from which a reduction streams its loads: 40 MB (f32), 64 MB with the ReLU gradient, 128 MB
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("mbytes", [39, 41, 63, 65, 126, 130])
def test_reductions_of_large_sources_are_exact(hip, dtype, mbytes):
    """small integers: every order of the sums gives the same value"""
    cols = 2052
    rows = mbytes * (1 << 20) // (cols * np.dtype(dtype).itemsize)
    r = np.random.default_rng(mbytes)
    a = r.integers(-4, 5, (rows, cols)).astype(dtype)
    x = r.integers(-1, 2, (rows, cols)).astype(dtype)
    for off in (0, 1):
        m = offset_matrix(hip, a, off)
        same(m.sum(0).to_numpy(), a.sum(0, dtype=np.float64), ("column sums", off))
        same(m.sum(1).to_numpy(), a.sum(1, dtype=np.float64), ("row sums", off))
        same(np.array(m.max_axis_idx_ravel(0)), a.argmax(0), ("rows of the column maxima", off))
        same(np.array(m.max_axis_idx_ravel(1)), a.argmax(1), ("columns of the row maxima", off))
        pieces = hip.Matrix(m.buf, m.offset, (rows, cols // 9, 9), (cols, 9, 1), dtype)
        out = hip.Matrix.from_numpy(np.full((1, cols // 9, 1), 7, dtype))
        hip.sum_to(pieces, out)
        same(out.to_numpy().reshape(-1), a.reshape(rows, cols // 9, 9).sum((0, 2), dtype=np.float64), ("sums over pieces", off))
        gx, gb = hip.Matrix.from_numpy(np.zeros((rows, cols), dtype)), hip.Matrix.from_numpy(np.zeros(cols, dtype))
        gx.relu_backward_bias_grad(gb, m, offset_matrix(hip, x, off), 0.0)
        g = np.where(x > 0, a, dtype(0))
        same(gx.to_numpy(), g, ("ReLU gradient", off))
        same(gb.to_numpy(), g.sum(0, dtype=np.float64), ("bias gradient", off))


# Copies with a short side by the positions a workgroup takes, 2^7 to 2^11 of them (see the rule where ew_thin_kernel is
# launched), last workgroups that are not full, 16 KB of a workgroup filled and not, and sizes on both sides of those from
# which the stores stream and from which the loads do
THIN = [(128, 3, 12545), (600, 2, 1027), (300, 2, 20001), (200, 8, 3137), (64, 8, 3137), (16, 24, 12547), (90, 5, 9001), (150, 16, 2051), (128, 3, 32769), (270, 3, 32771)]


def thin_log_run(n, short, long, size):
    log_run = 6
    while short * size << (log_run + 1) <= 16384:
        log_run += 1
    while log_run > 6 and n * -(-long // (1 << log_run)) < 4 * 256:
        log_run -= 1
    return log_run


def test_short_sides_reach_every_length_of_run():
    assert {thin_log_run(*s, 4) for s in THIN} >= {7, 8, 9, 10, 11} and {thin_log_run(*s, 8) for s in THIN} >= {6, 7, 8, 9, 10}


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", THIN, ids=str)
def test_copies_with_one_short_side_and_long_runs(hip, dtype, shape):
    n, short, long = shape
    a = np.random.default_rng(long).standard_normal(shape, dtype=np.float32).astype(dtype)
    flipped = np.ascontiguousarray(a.transpose(0, 2, 1))
    for off, end in ((0, 0), (1, 2)):
        def framed(x):
            m = hip.Matrix.from_numpy(np.concatenate([np.full(off, 7, dtype), x.reshape(-1), np.full(9, 7, dtype)]))
            return hip.Matrix(m.buf, off, x.shape, hip.default_stride(x.shape), dtype)

        def frame_is_whole(m):
            ends = hip.Matrix(m.buf, 0, (off + a.size + 9,), (1,), dtype).to_numpy()
            return np.all(ends[:off] == 7) and np.all(ends[-9:] == 7)
        A, out, back = framed(a), framed(np.zeros_like(flipped)), framed(np.zeros_like(a))
        out.copy_from(A.transpose())
        same(out.to_numpy(), flipped, ("into the short side", off))
        back.copy_from(out.transpose())
        same(back.to_numpy(), a, ("out of it", off))
        assert frame_is_whole(out) and frame_is_whole(back)


# Elementwise kernels by the way their operands pass the caches: megabytes of one operand such that one and two inputs are
# cached, kept, fed to the next call and streamed (32 MB moved; 72 MB of inputs; 192 MB moved)
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("mbytes", [13, 20, 38, 80, 105])
def test_elementwise_calls_of_every_size_class(hip, dtype, mbytes):
    cols = 2052
    rows = mbytes * (1 << 20) // (cols * np.dtype(dtype).itemsize) // 9 * 9 + 9
    r = np.random.default_rng(mbytes)
    shape, (n, c, hw) = (rows, cols), (rows // 9, 12, 9 * cols // 12)
    a, b = (r.standard_normal(shape, dtype=np.float32).astype(dtype) for _ in range(2))
    row, column, channel = (r.standard_normal(k, dtype=np.float32).astype(dtype) for k in ((cols,), (rows, 1), (1, c, 1)))
    for off in (0, 1):
        out = hip.Matrix.from_numpy(np.full(rows * cols + 16, 7, dtype))

        def into(s):
            return hip.Matrix(out.buf, off, s, hip.default_stride(s), dtype)

        def check(fn, exp, what):
            m = into(exp.shape)
            fn(m)
            same(m.to_numpy(), exp, (what, off))
            ends = hip.Matrix(out.buf, 0, (off + exp.size + 8,), (1,), dtype).to_numpy()
            assert np.all(ends[:off] == 7) and np.all(ends[-8:] == 7), (what, off)
        A, B = offset_matrix(hip, a, off), offset_matrix(hip, b, off)
        Row, Column, Channel = (hip.Matrix.from_numpy(x) for x in (row, column, channel))
        images = hip.Matrix(A.buf, off, (n, c, hw), hip.default_stride((n, c, hw)), dtype)
        check(lambda m: m.add_array(A, B), a + b, "a + b")
        check(lambda m: m.copy_from(A), a, "copy")
        check(lambda m: m.abs_array(A), np.abs(a), "abs")
        check(lambda m: m.relu(A, 0.5), np.where(a > 0, a, a * dtype(0.5)), "relu")
        check(lambda m: m.relu_backward(B, A, 0.5), b * np.where(a > 0, dtype(1), dtype(-0.5)), "relu backward")
        check(lambda m: m.add_array(A, Row), a + row, "a + row")
        check(lambda m: m.mul_array(A, Column), a * column, "a * column")
        check(lambda m: m.add_array(images, Channel), a.reshape(n, c, hw) + channel, "images + channel")
        check(lambda m: m.broadcast(Row), np.broadcast_to(row, shape), "broadcast")
        turned = hip.Matrix(B.buf, off, (cols, rows), (rows, 1), dtype)
        check(lambda m: m.add_array(A, turned.transpose()), a + b.reshape(cols, rows).T, "a + b^T")
        check(lambda m: m.copy_from(turned.transpose()), np.ascontiguousarray(b.reshape(cols, rows).T), "transposed copy")
        check(lambda m: m.abs_array(turned.transpose()), np.abs(b.reshape(cols, rows).T), "transposed abs")
        check(lambda m: m.add_array(m, B), into(shape).to_numpy() + b, "in place")


def in_steps(x, lanes):
    """the lanes' sums added as the column kernels add them: lanes 0 .. 7 first take every eighth, then lane 0 the rest"""
    x = [x[i] for i in range(lanes)]
    if lanes > 8:
        for i in range(8):
            for w in range(i + 8, lanes, 8):
                x[i] = x[i] + x[w]
    for w in range(1, min(lanes, 8)):
        x[0] = x[0] + x[w]
    return x[0]


def column_sums_in_order(a, lanes, splits):
    """every `lanes` rows of a chunk of four times as many go to the lanes, the chunks to the splits in turn"""
    rows, cols = a.shape
    partial = []
    for s in range(splits):
        acc = np.zeros((lanes, cols), a.dtype)
        for b in range(s * 4 * lanes, rows, splits * 4 * lanes):
            for r in range(b, min(b + 4 * lanes, rows), lanes):
                part = a[r:r + lanes]
                acc[:len(part)] = acc[:len(part)] + part
        partial.append(in_steps(acc, lanes))
    if splits == 1:
        return partial[0]
    acc = np.zeros((lanes, cols), a.dtype)
    for s in range(splits):
        acc[s % lanes] = acc[s % lanes] + partial[s]
    return in_steps(acc, lanes)


# The order of column sums, with and without a launch of their own for the splits: (rows, columns, log2 of the lanes along a
# row, splits), lanes and splits as the rule of the dispatch has them on 256 CUs
ORDERS = {np.float32: [(1000, 640, 5, 16), (3000, 400, 5, 47), (3000, 200, 3, 12), (1100, 1500, 5, 18), (520, 2100, 5, 9), (30000, 65, 3, 118), (3001, 65, 3, 12)],
          np.float64: [(1000, 300, 5, 16), (3000, 400, 5, 47), (1100, 1500, 5, 18), (520, 2100, 5, 9), (30000, 33, 3, 118)]}


@pytest.mark.parametrize("dtype,geometry", [(d, g) for d in DTYPES for g in ORDERS[d]], ids=str)
def test_order_of_column_sums(hip, dtype, geometry):
    rows, cols, shift, splits = geometry
    r = np.random.default_rng(rows)
    a = (r.standard_normal((rows, cols)) * 10.0 ** r.integers(-3, 4, (rows, 1))).astype(dtype)
    a[5] = -0.0
    exp = column_sums_in_order(a, 256 >> shift, splits)
    m, out = hip.Matrix.from_numpy(a), hip.Matrix.zeros((cols,), dtype)
    hip.sum_to(m, out)
    got = out.to_numpy()
    same(got.view(np.uint8), exp.view(np.uint8), "column sums")
    gx, gb = hip.Matrix.zeros(a.shape, dtype), hip.Matrix.zeros((cols,), dtype)
    gx.relu_backward_bias_grad(gb, m, hip.Matrix.from_numpy(np.ones_like(a)), 0.0)
    same(gb.to_numpy().view(np.uint8), exp.view(np.uint8), "with the ReLU gradient")
