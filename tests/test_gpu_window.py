"""Windowed tiles (vnec_win.hip): what the learned mode, SpB_mxv and the
Build_VNEC_* plans run in place of merge-path, block and slice kernels.

Each matrix sits at an edge of the layout — a tile's end, a row cut by one or
many tile boundaries, rows without nonzeros, windows too sparse for 16-bit
lists, columns repeated or descending — and is checked per row against the
oracle's long-double sums, |y - y_ref| <= tol (|A||x|)_i: 1e-12 for FP64 and hi
+ lo values, 2^-23 for hi-only, the FP32 API's row gate for FP32; against the
general merge-path plan of the same matrix within twice that; and bit for bit
over repeated and replayed launches."""
import numpy as np
import pytest

import oracle as O
from vnec_amd import matgen as g
from vnec_amd import spb

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-12, "hilo": 1e-12, "hi": 2.0 ** -23}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if spb.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    spb.init()


def _windowed(p):
    return bool(spb.L.load().vnec_plan_windowed(p.h))


def _chosen(A, variant, ipt, lanes=64):
    """The plan the library makes of a shape it has chosen itself."""
    f = spb.L.load().vnec_plan_build_chosen
    f.argtypes = [spb.C.c_void_p] * 3
    p = spb.Plan.__new__(spb.Plan)
    p.A, p.h = A, spb.C.c_void_p()
    t = spb.L.Tuning(spb.VNEC_VAR[variant], ipt, lanes, spb.VNEC_ENC["fp64"], 1, -1)
    spb.L.check(f(spb.C.byref(p.h), A.h, spb.C.byref(t)), "vnec_plan_build_chosen")
    return p


def _items(p, m):
    """Nonzeros per thread of a windowed plan, from its tiles: each holds up to
    512 of these, rows weighing an eighth."""
    per = (m.nnz + m.nrows / 8) / p.info().ntiles / 512
    return next(i for i in (4, 8, 16) if per <= i)


def _rows(lens, ncols, seed, cols=None):
    """CSR of the given row lengths; columns random, ascending and distinct
    within a row unless given."""
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    if cols is None:
        cols = np.concatenate([np.sort(rng.choice(ncols, n, replace=False)) for n in lens] or [np.zeros(0)])
    return g.from_pattern(len(lens), ncols, ptr, cols.astype(np.int32), seed=seed)


def _tile_edge(n):  # n nonzeros in rows of one, then a last row of three
    return _rows([1] * (n - 3) + [3], 4096, n)


def _cut_rows():  # rows over 1, 2, 3, 5, 9 and 40 tiles of 2048, short and empty ones between
    lens = []
    for k in (1, 2, 3, 5, 9, 40):
        lens += [0, 2, 2048 * k - 7, 1, 0, 0, 5]
    return _rows(lens, 100000, 5)


def _empty_stretches():
    return _rows([0] * 5000 + [3, 0, 4] * 40 + [0] * 70000 + [64, 0, 1] + [0] * 3000, 2000, 6)


def _sparse_window():  # 64 neighbouring window entries lie half a million columns apart
    return _rows([3] * 400, 8_000_000, 7)


def _repeated_descending():
    rng = np.random.default_rng(8)
    lens = rng.integers(0, 40, 3000)
    return _rows(lens, 500, 8, cols=np.concatenate(
        [np.sort(np.repeat(rng.integers(0, 500, n), 1))[::-1] for n in lens]))


def _lds_limit():  # rows of one nonzero, then rows of six
    rng = np.random.default_rng(13)
    lens = np.repeat([1, 6], [300000, 220000])
    return _rows(lens, 1 << 20, 13, cols=rng.integers(0, 1 << 20, int(lens.sum())))


def _mixed_wide():  # long rows of consecutive columns beside rows over eight million columns
    rng = np.random.default_rng(14)
    lens = [3] * 900 + [9000] + [3] * 900 + [70] * 60 + [2] * 40
    cols = [np.sort(rng.integers(0, 8_000_000 if n == 3 else 20_000, n)) if n < 9000 else np.arange(n) for n in lens]
    return _rows(lens, 8_000_000, 14, cols=np.concatenate(cols))


def _large_x(ncols):
    """400 rows over the whole of ncols columns, the first and the last one
    among them: row offsets, columns, the columns used, the columns' positions
    among those, values."""
    rng = np.random.default_rng(16)
    col = rng.integers(0, ncols, 400 * 7)
    col[[0, -1]] = 0, ncols - 1
    used, inv = np.unique(col, return_inverse=True)
    return (np.arange(0, len(col) + 1, 7), col.astype(np.int32), used, inv.astype(np.int32).ravel(),
            rng.uniform(-1, 1, len(col)))


MATRICES = {
    "one": lambda: _rows([1], 1, 1),
    "edge2047": lambda: _tile_edge(2047), "edge2048": lambda: _tile_edge(2048), "edge2049": lambda: _tile_edge(2049),
    "cut_rows": _cut_rows, "empty_stretches": _empty_stretches, "sparse_window": _sparse_window,
    "mixed_wide": _mixed_wide,
    "repeated_descending": _repeated_descending,
    "ipt8": lambda: g.powerlaw(60013, 2.2, 3, 20000, seed=9),   # 4096-item tiles, long rows
    "ipt16": lambda: g.rmat(17, 12, seed=10),                   # 8192-item tiles
    "short_rows": lambda: g.uniform(393241, 3, seed=11),        # a row end every two or three nonzeros
    "lds_limit": _lds_limit,                                    # 8192-item tiles of FP64 leave no room for two
    "dense_row": lambda: g.skew(13, 80, 2, 8000, seed=12),
}
ITEMS = {"cut_rows": (4, 4), "ipt8": (8, 8), "ipt16": (16, 16), "short_rows": (4, 4), "lds_limit": (8, 16)}  # FP64, FP32


def _check(m, y, enc, ref=None):
    if enc == "fp32":
        v, x = m.val.astype(np.float32), m.x.astype(np.float32)
        ax, _ = O.spmv_abs(m.ptr, m.col, v.astype(np.float64), x.astype(np.float64))
        return O.check_rows_f32(y, O.spmv_serial_f32(m.ptr, m.col, v, x) if ref is None else ref, m.ptr, ax)
    ax, yl = O.spmv_abs(m.ptr, m.col, m.val, m.x)
    return O.check_rows(y, yl if ref is None else ref, ax, TOL[enc] * (1 if ref is None else 2))


@pytest.mark.parametrize("enc", ["fp64", "hilo", "hi", "fp32"])
@pytest.mark.parametrize("name", list(MATRICES))
def test_windowed_plan_matches_oracle_and_general_plan(name, enc):
    m = MATRICES[name]()
    dt = np.float32 if enc == "fp32" else np.float64
    print(f"windowed {name} {enc}: {m.nrows} x {m.ncols}, {m.nnz} nonzeros", flush=True)
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val.astype(dt), dtype=dt)
    p = spb.Plan(A, "learned", encoding=enc)
    if p.info().variant == "G":
        pytest.fail("a pattern matrix: not what this test is for")
    assert _windowed(p), p.info()
    if name in ITEMS:
        assert _items(p, m) == ITEMS[name][enc == "fp32"]
    q = spb.Plan(A, "L", 7, encoding=enc, grid=-1)  # a named shape keeps its kernel
    assert not _windowed(q)
    dx = spb.DeviceArray.from_array(m.x.astype(dt))
    ys = []
    for run in (p.spmv_dev, p.spmv_dev, p.spmv_graph, p.spmv_graph, q.spmv_dev):
        dy = spb.DeviceArray.from_array(np.full(m.nrows, np.nan, dt))
        run(dx.ptr, dy.ptr)
        ys.append(dy.to_array(dt, m.nrows))
        dy.free()
    for y in ys[1:4]:
        assert np.array_equal(y.view(np.uint8), ys[0].view(np.uint8)), "repeated SpMV changed bits"
    ok, worst = _check(m, ys[0], enc)
    assert ok, worst
    ok, worst = _check(m, ys[0], enc, ref=ys[4])
    assert ok, worst
    fb, _ = p.format_bytes()
    assert fb >= (4 if enc in ("hi", "fp32") else 8) * m.nnz
    for h in (p, q):
        h.free()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_windowed_infinities_and_nan_stay_in_their_rows(dt):
    """x entries of +Inf, -Inf and NaN reach exactly the rows that hold their
    columns — not the slots a tile leaves unused, nor the next launch through
    the partial sums of rows that many tiles share — and the sums agree with
    the general plan's class by class."""
    m = _cut_rows()
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val.astype(dt), dtype=dt)
    p, q = spb.Plan(A, "learned"), spb.Plan(A, "L", 7, grid=-1)
    assert _windowed(p)
    long_row = int(np.argmax(np.diff(m.ptr)))
    lo = int(m.ptr[long_row])
    clean = m.x.astype(dt)
    want = None
    for bad in ({}, {m.col[lo]: np.inf}, {m.col[lo]: np.nan, m.col[lo + 5000]: -np.inf, 0: np.inf}, {}):
        x = clean.copy()
        for c, v in bad.items():
            x[c] = v
        dx = spb.DeviceArray.from_array(x)
        out = []
        for plan in (p, q):
            dy = spb.DeviceArray.from_array(np.zeros(m.nrows, dt))
            plan.spmv_dev(dx.ptr, dy.ptr)
            out.append(dy.to_array(dt, m.nrows))
            dy.free()
        dx.free()
        assert np.array_equal(np.isnan(out[0]), np.isnan(out[1]))
        assert np.array_equal(np.isinf(out[0]), np.isinf(out[1]))
        assert np.array_equal(np.sign(out[0][np.isinf(out[0])]), np.sign(out[1][np.isinf(out[1])]))
        if not bad:
            want = out[0] if want is None else want
            assert np.array_equal(out[0], want)
    p.free()
    q.free()


@pytest.mark.parametrize("kind", ["L", "D", "S"])
def test_reference_entries_run_windowed_tiles(kind):
    """Build_VNEC_L / D / S on scattered columns run windowed tiles; y matches
    the oracle's rows."""
    m = g.rmat(13, 16, seed=14)
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    plan = spb.build_vnec(kind, A)
    lib = spb.L.load()
    assert lib.vnec_plan_windowed(spb.C.c_void_p(lib.VNEC_plan_of_ext(spb.C.cast(plan, spb.C.c_void_p))))
    y = spb.Vector(m.nrows)
    assert spb.spmv_vnec(kind, y, A, spb.Vector.from_array(m.x), plan) == ""
    ok, worst = _check(m, y.to_array(), "fp64")
    assert ok, worst
    spb.free_vnec(kind, plan)


def test_window_relabelled_columns_beyond_the_training_sizes():
    """Above 2^24 nonzeros and 2 MiB of x the learned mode measures windowed
    tiles over relabelled columns too: the sums are right whichever it keeps."""
    m = g.uniform(2_100_011, 8, seed=15)
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    assert m.nnz > 1 << 24
    p = spb.Plan(A, "learned")
    assert _windowed(p)
    dx = spb.DeviceArray.from_array(m.x)
    dy = spb.DeviceArray(8 * m.nrows)
    p.spmv_dev(dx.ptr, dy.ptr)
    ok, worst = _check(m, dy.to_array(np.float64, m.nrows), "fp64")
    assert ok, (p.info(), worst)
    p.free()


@pytest.mark.parametrize("m", [g.rmat(12, 8, seed=19), g.rmat(17, 12, seed=10)], ids=["4_a_thread", "16_a_thread"])
def test_windowed_tiles_over_relabelled_columns(m):
    """Hot-first relabelled columns and a permuted x: the plain plan's bits,
    direct and replayed."""
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    plain, rel = _chosen(A, "L", 7), _chosen(A, "L", 7, spb.LANES_RELABEL)
    assert _windowed(plain) and _windowed(rel)
    assert rel.info().lanes & spb.LANES_RELABEL and not plain.info().lanes & spb.LANES_RELABEL
    dx, ys = spb.DeviceArray.from_array(m.x), []
    for run in (plain.spmv_dev, rel.spmv_dev, rel.spmv_graph, rel.spmv_graph):
        dy = spb.DeviceArray.from_array(np.full(m.nrows, np.nan))
        run(dx.ptr, dy.ptr)
        ys.append(dy.to_array(np.float64, m.nrows))
    ok, worst = _check(m, ys[0], "fp64")
    assert ok, worst
    for y in ys[1:]:
        assert np.array_equal(y.view(np.uint64), ys[0].view(np.uint64))


@pytest.mark.parametrize("n,hb,windowed", [(29999, 10, True), (30000, 10, False), (14425, 9, False)])
def test_short_pattern_matrices_run_windowed_tiles(n, hb, windowed):
    """Pattern matrices below 30000 rows of at least 20 entries: windowed tiles
    where the library has chosen pattern slices, pattern slices where they are
    named."""
    m = g.banded(n, hb, seed=17)
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    p, q = _chosen(A, "G", 8), spb.Plan(A, "G")
    assert p.info().variant == q.info().variant == "G"
    assert _windowed(p) == windowed and not _windowed(q)
    dx = spb.DeviceArray.from_array(m.x)
    for plan in (p, q):
        dy = spb.DeviceArray.from_array(np.full(m.nrows, np.nan))
        plan.spmv_dev(dx.ptr, dy.ptr)
        ok, worst = _check(m, dy.to_array(np.float64, m.nrows), "fp64")
        assert ok, worst
        dy.free()
        plan.free()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_windowed_large_x(dt):
    """x of 4 GiB and more, whose tiles read 32-bit column lists throughout:
    the same columns as in a small matrix, the same bits."""
    ncols = (1 << 32) // np.dtype(dt).itemsize + 999
    print(f"windowed large x: {ncols} columns, {np.dtype(dt)}", flush=True)
    ptr, col, used, inv, val = _large_x(ncols)
    n, xs = len(ptr) - 1, np.random.default_rng(1).uniform(-1, 1, len(used)).astype(dt)
    y = []
    for nc, c in ((ncols, col), (len(used), inv)):
        A = spb.Matrix.from_csr(n, nc, ptr, c, val.astype(dt), dtype=dt)
        p = spb.Plan(A, "learned")
        assert _windowed(p)
        dx, dy = spb.DeviceArray(xs.itemsize * nc), spb.DeviceArray.from_array(np.full(n, np.nan, dt))
        for at, v in zip(used if nc == ncols else range(nc), xs.reshape(-1, 1)):
            spb.L.check(spb.L.load().vnec_memcpy_h2d_ext(dx.ptr + xs.itemsize * int(at), v.ctypes.data, v.nbytes), "h2d")
        p.spmv_dev(dx.ptr, dy.ptr)
        y.append(dy.to_array(dt, n))
        for h in (p, dx, dy):
            h.free()
    assert np.array_equal(y[0].view(np.uint8), y[1].view(np.uint8))
    ax, ref = O.spmv_abs(ptr, inv, val.astype(dt).astype(np.float64), xs.astype(np.float64))
    if dt == np.float32:
        ok, worst = O.check_rows_f32(y[0], O.spmv_serial_f32(ptr, inv, val.astype(dt), xs), ptr, ax)
    else:
        ok, worst = O.check_rows(y[0], ref, ax, TOL["fp64"])
    assert ok, worst


class _FuncAttributes(spb.C.Structure):  # hipFuncAttributes
    _fields_ = [("binaryVersion", spb.C.c_int), ("cacheModeCA", spb.C.c_int), ("constSizeBytes", spb.C.c_size_t),
                ("localSizeBytes", spb.C.c_size_t), ("maxDynamicSharedSizeBytes", spb.C.c_int),
                ("maxThreadsPerBlock", spb.C.c_int), ("numRegs", spb.C.c_int), ("preferredShmemCarveout", spb.C.c_int),
                ("ptxVersion", spb.C.c_int), ("sharedSizeBytes", spb.C.c_size_t)]


def test_plans_of_one_kernel_keep_its_lds_limit():
    """A plan with a small window, built while one with a large window of the
    same kernel is alive, leaves the kernel's LDS limit and the first plan's
    results alone."""
    lib, hip = spb.L.load(), spb.C.CDLL("libamdhip64.so")

    def limit():
        a = _FuncAttributes()
        kernel = spb.C.addressof(spb.C.c_char.in_dll(lib, "_Z10k_spmv_winILi16ELi0ELb1EEv13vnec_win_argsi"))
        assert hip.hipFuncGetAttributes(spb.C.byref(a), spb.C.c_void_p(kernel)) == 0
        return a.maxDynamicSharedSizeBytes

    big = g.rmat(17, 12, seed=10)
    n = 20011  # rows of 80 among 2000 columns, no two of them neighbours
    cols = 2 * np.sort(np.random.default_rng(18).integers(0, 2000, (n, 80)), axis=1)
    small = _rows([80] * n, 4000, 18, cols=cols.ravel())
    A = spb.Matrix.from_csr(big.nrows, big.ncols, big.ptr, big.col, big.val)
    p = spb.Plan(A, "learned")
    dx, dy = spb.DeviceArray.from_array(big.x), spb.DeviceArray(8 * big.nrows)
    p.spmv_dev(dx.ptr, dy.ptr)
    want, before = dy.to_array(np.float64, big.nrows), limit()
    B = spb.Matrix.from_csr(small.nrows, small.ncols, small.ptr, small.col, small.val)
    q = spb.Plan(B, "learned")
    for plan, m in ((p, big), (q, small)):  # 16 nonzeros a thread, both
        assert _windowed(plan) and plan.info().ntiles < m.nnz / 4096
    assert limit() == before >= 128 << 10
    for run in (p.spmv_dev, p.spmv_graph, p.spmv_graph):
        dy = spb.DeviceArray.from_array(np.full(big.nrows, np.nan))
        run(dx.ptr, dy.ptr)
        assert np.array_equal(dy.to_array(np.float64, big.nrows).view(np.uint64), want.view(np.uint64))
    dx, dy = spb.DeviceArray.from_array(small.x), spb.DeviceArray(8 * small.nrows)
    q.spmv_dev(dx.ptr, dy.ptr)
    ok, worst = _check(small, dy.to_array(np.float64, small.nrows), "fp64")
    assert ok, worst
