"""Stream tiles (vnec_spmm.hip): what plans of several right-hand sides run
where the library chooses the kernel (FP64, k = 2, 4, 8, 16).

Matrices at the edges of the layout — one nonzero, a tile's end, rows cut by
many tiles, stretches of empty rows, the size at which streams lengthen — are
checked per row and column against the oracle's sums, |y - y_ref| <= 1e-12
(|A||x|)_i, and bit for bit over repeated, replayed and column-major
launches."""
import numpy as np
import pytest

import oracle as O
from test_gpu_window import _cut_rows, _empty_stretches, _large_x, _repeated_descending, _rows, _windowed
from vnec_amd import matgen as g
from vnec_amd import spb

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if spb.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    spb.init()


MATRICES = {
    "one": lambda: _rows([1], 1, 1),
    "edge": lambda: _rows([1] * 700 + [7] * 180 + [2], 4096, 2),
    "cut_rows": _cut_rows,
    "empty_stretches": _empty_stretches,
    "repeated_descending": _repeated_descending,
    "one_row": lambda: _rows([70001], 80000, 3),
    "long_streams": lambda: g.uniform(530_003, 16, seed=4),  # 8.5M: streams of 32 at k = 4 and 8
    "short_rows": lambda: g.uniform(600_011, 1, seed=5),
}


def _run(f, x, n):
    dx = spb.DeviceArray.from_array(x)
    dy = spb.DeviceArray.from_array(np.full(n, np.nan))
    f(dx.ptr, dy.ptr)
    y = dy.to_array(np.float64, n)
    dx.free()
    dy.free()
    return y


@pytest.mark.parametrize("k", [2, 4, 8, 16])
@pytest.mark.parametrize("name", list(MATRICES))
def test_stream_tiles_match_oracle(name, k):
    m = MATRICES[name]()
    print(f"streams {name} k={k}: {m.nrows} x {m.ncols}, {m.nnz} nonzeros", flush=True)
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    p = spb.Plan(A, "learned", nrhs=k)
    assert _windowed(p) and p.info().variant == "L"
    X = np.random.default_rng(k).uniform(-1, 1, (m.ncols, k))
    n = m.nrows * k
    y = _run(p.spmv_dev, X.ravel(), n)
    for c in range(k):
        ax, ref = O.spmv_abs(m.ptr, m.col, m.val, np.ascontiguousarray(X[:, c]))
        ok, worst = O.check_rows(np.ascontiguousarray(y[c::k]), ref, ax, TOL)
        assert ok, (c, worst)
    for f in (p.spmv_dev, p.spmv_graph, p.spmv_graph):
        assert np.array_equal(_run(f, X.ravel(), n).view(np.uint64), y.view(np.uint64))
    yc = _run(p.spmm_colmajor_dev, np.ascontiguousarray(X.T).ravel(), n)
    assert np.array_equal(yc.reshape(k, -1).T.ravel().view(np.uint64), y.view(np.uint64))


@pytest.mark.parametrize("k", [2, 4, 8, 16])
def test_stream_tiles_unaligned_vectors_and_infinities(k):
    """Vectors only 8-byte aligned run the merge-path kernel; infinities and
    NaN of x reach the rows that hold their columns and no other, whichever
    kernel runs, and leave nothing behind for the next launch."""
    m = _cut_rows()
    A = spb.Matrix.from_csr(m.nrows, m.ncols, m.ptr, m.col, m.val)
    p = spb.Plan(A, "learned", nrhs=k)
    clean = np.random.default_rng(k).uniform(-1, 1, (m.ncols, k))
    lo = int(m.ptr[int(np.argmax(np.diff(m.ptr)))])
    lib, n, first = spb.L.load(), m.nrows * k, None
    for bad in ({}, {(m.col[lo], 0): np.inf}, {(m.col[lo], 1): np.nan, (m.col[lo + 5000], 0): -np.inf,
                                               (0, k - 1): np.inf}, {}):
        x = clean.copy()
        for at, v in bad.items():
            x[at] = v
        y = _run(p.spmv_dev, x.ravel(), n)
        dx = spb.DeviceArray(8 * m.ncols * k + 16)
        dy = spb.DeviceArray(8 * n + 16)
        spb.L.check(lib.vnec_memcpy_h2d_ext(dx.ptr + 8, np.ascontiguousarray(x).ctypes.data, x.nbytes), "h2d")
        p.spmv_dev(dx.ptr + 8, dy.ptr + 8)
        u = dy.to_array(np.float64, n + 1)[1:]
        assert np.array_equal(np.isnan(y), np.isnan(u))
        assert np.array_equal(np.isinf(y), np.isinf(u))
        assert np.array_equal(np.sign(y[np.isinf(y)]), np.sign(u[np.isinf(u)]))
        fin = np.isfinite(y)
        for c in range(k):
            ax, _ = O.spmv_abs(m.ptr, m.col, m.val, np.ascontiguousarray(np.nan_to_num(x[:, c], posinf=0, neginf=0)))
            d = np.abs(y[c::k][fin[c::k]] - u[c::k][fin[c::k]])
            assert (d <= 2 * TOL * ax[fin[c::k]]).all()
        if not bad:
            first = y if first is None else first
            assert np.array_equal(y, first)


@pytest.mark.parametrize("k", [2, 4, 8, 16])
@pytest.mark.parametrize("gib", [3, 4], ids=["32_bit_offsets", "64_bit_offsets"])
def test_stream_tiles_large_x(gib, k):
    """x beyond 2 GiB, where an offset does not fit an int, and from 4 GiB on,
    where it does not fit 32 bits: the same columns as in a small matrix, the
    same bits."""
    print(f"streams large x: {gib} GiB, k={k}", flush=True)
    ncols = (gib << 30) // (8 * k) + 999
    ptr, col, used, inv, val = _large_x(ncols)
    xs = np.random.default_rng(k).uniform(-1, 1, (len(used), k))
    y = []
    for n, c in ((ncols, col), (len(used), inv)):
        A = spb.Matrix.from_csr(len(ptr) - 1, n, ptr, c, val)
        p = spb.Plan(A, "learned", nrhs=k)
        assert _windowed(p)
        dx, dy = spb.DeviceArray(8 * n * k), spb.DeviceArray.from_array(np.full((len(ptr) - 1) * k, np.nan))
        for at, row in zip(used if n == ncols else range(n), xs):
            spb.L.check(spb.L.load().vnec_memcpy_h2d_ext(dx.ptr + 8 * k * int(at), row.ctypes.data, row.nbytes), "h2d")
        p.spmv_dev(dx.ptr, dy.ptr)
        y.append(dy.to_array(np.float64, (len(ptr) - 1) * k))
        for h in (p, dx, dy):
            h.free()
    assert np.array_equal(y[0].view(np.uint64), y[1].view(np.uint64))
    for c in range(k):
        ax, ref = O.spmv_abs(ptr, inv, val, np.ascontiguousarray(xs[:, c]))
        ok, worst = O.check_rows(np.ascontiguousarray(y[0][c::k]), ref, ax, TOL)
        assert ok, (c, worst)
