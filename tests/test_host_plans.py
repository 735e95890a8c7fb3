"""Which kernel a plan the library chooses runs, decided on the CPU: the host
sources over a device made of host memory and planted kernel times
(host_stubs.c)."""
import ctypes as C
import gc
import os
import subprocess

import numpy as np
import pytest

from vnec_amd import _lib as L
from vnec_amd import spb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "vnec_amd", "csrc", "host")


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    cc = ["gcc", "-O1", "-std=gnu11", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
          "-I" + os.path.join(ROOT, "include"), "-I" + HOST]
    srcs = [os.path.join(HOST, f) for f in sorted(os.listdir(HOST)) if f.endswith(".c")]
    srcs.append(os.path.join(ROOT, "tests", "host_stubs.c"))
    subprocess.run(cc + ["-c"] + srcs, cwd=d, check=True)
    objs = sorted(str(p) for p in d.glob("*.o"))
    names = {True: set(), False: set()}
    for line in subprocess.run(["nm", *objs], capture_output=True, text=True, check=True).stdout.splitlines():
        f = line.split()
        if len(f) >= 2 and f[-1].startswith(("hip", "vnec_hip_")):
            names[f[-2] == "U"].add(f[-1])
    (d / "rest.c").write_text("".join(f"int {n}(void) {{ return 0; }}\n" for n in sorted(names[True] - names[False])))
    so = str(d / "libstub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-o", so, str(d / "rest.c"), *objs, "-lm"], check=True)
    return so


@pytest.fixture
def stub(stub_path, monkeypatch):
    lib = C.CDLL(stub_path)
    for name, (res, args) in L.SIGNATURES.items():
        if hasattr(lib, name):
            getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    monkeypatch.setattr(L, "_lib", lib)
    monkeypatch.setattr(spb, "_init", False)
    spb.init()
    yield lib
    gc.collect()  # handles of this library, before the other one is back


def _plant(lib, **values):
    for name, v in {"largest": C.c_size_t(-1).value, "layout_error": 0, "choice": 4, "win_us": 1.0, "tiles_us": 1.0,
                    "other_us": 1.0, "win_launches": 0, "other_launches": 0, "x_changes": 0, **values}.items():
        t = C.c_size_t if name == "largest" else C.c_double if name.endswith("us") else C.c_int
        t.in_dll(lib, "stub_" + name).value = v


def _matrix(dtype=np.float64):
    rng = np.random.default_rng(1)
    n, k = 4000, 8
    col = np.sort(rng.integers(0, n, (n, k)), axis=1)
    return spb.Matrix.from_csr(n, n, np.arange(0, n * k + 1, k), col.ravel(), np.ones(n * k, dtype), dtype=dtype)


def _windowed(p):
    return bool(L.load().vnec_plan_windowed(p.h))


@pytest.mark.parametrize("nrhs", [1, 4])
def test_no_room_for_the_layout_falls_back(stub, nrhs):
    """Windowed and stream tiles need more device memory than the kernels that
    read the matrix in place: these run where it does not suffice."""
    A = _matrix()
    _plant(stub)
    assert _windowed(spb.Plan(A, "learned", nrhs=nrhs))
    _plant(stub, largest=8 * A.nnz)  # the matrix itself and no padded copy of it
    p = spb.Plan(A, "learned", nrhs=nrhs)
    assert not _windowed(p) and p.info().variant == "L"


@pytest.mark.parametrize("nrhs", [1, 4])
def test_other_failures_reach_the_caller(stub, nrhs):
    """A layout that fails for any other reason is an error, with its message,
    and not a slower plan."""
    A = _matrix()
    _plant(stub, layout_error=719)
    with pytest.raises(RuntimeError, match="layout: HIP error 719"):
        spb.Plan(A, "learned", nrhs=nrhs)


@pytest.mark.parametrize("win_us,other_us", [(9.0, 5.0), (5.0, 9.0)], ids=["named_faster", "windowed_faster"])
@pytest.mark.parametrize("enc", ["fp64", "hilo", "hi", "fp32"])
def test_autotune_keeps_the_fastest_it_timed(stub, enc, win_us, other_us):
    """The autotune mode times windowed tiles beside the named shapes and runs
    whichever was faster, also from the cached comparison."""
    A = _matrix(np.float32 if enc == "fp32" else np.float64)
    _plant(stub, win_us=win_us, other_us=other_us)
    for _ in range(2):
        p = spb.Plan(A, "autotune", encoding=enc)
        launches = [C.c_int.in_dll(stub, "stub_" + k).value for k in ("win_launches", "other_launches")]
        assert min(launches) > 0, "both were timed"
        assert _windowed(p) == (win_us < other_us)
        x, y = spb.DeviceArray(8 * A.ncols), spb.DeviceArray(8 * A.nrows)
        assert p.time(x.ptr, y.ptr, 20) == pytest.approx(min(win_us, other_us) * 1e-3)
        for h in (p, x, y):
            h.free()


@pytest.mark.parametrize("tiles_us,kernel", [(9.0, "merge"), (2.0, "tiles")])
@pytest.mark.parametrize("nrhs", [2, 4, 8, 16])
def test_autotune_of_several_right_hand_sides(stub, nrhs, tiles_us, kernel):
    """Stream tiles where they were faster than the merge-path kernel at its
    best granularity; that granularity either way, since vectors aligned to 8
    bytes only run it."""
    A = _matrix()
    _plant(stub, tiles_us=tiles_us)
    (C.c_double * 16).in_dll(stub, "stub_merge_us")[3:8] = [3.0, 0, 6.0, 0, 5.0]
    for _ in range(2):
        p = spb.Plan(A, "autotune", nrhs=nrhs)
        assert p.info().ipt == 3 and _windowed(p) == (kernel == "tiles")
        x, y = (spb.DeviceArray(8 * (n * nrhs + 2)) for n in (A.ncols, A.nrows))
        assert p.time(x.ptr, y.ptr, 20) == pytest.approx(min(tiles_us, 3.0) * 1e-3)
        assert p.time(x.ptr + 8, y.ptr + 8, 20) == pytest.approx(3.0e-3)
        for h in (p, x, y):
            h.free()


def test_kernel_times_of_relabelled_windowed_tiles_read_the_permuted_x(stub):
    A = _matrix()
    _plant(stub)
    t = L.Tuning(spb.VNEC_VAR["L"], 7, spb.LANES_RELABEL, spb.VNEC_ENC["fp64"], 1, -1)
    h = C.c_void_p()
    stub.vnec_plan_build_windowed.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    L.check(stub.vnec_plan_build_windowed(C.byref(h), A.h, C.byref(t)), "build")
    x, y = spb.DeviceArray(8 * A.ncols), spb.DeviceArray(8 * A.nrows)
    L.check(stub.vnec_spmv_dev_ext(h, x.ptr, y.ptr), "SpMV")
    a, b = C.c_double(), C.c_double()
    _plant(stub)
    L.check(stub.vnec_time_kernels_ext(h, x.ptr, y.ptr, 5, C.byref(a), C.byref(b)), "time")
    assert C.c_int.in_dll(stub, "stub_win_launches").value == 7 and C.c_int.in_dll(stub, "stub_x_changes").value == 0
    L.check(stub.vnec_plan_free_ext(C.byref(h)), "free")
