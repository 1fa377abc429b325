"""rsg_cov_Calculate_noalloc (the allocation-free scoring entry point) through the C-ABI against
rsg_cov_Calculate: identical COV and extremes on two calls in a row, the second on a smaller
alignment, and a clear error beyond the fixed scratch size.  Device buffers for the input codes
and the output matrix come from the HIP runtime (hipMalloc through ctypes)."""
import ctypes as C
import time

import numpy as np
import pytest

import rscape_amd as R
from rscape_amd import synth

pytestmark = pytest.mark.gpu

_hip = None


def hip():
    global _hip
    if _hip is None:
        _hip = C.CDLL("libamdhip64.so")
        _hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        _hip.hipFree.argtypes = [C.c_void_p]
        _hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        _hip.hipDeviceSynchronize.argtypes = []
    return _hip


H2D, D2H = 1, 2


class DevBuf:
    def __init__(self, nbytes):
        self.p = C.c_void_p()
        assert hip().hipMalloc(C.byref(self.p), nbytes) == 0
        self.n = nbytes

    def put(self, a):
        a = np.ascontiguousarray(a)
        assert a.nbytes <= self.n
        assert hip().hipMemcpy(self.p, a.ctypes.data_as(C.c_void_p), a.nbytes, H2D) == 0

    def get(self, shape, dtype):
        out = np.empty(shape, dtype)
        assert hip().hipMemcpy(out.ctypes.data_as(C.c_void_p), self.p, out.nbytes, D2H) == 0
        return out

    def free(self):
        if self.p:
            hip().hipFree(self.p)
            self.p = C.c_void_p()


def _declare():
    L = R.lib()
    f = L.rsg_cov_Calculate_noalloc
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int,
                  C.c_int, C.c_double, C.c_void_p, C.POINTER(C.c_double), C.POINTER(C.c_double), C.c_char_p]
    return f


def noalloc(ctx, d_ax, N, L, d_cov, covtype, prec):
    f = _declare()
    mn, mx = C.c_double(), C.c_double()
    err = C.create_string_buffer(128)
    rc = f(ctx.h, d_ax.p, N, L, R.COV[covtype], R.CSELECT, prec, None, 8, 50, 1e-6, d_cov.p, C.byref(mn),
           C.byref(mx), err)
    return rc, mn.value, mx.value, err.value.decode()


def test_noalloc_matches_cov_calculate(ctx):
    cases = [(1500, 700, "GTp", R.STAT_FP64, 1), (200, 120, "MIa", R.STAT_FP32, 2)]   # the second is smaller
    d_ax = DevBuf(1500 * 700)
    d_cov = DevBuf(8 * 700 * 700)
    try:
        for N, L, covtype, prec, seed in cases:
            print("no-alloc case N=%d L=%d %s prec %d" % (N, L, covtype, prec), flush=True)
            ax = synth.config(0, seed=seed, N=N, L=L)["ax"]
            m = ctx.msa(ax)
            mn0, mx0 = m.calculate(covtype, prec=prec)
            ref = m.get_cov()[0]
            m.close()
            d_ax.put(ax)
            rc, mn, mx, err = noalloc(ctx, d_ax, N, L, d_cov, covtype, prec)
            assert rc == 0, err
            got = d_cov.get((L, L), np.float64)
            assert np.array_equal(got, ref)
            assert (mn, mx) == (mn0, mx0)
    finally:
        d_ax.free()
        d_cov.free()


@pytest.mark.parametrize("N,L,covtype,prec", [(1, 2, "GTp", R.STAT_FP64), (30, 1, "GT", R.STAT_FP64),
                                              (65, 768, "MIgp", R.STAT_FP32), (65, 769, "MIgp", R.STAT_FP32),
                                              (130, 992, "GTp", R.STAT_FP64), (130, 993, "GTp", R.STAT_FP64),
                                              (257, 1024, "CHIa", R.STAT_FP64), (4096, 1024, "GTp", R.STAT_FP64)])
def test_noalloc_to_its_limits(ctx, N, L, covtype, prec):
    """Up to RSG_NA_MAXN sequences and RSG_NA_MAXL columns, on either side of where the Gram's tiles
    stop fitting the device at once (992 columns): rsg_cov_Calculate's scores bit for bit."""
    ax = synth.random_msa(N, L, np.random.default_rng(N + L), gap=0.1)
    m = ctx.msa(ax)
    mn0, mx0 = m.calculate(covtype, prec=prec)
    ref = m.get_cov()[0]
    m.close()
    d_ax, d_cov = DevBuf(N * L), DevBuf(8 * L * L)
    try:
        d_ax.put(ax)
        rc, mn, mx, err = noalloc(ctx, d_ax, N, L, d_cov, covtype, prec)
        assert rc == 0, err
        assert np.array_equal(d_cov.get((L, L), np.float64), ref)
        assert (mn, mx) == (mn0, mx0)
    finally:
        d_ax.free()
        d_cov.free()


@pytest.mark.parametrize("covtype", ["GT", "GTp", "GTa"])
def test_noalloc_stamp_waits(ctx, covtype):
    """The chain's three ends (the statistic's own extremes, APC, ASC) with the completion stamp waited
    for, given up on after a microsecond, and not waited for: the same bits."""
    N, L = 300, 130
    ax = synth.config(0, seed=4, N=N, L=L)["ax"]
    m = ctx.msa(ax)
    mn0, mx0 = m.calculate(covtype)
    ref = m.get_cov()[0]
    m.close()
    d_ax, d_cov = DevBuf(N * L), DevBuf(8 * L * L)
    try:
        d_ax.put(ax)
        for wait in (2000, 1, 0):
            ctx.set_stamp_wait(wait)
            d_cov.put(np.zeros((L, L)))
            rc, mn, mx, err = noalloc(ctx, d_ax, N, L, d_cov, covtype, R.STAT_FP64)
            assert rc == 0, err
            assert (mn, mx) == (mn0, mx0) and np.array_equal(d_cov.get((L, L), np.float64), ref), wait
    finally:
        ctx.set_stamp_wait(0)
        d_ax.free()
        d_cov.free()


def test_noalloc_leaves_no_work_behind():
    """The call's own wait covers its work, however it waits: a device synchronisation behind it costs
    what one on an idle device does, within 4 us (medians of 101; 9 us more when the call returned with
    its commands not yet retired)."""
    N, L = 200, 120
    ax = synth.config(0, seed=5, N=N, L=L)["ax"]
    d_ax, d_cov = DevBuf(N * L), DevBuf(8 * L * L)
    c = R.Context(0)
    d_ax.put(ax)

    def sync():
        t = time.perf_counter()
        assert hip().hipDeviceSynchronize() == 0
        return time.perf_counter() - t

    def behind_call():
        assert noalloc(c, d_ax, N, L, d_cov, "GTp", R.STAT_FP64)[0] == 0
        return sync()

    try:
        for wait in (None, 2000):
            if wait is not None:
                c.set_stamp_wait(wait)
            behind_call()
            idle = np.median([sync() for _ in range(101)])
            assert np.median([behind_call() for _ in range(101)]) < idle + 4e-6, wait
    finally:
        c.close()
        d_ax.free()
        d_cov.free()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_noalloc_beside_a_capture(ctx, mode):
    """The call on its own stream while the caller captures another one (global, thread-local and
    relaxed capture): it scores, and the capture ends with its graph."""
    N, L = 200, 120
    ax = synth.config(0, seed=6, N=N, L=L)["ax"]
    m = ctx.msa(ax)
    m.calculate("GTp")
    ref = m.get_cov()[0]
    m.close()
    d_ax, d_cov = DevBuf(N * L), DevBuf(8 * L * L)
    st, graph = C.c_void_p(), C.c_void_p()
    h = hip()
    try:
        d_ax.put(ax)
        assert h.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        assert h.hipStreamBeginCapture(st, mode) == 0
        rc, _, _, err = noalloc(ctx, d_ax, N, L, d_cov, "GTp", R.STAT_FP64)
        assert h.hipStreamEndCapture(st, C.byref(graph)) == 0 and graph.value
        assert rc == 0, err
        assert np.array_equal(d_cov.get((L, L), np.float64), ref)
    finally:
        if graph.value:
            h.hipGraphDestroy(graph)
        if st.value:
            h.hipStreamDestroy(st)
        d_ax.free()
        d_cov.free()


def test_noalloc_rejects_oversize_and_unsupported(ctx):
    d = DevBuf(64)
    try:
        rc, _, _, err = noalloc(ctx, d, 10, 1025, d, "GTp", R.STAT_FP64)
        assert rc != 0 and "exceeds the fixed scratch" in err
        rc, _, _, err = noalloc(ctx, d, 4097, 10, d, "GTp", R.STAT_FP64)
        assert rc != 0 and "exceeds the fixed scratch" in err
        rc, _, _, err = noalloc(ctx, d, 10, 10, d, "RAFS", R.STAT_FP64)
        assert rc != 0 and "not available" in err
    finally:
        d.free()
