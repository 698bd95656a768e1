"""Objects that come and go while another thread's stream is captured: what
hipMalloc and hipFree leave alone, the library's block cache leaves alone too."""
import ctypes as C
import threading

import numpy as np
import pytest

from gpu_cases import announce

pytestmark = pytest.mark.gpu


GLOBAL, THREAD_LOCAL, RELAXED = 0, 1, 2  # hipStreamCaptureMode


@pytest.mark.parametrize("what", ["destroy", "create"])
@pytest.mark.parametrize("mode,thread", [(THREAD_LOCAL, True), (RELAXED, True), (RELAXED, False)])
def test_capture_survives_other_objects(gpu, mode, thread, what):
    from matrix_format_performance_amd import _lib as L
    lib = L.load()  # finds the HIP runtime's functions too

    def hip(name, *args):
        status = getattr(lib, name)(*args)
        assert status == 0, (name, status)

    announce(f"capture mode={mode} thread={thread} what={what}")
    rng = np.random.default_rng(0)

    def matrix():
        rp = np.concatenate([[0], np.cumsum(rng.integers(1, 30, 40000))]).astype(np.uint32)
        ci = rng.integers(0, 40000, rp[-1]).astype(np.uint32)
        return gpu.DeviceMatrix.from_csr(rp, ci, rng.random(ci.size).astype(np.float32), 40000)

    A, B = matrix(), matrix()
    P, Q = gpu.Plan(A, "ell"), gpu.Plan(B, "ell")
    gpu.Plan(B, "coo").destroy()  # blocks for the plan that is created
    x = gpu.DeviceArray.from_host(rng.random(40000).astype(np.float32))
    y = gpu.DeviceArray(40000, np.dtype(np.float32))
    P.spmv(x, y)
    gpu.synchronize()
    want, made = y.to_host(), []

    def act():
        if what == "destroy":
            Q.destroy()
        else:
            made.append(gpu.Plan(B, "coo"))

    s, g, e = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip("hipStreamCreateWithFlags", C.byref(s), C.c_uint(1))
    hip("hipStreamBeginCapture", s, C.c_int(mode))
    P.spmv(x, y, stream=s)
    if thread:
        t = threading.Thread(target=act)
        t.start()
        t.join()
    else:
        act()
    P.spmv(x, y, stream=s)
    hip("hipStreamEndCapture", s, C.byref(g))
    hip("hipGraphInstantiate", C.byref(e), g, None, None, C.c_size_t(0))
    for _ in range(3):
        y.fill(np.nan)
        gpu.synchronize()
        hip("hipGraphLaunch", e, s)
        hip("hipStreamSynchronize", s)
        assert np.array_equal(y.to_host(), want)
    hip("hipGraphExecDestroy", e)
    hip("hipGraphDestroy", g)
    hip("hipStreamDestroy", s)
    if what == "create":
        assert made
        made[0].destroy()
        Q.destroy()
    P.destroy()
    A.destroy()
    B.destroy()


# CSR-vector plans are made and destroyed beside a capture in any mode (they need
# no arrays).  Long rows side by side, so that the plan lists their blocks.
@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL, RELAXED])
@pytest.mark.parametrize("thread", [False, True])
def test_csr_vector_plans_within_a_capture(gpu, mode, thread):
    from matrix_format_performance_amd import _lib as L
    lib = L.load()

    def hip(name, *args):
        status = getattr(lib, name)(*args)
        assert status == 0, (name, status)

    announce(f"CSR-vector in a capture mode={mode} thread={thread}")
    rng = np.random.default_rng(0)
    lens = np.full(300007, 6)
    lens[100000:100256] = 1500
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    ci = np.sort(rng.integers(0, 300007, rp[-1])).astype(np.uint32)
    va = rng.integers(-3, 4, ci.size).astype(np.float32)
    A, B = (gpu.DeviceMatrix.from_csr(rp, ci, va, 300007) for _ in range(2))
    xh = rng.integers(-5, 6, 300007).astype(np.float32)
    x, y = gpu.DeviceArray.from_host(xh), gpu.DeviceArray(300007, np.dtype(np.float32))
    sums = np.concatenate([[0], np.cumsum(va.astype(np.int64) * xh.astype(np.int64)[ci])])
    want = (sums[rp[1:]] - sums[rp[:-1]]).astype(np.float32)
    old, made = gpu.Plan(B, "csr_vector", lanes=8), []
    s, g, e = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip("hipStreamCreateWithFlags", C.byref(s), C.c_uint(1))

    def act():
        old.destroy()
        made.append(gpu.Plan(A, "csr_vector", lanes=8))

    gpu.synchronize()
    hip("hipStreamBeginCapture", s, C.c_int(mode))
    try:
        if thread:
            t = threading.Thread(target=act)
            t.start()
            t.join()
        else:
            act()
        made[0].spmv(x, y, stream=s)
    finally:
        ended = lib.hipStreamEndCapture(s, C.byref(g))
    assert ended == 0
    hip("hipGraphInstantiate", C.byref(e), g, None, None, C.c_size_t(0))
    for _ in range(3):
        y.fill(np.nan)
        gpu.synchronize()
        hip("hipGraphLaunch", e, s)
        hip("hipStreamSynchronize", s)
        assert np.array_equal(y.to_host(), want)
    hip("hipGraphExecDestroy", e)
    hip("hipGraphDestroy", g)
    hip("hipStreamDestroy", s)
    for o in (made[0], A, B):
        o.destroy()


def test_trim_gives_kept_memory_to_other_allocators(gpu):
    from matrix_format_performance_amd import _lib as L
    lib = L.load()

    def raw_free():
        free, total = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n = 1 << 20  # 500 MB of ELL arrays, and the matrix lives on
    rp = (np.arange(n + 1) * 8).astype(np.uint32)
    A = gpu.DeviceMatrix.from_csr(rp, (np.arange(8 * n) % n).astype(np.uint32), np.ones(8 * n, np.float32), n)
    gpu.trim()
    before = raw_free()
    gpu.Plan(A, "ell", ell_width=60).destroy()
    assert gpu.device_info()["free_mem"] >= before - (8 << 20)  # what is kept counts as free
    gpu.trim()
    assert abs(raw_free() - before) < 64 << 20
    A.destroy()
