"""Device-to-host reads (des-alm_amd/csrc/host_copy.hip) against a CPU
stand-in for the runtime: which copies take the pinned ring, and what a read
waits for while it holds it."""
import ctypes
import os
import shutil
import subprocess
import threading
import time

import numpy as np
import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
LARGE = (37 << 20) // 8 + 5  # doubles: 19 chunks of 2 MiB, more than the ring's eight slots
SMALL = 1 << 10


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or no HIP headers")
    so = str(tmp_path_factory.mktemp("hc") / "libhc.so")
    csrc = os.path.join(ROOT, "des-alm_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                           "-I", os.path.join(ROCM, "include"), "-I", csrc, "-o", so,
                           "-x", "c++", os.path.join(csrc, "host_copy.hip"),
                           os.path.join(ROOT, "tests", "host_copy_stub.cpp")])
    L = ctypes.CDLL(so)
    vp = ctypes.c_void_p
    L.hc_read.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int]
    L.hc_know.argtypes = [vp]
    L.hc_direct.restype = ctypes.c_long
    L.hc_users(1)
    yield L
    L.hc_users(-1)


def read(hc, dst, src, stream=0):
    assert hc.hc_read(dst.ctypes.data, src.ctypes.data, src.nbytes, stream) == 0


@pytest.mark.parametrize("n,direct", [(SMALL, 1), (LARGE, 0)])
def test_bytes_arrive(hc, n, direct):
    src = np.random.default_rng(n).standard_normal(n)
    dst = np.zeros(n)
    hc.hc_direct()
    read(hc, dst, src)
    assert np.array_equal(dst, src)
    assert hc.hc_direct() == direct


def test_read_does_not_wait_for_another_streams_work(hc):
    """A read behind a stream's pending kernels leaves the ring to reads of
    other streams until those kernels are done."""
    src = [np.random.default_rng(k).standard_normal(LARGE) for k in range(2)]
    dst = [np.zeros(LARGE) for _ in range(2)]
    t = [threading.Thread(target=read, args=(hc, dst[k], src[k], k), daemon=True) for k in range(2)]
    hc.hc_busy(0, 1)
    try:
        t[0].start()
        end = time.monotonic() + 30
        while not hc.hc_waiting(0) and time.monotonic() < end:
            time.sleep(0.001)
        assert hc.hc_waiting(0)
        t[1].start()
        t[1].join(10)
        done = not t[1].is_alive()
    finally:
        hc.hc_busy(0, 0)
    t[0].join(30)
    t[1].join(30)
    assert done
    assert all(np.array_equal(d, s) for d, s in zip(dst, src))


def test_memory_the_runtime_knows_is_copied_into_directly(hc):
    """Pinned (or any other registered) destinations take one copy and no
    pass through the ring."""
    src = np.random.default_rng(7).standard_normal(LARGE)
    dst = np.zeros(LARGE)
    hc.hc_know(dst.ctypes.data)
    hc.hc_direct()
    read(hc, dst, src)
    assert np.array_equal(dst, src)
    assert hc.hc_direct() == 1
