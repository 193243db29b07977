"""host_copy (csrc/hostcopy.hip) on the CPU, against a HIP runtime that runs
copies of pinned memory as late as a runtime may (host_copy_runtime.cpp): the
same C++ source as the library's, compiled for the host alone."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "leeds-code_amd", "csrc")
ROCM = "/opt/rocm/include"
MB = 1 << 20

pytestmark = pytest.mark.skipif(not (shutil.which("g++") and os.path.isdir(ROCM)), reason="needs g++ and HIP's headers")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hc") / "host_copy.so")
    # (g++ has no __bf16 here; hostcopy.hip uses no value of that type)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__",
                    "-D__bf16=short", "-I" + ROCM, "-o", so, "-x", "c++", os.path.join(CSRC, "hostcopy.hip"),
                    os.path.join(HERE, "host_copy_runtime.cpp")], check=True)
    return ctypes.CDLL(so)


def copy(lib, host, dev, to_host, pin=False, delay=0, ok=-1, oom=False, nopin=False):
    n = len(host)
    P, S = ctypes.c_void_p * n, ctypes.c_size_t * n
    return lib.fake_host_copy(n, P(*[a.ctypes.data for a in host]), P(*[a.ctypes.data for a in dev]),
                              S(*[a.nbytes for a in host]), int(to_host), int(pin), delay, ok, int(oom),
                              int(nopin))


# below and above the sizes of the chunked copies (2 MiB of results, 24 MiB of
# uploads), last chunks of 1 byte and of all but one, several parts
SIZES = [(1,), (2 * MB - 1,), (2 * MB,), (5 * MB + 1,), (9 * MB - 1,), (MB, 3 * MB, 1), (4 * MB + 5, 7, 6 * MB),
         (24 * MB - 1,), (24 * MB + 1,), (12 * MB + 5, 7, 13 * MB - 1)]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("to_host", [True, False])
@pytest.mark.parametrize("pin", [False, True])
def test_all_bytes(lib, sizes, to_host, pin):
    rng = np.random.default_rng(1)
    src = [rng.integers(0, 256, n, dtype=np.uint8) for n in sizes]
    dst = [np.zeros(n, dtype=np.uint8) for n in sizes]
    host, dev = (dst, src) if to_host else (src, dst)
    assert copy(lib, host, dev, to_host, pin) == 0
    lib.fake_run()
    for a, b in zip(src, dst):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("offset", [0, MB + 3])
@pytest.mark.parametrize("delay", [0, 20])
def test_overlapping_results(lib, offset, delay):
    """Result arrays that share memory hold what the last of them brings, as
    copies one after another leave it (a caller that wants one of two results
    may pass the same array for both)."""
    n = 5 * MB
    dev = [np.full(n, 1 + k, dtype=np.uint8) for k in range(2)]
    buf = np.zeros(n + offset, dtype=np.uint8)
    assert copy(lib, [buf[:n], buf[offset:]], dev, True, delay=delay) == 0
    assert np.all(buf[offset:] == 2) and np.all(buf[:offset] == 1)


@pytest.mark.parametrize("to_host", [True, False])
def test_no_memory_for_threads(lib, to_host):
    """Without memory for a thread's state the calling thread does the work: no
    exception leaves the copy."""
    src = np.random.default_rng(2).integers(0, 256, 25 * MB + 1, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    assert copy(lib, [host], [dev], to_host, oom=True) == 0
    assert np.array_equal(src, dst)


@pytest.mark.parametrize("to_host", [True, False])
def test_no_pinned_memory(lib, to_host):
    """Without pinned memory for the chunks the copy is a plain one."""
    src = np.random.default_rng(4).integers(0, 256, 25 * MB + 1, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    assert copy(lib, [host], [dev], to_host, nopin=True) == 0
    assert np.array_equal(src, dst)


@pytest.mark.parametrize("to_host", [True, False])
@pytest.mark.parametrize("ok", [0, 3])
def test_failing_copy(lib, to_host, ok):
    """A copy that the runtime refuses is reported."""
    src = np.ones(25 * MB + 1, dtype=np.uint8)
    dst = np.zeros_like(src)
    host, dev = (dst, src) if to_host else (src, dst)
    assert copy(lib, [host], [dev], to_host, ok=ok) != 0
