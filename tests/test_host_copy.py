"""The host side of jpp_copy_h2d / jpp_copy_d2h (csrc/host_copy.hip) over a stand-in for the HIP runtime in which device
memory is host memory: what a call does without pinned memory, for two devices in turn, beside a call of
another thread, and in a forked process."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from jaxpp_amd import build

HIP = r"""
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>
#include <atomic>
#include <thread>
extern "C" {
std::atomic<int> pinned_left{1 << 20}, pinned_made{0}, streams_made{0}, sync_copies{0}, blocked{0}, waiting{0}, last{0};
static thread_local int t_device = 0;
int hold(int v) { return blocked = v; }             // asynchronous copies wait while it is set
int waiters() { return waiting; }
int pinned_limit(int v) { pinned_made = 0; return pinned_left = v; }
int count(int what) { return what == 0 ? pinned_made : what == 1 ? streams_made : what == 2 ? sync_copies : last; }
hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (pinned_left-- <= 0) { last = hipErrorOutOfMemory; return hipErrorOutOfMemory; }
  ++pinned_made; *p = malloc(n); return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { ++streams_made; *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  ++waiting; while (blocked) std::this_thread::yield(); --waiting;
  memcpy(d, s, n); return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { ++sync_copies; memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetLastError() { return (hipError_t)last.exchange(0); }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
}
int jpp_set_error(int code, const char*, ...) { return code; }
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("host_copy")
    (d / "hip.cpp").write_text(HIP)
    objs = []
    for src in (os.path.join(build.CSRC, "host_copy.hip"), str(d / "hip.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-I", build.CSRC,
                        "-c", src, "-o", objs[-1]], check=True, stderr=subprocess.DEVNULL)
    out = str(d / "libhost_copy.so")
    subprocess.run(["g++", "-shared", "-pthread", "-o", out, *objs], check=True)
    return out


def run(library, body):
    """`body` in a process of its own, which loads the library; a call that waits for ever ends it."""
    head = f"""
        import ctypes as C, os, sys, threading, time
        import numpy as np
        from jaxpp_amd import runtime as rt
        lib = C.CDLL({library!r})
        lib.jpp_copy_h2d.argtypes = lib.jpp_copy_d2h.argtypes = [C.c_int, C.POINTER(rt.CopyItem), C.c_int]

        def items(arrays, at, es):
            q = (rt.CopyItem * len(arrays))()
            for i, a in zip(q, arrays):
                i.host, i.device, i.count = a.ctypes.data, at, a.size
                at += es * a.size
            return q

        def round_trip(sizes, bf16, seed=0):
            rng, es = np.random.default_rng(seed), 2 if bf16 else 4
            device = np.zeros(es * sum(sizes), np.uint8)
            arrays = [rng.standard_normal(n, dtype=np.float32) for n in sizes]
            assert lib.jpp_copy_h2d(len(sizes), items(arrays, device.ctypes.data, es), bf16) == 0
            flat = np.concatenate(arrays)
            want = rt.to_bf16_bits(flat) if bf16 else flat.view(np.uint32)
            np.testing.assert_array_equal(device.view(want.dtype), want)
            outs = [np.empty(n, np.float32) for n in sizes]
            assert lib.jpp_copy_d2h(len(sizes), items(outs, device.ctypes.data, es), bf16) == 0
            np.testing.assert_array_equal(np.concatenate(outs), rt.from_bf16_bits(want) if bf16 else flat)

        SIZES = [[5], [70000, 3, 0, 900000], [3 << 20], [1000] * 50]
    """
    src = textwrap.dedent(head) + textwrap.dedent(body)
    p = subprocess.run([sys.executable, "-c", src], timeout=60, capture_output=True, text=True,
                       cwd=os.path.dirname(build.HERE))
    assert p.returncode == 0, p.stderr[-3000:]


@pytest.mark.parametrize("slots", [0, 1, 2, 3, 5])
def test_copies_with_the_pinned_memory_there_is(library, slots):
    """With slots for no lane, one or two: the same bytes, and no error left for the next GPU call to report."""
    run(library, f"""
        for sizes in SIZES:
            for bf16 in (0, 1):
                lib.pinned_limit({slots})
                round_trip(sizes, bf16)
                assert lib.count(3) == 0
                lib.pinned_limit(1 << 20)
                lib.jpp_copy_release()
        lib.pinned_limit({slots})
        round_trip(SIZES[2], 0)
        assert (lib.count(2) > 0) == ({slots} < 2)
        lib.pinned_limit(1 << 20)              # there is more again: the lanes that were missing are made
        round_trip(SIZES[2], 0)
    """)


def test_two_devices_in_turn_keep_their_lanes(library):
    run(library, """
        for device in (0, 1, 0, 1):
            lib.hipSetDevice(device)
            round_trip(SIZES[2], 0)
            if device: made = lib.count(0), lib.count(1)
        for device in (0, 1) * 3:
            lib.hipSetDevice(device)
            round_trip(SIZES[2], 0)
        assert (lib.count(0), lib.count(1)) == made, (made, lib.count(0), lib.count(1))
        assert lib.jpp_copy_release() == 0
        round_trip(SIZES[2], 1)
    """)


def test_a_copy_beside_another_threads_does_not_wait_for_it(library):
    run(library, """
        lib.hold(1)
        first = threading.Thread(target=round_trip, args=(SIZES[2], 0))
        first.start()
        while lib.waiters() == 0:
            time.sleep(0.001)
        for sizes in SIZES:
            for bf16 in (0, 1):
                round_trip(sizes, bf16, 1)     # (while the first one's copies are held)
        assert first.is_alive() and lib.count(2) > 0
        lib.hold(0)
        first.join()
    """)


def test_a_forked_process_ends_and_its_copies_are_refused(library):
    """Also one forked while a copy of another thread was under way, whose locks nobody gives back there."""
    run(library, """
        lib.hold(1)
        first = threading.Thread(target=round_trip, args=(SIZES[2], 0))
        first.start()
        while lib.waiters() == 0:
            time.sleep(0.001)
        child = os.fork()
        if child == 0:
            a = np.zeros(4, np.float32)
            refused = lib.jpp_copy_h2d(1, items([a], a.ctypes.data, 4), 0) != 0
            os._exit(0 if refused and lib.jpp_copy_release() == 0 else 1)
        for _ in range(1000):
            pid, status = os.waitpid(child, os.WNOHANG)
            if pid:
                break
            time.sleep(0.01)
        lib.hold(0)
        first.join()
        if not pid:
            os.kill(child, 9)
        assert pid and status == 0, (pid, status)
    """)
