"""Copies of many tensors in one call (jpp_copy_h2d / jpp_copy_d2h), at the edges of their chunks and lanes: empty
and one-element tensors, sizes around a chunk's, tensors that do and do not lie one behind the other on
the device, both element kinds.  Every byte is compared, what lies between and behind the tensors too."""
import ctypes
import threading

import numpy as np
import pytest

from jaxpp_amd import runtime as rt

pytestmark = pytest.mark.gpu

CHUNK = (1 << 20) // 4        # elements of the largest chunk


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def specials(rng, n):
    a = rng.standard_normal(n, dtype=np.float32)
    a[::7] = rng.integers(0, 1 << 32, a[::7].size, dtype=np.uint64).astype(np.uint32).view(np.float32)   # any bits
    return a


@pytest.mark.parametrize("gap", [0, 12], ids=["adjacent", "apart"])
@pytest.mark.parametrize("bf16", [False, True], ids=["words", "bf16"])
@pytest.mark.parametrize("sizes", [[1], [0, 3, 0, 5], [65535, 1, 65537], [CHUNK - 1, 2, CHUNK + 1, 7],
                                   [20 * CHUNK + 3], [1000] * 900], ids=lambda s: f"{len(s)}x{max(s)}")
def test_tensors_arrive_whole(sizes, bf16, gap):
    print(f"{len(sizes)} tensors of up to {max(sizes)}, bf16 {bf16}, gap {gap}", flush=True)
    rng = np.random.default_rng(len(sizes) + sizes[0])
    es, dt = (2, np.uint16) if bf16 else (4, np.uint32)
    at = [64 + sum(sizes[:i]) + gap * i for i in range(len(sizes))]
    total = at[-1] + sizes[-1] + 64
    arrays = [specials(rng, n) for n in sizes]
    want = np.full(total, 0x3a3a if bf16 else 0x3a3a3a3a, dt)
    buf = rt.DeviceBuffer.from_numpy(want)
    for a, i in zip(arrays, at):
        want[i:i + a.size] = rt.to_bf16_bits(a) if bf16 else a.view(np.uint32)
    rt.copy_in([(a, buf.ptr + es * i) for a, i in zip(arrays, at)], bf16)
    raw = np.empty(total, dt)
    rt.check(rt.load().jpp_memcpy_d2h(raw.ctypes.data, buf.ptr, raw.nbytes))
    np.testing.assert_array_equal(raw, want)
    outs = [np.empty(n, np.float32) for n in sizes]
    rt.copy_out([(o, buf.ptr + es * i) for o, i in zip(outs, at)], bf16)
    for o, a in zip(outs, arrays):
        np.testing.assert_array_equal(o.view(np.uint32),
                                      rt.from_bf16_bits(rt.to_bf16_bits(a)).view(np.uint32) if bf16 else a.view(np.uint32))


def test_copies_follow_the_null_stream_and_several_threads_may_copy():
    """A copy out sees what was queued before it; threads that copy at once, with the pool given back in
    between, each get their own data."""
    n = 3 * CHUNK + 1
    buf = rt.DeviceBuffer(4 * n)
    for value in range(1, 20):
        rt.check(rt.load().jpp_fill_u32(buf.ptr, value, n, None))
        out = np.empty(n, np.uint32)
        rt.copy_out([(out, buf.ptr)])
        assert (out == value).all()
    wrong = []

    def work(seed):
        rng, own = np.random.default_rng(seed), rt.DeviceBuffer(4 * n)
        for _ in range(8):
            a, out = rng.standard_normal(n, dtype=np.float32), np.empty(n, np.float32)
            rt.copy_in([(a, own.ptr)])
            if seed == 0:
                rt.check(rt.load().jpp_copy_release())
            rt.copy_out([(out, own.ptr)])
            if not np.array_equal(a, out):
                wrong.append(seed)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


def test_bad_items_are_refused():
    lib, item = rt.load(), (rt.CopyItem * 1)()
    assert ctypes.sizeof(rt.CopyItem) == 24
    item[0].count = 4                                     # null pointers
    assert lib.jpp_copy_h2d(1, item, 0) == -1 and b"item 0" in lib.jpp_last_error()
    assert lib.jpp_copy_d2h(1, None, 0) == -1 and lib.jpp_copy_h2d(0, None, 2) == -1
    item[0].count = 0
    assert lib.jpp_copy_h2d(1, item, 1) == 0 and lib.jpp_copy_d2h(0, None, 0) == 0
