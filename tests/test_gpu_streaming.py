"""The streaming kernels at the edges of what a wave or a workgroup takes: fills of every remainder and alignment,
Adam on tensors whose last wave is cut short in its first or its second half."""
import numpy as np
import pytest

import test_gpu_optimizer as optimizer
from jaxpp_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("count", [1, 3, 4, 5, 1023, 4095, 4096, 4099, 16385])
def test_fill_of_any_count_and_alignment(count, offset):
    buf = rt.DeviceBuffer.from_numpy(np.full(count + 8, 7, np.uint32))
    rt.check(rt.load().jpp_fill_u32(buf.ptr + 4 * offset, 0xabcd1234, count, None))
    got = buf.download(np.uint32, (count + 8,))
    assert (got[offset:offset + count] == 0xabcd1234).all()
    assert (got[:offset] == 7).all() and (got[offset + count:] == 7).all()


@pytest.mark.parametrize("count", [8, 248, 256, 264, 504, 8 * 64, 8 * 65, 8 * 255 + 3, 8 * 257])
@pytest.mark.parametrize("with_master", [True, False])
def test_adam_of_partial_waves(count, with_master):
    optimizer.test_adam_flat(count, with_master)


def test_fill_of_more_than_the_largest_grid_takes_in_one_trip():
    """128 GiB are a workgroup's single trip in the largest grid; 24 KB and 12 bytes more, a second trip for some."""
    count = (1 << 35) + 6 * 1024 + 3
    print(f"fill {count}", flush=True)
    buf = rt.DeviceBuffer(4 * (count + 1))
    rt.check(rt.load().jpp_fill_u32(buf.ptr, 5, count + 1, None))
    rt.check(rt.load().jpp_fill_u32(buf.ptr, 0xabcd1234, count, None))
    for at in (0, (1 << 34) - 4096, (1 << 35) - 8192, (1 << 35) - 4, count - 6000):
        n = min(16384, count - at)
        assert (buf.download(np.uint32, (n,), 4 * at) == 0xabcd1234).all(), at
    assert buf.download(np.uint32, (1,), 4 * count)[0] == 5
    buf.free()


CACHED_BYTES = 192 << 20


@pytest.mark.parametrize("with_master,with_param", [(True, True), (True, False), (False, True)])
def test_adam_through_the_caches_and_past_them(with_master, with_param):
    """Up to 192 MiB of tensors a step goes through the caches, larger ones past them: the form on either side of the
    line, and the same bits from one call past them and two through them over the halves."""
    per = 12 + 4 * with_master + 2 * with_param
    line = CACHED_BYTES // per // 8 * 8
    n = line + 8
    print(f"adam {n} parameters, master {with_master}, param {with_param}", flush=True)
    block = np.random.default_rng(per).standard_normal(1 << 20, dtype=np.float32)
    long = np.resize(block, 4 * n)
    start = {"grad": long[:n], "m": long[n // 2:n // 2 + n] * np.float32(0.1), "v": np.abs(long[7:7 + n]) * np.float32(0.01),
             "master": long[n // 3:n // 3 + n], "param": rt.to_bf16_bits(long[n // 3:n // 3 + n])}

    def run(parts):
        b = {k: rt.DeviceBuffer.from_numpy(a) for k, a in start.items()}
        for at, count, form in parts:
            with rt.probe(form) as p:
                rt.adam_step(count, b["grad"].ptr + 4 * at, b["m"].ptr + 4 * at, b["v"].ptr + 4 * at, 3,
                             master=b["master"].ptr + 4 * at if with_master else None,
                             param=b["param"].ptr + 2 * at if with_param else None, zero_grad=True)
            assert p.launches == 1, (count, form)
        return {k: b[k].download(a.dtype, a.shape) for k, a in start.items()}

    half = n // 16 * 8
    one = run([(0, n, "adam_streamed")])
    two = run([(0, half, "adam_cached"), (half, n - half, "adam_cached")])
    for k in start:
        np.testing.assert_array_equal(one[k], two[k], err_msg=k)
    assert (one["grad"] == 0).all() and not np.array_equal(one["m"], start["m"])
    run([(0, line, "adam_cached")])
