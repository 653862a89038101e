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
