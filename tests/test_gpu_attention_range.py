"""Problems of more than one workgroup of 16 rows per CU that still run as 16 rows per workgroup, by the
estimate of their time: many query heads per key head, several rounds of workgroups, 384 and 640 positions (which
leave some of the eight waves without a last step).  Against the kernels for whole blocks, with that
comparison's bounds; and the estimate's two sides."""
import ctypes as C

import pytest

import test_gpu_attention_small as small
from jaxpp_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


@pytest.mark.parametrize("d,causal,H,K,B,S", [(128, 1, 16, 4, 1, 512), (64, 1, 32, 8, 1, 640), (128, 0, 8, 1, 1, 1024),
                                              (64, 0, 16, 4, 2, 512), (64, 0, 12, 12, 1, 384), (128, 1, 4, 1, 2, 128)])
@pytest.mark.parametrize("pad,rope", [(0, False), (8, True)])
def test_larger_problems_of_16_rows_equal_whole_blocks(d, causal, H, K, B, S, pad, rope):
    small.test_small_attention_equals_whole_blocks(d, causal, H, K, B, S, pad, rope)


@pytest.mark.parametrize("d,causal,H,K,B,S,own", [
    (64, 0, 16, 16, 8, 512, False), (128, 1, 32, 8, 1, 4096, False), (64, 1, 16, 16, 8, 128, False),
    (128, 1, 16, 4, 1, 512, True), (64, 0, 2, 2, 1, 128, True)])
def test_side_of_the_estimate(d, causal, H, K, B, S, own):
    """Large problems keep the blocks, small ones take 16 rows, in the backward."""
    T, w = B * S, (H + 2 * K) * d
    b = [rt.DeviceBuffer(n) for n in (2 * T * w, 2 * T * H * d, 2 * T * H * d, 2 * T * w, 4 * T * H, 8 * T * H)]
    for q in b:
        q.zero()
    at = (0, H * d * 2, (H + K) * d * 2)
    a = rt.AttnArgs(*(b[0].ptr + x for x in at), b[1].ptr, b[4].ptr, b[2].ptr, *(b[3].ptr + x for x in at), b[5].ptr,
                    w, w, w, H * d, H * d, w, w, w, B, S, H, K, d, causal)
    with rt.probe("*") as p:
        rt.check(rt.load().jpp_attn_bwd(None, C.byref(a)))
        rt.sync()
    assert ("attn_bwd_small" in p.classes) == own, p.classes


@pytest.mark.parametrize("d,causal,H,K,B,S,own", [
    # many sequences of a head or two (more workgroups of keys than CUs), and beyond every measured size
    (64, 1, 1, 1, 64, 256, False), (128, 1, 2, 2, 16, 384, False), (128, 1, 1, 1, 32, 384, False),
    (64, 0, 1, 1, 130, 128, False),
    # where the estimates are close and a round of workgroups more makes the 16 rows the slower side
    (64, 0, 3, 3, 3, 1536, False), (128, 0, 5, 5, 2, 1280, False), (64, 1, 23, 23, 1, 640, False),
    # the sizes up to 4096 rows keep their side, and long sequences of one head theirs
    (64, 0, 2, 2, 8, 256, True), (128, 0, 4, 1, 1, 2048, True), (128, 1, 1, 1, 1, 8192, True)])
def test_side_of_the_estimate_with_many_rows(d, causal, H, K, B, S, own):
    test_side_of_the_estimate(d, causal, H, K, B, S, own)
