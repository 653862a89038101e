"""Attention problems that run as 16 rows per workgroup against the same sequences inside a batch
large enough to run on the kernels for whole blocks.

Both round the probabilities and the score cotangents to bf16 where they become matrix operands
and the results once more, so an element differs by a few of those roundings: 2e-2 of the largest
magnitude, the bound the kernels are held to against the oracle, and 1e-2 in the 2-norm (2^-9 of
each of the at most four roundings, all one way)."""
import ctypes as C

import numpy as np
import pytest

from jaxpp_amd import runtime as rt
from oracle import layers as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def run(q, k, v, do, causal, pad, rope):
    B, S, H, d = q.shape
    K, T = k.shape[2], B * S
    w = (H + 2 * K) * d + pad
    qkv = np.zeros((T, w), np.float32)
    qkv[:, :(H + 2 * K) * d] = np.concatenate([x.reshape(T, -1) for x in (q, k, v)], 1)
    bq, bdo = (rt.DeviceBuffer.from_f32_as_bf16(x) for x in (qkv, do.reshape(T, -1)))
    bo, bd = rt.DeviceBuffer(T * H * d * 2), rt.DeviceBuffer(T * w * 2)
    lse, delta = rt.DeviceBuffer(T * H * 4), rt.DeviceBuffer(T * H * 8)
    bd.zero()
    at = (0, H * d * 2, (H + K) * d * 2)
    a = rt.AttnArgs(*(bq.ptr + x for x in at), bo.ptr, lse.ptr, bdo.ptr, *(bd.ptr + x for x in at),
                    delta.ptr, w, w, w, H * d, H * d, w, w, w, B, S, H, K, d, causal)
    tabs = [rt.DeviceBuffer.from_numpy(t) for t in L.rope_tables(S, d, 5e5, np.float32)]
    if rope:
        a.rope_cos, a.rope_sin = tabs[0].ptr, tabs[1].ptr
    lib = rt.load()
    rt.check(lib.jpp_attn_fwd(None, C.byref(a)))
    rt.check(lib.jpp_attn_bwd(None, C.byref(a)))
    rt.sync()
    d_all = bd.download_bf16((T, w))
    assert (d_all[:, (H + 2 * K) * d:] == 0).all()     # nothing beside the rows' own columns
    return (bo.download_bf16((B, S, H * d)), d_all[:, :(H + 2 * K) * d].reshape(B, S, -1),
            lse.download(np.float32, (B, H, S)))


@pytest.mark.parametrize("d,causal,H,K,B,S", [
    (64, 0, 1, 1, 1, 128), (128, 1, 2, 2, 1, 128), (64, 1, 4, 1, 2, 128), (128, 0, 8, 2, 1, 256),
    # one workgroup of 16 rows per CU exactly; three 128-blocks; the longest of the range
    (128, 1, 8, 8, 2, 256), (64, 0, 3, 3, 3, 384), (64, 1, 2, 2, 1, 2048), (128, 0, 2, 1, 1, 1152),
])
@pytest.mark.parametrize("pad,rope", [(0, False), (8, True)])
def test_small_attention_equals_whole_blocks(d, causal, H, K, B, S, pad, rope):
    print(f"attention d={d} causal={causal} heads={H}/{K} b={B} s={S} pad={pad} rope={rope}", flush=True)
    rng = np.random.default_rng(d + S + H)
    more = 16384 // (K * S) + 1     # (the blocks' side of both rules; the launches below are checked)
    draw = lambda h: L.bf16_round(rng.standard_normal((B + more, S, h, d), dtype=np.float32))
    q, k, v, do = draw(H), draw(K), draw(K), draw(H)
    with rt.probe("*") as p:
        small = run(*(x[:B] for x in (q, k, v, do)), causal, pad, rope)
    assert "attn_bwd_small" in p.classes and "attn_bwd_dq" not in p.classes, p.classes
    with rt.probe("*") as p:
        large = run(q, k, v, do, causal, pad, rope)
    assert "attn_bwd_small" not in p.classes and p.classes["attn_bwd_dq"][0] == 1, p.classes
    for name, s, g in zip(("o", "dqkv"), small, large):
        g = g[:B]
        assert np.abs(s - g).max() <= 2e-2 * np.abs(g).max(), name
        assert np.linalg.norm(s - g) <= 1e-2 * np.linalg.norm(g), name
    np.testing.assert_allclose(small[2], large[2][:B], rtol=0, atol=2e-4)
