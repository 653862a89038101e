"""Products of few tiles, whose waves each stage their own share of the contraction: fewer K-steps
than waves, than stages, remainders of both; tile rows that do not fill a group of the tile
walk, the last sizes of the range and the first behind it, leading dimensions larger than the extents.

Against float64 on the same bf16-valued operands.  A sum of k products is within (k + 8) 2^-24 of
the sum of their magnitudes in any order; it is rounded once to bf16 (2^-8 of its magnitude).
GELU and its derivative are evaluated in fp32 on the unrounded sum (slope at most 1.13), to 6e-7
times the argument (jaxpp_amd/csrc/gemm_wave.h)."""
import math

import numpy as np
import pytest

from jaxpp_amd import runtime as rt
from oracle import layers as L

pytestmark = pytest.mark.gpu
U = 2.0 ** -24
erf = np.vectorize(math.erf)


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def padded(x, pad):
    h = np.zeros((x.shape[0], x.shape[1] + pad), np.float32)
    h[:, :x.shape[1]] = x
    return rt.DeviceBuffer.from_f32_as_bf16(h), h.shape[1]


@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (128, 128, 192), (128, 384, 576), (384, 128, 320),
                                   (640, 768, 832), (512, 1024, 1088), (128, 2048, 128),
                                   (256, 2048, 64), (256, 2176, 64), (128, 256, 960)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("kind", ["nn", "nt", "gelu", "dgelu"])
@pytest.mark.parametrize("pad,tanh", [(0, 0), (8, 1)])
def test_wave_products(kind, m, n, k, pad, tanh):
    print(f"gemm {kind} {m}x{n}x{k} pad={pad} tanh={tanh}", flush=True)
    rng = np.random.default_rng(m + n + k)
    tb = kind in ("nn", "gelu")
    draw = lambda *s: L.bf16_round(rng.standard_normal(s, dtype=np.float32))
    A, B, bias, R = draw(m, k), L.bf16_round(draw(n, k) / np.float32(np.sqrt(k))), draw(n), draw(m, n)
    a, lda = padded(A, pad)
    b, ldb = padded(B.T if tb else B, pad)
    r, ldr = padded(R, pad)
    c, ldc = padded(np.zeros((m, n), np.float32), pad)
    c2, _ = padded(np.zeros((m, n), np.float32), pad)
    bb = rt.DeviceBuffer.from_f32_as_bf16(bias)
    s = A.astype(np.float64) @ B.astype(np.float64).T
    err = (k + 8) * U * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T + 8)
    kw = dict(nn=dict(bias=bb.ptr, resid=r.ptr, ldresid=ldr), nt=dict(resid=r.ptr, ldresid=ldr),
              gelu=dict(bias=bb.ptr, c2=c2.ptr, ldc2=ldc, gelu_tanh=tanh),
              dgelu=dict(aux=r.ptr, ldaux=ldr, gelu_tanh=tanh))[kind]
    epi = {"gelu": rt.EPI_GELU, "dgelu": rt.EPI_DGELU}.get(kind, rt.EPI_BF16)
    rt.gemm(a.ptr, b.ptr, c.ptr, m, n, k, lda, ldb, ldc, 0, int(tb), epi, **kw)
    rt.sync()
    got = c.download_bf16((m, ldc))
    assert (got[:, n:] == 0).all()
    got = got[:, :n]

    def near(x, want, slack):
        assert (np.abs(x - want) <= 2.0 ** -8 * np.abs(want) + slack).all()

    if kind in ("nn", "nt"):
        near(got, s + R + (bias if kind == "nn" else 0), err)
        return
    u = (s + bias if kind == "gelu" else R).astype(np.float64)
    if tanh:
        t = np.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3))
        g, dg = 0.5 * u * (1 + t), 0.5 * (1 + t) + 0.5 * u * (1 - t * t) * 0.7978845608028654 * (1 + 0.134145 * u * u)
    else:
        g = 0.5 * u * (1 + erf(u / math.sqrt(2)))
        dg = 0.5 * (1 + erf(u / math.sqrt(2))) + u * np.exp(-0.5 * u * u) / math.sqrt(2 * math.pi)
    if kind == "gelu":
        near(got, u, err)
        near(c2.download_bf16((m, ldc))[:, :n], g, 1.13 * err + 2e-6 * (1 + np.abs(u)))
    else:
        near(got, s * dg, 1.13 * err + 4e-6 * np.abs(s))
