"""Accumulated weight gradients in 128x128 tiles, two workgroups on a CU, at the edges of that form: more
tiles than CUs, contractions shorter than the two LDS stages and long ones, whose old values all
tiles of this size add at the end.  Against numpy in float64, prev + a^T b; fp32 accumulation errs by 6e-8
sqrt(K) of terms of size 0.3, the bar is 1e-4 sqrt(K)."""
import math

import numpy as np
import pytest

from jaxpp_amd import runtime as rt
from test_gpu_kernels import close, dev_bf16, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 128, 192, 1344])
@pytest.mark.parametrize("m,n", [(2176, 2048), (4352, 2048)])   # 272 and 544 tiles; the first are not whole 256s
def test_two_stage_128x128_weight_gradients(m, n, k):
    print(f"128x128 weight gradient {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + k)
    a, b = rnd(rng, k, m), rnd(rng, k, n, scale=0.3)
    prev = rng.standard_normal((m, n)).astype(np.float32)
    want = prev + a.astype(np.float64).T @ b.astype(np.float64)
    da, db = dev_bf16(a), dev_bf16(b)
    one, both = rt.DeviceBuffer.from_numpy(prev), rt.DeviceBuffer.from_numpy(prev)
    small = rt.DeviceBuffer.from_numpy(prev[:128, :256])
    rt.gemm(da.ptr, db.ptr, one.ptr, m, n, k, m, n, n, 1, 1, rt.EPI_ACC_F32, tile=1)
    # beside another product in one launch, the tile left to the library
    rt.gemm_multi([dict(a=da.ptr, b=db.ptr, c=small.ptr, m=128, n=256, k=k, lda=m, ldb=n, ldc=256),
                   dict(a=da.ptr, b=db.ptr, c=both.ptr, m=m, n=n, k=k, lda=m, ldb=n, ldc=n)])
    rt.sync()
    bar = 1e-4 * math.sqrt(k)
    close(one.download(np.float32, (m, n)), want, bar, "by itself")
    close(both.download(np.float32, (m, n)), want, bar, "in a launch of two")
    close(small.download(np.float32, (128, 256)), want[:128, :256], bar, "the other product")


@pytest.mark.parametrize("m,n,k,form", [
    (4096, 4096, 128, "128x128w8"), (8192, 4096, 256, "128x128w8"),   # few K-steps: two tiles' traffic on a CU
    (4096, 4096, 8192, "256x256w8"), (768, 1024, 256, "64x64k2")])
def test_form_of_a_weight_gradient(m, n, k, form):
    """The form that the estimate names runs, with whole 256x256 tiles too."""
    print(f"weight gradient {m}x{n}x{k}: {form}", flush=True)
    a, b, c = (rt.DeviceBuffer(q) for q in (2 * k * m, 2 * k * n, 4 * m * n))
    for q in (a, b, c):
        q.zero()
    with rt.probe("*") as p:
        rt.gemm(a.ptr, b.ptr, c.ptr, m, n, k, m, n, n, 1, 1, rt.EPI_ACC_F32)
        rt.sync()
    assert list(p.classes) == [f"gemm_tn_accf32_{form}"], p.classes


@pytest.mark.parametrize("epi,name", [(rt.EPI_BF16, "bf16"), (rt.EPI_F32, "f32")])
@pytest.mark.parametrize("m,n,k,form", [(2304, 768, 256, "64x64k2"), (6912, 1792, 704, "256x256w8"),
                                        (640, 3200, 64, "64x64k2"), (1024, 1024, 1024, "64x64s4k2")])
def test_form_of_a_weight_gradient_that_is_not_accumulated(m, n, k, form, epi, name):
    """Products of the same layout without an old value go by the estimate of products without one; the bits are
    those of the tile asked for by name, and the values float64's to a bf16 rounding (fp32 sums of terms of
    size 0.3: 1e-4 sqrt(K))."""
    print(f"weight gradient {m}x{n}x{k} {name}: {form}", flush=True)
    rng = np.random.default_rng(m + k)
    a, b = rnd(rng, k, m), rnd(rng, k, n, scale=0.3)
    da, db = dev_bf16(a), dev_bf16(b)
    es = 2 if epi == rt.EPI_BF16 else 4
    own, named = rt.DeviceBuffer(es * m * n), rt.DeviceBuffer(es * m * n)
    with rt.probe("*") as p:
        rt.gemm(da.ptr, db.ptr, own.ptr, m, n, k, m, n, n, 1, 1, epi)
        rt.sync()
    assert list(p.classes) == [f"gemm_tn_{name}_{form}"], p.classes
    rt.gemm(da.ptr, db.ptr, named.ptr, m, n, k, m, n, n, 1, 1, epi, tile={"64": 5, "128": 1, "256": 4}[form.split("x")[0]])
    rt.sync()
    dt = np.uint16 if es == 2 else np.uint32
    np.testing.assert_array_equal(own.download(dt, (m, n)), named.download(dt, (m, n)))
    got = own.download_bf16((m, n)) if es == 2 else own.download(np.float32, (m, n))
    want = a.astype(np.float64).T @ b.astype(np.float64)
    assert (np.abs(got - want) <= 1e-4 * math.sqrt(k) + (2.0 ** -8 * np.abs(want) if es == 2 else 0)).all()
