"""The f32 operators at the edges of their tiles: contractions of fewer steps than waves or
prefetch stages, each output tile height in each orientation, leading dimensions and addresses
that are multiples of 4 bytes only, column sums over ragged rows and columns, attention whose
key tiles are fewer than the waves that share them.

Bounds are a sum's own: each of n products is rounded once on its way into an fp32 chain, so an
element is within (n + 4) 2^-24 of the sum of its terms' magnitudes."""
import ctypes as C

import numpy as np
import pytest

import parity
from jaxpp_amd import runtime as rt
from jaxpp_amd import schedules as S
from jaxpp_amd.model import LayerSpec, init_layer_params
from jaxpp_amd.plan import make_rank_plan
from test_gpu_stage import run_on_gpu, run_on_oracle

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def dev(a):
    return rt.DeviceBuffer.from_numpy(np.ascontiguousarray(a, dtype=np.float32))


def padded(x, pad, at=4):
    """x in rows of a leading dimension `pad` larger, and a device copy `at` bytes past an
    aligned address."""
    ld = x.shape[1] + pad
    h = np.zeros(x.shape[0] * ld + at // 4, np.float32)
    h[at // 4:].reshape(x.shape[0], ld)[:, :x.shape[1]] = x
    return dev(h), ld


# strips of 16 x 64: fewer than a CU each (16-row tiles), two each (32), four each (64)
SHAPES = [(64, 64, 16), (64, 64, 32), (64, 128, 48), (128, 64, 80), (128, 128, 416), (512, 1024, 144),
          (512, 1024, 160), (1024, 1024, 64), (1024, 1088, 208)]


@pytest.mark.parametrize("aligned", [False, True])
@pytest.mark.parametrize("lay", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_gemm_f32_tiles(lay, m, n, k, aligned):
    print(f"gemm_f32 {lay} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    ta, tb = {"nn": (0, 1), "nt": (0, 0), "tn": (1, 1), "tt": (1, 0)}[lay]
    A, B = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
    c0 = rng.standard_normal((m, n), dtype=np.float32)
    at = 0 if aligned else 4        # the operands' distance from an aligned address
    da, lda = padded(A.T if ta else A, 4 if aligned else 3, at)
    db, ldb = padded(B.T if tb else B, 8 if aligned else 5, at)
    dc, ldc = padded(c0, 1)
    rt.gemm(da.ptr + at, db.ptr + at, dc.ptr + 4, m, n, k, lda, ldb, ldc, ta, tb, rt.EPI_ACC_F32, f32=True)
    rt.sync()
    raw = dc.download(np.float32, (m * ldc + 1,))
    got = raw[1:].reshape(m, ldc)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    bound = (k + 4) * U * (np.abs(A64) @ np.abs(B64).T + np.abs(c0))
    assert (np.abs(got[:, :n] - (c0 + A64 @ B64.T)) <= bound).all()
    assert raw[0] == 0 and (got[:, n:] == 0).all()      # nothing beside the output is written


@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 17), (64, 16), (513, 100), (1000, 256)])
def test_norm_bwd_and_column_sums_f32_ragged(rows, cols):
    rng = np.random.default_rng(rows + cols)
    x, dy, resid = (rng.standard_normal((rows, cols), dtype=np.float32) for _ in range(3))
    gamma, dg0, db0 = (rng.standard_normal(cols, dtype=np.float32) for _ in range(3))
    mean = rng.standard_normal(rows, dtype=np.float32)
    rstd = rng.random(rows, dtype=np.float32) + np.float32(0.5)
    bufs = {k: dev(v) for k, v in dict(x=x, dy=dy, resid=resid, gamma=gamma, mean=mean, rstd=rstd,
                                       dgamma=dg0, dbeta=db0, dx=np.zeros_like(x)).items()}
    lib = rt.load()
    a = rt.NormArgs()
    for k, v in bufs.items():
        setattr(a, k, v.ptr)
    a.rows, a.cols, a.eps = rows, cols, 1e-5
    rt.check(lib.jpp_norm_bwd_f32(None, C.byref(a)))
    acc = dev(db0)
    rt.check(lib.jpp_colsum_accum_f32(None, bufs["dy"].ptr, cols, rows, cols, acc.ptr))
    rt.sync()
    d, xh = dy.astype(np.float64), (x.astype(np.float64) - mean[:, None]) * rstd[:, None]
    n = rows + 4
    # (a term of dgamma is itself rounded three times)
    assert (np.abs(bufs["dgamma"].download(np.float32, (cols,)) - (dg0 + (d * xh).sum(0))) <=
            (n + 3) * U * (np.abs(dg0) + np.abs(d * xh).sum(0) +
                           (np.abs(d) * np.abs(mean)[:, None] * rstd[:, None]).sum(0))).all()
    for got in (bufs["dbeta"], acc):
        assert (np.abs(got.download(np.float32, (cols,)) - (db0 + d.sum(0))) <=
                n * U * (np.abs(db0) + np.abs(d).sum(0))).all()
    w = d * gamma
    want = (w - w.mean(1, keepdims=True) - xh * (w * xh).mean(1, keepdims=True)) * rstd[:, None] + resid
    mag = (np.abs(w) + np.abs(w).mean(1, keepdims=True) +
           (np.abs(x) + np.abs(mean)[:, None]) * rstd[:, None] * (1 + np.abs(w * xh).mean(1, keepdims=True)) *
           (1 + np.abs(xh))) * rstd[:, None] + np.abs(resid)
    assert (np.abs(bufs["dx"].download(np.float32, (rows, cols)) - want) <= (cols + 12) * U * mag).all()


@pytest.mark.parametrize("ln", [True, False])
@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 63), (6, 64), (7, 65), (512, 256), (9, 257), (66, 512), (3, 513),
                                       (130, 1024), (11, 1025), (65, 4100)])
def test_norm_fwd_f32_row_lengths(rows, cols, ln):
    """Rows a lane holds in 4, 8 or 16 registers, the last and first lengths of each, and longer ones.  The mean and
    the mean square are sums of cols terms, each within (cols + 3) 2^-24 of its terms' magnitudes."""
    rng = np.random.default_rng(rows * 3 + cols)
    x = rng.standard_normal((rows, cols), dtype=np.float32) + np.float32(0.5)
    gamma, beta = (rng.standard_normal(cols, dtype=np.float32) for _ in range(2))
    bufs = dict(x=dev(x), gamma=dev(gamma), y=dev(np.zeros((rows + 1, cols))), rstd=dev(np.zeros(rows)))
    if ln:
        bufs.update(beta=dev(beta), mean=dev(np.zeros(rows)))
    a = rt.NormArgs()
    for k, b in bufs.items():
        setattr(a, k, b.ptr)
    a.rows, a.cols, a.eps = rows, cols, 1e-3
    rt.check(rt.load().jpp_norm_fwd_f32(None, C.byref(a)))
    rt.sync()
    x64 = x.astype(np.float64)
    mean = x64.mean(1, keepdims=True) if ln else np.zeros((rows, 1))
    d = x64 - mean
    var = (d * d).mean(1, keepdims=True) + a.eps
    rstd = 1 / np.sqrt(var)
    e = (cols + 3) * U                       # of the mean, of the variance, and half of it of rstd
    em = e * np.abs(x64).mean(1, keepdims=True) if ln else 0.0
    er = e + (2 * em * np.abs(d).mean(1, keepdims=True) + em * em) / var + 4 * U
    y = bufs["y"].download(np.float32, (rows + 1, cols))
    want = d * rstd * gamma + (beta if ln else 0)
    mag = np.abs(gamma) * rstd
    assert (np.abs(y[:rows] - want) <= mag * (em + np.abs(d) * (er + 4 * U)) + 2 * U * np.abs(want) + 1e-30).all()
    assert (y[rows] == 0).all()
    assert (np.abs(bufs["rstd"].download(np.float32, (rows,)) - rstd[:, 0]) <= (er * rstd)[:, 0]).all()
    if ln:
        assert (np.abs(bufs["mean"].download(np.float32, (rows,)) - mean[:, 0]) <= em[:, 0]).all()


@pytest.mark.parametrize("d,hq,hk,seq,causal", [(64, 2, 1, 64, 1), (64, 3, 3, 192, 0), (128, 4, 2, 64, 0),
                                                (128, 2, 2, 320, 1)])
def test_attention_f32_tiles(d, hq, hk, seq, causal):
    """Against float64; a difference of 2^-24 (d + 4) of the largest score moves a probability by
    that share, and a result is a sum of d or seq terms of that error: 1e-5 of the largest
    magnitude covers the sizes here."""
    print(f"attention_f32 d={d} heads={hq}/{hk} seq={seq} causal={causal}", flush=True)
    rng = np.random.default_rng(d + seq)
    B, g = 2, hq // hk
    q, do = (rng.standard_normal((B, seq, hq, d), dtype=np.float32) for _ in range(2))
    k, v = (rng.standard_normal((B, seq, hk, d), dtype=np.float32) for _ in range(2))
    qd, kd, vd, dod = dev(q), dev(k), dev(v), dev(do)
    o, dq = (rt.DeviceBuffer(q.nbytes) for _ in range(2))
    dk, dv = (rt.DeviceBuffer(k.nbytes) for _ in range(2))
    lse, delta = rt.DeviceBuffer(B * hq * seq * 4), rt.DeviceBuffer(B * hq * seq * 4)
    a = rt.AttnArgs()
    a.q, a.k, a.v, a.o, a.lse, a.d_o, a.dq, a.dk, a.dv, a.delta = (
        qd.ptr, kd.ptr, vd.ptr, o.ptr, lse.ptr, dod.ptr, dq.ptr, dk.ptr, dv.ptr, delta.ptr)
    a.ldq = a.ldo = a.lddo = a.lddq = hq * d
    a.ldk = a.ldv = a.lddk = a.lddv = hk * d
    a.batch, a.seq, a.n_heads, a.n_kv_heads, a.head_dim, a.causal = B, seq, hq, hk, d, causal
    lib = rt.load()
    rt.check(lib.jpp_attn_fwd_f32(None, C.byref(a)))
    rt.check(lib.jpp_attn_bwd_f32(None, C.byref(a)))
    rt.sync()
    q, k, v, do = (x.astype(np.float64).transpose(0, 2, 1, 3) for x in (q, k, v, do))
    k, v = k.repeat(g, 1), v.repeat(g, 1)
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(d)
    if causal:
        s = np.where(np.tril(np.ones((seq, seq), bool)), s, -np.inf)
    mx = s.max(-1, keepdims=True)
    e = np.exp(s - mx)
    p = e / e.sum(-1, keepdims=True)
    out = p @ v
    dp = do @ v.transpose(0, 1, 3, 2)
    ds = p * (dp - (do * out).sum(-1, keepdims=True)) / np.sqrt(d)
    want = {"o": out, "dq": ds @ k}
    want["dk"], want["dv"] = (x.reshape(B, hk, g, seq, d).sum(2) for x in
                              (ds.transpose(0, 1, 3, 2) @ q, p.transpose(0, 1, 3, 2) @ do))
    for name, buf in (("o", o), ("dq", dq), ("dk", dk), ("dv", dv)):
        w = want[name].transpose(0, 2, 1, 3)
        assert np.abs(buf.download(np.float32, w.shape) - w).max() <= 1e-5 * np.abs(w).max(), name
    w = (mx + np.log(e.sum(-1, keepdims=True)))[..., 0]
    assert np.abs(lse.download(np.float32, w.shape) - w).max() <= 1e-5 * np.abs(w).max()


# 16 x 64 strips of a layer's weight gradients: 128 (16-row tiles), 384 (32), 768 and more (64), 400 (32)
@pytest.mark.parametrize("family,h,heads,f,seq", [
    ("bert", 128, 2, 256, 128), ("bert", 256, 4, 256, 256), ("bert", 256, 4, 1024, 384),
    ("decoder", 384, 6, 640, 128), ("llama", 256, 4, 128, 128)])
def test_layer_weight_and_bias_gradients_in_one_launch_f32(family, h, heads, f, seq):
    """On one stream a layer's bias gradients go with its weight gradients, on two they go before them: the same
    sums, whichever launch adds them up, and those of the oracle."""
    print(f"wgrads_f32 {family} {h} {f} {seq}", flush=True)
    spec = LayerSpec(family, h, heads, f, seq, 1, n_kv_heads=heads, head_dim=64, causal=family != "bert", eps=1e-5,
                     dtype="f32")
    sched = S.Std1F1B(1)
    plan = make_rank_plan(sched, 2, 0)
    params = {0: [init_layer_params(spec, 3, li, perturb=True) for li in range(2)]}
    _, _, apart = run_on_gpu(spec, plan, 2, params, two_streams=True)
    _, _, here = run_on_gpu(spec, plan, 2, params, two_streams=False)
    _, _, want = run_on_oracle(spec, plan, params, S.preprocess_schedule_tasks(sched.tasks(2), 0, False)[0])
    for li in range(2):
        for name, w in want[0][li].items():
            assert np.array_equal(here[0][li][name], apart[0][li][name]), name
            parity.close(here[0][li][name], w.reshape(here[0][li][name].shape).astype(np.float64), 1e-4, name)


# workgroups (rows / 16 x heads of both kinds): 16, 128, 192, 256, 384
@pytest.mark.parametrize("d,hq,hk,seq,batch,causal", [(64, 2, 2, 64, 1, 0), (64, 6, 2, 128, 2, 1), (64, 4, 4, 128, 4, 0),
                                                      (128, 2, 1, 128, 8, 1), (128, 3, 3, 64, 4, 0), (64, 8, 4, 256, 2, 0)])
def test_attention_backward_f32_at_once_and_in_two(d, hq, hk, seq, batch, causal):
    """Few workgroups: dQ, dK and dV in one launch, where they lie apart from the inputs; dK over K and dV over V keep
    the two.  The same bits, with the results interleaved or not."""
    print(f"attention_bwd_f32 d={d} heads={hq}/{hk} {batch}x{seq} causal={causal}", flush=True)
    rng = np.random.default_rng(d + seq + hq)
    T, W = batch * seq, (hq + 2 * hk) * d
    qkv, o, do = (rng.standard_normal((T, w), dtype=np.float32) for w in (W, hq * d, hq * d))
    lib = rt.load()
    got = []
    for over in (False, True):
        bufs = dict(qkv=dev(qkv), o=dev(o), d_o=dev(do), lse=dev(np.zeros(batch * hq * seq)),
                    delta=dev(np.zeros(2 * batch * hq * seq)), g=dev(np.zeros((T, W))))
        a = rt.AttnArgs()
        a.q, a.k, a.v = (bufs["qkv"].ptr + 4 * d * n for n in (0, hq, hq + hk))
        a.dq, a.dk, a.dv = (bufs["g"].ptr + 4 * d * n for n in (0, hq, hq + hk))
        a.ldq = a.ldk = a.ldv = a.lddq = a.lddk = a.lddv = W
        a.ldo = a.lddo = hq * d
        a.o, a.d_o, a.lse, a.delta = (bufs[k].ptr for k in ("o", "d_o", "lse", "delta"))
        a.batch, a.seq, a.n_heads, a.n_kv_heads, a.head_dim, a.causal = batch, seq, hq, hk, d, causal
        rt.check(lib.jpp_attn_fwd_f32(None, C.byref(a)))
        if over:
            a.dk, a.dv = a.k, a.v
        rt.check(lib.jpp_attn_bwd_f32(None, C.byref(a)))
        rt.sync()
        g = bufs["g"].download(np.float32, (T, W))
        if over:
            g[:, hq * d:] = bufs["qkv"].download(np.float32, (T, W))[:, hq * d:]
        got.append(g)
    assert np.array_equal(*got) and np.isfinite(got[0]).all() and (got[0] != 0).mean() > 0.9


# a layer's ways: a launch per product; one launch, on tiles of 16 / 32 / 64 rows, with the sums along or behind
@pytest.mark.parametrize("h,heads,f,seq,way", [
    (512, 8, 2048, 1024, None), (128, 2, 256, 128, "along"), (128, 2, 512, 1152, "apart"), (256, 4, 512, 256, "along"),
    (256, 4, 512, 1024, "apart"), (256, 4, 1024, 512, "apart"), (512, 8, 1024, 512, "along"), (384, 6, 768, 1024, "along"),
    (512, 8, 1024, 1024, "apart")])
def test_ways_of_a_layers_weight_gradients_f32(h, heads, f, seq, way):
    """The way that the sizes choose, and the bits of the same gradients with the sums in front of them, on two
    streams."""
    print(f"wgrads_f32 {h} {f} {seq} {way}", flush=True)
    spec = LayerSpec("bert", h, heads, f, seq, 1, n_kv_heads=heads, head_dim=64, causal=False, eps=1e-5, dtype="f32")
    sched = S.Std1F1B(1)
    plan = make_rank_plan(sched, 1, 0)
    params = {0: [init_layer_params(spec, 3, 0, perturb=True)]}
    _, _, two = run_on_gpu(spec, plan, 1, params, two_streams=True)
    with rt.probe("*") as p:
        _, _, one = run_on_gpu(spec, plan, 1, params, two_streams=False)
    assert {k: v[0] for k, v in p.classes.items() if k.startswith("wgrads_f32")} == (
        {} if way is None else {"wgrads_f32_sums" if way == "along" else "wgrads_f32": 1}), p.classes
    _, _, want = run_on_oracle(spec, plan, params, S.preprocess_schedule_tasks(sched.tasks(1), 0, False)[0])
    for name, w in want[0][0].items():
        got = one[0][0][name]
        assert np.array_equal(got, two[0][0][name]), name
        parity.close(got, w.reshape(got.shape).astype(np.float64), 1e-4, name)
