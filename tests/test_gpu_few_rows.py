"""A norm's backward and the column sums on few rows (one launch, sums by 64 columns): ragged
rows and columns, with and without residual, dx over dy, several tensors in one launch.

Against float64 on the same bf16-valued inputs.  A sum of n terms, each rounded at most four
times on its way, is within (n + 8) 2^-24 of the sum of their magnitudes; dx is such a result
rounded once more to bf16 (2^-8 of its magnitude)."""
import ctypes as C

import numpy as np
import pytest

from jaxpp_amd import runtime as rt
from jaxpp_amd import schedules as S
from jaxpp_amd.model import LayerSpec, init_layer_params
from jaxpp_amd.plan import make_rank_plan
from oracle import layers as L
from test_gpu_stage import run_on_gpu

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def bf16(a):
    return rt.DeviceBuffer.from_f32_as_bf16(a)


def f32(a):
    return rt.DeviceBuffer.from_numpy(np.ascontiguousarray(a, np.float32))


@pytest.mark.parametrize("ln", [True, False])
@pytest.mark.parametrize("rows,cols,resid,in_place", [
    (1, 8, False, False), (7, 72, True, False), (65, 136, True, True), (128, 128, False, False),
    (515, 1024, True, False), (300, 1032, False, True), (256, 2048, True, False), (40, 4088, True, False),
    # the last sizes of the range and the first behind it
    (1024, 512, False, False), (1025, 512, False, False), (1536, 520, True, False), (1537, 520, True, False)])
def test_norm_backward(ln, rows, cols, resid, in_place):
    print(f"norm_bwd ln={ln} {rows}x{cols} resid={resid} in_place={in_place}", flush=True)
    rng = np.random.default_rng(rows + cols)
    x, dy, res = (L.bf16_round(rng.standard_normal((rows, cols), dtype=np.float32)) for _ in range(3))
    gamma = L.bf16_round(rng.standard_normal(cols, dtype=np.float32))
    mean = rng.standard_normal(rows, dtype=np.float32) if ln else np.zeros(rows, np.float32)
    rstd = rng.random(rows, dtype=np.float32) + np.float32(0.5)
    g0, b0 = (rng.standard_normal(cols, dtype=np.float32) for _ in range(2))
    bx, bdy, bres, bg = bf16(x), bf16(dy), bf16(res), bf16(gamma)
    bm, br, dg, db = f32(mean), f32(rstd), f32(g0), f32(b0)
    part = rt.DeviceBuffer(2 * 4 * rt.NORM_PARTIALS * cols)
    bdx = bdy if in_place else rt.DeviceBuffer(rows * cols * 2)
    a = rt.NormArgs()
    a.x, a.dy, a.gamma, a.rstd, a.dx, a.dgamma, a.partial = (
        bx.ptr, bdy.ptr, bg.ptr, br.ptr, bdx.ptr, dg.ptr, part.ptr)
    if ln:
        a.mean, a.dbeta = bm.ptr, db.ptr
    if resid:
        a.resid = bres.ptr
    a.rows, a.cols, a.eps = rows, cols, 1e-5
    rt.check(rt.load().jpp_norm_bwd(None, C.byref(a)))
    rt.sync()
    d = dy.astype(np.float64)
    xh = (x.astype(np.float64) - mean[:, None]) * rstd[:, None]
    term = (np.abs(x) + np.abs(mean)[:, None]) * rstd[:, None]
    assert (np.abs(dg.download(np.float32, (cols,)) - (g0 + (d * xh).sum(0))) <=
            (rows + 8) * U * (np.abs(g0) + (np.abs(d) * term).sum(0))).all()
    want_b = b0 + d.sum(0) if ln else b0
    assert (np.abs(db.download(np.float32, (cols,)) - want_b) <=
            (rows + 8) * U * (np.abs(b0) + np.abs(d).sum(0))).all()
    w = d * gamma
    want = (w - (w.mean(1, keepdims=True) if ln else 0) - xh * (w * xh).mean(1, keepdims=True)) * rstd[:, None]
    mag = (np.abs(w) + np.abs(w).mean(1, keepdims=True) +
           (1 + term) * (np.abs(w) * term).mean(1, keepdims=True) * 2) * rstd[:, None]
    if resid:
        want, mag = want + res, mag + np.abs(res)
    got = bdx.download_bf16((rows, cols))
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + (cols + 16) * U * mag).all()


@pytest.mark.parametrize("rows,cols", [(1, (8,)), (129, (64, 72)), (130, (8, 256, 1032)), (1100, (768, 3072, 768, 2304)), (4096, (64,)), (4097, (64, 8))])
def test_column_sums(rows, cols):
    print(f"colsum {rows} x {cols}", flush=True)
    rng = np.random.default_rng(rows)
    xs = [L.bf16_round(rng.standard_normal((rows, c + 8), dtype=np.float32)) for c in cols]
    acc0 = [rng.standard_normal(c, dtype=np.float32) for c in cols]
    bufs, accs = [bf16(x) for x in xs], [f32(a) for a in acc0]
    items = (rt.ColsumItem * len(cols))()
    for it, b, a, c in zip(items, bufs, accs, cols):
        it.x, it.ld, it.cols, it.acc = b.ptr, c + 8, c, a.ptr
    part = rt.DeviceBuffer(4 * rt.NORM_PARTIALS * sum(cols))
    rt.check(rt.load().jpp_colsum_accum_multi(None, len(cols), items, rows, part.ptr))
    rt.sync()
    for x, a0, a, c in zip(xs, acc0, accs, cols):
        x = x[:, :c].astype(np.float64)
        assert (np.abs(a.download(np.float32, (c,)) - (a0 + x.sum(0))) <=
                (rows + 8) * U * (np.abs(a0) + np.abs(x).sum(0))).all()


# weight gradients on 64x64 tiles (few and many K-steps), on 128x128 ones, on 256x256 ones, some of them
# apart; the last rows that are few and the first that are not
@pytest.mark.parametrize("family,h,heads,f,seq,batch", [
    ("bert", 128, 2, 512, 128, 1), ("decoder", 128, 2, 384, 384, 5), ("bert", 640, 10, 1280, 128, 3),
    ("decoder", 1024, 8, 4096, 512, 1), ("bert", 768, 6, 3072, 512, 4), ("bert", 1024, 16, 4096, 512, 3),
    ("decoder", 1408, 11, 5632, 128, 9), ("bert", 128, 2, 256, 512, 8), ("decoder", 128, 2, 256, 1408, 3)])
def test_bias_gradients_beside_weight_gradients(family, h, heads, f, seq, batch):
    """On one stream a layer's bias gradients go with its weight gradients, on two they go before them: the same
    sums to the last bit, whichever launch adds them up."""
    print(f"bias gradients {family} {h} {f} {seq} x {batch}", flush=True)
    spec = LayerSpec(family, h, heads, f, seq, batch, head_dim=h // heads, causal=family == "decoder", eps=1e-5)
    plan = make_rank_plan(S.Std1F1B(1), 2, 0)
    params = {0: [init_layer_params(spec, 3, li, perturb=True) for li in range(2)]}
    _, _, apart = run_on_gpu(spec, plan, 2, params, two_streams=True)
    _, _, here = run_on_gpu(spec, plan, 2, params, two_streams=False)
    for li in range(2):
        for name, w in apart[0][li].items():
            assert np.abs(w).max() > 0 and np.array_equal(here[0][li][name], w), name


@pytest.mark.parametrize("family,h,heads,f,seq", [("bert", 128, 2, 512, 128), ("decoder", 1024, 8, 4096, 512)])
def test_probe_counts_the_sums_that_go_along(family, h, heads, f, seq):
    """Their reads are bytes of the launch that they are part of."""
    spec = LayerSpec(family, h, heads, f, seq, 1, head_dim=h // heads, causal=family == "decoder", eps=1e-5)
    params = {0: [init_layer_params(spec, 3, 0, perturb=True)]}
    with rt.probe("*") as p:
        run_on_gpu(spec, make_rank_plan(S.Std1F1B(1), 1, 0), 1, params, two_streams=False)
    (name, (launches, _, _, got)), = ((k, v) for k, v in p.classes.items() if k.endswith("_multi"))
    shapes = [(f, h), (h, f), (h, h), (h, 3 * h)]
    want = sum(2 * seq * (m + n) + 8 * m * n for m, n in shapes) + sum(2 * seq * n for _, n in shapes)
    assert launches == 1 and "colsum" not in p.classes and got == want, (name, launches, got, want)
