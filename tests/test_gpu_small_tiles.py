"""Products with fewer tiles than the device has CUs: the 64x64 tile whose two wave groups take
the K-steps in turn, its 64x128 form for rotated heads of 128, the five-stage 128x128 tile, and
several weight gradients in one grid of small tiles - at the sizes where they can go wrong: one
K-step (a group without work), odd numbers of steps, fewer steps than LDS stages, more tiles than
one round.  Against numpy in float64; the bar for fp32 outputs is 1e-4 sqrt(K) of N(0, 1) x
N(0, 0.3) products (fp32 accumulation errs by 6e-8 sqrt(K) of terms of size 0.3), for bf16 ones
1e-2 (an ulp is 4e-3 of the element)."""
import math

import numpy as np
import pytest

from jaxpp_amd import runtime as rt
import test_gpu_kernels as K
import test_gpu_random_kernels as R
from test_gpu_kernels import close, dev_bf16, rnd
from oracle import layers as L

pytestmark = pytest.mark.gpu

LAYOUT = {"nn": (0, 1), "nt": (0, 0), "tn": (1, 1)}
SIZES = [(128, 128, 64), (128, 256, 192), (256, 128, 320), (128, 384, 1088),  # 64x64, deep stages
         (1152, 1280, 128), (1152, 1280, 448),                                  # more than 256 of them
         (384, 128, 64)]


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("lay", LAYOUT)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_small_tiles(lay, m, n, k, tile):
    print(f"small tile {tile} {lay} {m}x{n}x{k}", flush=True)
    ta, tb = LAYOUT[lay]
    rng = np.random.default_rng(m + n + k + tile)
    a, b = rnd(rng, m, k), rnd(rng, n, k, scale=0.3)
    want = a.astype(np.float64) @ b.astype(np.float64).T
    a_h, b_h = (np.ascontiguousarray(x.T) if t else x for x, t in ((a, ta), (b, tb)))
    da, db = dev_bf16(a_h), dev_bf16(b_h)
    args = (da.ptr, db.ptr)
    dims = (m, n, k, a_h.shape[1], b_h.shape[1], n, ta, tb)
    if lay != "nt":
        prev = rng.standard_normal((m, n)).astype(np.float32)
        dc = rt.DeviceBuffer.from_numpy(prev)
        rt.gemm(*args, dc.ptr, *dims, rt.EPI_ACC_F32, tile=tile)
        rt.sync()
        close(dc.download(np.float32, (m, n)), prev + want, 1e-4 * math.sqrt(k), "accumulated")
    dc = rt.DeviceBuffer(2 * m * n)
    rt.gemm(*args, dc.ptr, *dims, rt.EPI_BF16, tile=tile)
    rt.sync()
    close(dc.download_bf16((m, n)), want, 1e-2, "bf16")


# (few tiles with two and with four stages; one K-step; more tiles than CUs)
@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (256, 384, 320), (384, 512, 704), (1152, 1280, 448)])
@pytest.mark.parametrize("ta,tb,epi", K.GEMM_CASES)
def test_every_epilogue_on_64x64_tiles(ta, tb, epi, m, n, k):
    K.test_gemm(ta, tb, epi, 5, m, n, k)


@pytest.mark.parametrize("m,f,k", [(128, 128, 64), (256, 640, 640), (1152, 640, 128)])
def test_swiglu_epilogues_on_64x64_tiles(m, f, k):
    K.test_gemm_swiglu_epilogues(5, m, f, k)


@pytest.mark.parametrize("seed", range(24))
def test_random_products_on_64x64_tiles(seed, monkeypatch):
    """The random products (padded leading dimensions, bias and residual or not, operand pairs) with
    tile 5 in the place of the tile drawn."""
    gemm = rt.gemm
    monkeypatch.setattr(rt, "gemm", lambda *a, **kw: gemm(*a, **{**kw, "tile": 5}))
    R.test_random_gemm(100 + seed)


@pytest.mark.parametrize("k", [64, 448])
def test_rotated_heads_of_128_on_small_tiles(k):
    """The rotated product is the plain one's bits rotated, whichever tile either takes."""
    batch, seq, heads, rot, d = 1, 128, 5, 3, 128
    rng = np.random.default_rng(k)
    m, n = batch * seq, heads * d
    da, dw = dev_bf16(rnd(rng, m, k)), dev_bf16(rnd(rng, k, n, scale=0.1))
    cos, sin = (rt.DeviceBuffer.from_numpy(t) for t in L.rope_tables(seq, d, 5e5, np.float32))
    plain, fused = rt.DeviceBuffer(2 * m * n), rt.DeviceBuffer(2 * m * n)
    rt.gemm(da.ptr, dw.ptr, plain.ptr, m, n, k, k, n, n, 0, 1)
    rt.check(rt.load().jpp_rope(None, plain.ptr, n, cos.ptr, sin.ptr, batch, seq, rot, d, 0))
    rt.gemm(da.ptr, dw.ptr, fused.ptr, m, n, k, k, n, n, 0, 1, rope=(cos.ptr, sin.ptr, rot * d, seq, d))
    rt.sync()
    np.testing.assert_array_equal(fused.download_bf16((m, n)), plain.download_bf16((m, n)))


@pytest.mark.parametrize("batch,heads,rot,k", [(1, 4, 2, 64), (2, 10, 7, 448), (9, 20, 20, 64)])
def test_rotated_heads_of_64_on_64x64_tiles(batch, heads, rot, k):
    """Tile 5 holds a head of 64 whole (odd tile columns and rows among them, more tiles than
    CUs); a rotated head of 128 is refused, tests/test_abi.py."""
    seq, d = 128, 64
    print(f"gemm+rope on 64x64 tiles, {batch} x {heads}/{rot} heads, k={k}", flush=True)
    rng = np.random.default_rng(batch + k)
    m, n = batch * seq, heads * d
    da, dw = dev_bf16(rnd(rng, m, k)), dev_bf16(rnd(rng, k, n, scale=0.1))
    cos, sin = (rt.DeviceBuffer.from_numpy(t) for t in L.rope_tables(seq, d, 5e5, np.float32))
    plain, fused = rt.DeviceBuffer(2 * m * n), rt.DeviceBuffer(2 * m * n)
    rt.gemm(da.ptr, dw.ptr, plain.ptr, m, n, k, k, n, n, 0, 1, tile=5)
    rt.check(rt.load().jpp_rope(None, plain.ptr, n, cos.ptr, sin.ptr, batch, seq, rot, d, 0))
    rt.gemm(da.ptr, dw.ptr, fused.ptr, m, n, k, k, n, n, 0, 1, tile=5, rope=(cos.ptr, sin.ptr, rot * d, seq, d))
    rt.sync()
    np.testing.assert_array_equal(fused.download_bf16((m, n)), plain.download_bf16((m, n)))


@pytest.mark.parametrize("parts,k,shapes", [
    (1, 64, [(128, 384), (128, 128), (128, 256), (256, 128)]),          # 28 tiles of 64x64
    (3, 192, [(384, 128), (128, 640)]),                                  # nine steps over three pairs
    (2, 128, [(768, 2304), (768, 768), (3072, 768)]),                    # more than 256 of 64x64
    (1, 128, [(1408, 1408), (1408, 2816), (2816, 1408), (640, 1408)])])  # 128x128
def test_small_weight_gradients_in_one_launch(parts, k, shapes):
    rng = np.random.default_rng(parts + k)
    probs, keep, wants = [], [], []
    for m, n in shapes:
        As = [rnd(rng, k, m) for _ in range(parts)]
        Bs = [rnd(rng, k, n, scale=0.3) for _ in range(parts)]
        prev = rng.standard_normal((m, n)).astype(np.float32)
        wants.append(prev + sum(a.astype(np.float64).T @ b.astype(np.float64) for a, b in zip(As, Bs)))
        dA, dB, dc = [dev_bf16(a) for a in As], [dev_bf16(b) for b in Bs], rt.DeviceBuffer.from_numpy(prev)
        keep.append((dA, dB, dc))
        probs.append(dict(a=dA[0].ptr, b=dB[0].ptr, c=dc.ptr, m=m, n=n, k=k, lda=m, ldb=n, ldc=n,
                          more=[(a.ptr, b.ptr) for a, b in zip(dA[1:], dB[1:])]))
    print(f"multi {parts} x {k} {shapes}", flush=True)
    rt.gemm_multi(probs)
    rt.sync()
    for (_, _, dc), want, shape in zip(keep, wants, shapes):
        close(dc.download(np.float32, shape), want, 1e-4 * math.sqrt(k * parts), f"multi {shape}")


@pytest.mark.parametrize("rows,cols", [(1, c) for c in range(1, 18)] + [(9, 5), (10, 5), (17, 3), (3, 19),
                                                                                 (32, 4), (128, 8)])
def test_every_tile_of_a_grid_is_computed_once(rows, cols):
    """Grids of every remainder by the 8 XCDs, fewer tiles than XCDs, groups of tile rows that do
    not come out even, tall ones (columns split over the XCDs), plain and as the second problem
    of a launch: C += A B with 0/1 operands is exact, and a tile left out or taken twice shows."""
    m, n, k = 128 * rows, 128 * cols, 64
    print(f"{rows} x {cols} tiles", flush=True)
    rng = np.random.default_rng(rows + cols)
    a, b = (rng.integers(0, 2, s).astype(np.float32) for s in ((k, m), (k, n)))
    c0 = rng.integers(0, 9, (m, n)).astype(np.float32)
    da, db, want = dev_bf16(a), dev_bf16(b), c0 + a.T @ b
    for tile in (1, 5):
        dc = rt.DeviceBuffer.from_numpy(c0)
        rt.gemm(da.ptr, db.ptr, dc.ptr, m, n, k, m, n, n, 1, 1, rt.EPI_ACC_F32, tile=tile)
        rt.sync()
        np.testing.assert_array_equal(dc.download(np.float32, (m, n)), want)
    first, dc = rt.DeviceBuffer.from_numpy(c0[:128, :128]), rt.DeviceBuffer.from_numpy(c0)
    rt.gemm_multi([dict(a=da.ptr, b=db.ptr, c=first.ptr, m=128, n=128, k=k, lda=m, ldb=n, ldc=128),
                   dict(a=da.ptr, b=db.ptr, c=dc.ptr, m=m, n=n, k=k, lda=m, ldb=n, ldc=n)])
    rt.sync()
    np.testing.assert_array_equal(dc.download(np.float32, (m, n)), want)
    np.testing.assert_array_equal(first.download(np.float32, (128, 128)), want[:128, :128])


@pytest.mark.parametrize("m,n", [(128, 128), (128, 256), (256, 128), (768, 384), (384, 768), (256, 512)])
def test_operand_pairs_of_every_extent(m, n):
    """A weight gradient over three operand pairs, tile left to the library, whichever of M and N
    are multiples of 256."""
    k, parts = 192, 3
    print(f"{parts} operand pairs {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + n)
    As, Bs = [rnd(rng, k, m) for _ in range(parts)], [rnd(rng, k, n, scale=0.3) for _ in range(parts)]
    prev = rng.standard_normal((m, n)).astype(np.float32)
    dA, dB, dc = [dev_bf16(a) for a in As], [dev_bf16(b) for b in Bs], rt.DeviceBuffer.from_numpy(prev)
    rt.gemm(dA[0].ptr, dB[0].ptr, dc.ptr, m, n, k, m, n, n, 1, 1, rt.EPI_ACC_F32,
            more=[(a.ptr, b.ptr) for a, b in zip(dA[1:], dB[1:])])
    rt.sync()
    want = prev + sum(a.astype(np.float64).T @ b.astype(np.float64) for a, b in zip(As, Bs))
    close(dc.download(np.float32, (m, n)), want, 1e-4 * math.sqrt(k * parts), "operand pairs")


@pytest.mark.parametrize("counts", [[70, 0, 256, 3], [300, 1, 64, 129]])
def test_small_grouped_products(counts):
    """Row-grouped and contraction-grouped products that state how many rows hold data: small
    ones leave the 256x256 tile."""
    print(f"small groups {counts}", flush=True)
    E, h, f = len(counts), 256, 512
    rng = np.random.default_rng(sum(counts))
    seg = np.concatenate([[0], np.cumsum([(c + 255) // 256 * 256 for c in counts])]).astype(np.int32)
    cap = int(seg[-1]) + 256
    x, dy = np.zeros((cap, h), np.float32), np.zeros((cap, f), np.float32)
    for e, c in enumerate(counts):
        x[seg[e]:seg[e] + c], dy[seg[e]:seg[e] + c] = rnd(rng, c, h), rnd(rng, c, f)
    w = rnd(rng, E * h, f, scale=0.1)
    b_seg = rt.DeviceBuffer.from_numpy(seg)
    b_rows = rt.DeviceBuffer.from_numpy(np.asarray(counts, np.int32))
    dx, ddy, dw, dc = dev_bf16(x), dev_bf16(dy), dev_bf16(w), rt.DeviceBuffer(2 * cap * f)
    dc.zero()
    rt.gemm(dx.ptr, dw.ptr, dc.ptr, cap, f, h, h, f, f, 0, 1, seg=b_seg.ptr, n_seg=E, group_mode=1,
            stride_b=h * f, group_rows=sum(counts), seg_rows=b_rows.ptr)
    acc = rng.standard_normal((E, h, f)).astype(np.float32)
    dacc = rt.DeviceBuffer.from_numpy(acc)
    rt.gemm(dx.ptr, ddy.ptr, dacc.ptr, h, f, 0, h, f, f, 1, 1, rt.EPI_ACC_F32, seg=b_seg.ptr, n_seg=E,
            group_mode=2, stride_c=h * f, group_rows=2 * sum(counts), seg_rows=b_rows.ptr,
            more=[(dx.ptr, ddy.ptr)], more_seg=[(b_seg.ptr, b_rows.ptr)])
    rt.sync()
    got = dc.download_bf16((cap, f))
    assert not got[seg[E]:].any(), "rows past the last group are not written"
    for e, c in enumerate(counts):
        rows = slice(seg[e], seg[e] + c)
        want = x[rows].astype(np.float64) @ w[e * h:(e + 1) * h].astype(np.float64)
        if c:
            close(got[rows], want, 1e-2, f"rows of group {e}")
        want = acc[e] + 2 * x[rows].astype(np.float64).T @ dy[rows].astype(np.float64)
        close(dacc.download(np.float32, (E, h, f))[e], want, 1e-4 * math.sqrt(2 * max(c, 1)), f"dW of group {e}")


@pytest.mark.parametrize("rows,form", [(448, ""), (512, "s4")])
def test_grouped_contraction_runs_in_the_form_that_was_priced(rows, form):
    """At most one 64x64 tile per CU takes the tile's four-stage form from 9 K-steps on - by the
    groups' rows (and one step more), not by k, which is unused - as the choice of the tile
    assumes."""
    E, h, f = 8, 256, 256
    print(f"grouped contraction of {rows} rows", flush=True)
    rng = np.random.default_rng(2)
    per = (rows + 255) // 256 * 256
    seg, cnt = np.arange(E + 1, dtype=np.int32) * per, np.full(E, rows, np.int32)
    x, dy = np.zeros((E * per, h), np.float32), np.zeros((E * per, f), np.float32)
    for e in range(E):
        x[seg[e]:seg[e] + rows], dy[seg[e]:seg[e] + rows] = rnd(rng, rows, h), rnd(rng, rows, f, scale=0.3)
    dx, ddy, b_seg, b_cnt = dev_bf16(x), dev_bf16(dy), rt.DeviceBuffer.from_numpy(seg), rt.DeviceBuffer.from_numpy(cnt)
    dacc = rt.DeviceBuffer(4 * E * h * f)
    dacc.zero()
    with rt.probe("*") as p:
        rt.gemm(dx.ptr, ddy.ptr, dacc.ptr, h, f, 0, h, f, f, 1, 1, rt.EPI_ACC_F32, stride_c=h * f, seg=b_seg.ptr,
                n_seg=E, group_mode=2, group_rows=E * rows, seg_rows=b_cnt.ptr)
        rt.sync()
    got = dacc.download(np.float32, (E, h, f))
    for e in range(E):
        r = slice(seg[e], seg[e] + rows)
        close(got[e], x[r].astype(np.float64).T @ dy[r], 1e-4 * math.sqrt(rows), f"gradient {e}")
    assert list(p.classes) == [f"gemm_tn_accf32_64x64{form}k2"], p.classes
