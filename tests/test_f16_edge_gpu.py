"""The f16 contraction's edge kernel (gemm_f16_edge) around its tiles, slices and alignments.

On halves of a 2^-10 grid every sum is exact in f64, so each output is the exact value rounded
once, which numpy's float64 -> float16 conversion gives."""
import numpy as np
import pytest

from helpers import Layout, rng
from linalg_hip import contraction as C
from test_contraction_f16_gpu import Half, f16_bits_equal, grid_halves

pytestmark = pytest.mark.gpu


# 32x32 tiles: one short of, at and past a tile and a slice; 64x64: K under one slice, or 552
# ragged tiles; stride 2 leaves no unit stride, offset 1 no alignment.
@pytest.mark.parametrize("m,n,k", [(32, 32, 64), (31, 33, 65), (65, 97, 127), (1, 700, 191), (247, 130, 128),
                                   (70, 66, 63), (33, 40, 17), (1450, 1473, 64), (1409, 1475, 71)])
@pytest.mark.parametrize("at,bt,stride,offset", [(False, False, 1, 0), (True, True, 1, 1), (False, True, 1, 1),
                                                 (True, False, 2, 0)])
def test_edges_round_once(ctx, pool, m, n, k, at, bt, stride, offset):
    if stride == 2 and m > 1000:
        pytest.skip("covered by the smaller shapes")
    g = rng(8700 + m + n + k)
    alpha, beta = [(1.0, 0.0), (0.5, -0.25)][(m + k) % 2]
    pick = lambda t, r, c, s, o: Layout(o, [r, c], [s, r * s] if t else [c * s, s])
    la, lb = pick(at, m, k, stride, offset), pick(bt, k, n, 1, offset)
    a, b = Half(pool, la, grid_halves(g, la.span())), Half(pool, lb, grid_halves(g, lb.span()))
    c0 = grid_halves(g, m * n) if beta else np.full(m * n, np.nan, np.float16)
    c = Half(pool, Layout.dense([m, n]), c0)
    C.gemm(ctx, alpha, a.view(), b.view(), beta, c.view())
    # Less than a slice of K: only operands that both lie along it.
    edge = k >= 64 or (not at and bt)
    assert ctx.launches()[-1].startswith("gemm_f16_edge" if edge else "gemm_f16_f64mfma")
    want = alpha * (a.logical().astype(np.float64) @ b.logical().astype(np.float64))
    if beta:
        want = want + beta * c0.reshape(m, n).astype(np.float64)
    assert f16_bits_equal(c.read()[: m * n].reshape(m, n), want.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,edge", [(72, 1528, ()), (1000, 1001, ()), (2001, 1999, ((False, False), (True, True))),
                                      (2000, 2000, ())])
def test_short_k_keeps_the_tile_kernel(ctx, pool, m, n, edge, at, bt):
    """K of half a slice: the edge kernel where both operands lie along K, or one on a large grid of unaligned
    rows; elsewhere its predicated element loads took up to 28 % longer than the tile kernel."""
    k = 31
    g = rng(8750 + m)
    la = Layout(0, [m, k], [1, m] if at else [k, 1])
    lb = Layout(0, [k, n], [1, k] if bt else [n, 1])
    a, b = Half(pool, la, grid_halves(g, la.span())), Half(pool, lb, grid_halves(g, lb.span()))
    c = Half(pool, Layout.dense([m, n]), np.full(m * n, np.nan, np.float16))
    C.gemm(ctx, 1.0, a.view(), b.view(), 0.0, c.view())
    along_k = not at and bt
    assert ctx.launches()[-1] == ("gemm_f16_edge" if along_k or (at, bt) in edge else "gemm_f16_f64mfma")
    want = a.logical().astype(np.float64) @ b.logical().astype(np.float64)
    assert f16_bits_equal(c.read()[: m * n].reshape(m, n), want.astype(np.float16).view(np.uint16))
