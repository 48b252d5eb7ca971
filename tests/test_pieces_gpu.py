"""The f32 GEMM on three bf16 pieces per element (gemm_f32_b3), at the edges of its tiles, slices and range.

Every product is compared with the exact one in f64 under the bound of an f32 dot product,
(K + 2) u sum |a||b| plus C's own rounding.
"""
import time

import numpy as np
import pytest

from linalg_hip import contraction as C
from helpers import Layout, Tensor, rng

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _product(ctx, pool, a, b, ta, tb, alpha=1.0, beta=0.0, c0=None, stride=1):
    """alpha * a @ b + beta * c0 through the library; `ta` / `tb` store an operand column-major,
    `stride` 2 leaves no unit stride in A."""
    m, k = a.shape
    n = b.shape[1]
    la = Layout.transposed(m, k) if ta else Layout.dense([m, k])
    stored = (a.T if ta else a).ravel()
    if stride == 2:
        la = Layout(0, [m, k], [2, 2 * m] if ta else [2 * k, 2])
        stored = np.repeat(stored, 2)[:-1]
    lb = Layout.transposed(k, n) if tb else Layout.dense([k, n])
    A = Tensor(pool, la, np.ascontiguousarray(stored))
    B = Tensor(pool, lb, np.ascontiguousarray((b.T if tb else b).ravel()))
    c = np.full((m, n), np.nan, np.float32) if c0 is None else c0.astype(np.float32)
    Cc = Tensor(pool, Layout.dense([m, n]), c.ravel().copy())
    C.gemm(ctx, alpha, A.view(), B.view(), beta, Cc.view())
    name = [x for x in ctx.launches() if x.startswith("gemm")][-1]
    return Cc.read()[: m * n].reshape(m, n).copy(), name


def _check(got, a, b, alpha, beta, c0):
    k = a.shape[1]
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = alpha * (a64 @ b64)
    bound = (k + 2) * U * abs(alpha) * (np.abs(a64) @ np.abs(b64)) + 1e-44
    if beta:
        want = want + beta * c0
        bound = bound + 2 * U * np.abs(beta * c0) + U * np.abs(want)
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))


@pytest.mark.parametrize("m,n,k,ta,tb,stride", [
    (2045, 1930, 77, False, False, 1),    # odd rows and pitches: 4-byte aligned 128-bit loads, K tail of 13
    (2045, 1929, 64, True, True, 1),      # A along M, B along K, the shortest K, one ragged column
    (1921, 2048, 65, True, False, 1),     # one row past a tile, K tail of 1
    (2048, 1923, 79, False, True, 1),     # three columns past a tile, K tail of 15
    (1924, 1924, 96, True, False, 1),     # whole quads past a tile
    (2048, 2048, 80, False, False, 1),    # full tiles, five slices
    (2048, 2048, 90, True, True, 2),      # no unit stride in A
    (1921, 1925, 67, False, False, 2),
    (3001, 2011, 77, False, True, 1),     # 384 tiles, odd rows: 128x128 all the same
    (130, 190, 20001, False, True, 1),     # 64x64 tiles split along K, the last chunk ragged
    (190, 130, 20011, True, False, 2),     # the same, strided, a wave with the chunk's short slice
    (1000, 1020, 1537, True, True, 1),    # 64x64 tiles, whole K, A along M
    (2300, 2304, 520, False, False, 1),   # 64x64 tiles of an uneven grid
    (2304, 2304, 256, True, True, 1),     # stream-K
])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-0.3, 0.75)])
def test_tile_edges(ctx, pool, m, n, k, ta, tb, stride, alpha, beta):
    g = rng(9100 + m + n + k)
    kernel = {130: "gemm_f32_b3kw", 190: "gemm_f32_b3kw", 1000: "gemm_f32_b3kw", 2300: "gemm_f32_b3kw",
              2304: "gemm_f32_b3sk"}.get(m, "gemm_f32_b3<")
    a = g.standard_normal((m, k)).astype(np.float32)
    b = g.standard_normal((k, n)).astype(np.float32)
    c0 = g.standard_normal((m, n)).astype(np.float32) if beta else None
    alpha = float(np.float32(alpha))
    got, name = _product(ctx, pool, a, b, ta, tb, alpha, beta, c0, stride)
    assert name.startswith(kernel), name
    _check(got, a, b, alpha, beta, c0)


@pytest.mark.parametrize("m,n,k,ta,tb,kernel", [
    (2048, 2048, 72, False, True, "gemm_f32_dl"),     # both along K, a tail of 8
    (2048, 2048, 84, False, True, "gemm_f32_b3<"),    # tails of 4, 8 and 12
    (2048, 2048, 88, False, True, "gemm_f32_b3<"),
    (2048, 2048, 92, False, True, "gemm_f32_b3<"),
    (2048, 2048, 72, False, False, "gemm_f32_b3<"),   # A along K alone
    (4096, 4096, 65, True, False, "gemm_f32_b3"),     # neither along K: tails of 1 and 15
    (4096, 4096, 79, True, False, "gemm_f32_b3"),
    (128, 262144, 64, False, False, "gemm_f32_pl"),   # one row of tiles, an output of 128 MB
    (128, 262144, 88, False, False, "gemm_f32_dl"),
    (128, 262144, 96, False, False, "gemm_f32_b3"),
    (128, 262144, 136, False, True, "gemm_f32_dl"),
    (256, 131072, 64, False, False, "gemm_f32_b3_256x256"),
    (128, 131072, 64, False, False, "gemm_f32_b3<"),  # and of 64 MB
])
def test_short_sums(ctx, pool, m, n, k, ta, tb, kernel):
    """Sums of a few slices on the kernel that is the faster one for them, their last slice partly filled."""
    g = rng(9300 + m + n + k)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    got, name = _product(ctx, pool, a, b, ta, tb)
    assert name.startswith(kernel), name
    columns = slice(n % 7, None, max(1, n // 4099))
    _check(got[:, columns], a, b[:, columns], 1.0, 0.0, None)


@pytest.mark.parametrize("dense", ["a", "b"])
def test_pieces_hold_the_element_whole(ctx, pool, dense):
    """A times a permutation matrix is A's columns, bit for bit, and a permutation matrix times B is B's rows, from f32's
    least subnormals to 2^103."""
    n = 2048
    g = rng(9200)
    x = np.ldexp(g.uniform(1, 2, (n, n)), g.integers(-149, 103, (n, n))).astype(np.float32)
    x *= g.choice([-1, 1], (n, n)).astype(np.float32)
    perm = g.permutation(n)
    one = np.zeros((n, n), np.float32)
    one[perm, np.arange(n)] = 1.0
    got, name = _product(ctx, pool, *((x, one) if dense == "a" else (one.T.copy(), x)), False, False)
    assert name.startswith("gemm_f32_b3"), name
    assert np.array_equal(got, x[:, perm] if dense == "a" else x[perm])


@pytest.mark.parametrize("shape", [(2045, 1930, 77), (1000, 1020, 1537), (2304, 2304, 256)])
@pytest.mark.parametrize("what", ["inf", "nan", "huge", "tiny", "subnormal", "zero"])
def test_elements_outside_the_pieces(ctx, pool, what, shape):
    """Infinities, NaNs, elements past bf16's largest and below what three pieces hold: the
    products of f32 arithmetic, wherever in K and in the tile they stand."""
    m, n, k = shape
    g = rng(9300)
    a = g.standard_normal((m, k)).astype(np.float32)
    b = g.standard_normal((k, n)).astype(np.float32)
    if what in ("inf", "nan"):
        v = np.float32(np.inf if what == "inf" else np.nan)
        a[5, k - 1], a[700, 0], a[m - 1, 30], b[40, n - 1] = v, -v, v, v
    elif what == "huge":
        a[5, k - 1] = a[m - 1, 3] = np.finfo(np.float32).max
        b *= np.float32(2.0 ** -10)
    elif what == "tiny":
        a *= np.float32(2.0 ** -115)
        b *= np.float32(2.0 ** 60)
    elif what == "subnormal":
        a[700] = (g.integers(1, 1 << 20, k) * 2.0 ** -149).astype(np.float32)
        b *= np.float32(2.0 ** 100)
        a[:700] = 0
        a[701:] = 0
    else:
        a[:] = 0
    got, name = _product(ctx, pool, a, b, m == 1000, False)
    assert name.startswith("gemm_f32_b3"), name
    with np.errstate(invalid="ignore", over="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        fine = np.isfinite(want)
        assert np.array_equal(np.isnan(want), np.isnan(got))
        assert np.array_equal(want[~fine & ~np.isnan(want)], got[~fine & ~np.isnan(want)])
        bound = (k + 2) * U * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)))
    assert np.all(np.abs(got[fine] - want[fine]) <= bound[fine] + 1e-44)


@pytest.mark.parametrize("shape", [(2045, 1930, 77), (1000, 1020, 1537), (2304, 2304, 256)])
@pytest.mark.parametrize("exponent", [-58, -64, -70, -74])
def test_products_below_the_normal_range(ctx, pool, shape, exponent):
    """Products of the later pieces, or all of them, are subnormal in f32: each of the up to 6 K sums
    may lose half of a least subnormal, and no more."""
    m, n, k = shape
    g = rng(9400)
    a = np.ldexp(g.standard_normal((m, k)), exponent).astype(np.float32)
    b = np.ldexp(g.standard_normal((k, n)), exponent).astype(np.float32)
    got, name = _product(ctx, pool, a, b, m == 1000, False)
    assert name.startswith("gemm_f32_b3"), name
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (k + 2) * U * (np.abs(a64) @ np.abs(b64)) + 6 * k * 2.0 ** -149
    assert np.all(np.abs(got - a64 @ b64) <= bound), float(np.max(np.abs(got - a64 @ b64) / bound))


# Every kernel of three pieces: its shape, and whether A is stored along M.
KERNELS = {"gemm_f32_b3_256x256": (4096, 4096, 64, False), "gemm_f32_b3_256x128": (4096, 2048, 64, False),
           "gemm_f32_b3<": (2045, 1930, 77, False), "gemm_f32_b3kw": (1000, 1020, 1537, True),
           "gemm_f32_b3sk": (2304, 2304, 256, False)}


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("where,bits", [("a", 1), ("a", 0x7fff), ("a", 0x8000), ("a", 0x8001), ("b", 1),
                                        ("b", 0x8000), ("alpha", 0x8000)])
def test_least_subnormals(ctx, pool, kernel, where, bits):
    """Operands of zeros and elements of at most `bits` least subnormals (2^-149), which bf16 rounds to
    zero up to 0x8000 of them, stored so or made by alpha: every product counts."""
    m, n, k, ta = KERNELS[kernel]
    g = rng(9500 + bits)
    small = lambda *s: np.ldexp(g.integers(-bits, bits + 1, s).astype(np.float64), -149).astype(np.float32)
    large = lambda *s: np.ldexp(g.standard_normal(s), 100).astype(np.float32)
    a, b = (large(m, k), small(k, n)) if where == "b" else (small(m, k), large(k, n))
    alpha = 1.0
    if where == "alpha":
        a, alpha = np.ldexp(a, 40), 2.0 ** -40
    got, name = _product(ctx, pool, a, b, ta, False, alpha)
    assert name.startswith(kernel), name
    _check(got, a, b, alpha, 0.0, None)


@pytest.mark.parametrize("shape,kernel", [((4096, 4096, 4096), "gemm_f32_b3_256x256"), ((3001, 2011, 1537), "gemm_f32_b3<"),
                                          ((2304, 2304, 2304), "gemm_f32_b3sk")])
@pytest.mark.parametrize("value,every,limit", [(1e-35, 16, 2.0), (np.inf, 64, 3.5)])
def test_time_with_elements_at_the_ends_of_the_range(ctx, pool, shape, kernel, value, every, limit):
    """One tiny element in every sixteenth row of A costs nothing and an infinity in every 64th, half of all rows
    of blocks, about one more pass: twice the time was measured, six to eleven times where whole tiles are computed again
    with nothing in flight."""
    m, n, k = shape
    g = rng(9600)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    B, Cc = Tensor(pool, Layout.dense([k, n]), b.ravel()), Tensor(pool, Layout.dense([m, n]), np.zeros(m * n, np.float32))
    times = []
    for special in (False, True):
        if special:
            a[::every, 7] = value
        A = Tensor(pool, Layout.dense([m, k]), a.ravel())
        best = np.inf
        for _ in range(12):
            t = time.perf_counter()
            C.gemm(ctx, 1.0, A.view(), B.view(), 0.0, Cc.view())
            best = min(best, time.perf_counter() - t)
        times.append(best)
        assert ctx.launches()[-1].startswith(kernel)
    assert times[1] < limit * times[0], times


@pytest.mark.parametrize("m,n,k,kernel", [(2048, 2048, 65536, "gemm_f32_b3<"), (2304, 2304, 65536, "gemm_f32_b3sk"),
                                          (3001, 2011, 16401, "gemm_f32_b3<"), (4096, 4096, 16384, "gemm_f32_b3_256x256")])
@pytest.mark.parametrize("what", ["normal", "positive"])
def test_long_sums_are_not_biased(ctx, pool, m, n, k, kernel, what):
    """Sums over a long K on unsplit tiles, of either sign or of one: no further from the exact ones than an f32
    chain's (1.8e-8 sqrt(K) of their norm), and neither high nor low. Rounding down throughout leaves a mean
    error of 3e-6 of the mean magnitude at K = 65536 (normal) and 4e-7 at 16384 (uniform)."""
    g = rng(9700 + k)
    draw = g.standard_normal if what == "normal" else g.random
    a, b = draw((m, k), dtype=np.float32), draw((k, n), dtype=np.float32)
    got, name = _product(ctx, pool, a, b, False, k == 16401)
    assert name.startswith(kernel), name
    rows = g.integers(0, m, 64)
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    err = got[rows] - want
    assert np.linalg.norm(err) <= 1.8e-8 * np.sqrt(k) * np.linalg.norm(want)
    # The mean over 64 n outputs of errors that are independent of each other strays by 2e-8 of the magnitude at
    # the most (an rms error of 1.4 1.8e-8 sqrt(K), over sqrt(64 n)); a turn's own share is 5e-8.
    assert abs(err.mean()) <= 1.2e-7 * np.abs(want).mean(), err.mean() / np.abs(want).mean()


@pytest.mark.parametrize("kernel", KERNELS)
def test_single_products(ctx, pool, kernel):
    """Rows of one element each, so that every output is one product of two full mantissas: the six products of pieces
    that are formed leave out 2^-24 of it at the most, the last addition cuts up to 2^-23 (or rounds), and
    the five before it are below 2^-7 of it and err by 2^-28 in all. Without any one of the six the worst output is 2^-17 off or more."""
    m, n, k, ta = KERNELS[kernel]
    g = rng(9900 + m)
    a, b = np.zeros((m, k), np.float32), g.uniform(1, 2, (k, n)).astype(np.float32)
    a[np.arange(m), np.arange(m) % k] = g.uniform(-2, 2, m)
    got, name = _product(ctx, pool, a, b, ta, False)
    assert name.startswith(kernel), name
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.max(np.abs(got - want) / np.abs(want)) <= 1.6 * 2.0 ** -23


@pytest.mark.parametrize("kernel", KERNELS)
def test_error_in_norm(ctx, pool, kernel):
    """Normal operands: the error's norm over the result's is an f32 chain's, 1.8e-8 sqrt(K), or less (measured: 1.1e-7 at
    K = 64, 3.5e-7 at 1537). Any five of the six products would leave 2.4e-6 or more at K = 64."""
    m, n, k, ta = KERNELS[kernel]
    g = rng(9950 + m)
    a, b = g.standard_normal((m, k)).astype(np.float32), g.standard_normal((k, n)).astype(np.float32)
    got, name = _product(ctx, pool, a, b, ta, False)
    assert name.startswith(kernel), name
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(got - want) <= 1.8e-8 * np.sqrt(k) * np.linalg.norm(want)
