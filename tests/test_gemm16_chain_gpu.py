"""The 16-bit Backend gemm on the f32 matrix cores (gemm16_chain): CpuBackend's bits at the
edges of its tiles and slices and of the range in which its products need no rounding."""
import time

import numpy as np
import pytest

import oracle
from helpers import rng
from test_backend_gpu import run16, same16, hb, up16  # noqa: F401  (hb: the backend fixture)

pytestmark = pytest.mark.gpu


def _bits(kind, x):
    x = np.ascontiguousarray(x, dtype=np.float32)
    return oracle.f32_to_f16(x) if kind == "f16" else oracle.f32_to_bf16(x)


def _check(hb, kind, layout, a, b, c, m, k, n, alpha, beta, kernel):
    """Bits against the oracle's, and the kernel that ran: a name, or the tile of the chain on the matrix cores."""
    a16, b16, c16 = _bits(kind, a.ravel()), _bits(kind, b.ravel()), _bits(kind, c.ravel())
    got = run16(hb, kind, layout, a16, b16, c16, m, k, n, alpha, beta)
    name = hb.debug_launches()[-1]
    assert name == (kernel if isinstance(kernel, str) else f"gemm_{kind}_chain{kernel}"), name
    want = oracle.gemm_seq_16(kind, alpha, beta, a16.reshape(m, k), b16.reshape(k, n), c16.reshape(m, n))
    assert same16(kind, got, want)


# 128x128 tiles (529 of them, ragged), 64x64 (552) and 32x32, with K around their slices of 16, 32
# and 64; rows along K are read 128 bits at a time whatever their alignment.
@pytest.mark.parametrize("m,k,n", [(2900, 16, 2820), (2817, 17, 2944), (2823, 40, 2900), (1500, 32, 1450),
                                   (1409, 33, 1473), (1481, 104, 1472), (70, 64, 45), (33, 65, 97),
                                   (31, 1, 32), (64, 136, 64), (1, 191, 700)])
@pytest.mark.parametrize("kind,layout", [("f16", "at"), ("f16", "bt"), ("bf16", "plain"), ("bf16", "bt")])
def test_tile_and_slice_edges(hb, kind, layout, m, k, n):
    g = rng(8800 + m + k + n)
    alpha, beta = [(1.0, 0.0), (-0.75, 0.3)][(m + k) % 2]
    _check(hb, kind, layout, g.standard_normal((m, k)), g.standard_normal((k, n)),
           g.standard_normal((m, n)), m, k, n, alpha, beta, 128 if m > 2000 else 64 if m > 1400 else 32)


@pytest.mark.parametrize("kind", ["f16", "bf16"])
def test_negative_zero_sums_survive_the_padding(hb, kind):
    m, k, n = 40, 19, 36
    a, b, c = -np.zeros((m, k), np.float32), np.ones((k, n), np.float32), -np.zeros((m, n), np.float32)
    _check(hb, kind, "plain", a, b, c, m, k, n, 1.0, 1.0, 32)


@pytest.mark.parametrize("alpha", [1.0, 2.0 ** -10, 1.9921875, 0.3])
@pytest.mark.parametrize("low,high", [(-126, -60), (-70, 70), (60, 127), (-56, -54), (61, 63)])
def test_bf16_exponents_whose_products_round(hb, alpha, low, high):
    """Products that underflow, overflow or lose bits keep their own rounding, a factor 2^(low..high)
    on either side, in one tile of several and in a last slice that is not full."""
    m, k, n = 70, 75, 100
    g = rng(8900 + low + high)
    a, b = g.standard_normal((m, k)), g.standard_normal((k, n))
    at = (g.integers(0, m, 40), g.integers(0, k, 40))
    a[at] = np.ldexp(a[at], g.integers(low, high + 1, 40))
    a[5] = np.ldexp(a[5], g.integers(low, high + 1, k))
    bt = (g.integers(0, k, 40), g.integers(0, n, 40))
    b[bt] = np.ldexp(b[bt], g.integers(low, high + 1, 40))
    with np.errstate(over="ignore"):
        _check(hb, "bf16", "bt", a, b, g.standard_normal((m, n)), m, k, n, alpha, 0.5,
               "gemm_bf16_seq" if alpha == 0.3 else 32)


@pytest.mark.parametrize("m,k,n", [(70, 330, 100), (1500, 167, 1450), (2900, 83, 2820)])
@pytest.mark.parametrize("layout", ["bt", "at"])
def test_bf16_slices_whose_products_round(hb, m, k, n, layout):
    """32x32, 64x64 and 128x128 tiles with such slices alone, in runs, first and last, among slices
    whose products need no rounding: either way of a slice continues the other's sums."""
    g = rng(8950 + m)
    a, b = g.standard_normal((m, k)), g.standard_normal((k, n))
    for k0, k1 in ((0, 1), (k // 3, k // 3 + 1), (k // 2, 3 * k // 4), (k - 1, k)):
        rows = g.integers(0, m, m // 8 + 1)
        a[rows, k0:k1] = np.ldexp(a[rows, k0:k1], -140)
        b[k0:k1, g.integers(0, n, 9)] *= 2.0 ** -60
    a[3] = np.ldexp(a[3], -100)  # sums of products below the normal range alone
    b[:, 5] = np.ldexp(b[:, 5], -40)
    _check(hb, "bf16", layout, a, b, g.standard_normal((m, n)), m, k, n, 0.75, 0.0, {70: 32, 1500: 64, 2900: 128}[m])


@pytest.mark.parametrize("m,k,n", [(2048, 1024, 4096), (1501, 1023, 1477)])
def test_time_with_bf16_elements_whose_products_round(hb, m, k, n):
    """One element of 1e-20 costs next to nothing (1.0 of the time without was measured), one in every slice
    of every tile the VALU's rate (2.2 to 2.4; whole tiles computed again took 4.5 times in both)."""
    g = rng(8960)
    a = np.ascontiguousarray(g.standard_normal((m, k), dtype=np.float32))
    b = up16(hb, "bf16", oracle.f32_to_bf16(g.standard_normal(k * n, dtype=np.float32)), (k, n))
    c = up16(hb, "bf16", np.zeros(m * n, np.uint16), (m, n))
    times = []
    for what in ("none", "one", "all"):
        if what == "one":
            a[m // 2, k // 2] = 1e-20
        elif what == "all":
            a[::16] = 1e-20
        t16 = up16(hb, "bf16", oracle.f32_to_bf16(a.ravel()), (m, k))
        hb.gemm(t16, b, c, 1.0, 0.0)
        hb.sync()
        best = np.inf
        for _ in range(12):
            t = time.perf_counter()
            for _ in range(4):
                hb.gemm(t16, b, c, 1.0, 0.0)
            hb.sync()
            best = min(best, time.perf_counter() - t)
        times.append(best)
    assert times[1] < 1.6 * times[0] and times[2] < 3.2 * times[0], times
