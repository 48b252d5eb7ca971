"""Row pitches of 2^20 elements and K strides of 2^23, where operand tiles outgrow the three-piece kernels' 32-bit
byte offsets and the kernels on the f32 instruction take over: either side of the line, the kernel that ran and every
output against the exact products."""
import numpy as np
import pytest

import linalg_hip as L
from helpers import rng
from linalg_hip import contraction as C

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
PITCH, KSTRIDE = 2 ** 20, 2 ** 23


@pytest.fixture(scope="module")
def big(ctx):
    buf = L.alloc_shared(ctx, "f32", 4200 * (PITCH + 64))  # 16 GiB of 288
    yield buf
    buf.free()


# wide: the operand and axis with the wide stride. past/below: the kernel at the line and just under it.
@pytest.mark.parametrize("m,n,k,wide,past,below", [
    (4096, 4096, 64, "a", "gemm_f32_pl2x<K,MN>", "gemm_f32_b3_256x256<K,MN>"),
    (4096, 2048, 64, "a", "gemm_f32_pl256<K,MN>", "gemm_f32_b3_256x128<K,MN>"),
    (4096, 2048, 64, "b", "gemm_f32_pl<MN,K>", "gemm_f32_b3<MN,K>"),
    (4096, 2048, 64, "ak", "gemm_f32_pl<MN,MN>", "gemm_f32_b3<MN,MN>"),
    (2048, 2048, 256, "a", "gemm_f32_pl32<K,MN>", "gemm_f32_b3<K,MN>"),
    (2304, 2304, 256, "a", "gemm_f32_sk<K,MN>", "gemm_f32_b3sk<K,MN>"),
    (4100, 4100, 72, "a", "gemm_f32_dl<K,MN>", "gemm_f32_b3_128x256<K,MN>"),
    (2040, 1932, 300, "a", "gemm_f32_dl<K,MN>", "gemm_f32_b3<K,MN>"),
    (2045, 1931, 77, "a", "gemm_f32_mfma<K,S>", "gemm_f32_b3<K,MN>"),
    (1000, 1020, 1537, "a", "gemm_f32_mfma<S,MN>", "gemm_f32_b3kw<K,MN>"),
])
@pytest.mark.parametrize("side", ["past", "below"])
def test_either_side_of_the_32_bit_line(ctx, pool, big, m, n, k, wide, past, below, side):
    g = rng(9800 + m + n + k)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    at, st = (KSTRIDE, k) if wide == "ak" else (PITCH, n if wide == "b" else m)
    at -= 4 if side == "below" else 0
    if m == 1000:
        at += 1  # no row aligned either
    for i, row in enumerate({"a": a, "b": b.T, "ak": a.T}[wide][:st]):
        big.write(np.ascontiguousarray(row), byte_offset=4 * i * at)

    def dense(x):
        buf = pool.alloc("f32", x.size)
        buf.write(np.ascontiguousarray(x).ravel())
        return buf
    if wide == "a":
        av, bv = L.TensorView(big, 0, [m, k], [at, 1]), L.TensorView(dense(b), 0, [k, n], [n, 1])
    elif wide == "b":
        av, bv = L.TensorView(dense(a.T), 0, [m, k], [1, m]), L.TensorView(big, 0, [k, n], [1, at])
    else:
        av, bv = L.TensorView(big, 0, [m, k], [1, at]), L.TensorView(dense(b), 0, [k, n], [n, 1])
    cbuf = dense(np.full((m, n), np.nan, np.float32))
    C.gemm(ctx, 1.0, av, bv, 0.0, L.TensorView.row_major(cbuf, 0, [m, n]))
    name = [x for x in ctx.launches() if x.startswith("gemm")][-1]
    assert name == (past if side == "past" else below), name
    got = cbuf.read(np.float32, count=m * n).reshape(m, n)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (k + 2) * U * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)
