"""Gathers with contiguous destination rows (perm_rows): every split of a 128-bit chunk over source
rows, at any alignment, word for word."""
import numpy as np
import pytest

import linalg_hip as L
from helpers import rng
from linalg_hip import permutation as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,perm", [([9, 11, 1], [1, 0, 2]), ([7, 13, 2], [1, 0, 2]), ([13, 9, 3], [1, 0, 2]),
                                        ([10, 6, 4], [1, 0, 2]), ([5, 7, 5], [1, 0, 2]), ([31, 3, 67], [1, 0, 2]),
                                        ([5, 6, 7, 9], [2, 0, 1, 3]), ([4, 3, 5, 33], [1, 0, 2, 3]), ([257, 129], [0, 1])])
@pytest.mark.parametrize("dtype,pad,offset", [("f32", 0, 0), ("u32", 3, 1), ("c64", 1, 1), ("conj", 2, 0)])
def test_rows_word_for_word(ctx, pool, shape, perm, dtype, pad, offset):
    kind = "c64" if dtype == "conj" else dtype
    words = 2 if kind == "c64" else 1
    strides, st = [0] * len(shape), 1
    for d in range(len(shape) - 1, -1, -1):
        strides[d] = st
        st *= shape[d] + (pad if d == len(shape) - 1 else 0)
    span = offset + 1 + sum((e - 1) * s for e, s in zip(shape, strides))
    x = rng(sum(shape) + pad).integers(0, 2 ** 32, span * words, dtype=np.uint64).astype(np.uint32)
    src_buf = pool.alloc(kind, span)
    src_buf.write(x)
    src = P.permute_view(L.TensorView(src_buf, offset, shape, strides, kind), perm)
    count = int(np.prod(shape))
    dst_buf = pool.alloc(kind, count + offset + 4)
    dst_buf.write(np.full((count + offset + 4) * words, 0xA5A5A5A5, np.uint32))
    dst = L.TensorView.row_major(dst_buf, offset, src.shape, kind)
    (P.conjugate if dtype == "conj" else P.materialize)(ctx, src, dst)
    got = dst_buf.read(np.uint32, count=(count + offset + 4) * words).reshape(-1, words)
    idx = np.full(src.shape, src.offset, np.int64)
    for d, (n, s) in enumerate(zip(src.shape, src.strides)):
        idx = idx + (np.arange(n) * s).reshape([n if i == d else 1 for i in range(len(src.shape))])
    want = x.reshape(-1, words)[idx.ravel()].copy()
    if dtype == "conj":
        want[:, 1] ^= 0x80000000
    assert np.array_equal(got[offset:offset + count], want)
    assert np.all(got[:offset] == 0xA5A5A5A5) and np.all(got[offset + count:] == 0xA5A5A5A5)
