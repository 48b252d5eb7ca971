// gfx950 permutation kernels: the tiled transpose (permutation_tile.h) instantiated at the
// library's tile geometry, and the gather copy.
//
// perm_copy: the destination is contiguous, so each thread produces 128 bits of it: a straight
// 128-bit copy of a fully contiguous source, else a strided gather (odometer over the source strides;
// perm_rows for the ranks and sizes that occur, perm_copy for the rest).
#include <hip/hip_runtime.h>

#include "lg_internal.h"
#include "permutation_tile.h"

namespace lg {
namespace {

using perm_detail::perm_tile;
using perm_detail::SIGN;
using perm_detail::u32x4;

template <int W, bool CONJ, bool NT>
__global__ __launch_bounds__(PERM_THREADS) void perm_copy(PermCopyArgs p) {
    constexpr int VE = 4 / W;
    const uint32_t* src = static_cast<const uint32_t*>(p.src);
    uint32_t* dst = static_cast<uint32_t*>(p.dst);
    const uint64_t step = static_cast<uint64_t>(gridDim.x) * PERM_THREADS * VE;
    const int rank = static_cast<int>(p.rank);
    for (uint64_t i0 = (static_cast<uint64_t>(blockIdx.x) * PERM_THREADS + threadIdx.x) * VE;
         i0 < p.count; i0 += step) {
        const bool full = i0 + VE <= p.count;
        u32x4 v;
        if (p.contiguous) {
            const uint64_t s0 = p.src_offset + i0;
            if (full) {
                v = perm_detail::load128<NT>(src + s0 * W);
            } else {
                for (int e = 0; e < VE; ++e)
                    if (i0 + e < p.count)
                        for (int w = 0; w < W; ++w) v[e * W + w] = src[(s0 + e) * W + w];
            }
        } else {
            // Decode i0 into a multi-index, then step the odometer VE times.
            uint64_t idx[PERM_MAX_RANK];
            uint64_t r = i0;
            int64_t soff = static_cast<int64_t>(p.src_offset);
            for (int d = rank - 1; d >= 0; --d) {
                const uint64_t q = r / p.shape[d];
                idx[d] = r - q * p.shape[d];
                soff += static_cast<int64_t>(idx[d]) * p.strides[d];
                r = q;
            }
            for (int e = 0; e < VE; ++e) {
                if (i0 + e >= p.count) break;
                for (int w = 0; w < W; ++w) v[e * W + w] = src[soff * W + w];
                for (int d = rank - 1; d >= 0; --d) {
                    soff += p.strides[d];
                    if (++idx[d] < p.shape[d]) break;
                    soff -= static_cast<int64_t>(p.shape[d]) * p.strides[d];
                    idx[d] = 0;
                }
            }
        }
        if constexpr (CONJ) {
            for (int e = 0; e < VE; ++e) v[e * W + 1] ^= SIGN;
        }
        const uint64_t d0 = p.dst_offset + i0;
        if (full && p.vec_dst) {
            perm_detail::store128<NT>(dst + d0 * W, v);
        } else {
            for (int e = 0; e < VE; ++e)
                if (i0 + e < p.count)
                    for (int w = 0; w < W; ++w) dst[(d0 + e) * W + w] = v[e * W + w];
        }
    }
}

// perm_copy of a gather whose rank after merging is 2 to 4 and whose elements number less than 2^32: the
// index is decoded with 32-bit divisions into registers (perm_copy's 64-bit ones, over a rank it learns at run time,
// bound it: 3.3 TB/s), and four neighbours of the source row, at any alignment, are one 128-bit load
// where they lie in one row. Bound: HBM where rows are long. us, before -> after: [116,108,60,136] by 0,2,1,3
// 249 -> 139 (5.9 TB/s), [64,128,2048] by 1,0,2 34 -> 21, [301,501,67] by 1,0,2 29 -> 19, [1000,1000,5] 42 -> 26.
template <int W, bool CONJ, int RANK>
__global__ __launch_bounds__(PERM_THREADS) void perm_rows(PermCopyArgs p) {
    constexpr uint32_t VE = 4 / W;
    const uint32_t* src = static_cast<const uint32_t*>(p.src);
    uint32_t* dst = static_cast<uint32_t*>(p.dst) + p.dst_offset * W;
    const uint32_t count = static_cast<uint32_t>(p.count);
    uint32_t shape[RANK];
#pragma unroll
    for (int d = 0; d < RANK; ++d) shape[d] = static_cast<uint32_t>(p.shape[d]);
    for (uint64_t at = (static_cast<uint64_t>(blockIdx.x) * PERM_THREADS + threadIdx.x) * VE; at < count;
         at += static_cast<uint64_t>(gridDim.x) * PERM_THREADS * VE) {
        const uint32_t i0 = static_cast<uint32_t>(at);
        uint32_t idx[RANK], r = i0;
        int64_t soff = static_cast<int64_t>(p.src_offset);
#pragma unroll
        for (int d = RANK - 1; d > 0; --d) {
            const uint32_t q = r / shape[d];
            idx[d] = r - q * shape[d];
            soff += idx[d] * p.strides[d];
            r = q;
        }
        idx[0] = r;
        soff += r * p.strides[0];
        const bool full = at + VE <= count;
        u32x4 v = {0, 0, 0, 0};
        if (p.strides[RANK - 1] == 1 && idx[RANK - 1] + VE <= shape[RANK - 1]) {
            v = perm_detail::load128u<false>(src + soff * W);
        } else {
#pragma unroll
            for (uint32_t e = 0; e < VE; ++e) {
                if (at + e < count) {
#pragma unroll
                    for (int w = 0; w < W; ++w) v[e * W + w] = src[soff * W + w];
                }
                // The next element: a carry runs up through the axes that end here.
                bool carry = true;
#pragma unroll
                for (int d = RANK - 1; d >= 0; --d) {
                    if (carry) {
                        soff += p.strides[d];
                        carry = ++idx[d] == shape[d];
                        if (carry) {
                            soff -= static_cast<int64_t>(shape[d]) * p.strides[d];
                            idx[d] = 0;
                        }
                    }
                }
            }
        }
        if constexpr (CONJ) {
#pragma unroll
            for (uint32_t e = 0; e < VE; ++e) v[e * W + 1] ^= SIGN;
        }
        uint32_t* q = dst + at * W;
        if (full) {
            perm_detail::store128u<false>(q, v);
        } else {
#pragma unroll
            for (uint32_t e = 0; e < VE; ++e)
                if (at + e < count)
                    for (int w = 0; w < W; ++w) q[e * W + w] = v[e * W + w];
        }
    }
}

constexpr uint64_t TILE_GRID_CAP = 1u << 22;
constexpr uint64_t COPY_GRID_CAP = 1u << 20;

// Streaming (operands beyond the Infinity Cache) tiles are 64 x 256 with 1024 threads, cached
// ones 64 x 64 with 512: measured best on configs 2b and 2a respectively (2b: 6.14 TB/s against
// 6.0 for 128 x 64 tiles of 256 threads, whose destination row segments are 256 B; the 1 GiB
// tensor [1024,1024,256] 5.89 against 5.62. 2a: 6.44 against 6.21 with 256 threads).
template <int W, bool CONJ, bool VEC, int TA, bool NT>
void tile_t(hipStream_t s, const PermTileArgs& a) {
    constexpr int threads = NT ? PERM_STREAM_THREADS : PERM_CACHED_THREADS;
    constexpr int TB = NT ? PERM_STREAM_TILE_B : PERM_TILE_B;
    const uint64_t g = perm_tile_workgroups(a.total_tiles);
    hipLaunchKernelGGL((perm_tile<W, CONJ, VEC, TA, TB, NT ? 3 : 0, threads>),
                       dim3(static_cast<uint32_t>(g)), dim3(threads), 0, s, a);
}

template <int W, bool CONJ, bool NT>
void copy_t(hipStream_t s, const PermCopyArgs& a) {
    const dim3 grid(static_cast<uint32_t>(perm_copy_workgroups(a.count, W)));
    hipLaunchKernelGGL((perm_copy<W, CONJ, NT>), grid, dim3(PERM_THREADS), 0, s, a);
}

template <int W, bool CONJ>
void rows_t(hipStream_t s, const PermCopyArgs& a) {
    const dim3 grid(static_cast<uint32_t>(perm_copy_workgroups(a.count, W)));
    if (a.rank == 2) hipLaunchKernelGGL((perm_rows<W, CONJ, 2>), grid, dim3(PERM_THREADS), 0, s, a);
    else if (a.rank == 3) hipLaunchKernelGGL((perm_rows<W, CONJ, 3>), grid, dim3(PERM_THREADS), 0, s, a);
    else hipLaunchKernelGGL((perm_rows<W, CONJ, 4>), grid, dim3(PERM_THREADS), 0, s, a);
}

}  // namespace

uint64_t perm_tile_workgroups(uint64_t total_tiles) {
    return total_tiles < TILE_GRID_CAP ? (total_tiles ? total_tiles : 1) : TILE_GRID_CAP;
}

uint64_t perm_copy_workgroups(uint64_t count, int words) {
    const uint64_t per = static_cast<uint64_t>(PERM_THREADS) * (4 / words);
    const uint64_t g = (count + per - 1) / per;
    return g < COPY_GRID_CAP ? (g ? g : 1) : COPY_GRID_CAP;
}

// The walk over a cached view's tiles. 0: (outer, ta, tb), tb fastest. 1: workgroups are dealt to the eight
// XCDs in turn, and each XCD takes one contiguous run of that order, so that the tiles on either side of a
// destination line that no tile boundary falls on (rows off the 128-byte grid) meet in one L2 instead of each
// writing a part of it. 2: runs with ta fastest, where few tiles along a would give whole XCDs the last,
// partly filled ones. Measured, us: 8191 x 4099 85 -> 65 (77 by order 2, so the limit), 2476 x 3864 16.8 -> 13.2,
// 4855 x 1187 13.1 -> 10.8 (11.8 by order 1; 7900 x 129 5.0 against 4.3). Runs lose where no destination line is
// cut: rows on the grid (77088 x 229 35.0 against 41.4), one tile per row ([28,1372,240] by 1,2,0 16.7
// against 18.8), streaming tiles (8192 x 4096 48.6 against 49.5); and on aligned rows of many planes
// ([100,180,16,36] by 2,0,3,1 22.9 against 24.6; unaligned [66,30,47,8] by 3,1,2,0 gains, 15.6 -> 12.9).
// Two tiles along a of which the last is at least half full, but not full, also lose (20001 x 112 7.6 by order 0 against 8.1 by
// order 2, 9922 x 120 5.6 against 6.2, 100001 x 96 18.5 against 20.1; 40003 x 120 alone 13.7 against 13.1); an emptier
// one gains (100001 x 88 19.2 against 17.4, 40003 x 80 9.2 against 8.5), and so does a full one (100001 x 128 19.5 against 16.9).
uint32_t perm_tile_order(const PermTileArgs& a, int words, bool vec, bool streaming) {
    constexpr uint32_t FEW = 32;
    if (streaming || a.tiles_b < 2 || (a.dst_sa * words) % 32 == 0 || (vec && a.outer_rank != 0) ||
        a.total_tiles > 0xffffffffull) {
        return 0;
    }
    const uint32_t last = a.ext_a % PERM_TILE_A;
    if (a.outer_rank == 0 && a.tiles_a == 2 && last >= PERM_TILE_A / 2) return 0;
    return a.outer_rank == 0 && a.tiles_b > a.tiles_a && a.tiles_a <= FEW ? 2 : 1;
}

void launch_perm_tile(Context* ctx, hipStream_t s, const PermTileArgs& args, int words, bool conj,
                      bool vec, bool streaming) {
    PermTileArgs a = args;
    a.order = perm_tile_order(a, words, vec, streaming);
    constexpr int TS = PERM_STREAM_TILE_A, TN = PERM_TILE_A;
    const char* name = nullptr;
    if (words == 1) {
        if (streaming) tile_t<1, false, true, TS, true>(s, a), name = "perm_tile_w1_v128_stream";
        else if (vec) tile_t<1, false, true, TN, false>(s, a), name = "perm_tile_w1_v128";
        else tile_t<1, false, false, TN, false>(s, a), name = "perm_tile_w1";
    } else if (!conj) {
        if (streaming) tile_t<2, false, true, TS, true>(s, a), name = "perm_tile_w2_v128_stream";
        else if (vec) tile_t<2, false, true, TN, false>(s, a), name = "perm_tile_w2_v128";
        else tile_t<2, false, false, TN, false>(s, a), name = "perm_tile_w2";
    } else {
        if (streaming) tile_t<2, true, true, TS, true>(s, a), name = "perm_tile_conj_w2_v128_stream";
        else if (vec) tile_t<2, true, true, TN, false>(s, a), name = "perm_tile_conj_w2_v128";
        else tile_t<2, true, false, TN, false>(s, a), name = "perm_tile_conj_w2";
    }
    check_hip(hipGetLastError(), "perm_tile launch");
    note_launch(ctx, name);
}

void launch_perm_copy(Context* ctx, hipStream_t s, const PermCopyArgs& a, int words, bool conj) {
    const bool nt = a.streaming != 0;
    const char* name;
    if (a.contiguous == 0 && a.rank >= 2 && a.rank <= 4 && a.count < (1ull << 32)) {
        if (words == 1) rows_t<1, false>(s, a), name = "perm_rows_w1";
        else if (!conj) rows_t<2, false>(s, a), name = "perm_rows_w2";
        else rows_t<2, true>(s, a), name = "perm_rows_conj_w2";
    } else if (words == 1) {
        if (nt) copy_t<1, false, true>(s, a), name = "perm_copy_w1_stream";
        else copy_t<1, false, false>(s, a), name = "perm_copy_w1";
    } else if (!conj) {
        if (nt) copy_t<2, false, true>(s, a), name = "perm_copy_w2_stream";
        else copy_t<2, false, false>(s, a), name = "perm_copy_w2";
    } else {
        if (nt) copy_t<2, true, true>(s, a), name = "perm_copy_conj_w2_stream";
        else copy_t<2, true, false>(s, a), name = "perm_copy_conj_w2";
    }
    check_hip(hipGetLastError(), "perm_copy launch");
    note_launch(ctx, name);
}

}  // namespace lg
