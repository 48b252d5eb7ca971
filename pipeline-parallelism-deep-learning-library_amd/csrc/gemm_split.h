// The fp32 GEMM on the bf16 matrix cores: every operand element as three bf16 pieces.
//
// An f32 has 24 significant bits and a bf16 has 8, so x = x0 + x1 + x2 with x0 = bf16(x),
// x1 = bf16(x - x0), x2 = x - x0 - x1, each step exact: the three pieces hold the f32 whole. A
// product is then six bf16 products, a0b0 + (a0b1 + a1b0) + (a1b1 + a0b2 + a2b0); the three left
// out add up to 2^-24 of it at the most. bf16 products are exact in f32 and one
// v_mfma_f32_32x32x16_bf16 adds sixteen of them into an f32 accumulator, so a sum over K is
// rounded about 6 K / 16 times instead of the K times of v_mfma_f32_32x32x2_f32. A sum of many terms is closer to
// the exact one for it; one of a single term, which that instruction rounds correctly, is up to 1.5 units in
// the last place off (measured: 1.48, one in five not the nearest f32).
//
// Elements are scaled by 2^23 before they are split and the sums by 2^-46 after: an f32, subnormals
// included, is a whole multiple of 2^-149, so a scaled one is a whole multiple of 2^-126 and each of its pieces
// zero or a normal bf16. So the pieces hold every element below 2^104 whole, whatever its size. Where
// scaled sums come out as anything but finite numbers (an infinity or a NaN in an operand, an element of
// 2^104 or more, a sum of 2^82 or more: x - x0 turns an infinity into NaN), the wave that holds them computes
// their row of 32x32 blocks again with the f32 matrix instruction on the operands themselves (b3_redo).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_pipe.h"

namespace lg {
namespace gemm_detail {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
// Four floats that are only known to be 4-byte aligned (global_load_dwordx4 needs no more).
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int B3_BK = 16;  // K depth of one slice

// LDS image of one operand's slice, R rows: three planes (one per piece), each of two chunks (k 0-7 and
// 8-15), each of four classes (row % 4), each of R / 4 rows of 16 bytes (eight bf16). A
// thread converts a block of four rows by four k: for each row of the block the wave writes 16
// neighbouring rows of one class, 8 bytes each. A fragment read takes 32 rows by 16 bytes:
// eight consecutive lanes are two neighbours in each of four classes, which the classes' 32-byte padding
// puts on distinct banks; the chunk's 64-byte padding does so for the two chunks of a write.
template <int R>
struct B3Geo {
    static constexpr int CLS = R * 4 + 64;
    static constexpr int CH = 4 * CLS + 64;
    static constexpr int PL = 2 * CH;
    static constexpr int BYTES = 3 * PL;
};

// The scale of the operands' elements, and that of the sums back (see the file's head). A test of the elements
// instead, with the tile computed again where one is too small, cost as much per element and 4096^3 with
// one element of 1e-35 4028 us, against 600 with the scale.
constexpr float B3_UP = 0x1p23f, B3_DOWN = 0x1p-46f;
// Slices after which a tile's sums change sign (see b3_sums): within the loop, a multiple of its unrolling, or by
// another loop around it for one wave per SIMD, whose schedule the first way disturbs (2304^3 on stream-K 148 ->
// 153 us) and whose registers take the second (all other tiles would spill: 2048^3 97 -> 112 us). That loop costs 3 %
// at K = 1024 (3072 x 3072 120 -> 124 us), so it has a kernel of its own for K beyond one turn.
constexpr uint32_t B3_TURN = 64, B3_TURN_ALONE = 256;
enum B3Turns { TURNS_INSIDE, TURNS_NONE, TURNS_AROUND };

// (x, y) -> three packed pairs of bf16 pieces. Eleven VALU instructions a pair and two for the scale, four
// cycles each, and up to six of them hide behind every MFMA. (v_dot2_f32_bf16 would do the subtraction and the
// unpacking in one, exactly, but it does not run beside an MFMA: two of them cost an MFMA's time and a half.)
__device__ __forceinline__ void b3_split(float x, float y, uint32_t (&q)[3]) {
    q[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x, y}, bf16x2));
    x = x - __builtin_bit_cast(float, q[0] << 16);
    y = y - __builtin_bit_cast(float, q[0] & 0xffff0000u);
    q[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x, y}, bf16x2));
    x = x - __builtin_bit_cast(float, q[1] << 16);
    y = y - __builtin_bit_cast(float, q[1] & 0xffff0000u);
    q[2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x, y}, bf16x2));
}

// One thread's 4 x 4 block of an operand slice (rows 4 rq .. 4 rq + 3, k 4 k4 .. 4 k4 + 3), in the order in
// which it is loaded: LOAD_K and LOAD_S v[row][k], LOAD_MN v[k][row].
struct B3Block {
    floatx4 v[4];
};

// Where a thread's block lies: byte offsets from the tile's first element of the slice, uniform strides,
// and the LDS byte address of each of its rows (EDGE: rows past the operand's end are
// the last ones again, and rows before the tile's first are written into their class's padding, which
// nothing reads: a branch there would part the conversion from the MFMAs that hide it).
template <int MODE, int R, bool EDGE>
struct B3Loader {
    using G = B3Geo<R>;
    const float* base;  // the operand at the tile's first row (EDGE, LOAD_MN: see init) and current k
    int64_t srow, sk;
    uint32_t off[4];   // byte offset of load i (one offset and uniform strides unless EDGE)
    uint32_t lds[4];   // byte address of row i in plane 0
    uint32_t k4;

    // p: the operand at (row 0 of the batch plane, first k). m0: the tile's first row, rows: the
    // operand's row count, t: the thread's number among the R threads that load this operand.
    __device__ __forceinline__ void init(const float* p, int64_t srow_, int64_t sk_, uint32_t m0,
                                         uint32_t rows, uint32_t t) {
        srow = srow_;
        sk = sk_;
        k4 = t & 3u;
        const uint32_t rq = t >> 2;
        const uint32_t at = (k4 >> 1) * G::CH + (k4 & 1u) * 8u;
        uint32_t row0 = m0 + 4 * rq;  // first row of the block
        uint32_t first = m0;          // row that `base` points at
        if constexpr (EDGE && MODE == LOAD_MN) {
            // A block that would cross the end starts four rows before it.
            row0 = min(row0, rows - 4);
            first = min(m0, rows - 4);
        }
        base = p + static_cast<int64_t>(first) * srow;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t row = EDGE && MODE != LOAD_MN ? min(row0 + i, rows - 1) : row0 + i;
            if constexpr (MODE == LOAD_MN) {
                off[i] = (row0 - first) * 4u;
            } else if constexpr (EDGE) {
                off[i] = static_cast<uint32_t>((row - first) * srow) * 4u;
            } else {
                off[i] = static_cast<uint32_t>((row0 - first) * srow) * 4u;
            }
            if constexpr (MODE != LOAD_MN) off[i] += k4 * 4u * static_cast<uint32_t>(sk) * 4u;
            else off[i] += k4 * 4u * static_cast<uint32_t>(sk) * 4u;
            const uint32_t r = EDGE && MODE == LOAD_MN ? row0 + i - m0 : 4 * rq + i;
            lds[i] = at + (r & 3u) * G::CLS + (static_cast<int32_t>(r) < 0 ? R * 4u : (r >> 2) * 16u);
        }
    }
    __device__ __forceinline__ const float* at(int i) const {
        // Load i's uniform part: row i of the block (LOAD_K, LOAD_S) or its k i (LOAD_MN).
        const float* b = base;
        if constexpr (MODE == LOAD_MN) b += i * sk;
        else if constexpr (!EDGE) b += i * srow;
        return b;
    }
    __device__ __forceinline__ void load(B3Block& x) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (MODE == LOAD_S) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    x.v[i][j] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(at(i) + j * sk) + off[i]);
                }
            } else {
                x.v[i] = *reinterpret_cast<const floatx4u*>(reinterpret_cast<const char*>(at(i)) + off[i]);
            }
        }
    }
    // The last slice's `left` < 16 k: zero past them, where the last one is loaded again. (A branch around each load,
    // and the tail again in place of every slice past it: 2048 x 2048 x 88 of both along K 17.5 us against 16.0, of A
    // alone 15.7 against 14.6, 3001 x 2011 x 1537 129 against 123-127, on 64x64 tiles 1000 x 1020 x 1537 31-40 against 29-35.)
    __device__ __forceinline__ void load_tail(B3Block& x, uint32_t left) const {
        __asm__ volatile("" : "+s"(left));  // no offsets held in registers through the loop
        uint32_t to[4];  // byte offset from k 4 k4 to that of the block's k j, modulo 2^32
#pragma unroll
        for (int j = 0; j < 4; ++j) to[j] = (min(4 * k4 + j, left - 1) - 4 * k4) * static_cast<uint32_t>(sk) * 4u;
        const char* from = reinterpret_cast<const char*>(base);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (MODE == LOAD_MN) {
                x.v[i] = *reinterpret_cast<const floatx4u*>(from + (off[i] + to[i]));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) x.v[i][j] = *reinterpret_cast<const float*>(from + (off[i] + to[j]));
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (4 * k4 + (MODE == LOAD_MN ? i : j) >= left) x.v[i][j] = 0.0f;
    }
    __device__ __forceinline__ void advance(int slices = 1) { base += slices * B3_BK * sk; }

    // Row i of the block: the pieces of its scaled elements into a stage.
    __device__ __forceinline__ void store_row(char* stage, const B3Block& x, int i, float scale) const {
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = scale * (MODE == LOAD_MN ? x.v[j][i] : x.v[i][j]);
        uint32_t lo[3], hi[3];
        b3_split(e[0], e[1], lo);
        b3_split(e[2], e[3], hi);
        char* q = EDGE && MODE == LOAD_MN ? stage + lds[i] : stage + lds[0] + i * G::CLS;
#pragma unroll
        for (int j = 0; j < 3; ++j) *reinterpret_cast<uintx2*>(q + j * G::PL) = uintx2{lo[j], hi[j]};
    }
};

// Every LDS access of this wave done, then the workgroup's barrier. Waves that load nothing store
// nothing either, and only the fences tell the compiler that what they read there changes.
__device__ __forceinline__ void b3_barrier() {
    __asm__ volatile("" ::: "memory");
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

template <int FM, int FN>
__device__ __forceinline__ void b3_zero(floatx16 (&acc)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
}

// One row of blocks: the six products of A block `a` with each B block, small ones first, each B piece
// for the last time as early as the order allows (piece 2 in the first product, piece 1 by the third).
template <int FN, typename F>
__device__ __forceinline__ void b3_block(const bf16x8 (&a)[3], const bf16x8 (&b)[FN][3], floatx16 (&acc)[FN], F&& after) {
    constexpr int ta[6] = {0, 1, 0, 2, 1, 0}, tb[6] = {2, 1, 1, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ta[t]], b[j][tb[t]], acc[j], 0, 0, 0);
        after(t);
    }
}

template <int FM, int FN>
__device__ __forceinline__ void b3_scale(floatx16 (&acc)[FM][FN], float by) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = by * acc[i][j][r];
}

// One (32 FM WM) x (32 FN WN) tile over k [0, klen) from A and B (batch plane, first k): acc, of the scaled
// elements, added to acc, and of the sign returned. `sign` is the first slices'. ALONE: one wave per SIMD, one sign.
template <int AM, int BMD, int WM, int WN, int FM, int FN, bool EDGE, bool ALONE>
__device__ __forceinline__ float b3_tile(const GemmArgs& p, char* smem, const float* A, const float* B,
                                        uint32_t m0, uint32_t n0, uint32_t klen, float sign, floatx16 (&acc)[FM][FN]) {
    constexpr int RA = 32 * FM * WM, RB = 32 * FN * WN;
    using GA = B3Geo<RA>;
    using GB = B3Geo<RB>;
    constexpr int ST = GA::BYTES + GB::BYTES;
    constexpr int WA = RA / 64, WB = RB / 64;  // waves that load A, then B
    constexpr int NX = FM == 4 ? 2 : 4, EARLY = FM == 4 ? 0 : 2;
    static_assert(WA + WB <= WM * WN, "one block of a slice per thread");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    // This lane's fragment addresses (row lane % 32 of a block, chunk lane / 32).
    const uint32_t fr = (lane & 3) * 1u, fq = ((lane & 31) >> 2) * 16u, fh = lane >> 5;
    const uint32_t fa = fr * GA::CLS + fq + fh * GA::CH + wm * FM * 128;
    const uint32_t fb = fr * GB::CLS + fq + fh * GB::CH + wn * FN * 128 + GA::BYTES;
    const uint32_t full = klen / B3_BK, left = klen - full * B3_BK;

    auto loop = [&](auto* loader, float scale, float turned, char* mine) __attribute__((always_inline)) {
        using LD = std::remove_pointer_t<decltype(loader)>;
        constexpr bool LOADS = !std::is_same_v<LD, void*>;
        // Slice s passes through the registers x[s % NX] into stage s % 2. Step s multiplies slice s. All
        // of stage s % 2 is read and all of slice s + 1 written when the last row of blocks
        // begins: the step's one barrier stands there, and behind it, among that row's MFMAs, the
        // first fragments of slice s + 1 are read and the first EARLY rows of slice s + 2
        // converted into the stage just read; the other rows are converted in step s + 1 before its
        // barrier, which ends with the loads of slice s + 2 + NX into the same registers. Past the last slice the
        // last one is loaded again (EDGE: nothing is; a tail costs more than a branch).
        const uint32_t slices = full + (left != 0);
        B3Block x[NX];
        auto fetch = [&](uint32_t s, B3Block& to) __attribute__((always_inline)) {
            if constexpr (LOADS) {
                if (EDGE && s >= slices) return;
                if (s != 0 && s < slices) loader->advance();
                if (EDGE && left != 0 && s + 1 == slices) loader->load_tail(to, left);
                else loader->load(to);
            }
        };
        // Row i of slice s's block, scaled by `scale` or, every other B3_TURN slices, `turned`.
        constexpr uint32_t TURN = ALONE ? 0 : B3_TURN;
        auto put_row = [&](int i, uint32_t s, int stage, const B3Block& from) __attribute__((always_inline)) {
            if constexpr (LOADS) loader->store_row(mine + stage * ST, from, i, (s & TURN) != 0 ? turned : scale);
        };
        auto turn = [&](uint32_t s) __attribute__((always_inline)) {
            if (TURN != 0 && s % B3_TURN == 0 && s != 0 && s < slices) b3_scale(acc, -1.0f);
        };
        bf16x8 a[2][3], b[FN][3];
        auto read_a = [&](bf16x8 (&to)[3], int i, int stage) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < 3; ++q) to[q] = *reinterpret_cast<const bf16x8*>(smem + fa + stage * ST + q * GA::PL + i * 128);
        };
        auto read_b = [&](int q, int stage) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j][q] = *reinterpret_cast<const bf16x8*>(smem + fb + stage * ST + q * GB::PL + j * 128);
        };
        auto step = [&](auto phase, uint32_t s) __attribute__((always_inline)) {
            constexpr int U = decltype(phase)::value, P = U & 1, X1 = (U + 1) % NX, X2 = (U + 2) % NX;
            constexpr int MG = 6 * FN;
            // VALU instructions after each MFMA: a row takes 26, and the loop's own a few more. One more behind
            // the barrier where nothing else covers a wave's wait there (4608 x 4608 x 512 on stream-K
            // 150 -> 146 us, 2304^3 151 -> 148; 256x128 tiles of two waves per SIMD 167 against 173).
            constexpr int V = LOADS ? ((4 - EARLY) * 28 + (FM - 1) * MG - 1) / ((FM - 1) * MG) : 0;
            constexpr int VL = LOADS ? (EARLY * 28 + MG - 1) / MG + (ALONE ? 1 : 0) : 0;
#pragma unroll
            for (int i = 0; i + 1 < FM; ++i) {
                read_a(a[(i + 1) & 1], i + 1, P);
                // This row of blocks' share of the conversion.
#pragma unroll
                for (int r = EARLY + i * (4 - EARLY) / (FM - 1); r < EARLY + (i + 1) * (4 - EARLY) / (FM - 1); ++r) {
                    put_row(r, s + 1, P ^ 1, x[X1]);
                }
                b3_block<FN>(a[i & 1], b, acc[i], [](int) {});
                // One read after each of the first MFMAs, the conversion's VALU work and writes spread over all.
#pragma unroll
                for (int q = 0; q < MG; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (q < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if constexpr (V > 0) {
                        __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
                        if (q % 3 == 2) __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            b3_barrier();
            constexpr int L = (FM - 1) & 1;
#pragma unroll
            for (int r = 0; r < EARLY; ++r) put_row(r, s + 2, P, x[X2]);
            b3_block<FN>(a[L], b, acc[FM - 1], [&](int t) {
                if (t == 0) read_b(2, P ^ 1);
                if (t == 2) {
                    read_b(1, P ^ 1);
                    read_a(a[L ^ 1], 0, P ^ 1);
                }
                if (t == 5) read_b(0, P ^ 1);
            });
            if constexpr (VL > 0) {
#pragma unroll
                for (int q = 0; q < MG; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (q > 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, VL, 0);
                    if (q % 3 == 2) __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
                }
            }
            if constexpr (L == 0) {
#pragma unroll
                for (int q = 0; q < 3; ++q) a[0][q] = a[1][q];
            }
            __builtin_amdgcn_sched_barrier(0);
            fetch(s + 1 + NX, x[X1]);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int s = 0; s < NX; ++s) fetch(s, x[s]);
#pragma unroll
        for (int r = 0; r < 4; ++r) put_row(r, 0, 0, x[0]);
#pragma unroll
        for (int r = 0; r < EARLY; ++r) put_row(r, 1, 1, x[1]);
        fetch(NX, x[0]);
        b3_barrier();
        read_a(a[0], 0, 0);
        read_b(2, 0);
        read_b(1, 0);
        read_b(0, 0);
        uint32_t s = 0;
        if constexpr (NX == 4) {
            for (; s + 3 < slices; s += 4) {
                turn(s);
                step(std::integral_constant<int, 0>{}, s);
                step(std::integral_constant<int, 1>{}, s + 1);
                step(std::integral_constant<int, 2>{}, s + 2);
                step(std::integral_constant<int, 3>{}, s + 3);
            }
            turn(s);
            if (s < slices) step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < slices) step(std::integral_constant<int, 1>{}, s + 1);
            if (s + 2 < slices) step(std::integral_constant<int, 2>{}, s + 2);
        } else {
            for (; s + 1 < slices; s += 2) {
                turn(s);
                step(std::integral_constant<int, 0>{}, s);
                step(std::integral_constant<int, 1>{}, s + 1);
            }
            turn(s);
            if (s < slices) step(std::integral_constant<int, 0>{}, s);
        }
    };
    if (wave < WA) {
        B3Loader<AM, RA, EDGE> ld;
        ld.init(A, p.a_sm, p.a_sk, m0, p.m, tid);
        const float scale = sign * (p.scale_b ? B3_UP : B3_UP * p.alpha);
        loop(&ld, scale, -scale, smem);
    } else if (wave < WA + WB) {
        B3Loader<BMD, RB, EDGE> ld;
        ld.init(B, p.b_sn, p.b_sk, n0, p.n, tid - RA);
        const float scale = p.scale_b ? B3_UP * p.alpha : B3_UP;
        loop(&ld, scale, scale, smem + GA::BYTES);
    } else {
        void* none = nullptr;
        loop(&none, 1.0f, 1.0f, smem);
    }
    return !ALONE && (full + (left != 0) - 1 & B3_TURN) != 0 ? -sign : sign;
}

// One wave's 32 x 32 FN outputs in plain f32 (v_mfma_f32_32x32x2_f32), straight from memory, for rows of
// blocks whose scaled sums are not finite: rows from m, columns from n. Half h of the wave takes k 8 g + 4 h ..
// 8 g + 4 h + 3 of group g, one 128-bit load an operand row where K is contiguous, four groups in
// flight (the MFMAs of one take 256 FN cycles). Bound: the f32 matrix rate over the rows of blocks concerned, which it
// reaches to about 60 %: 4096^3 with an infinity in one row of A 784 us, in every 64th 1270, with all of A NaN 1740
// (601 without; 32-bit loads with nothing in flight took 3720, the f32 instruction alone 930); 3001 x 2011 x 1537
// 238, 284 and 424 (132; 454), 2304^3 on stream-K 267, 317 and 481 (150; 190).
template <int AM, int BMD, int FN>
__device__ __forceinline__ void b3_redo(const GemmArgs& p, const float* A, const float* B, uint32_t m, uint32_t n,
                                        uint32_t klen, int lane, floatx16 (&acc)[FN]) {
    constexpr int D = 4;
    const uint32_t lr = lane & 31, h = lane >> 5;
    const float alpha_a = p.scale_b ? 1.0f : p.alpha, alpha_b = p.scale_b ? p.alpha : 1.0f;
    // Uniform first elements and 32-bit byte offsets of the lane's (rows past the end repeat the last one).
    A += static_cast<int64_t>(m) * p.a_sm;
    B += static_cast<int64_t>(n) * p.b_sn;
    const uint32_t ao = static_cast<uint32_t>((min(m + lr, p.m - 1) - m) * p.a_sm + 4 * h * p.a_sk) * 4u;
    uint32_t bo[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        bo[j] = static_cast<uint32_t>((min(n + j * 32 + lr, p.n - 1) - n) * p.b_sn + 4 * h * p.b_sk) * 4u;
    }
    const uint32_t groups = klen / 8;
    floatx4 a[D], b[D][FN];
    auto one = [](const float* q, uint32_t off) __attribute__((always_inline)) {
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(q) + off);
    };
    auto get = [&](auto mode, const float* q, int64_t sk, uint32_t off) __attribute__((always_inline)) {
        floatx4 x;
        if constexpr (decltype(mode)::value == LOAD_K) {
            x = *reinterpret_cast<const floatx4u*>(reinterpret_cast<const char*>(q) + off);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = one(q + e * sk, off);
        }
        return x;
    };
    auto load = [&](uint32_t g, int u) __attribute__((always_inline)) {
        const int64_t k = static_cast<int64_t>(min(g, groups - 1)) * 8;
        a[u] = get(std::integral_constant<int, AM>{}, A + k * p.a_sk, p.a_sk, ao);
#pragma unroll
        for (int j = 0; j < FN; ++j) b[u][j] = get(std::integral_constant<int, BMD>{}, B + k * p.b_sk, p.b_sk, bo[j]);
    };
    auto multiply = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(alpha_a * a[u][e], alpha_b * b[u][j][e], acc[j], 0, 0, 0);
            }
    };
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    if (groups > 0) {
#pragma unroll
        for (int u = 0; u < D; ++u) load(u, u);
        uint32_t g = 0;
        for (; g + D <= groups; g += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                multiply(u);
                load(g + D + u, u);
            }
        }
#pragma unroll
        for (int u = 0; u < D; ++u)
            if (g + u < groups) multiply(u);
    }
    if (groups * 8 < klen) {
        const int64_t k = static_cast<int64_t>(groups) * 8;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = groups * 8 + 4 * h + e < klen;
            a[0][e] = 0.0f;
            if (in) a[0][e] = one(A + (k + e) * p.a_sk, ao);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                b[0][j][e] = 0.0f;
                if (in) b[0][j][e] = one(B + (k + e) * p.b_sk, bo[j]);
            }
        }
        multiply(0);
    }
}

// A tile's sums over k [0, klen). Returns the wave's rows of blocks (bit i: row i) whose sums are not finite and
// that b3_redo has to compute. The bf16 instruction rounds down where its accumulator has no room, so a sum over
// one sign is a little low: 2.7e-7 of it at K = 4096 on normal operands, 1e-5 at 262144. `negative` sums the negated
// products and negates the sum, which is then a little high: every other split of K does, and so
// does every other B3_TURN slices of a longer K, and the errors cancel instead of adding up. Error against f64,
// normal operands, 2048^2 outputs, over one sign / now / f32 instruction: K = 4096 1.00e-6 / 0.97e-6 / 1.15e-6, 16384
// 2.1e-6 / 1.9e-6 / 2.3e-6, 65536 4.5e-6 / 3.5e-6 / 4.6e-6, 262144 1.1e-5 / 6.3e-6 / 9.2e-6.
template <int AM, int BMD, int WM, int WN, int FM, int FN, bool EDGE, B3Turns TURNS>
__device__ __forceinline__ uint32_t b3_sums(const GemmArgs& p, char* smem, const float* A, const float* B, uint32_t m0,
                                        uint32_t n0, uint32_t klen, bool negative, int wave, int lane,
                                        floatx16 (&acc)[FM][FN]) {
    float sign = negative ? -1.0f : 1.0f;
    if constexpr (TURNS == TURNS_AROUND) {
        for (uint32_t k = 0;;) {
            const uint32_t len = min(klen - k, B3_TURN_ALONE * B3_BK);
            b3_tile<AM, BMD, WM, WN, FM, FN, EDGE, true>(p, smem, A + static_cast<int64_t>(k) * p.a_sk,
                                                         B + static_cast<int64_t>(k) * p.b_sk, m0, n0, len, sign, acc);
            k += len;
            if (k == klen) break;
            b3_scale(acc, -1.0f);
            sign = -sign;
            b3_barrier();  // every wave is done with the stages
        }
    } else {
        sign = b3_tile<AM, BMD, WM, WN, FM, FN, EDGE, TURNS == TURNS_NONE>(p, smem, A, B, m0, n0, klen, sign, acc);
    }
    b3_scale(acc, sign * B3_DOWN);
    // x * 0 is 0 unless x is infinite or NaN. Rows and columns past the output's edge hold
    // whatever the stages held, and do not count.
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, h = lane >> 5;
    uint32_t bad = 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        float z = 0.0f;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float t = acc[i][j][r] * 0.0f;
                if (!EDGE || (m0 + (wm * FM + i) * 32 + (r >> 2) * 8 + h * 4 + (r & 3) < p.m &&
                              n0 + (wn * FN + j) * 32 + lr < p.n)) {
                    z = z + t;
                }
            }
        if (__any(z != 0.0f)) bad |= 1u << i;
    }
    return bad;
}

// gemm_f32_b3<AM, BMD, WM, WN, FM, FN, EDGE>: C = beta * C + sum_k (alpha * a) * b, or raw split-K partials,
// on (32 FM WM) x (32 FN WN) tiles of WM x WN waves: 256x256 and 256x128 and 128x256 tiles with eight waves
// (the first with 4 x 2 blocks each, so that a piece read from LDS feeds twice the products), 128x128 with
// four. EDGE: ragged tiles or a K that is no multiple of 16. Operands pass through registers, where
// they are split, so a load needs no alignment beyond its elements' and edges cost no second path.
//
// Bound: the chip's power. 1748 TFLOP/s of bf16 MFMA is what it sustains with nothing else running (1.74 of
// 2.4 GHz), 291 TFLOP/s of this product; the 256x256 tiles keep the matrix cores 79 % busy at 1.6-1.7 GHz (4096^3), the
// rest of the power going into fragment reads and conversions. 128x128 tiles are 48 % busy at 2.07 GHz on one workgroup per
// compute unit (2048^3), 62 % at 1.83 on many (2048 x 8192 x 2048): their two waves per SIMD or fewer wait. Fewer stalls alone do not help: the same
// kernel without a schedule was busy 69 % at 1.87 GHz and 3 % slower. Against v_mfma_f32_32x32x2_f32 on the same
// tiles: 4096^3 931 -> 570-580 us (148 -> 237 TFLOP/s), 32 x 1024^3 483 -> 310 us (142 -> 222), a layer's three
// products and elementwise work at 2048 x 2048 x 8192 1554 -> 1108 us. Error against f64 on
// normal operands: 1.0e-6 (4096^3), 4.9e-7 (K = 1024), before 1.1e-6 and 5.7e-7.
template <int AM, int BMD, int WM, int WN, int FM, int FN, bool EDGE>
__global__ __launch_bounds__(64 * WM * WN, WM * WN >= 8 ? 1 : 2) void gemm_f32_b3(GemmArgs p) {
    constexpr int RA = 32 * FM * WM, RB = 32 * FN * WN;
    constexpr int ST = B3Geo<RA>::BYTES + B3Geo<RB>::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[2 * ST];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t plane, tm, tn;
    decode_tile<RA == 256 ? 4 : 8>(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, &plane, &tm, &tn);
    const uint32_t bi = plane / p.splits, split = plane - bi * p.splits;
    const uint32_t m0 = tm * RA, n0 = tn * RB, kb = split * p.k_chunk;
    const uint32_t klen = min(p.k - kb, p.k_chunk);
    const float* A = p.a + static_cast<int64_t>(bi) * p.a_sb + static_cast<int64_t>(kb) * p.a_sk;
    const float* B = p.b + static_cast<int64_t>(bi) * p.b_sb + static_cast<int64_t>(kb) * p.b_sk;
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, h = lane >> 5;
    float* C = p.partial != nullptr ? p.partial + static_cast<int64_t>(plane) * p.m * p.n
                                    : p.c + static_cast<int64_t>(bi) * p.c_sb;
    const int64_t c_sm = p.partial != nullptr ? static_cast<int64_t>(p.n) : p.c_sm;
    const int64_t c_sn = p.partial != nullptr ? 1 : p.c_sn;
    const float beta = p.partial != nullptr ? 0.0f : p.beta;
    auto store = [&](uint32_t i, const floatx16 (&x)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const uint32_t col = n0 + (wn * FN + j) * 32 + lr;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = m0 + (wm * FM + i) * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
                if (EDGE && (row >= p.m || col >= p.n)) continue;
                float* q = C + row * c_sm + col * c_sn;
                float v = x[j][r];
                if (beta != 0.0f) v = beta * *q + v;
                *q = v;
            }
        }
    };
    floatx16 acc[FM][FN];
    b3_zero(acc);
    uint32_t bad = b3_sums<AM, BMD, WM, WN, FM, FN, EDGE, TURNS_INSIDE>(p, smem, A, B, m0, n0, klen, split & 1u, wave, lane, acc);
#pragma unroll
    for (int i = 0; i < FM; ++i)
        if ((bad >> i & 1u) == 0) store(i, acc[i]);
    while (bad != 0) {
        const uint32_t i = __builtin_ctz(bad);
        bad &= bad - 1;
        floatx16 t[FN];
        b3_redo<AM, BMD, FN>(p, A, B, m0 + (wm * FM + i) * 32, n0 + wn * FN * 32, klen, lane, t);
        store(i, t);
    }
}

// gemm_f32_b3kw<AM, BMD, EDGE>: a 64x64 tile per workgroup, each of four waves summing the whole tile
// over every fourth slice of the K chunk, for outputs of too few 128x128 tiles, or tiles that would spread
// unevenly. A wave's 2 x 2 blocks then read 12 fragments for 24 MFMAs, as 128x128 tiles do (waves
// of 32x32 sharing stages would read twice that, the LDS's whole rate), and nothing but its own loads
// and LDS accesses, which complete in order, holds it: no barrier before the end, one stage a wave. The price is the
// conversion, once per wave: 208 VALU instructions for 24 MFMAs, more than they hide, so two workgroups
// share a compute unit. The sums meet in LDS as (s0 + s1) + (s2 + s3), each wave storing one block. Bound: what a wave
// waits for, at 110-118 TFLOP/s: matrix cores 28 % busy, VALU 38 %, LDS 22 % (2300 x 2304 x 2304, 2.1 GHz). Against the
// f32 instruction: 1000 x 1020 x 1537 with odd rows 148-162 -> 29-34 us (32-bit loads before), 2300 x 2304 x 2304 274 -> 214,
// 320 x 352 x 97536 418 -> 224, 37^6 in rank 4 147 -> 56, 1000 x 1024 x 1024 with A along M 40 -> 27.
template <int AM, int BMD, bool EDGE>
__global__ __launch_bounds__(256, 2) void gemm_f32_b3kw(GemmArgs p) {
    constexpr int R = 64, W = 4;
    using G = B3Geo<R>;
    constexpr int ST = 2 * G::BYTES;
    // The stages, then the four sums: two workgroups per compute unit.
    constexpr int SM = W * (ST > R * R * 4 ? ST : R * R * 4);
    static_assert(SM <= 80 * 1024, "two workgroups per compute unit");
    __shared__ __attribute__((aligned(16))) char smem[SM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, h = lane >> 5;
    uint32_t plane, tm, tn;
    decode_tile(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, &plane, &tm, &tn);
    const uint32_t bi = plane / p.splits, split = plane - bi * p.splits;
    const uint32_t m0 = tm * R, n0 = tn * R, kb = split * p.k_chunk;
    const uint32_t klen = min(p.k - kb, p.k_chunk);
    const float* A = p.a + static_cast<int64_t>(bi) * p.a_sb + static_cast<int64_t>(kb) * p.a_sk;
    const float* B = p.b + static_cast<int64_t>(bi) * p.b_sb + static_cast<int64_t>(kb) * p.b_sk;
    char* mine = smem + wave * ST;
    const char* fa = mine + (lane & 3) * G::CLS + (lr >> 2) * 16 + h * G::CH;
    const char* fb = fa + G::BYTES;

    // This wave's slices: wave, wave + 4, ...; the chunk's last may hold `left` < 16 k.
    const uint32_t total = (klen + B3_BK - 1) / B3_BK, left = klen % B3_BK;
    const uint32_t slices = (total - wave + W - 1) / W;
    const bool tail = EDGE && left != 0 && (total - 1) % W == static_cast<uint32_t>(wave);
    B3Loader<AM, R, EDGE> la;
    B3Loader<BMD, R, EDGE> lb;
    la.init(A, p.a_sm, p.a_sk, m0, p.m, lane);
    lb.init(B, p.b_sn, p.b_sk, n0, p.n, lane);
    la.advance(wave);
    lb.advance(wave);
    // Waves 1 and 3 sum the negated products: see b3_sums.
    const float scale_a = (wave & 1 ? -B3_UP : B3_UP) * (p.scale_b ? 1.0f : p.alpha);
    const float scale_b = p.scale_b ? B3_UP * p.alpha : B3_UP, down = wave & 1 ? -B3_DOWN : B3_DOWN;
    floatx16 acc[2][2];
    b3_zero(acc);
    {
        B3Block xa[2], xb[2];
        auto fetch = [&](uint32_t s, int to) __attribute__((always_inline)) {
            if (EDGE && s >= slices) return;
            if (s != 0 && s < slices) {
                la.advance(W);
                lb.advance(W);
            }
            if (EDGE && tail && s + 1 == slices) {
                la.load_tail(xa[to], left);
                lb.load_tail(xb[to], left);
            } else {
                la.load(xa[to]);
                lb.load(xb[to]);
            }
        };
        auto put = [&](int from) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                la.store_row(mine, xa[from], r, scale_a);
                lb.store_row(mine + G::BYTES, xb[from], r, scale_b);
            }
        };
        // Other lanes read what a lane wrote: the compiler keeps their order, the LDS does by itself.
        auto in_order = [] { __asm__ volatile("" ::: "memory"); };
        auto step = [&](auto phase, uint32_t s) __attribute__((always_inline)) {
            constexpr int U = decltype(phase)::value;
            bf16x8 a[2][3], b[2][3];
            in_order();
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    a[i][q] = *reinterpret_cast<const bf16x8*>(fa + q * G::PL + i * 128);
                    b[i][q] = *reinterpret_cast<const bf16x8*>(fb + q * G::PL + i * 128);
                }
            in_order();
            put(U ^ 1);
#pragma unroll
            for (int i = 0; i < 2; ++i) b3_block<2>(a[i], b, acc[i], [](int) {});
#pragma unroll
            for (int q = 0; q < 24; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            fetch(s + 3, U ^ 1);
            __builtin_amdgcn_sched_barrier(0);
        };
        fetch(0, 0);
        fetch(1, 1);
        put(0);
        fetch(2, 0);
        uint32_t s = 0;
        for (; s + 1 < slices; s += 2) {
            step(std::integral_constant<int, 0>{}, s);
            step(std::integral_constant<int, 1>{}, s + 1);
        }
        if (s < slices) step(std::integral_constant<int, 0>{}, s);
    }

    __syncthreads();  // the stages are free
    {
        float* q = reinterpret_cast<float*>(smem) + wave * (R * R) + lane;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) q[((i * 2 + j) * 16 + r) * 64] = down * acc[i][j][r];
    }
    __syncthreads();
    const int bm = wave >> 1, bn = wave & 1;
    const uint32_t col = n0 + bn * 32 + lr;
    auto row_of = [&](int r) { return m0 + bm * 32 + (r >> 2) * 8 + h * 4 + (r & 3); };
    floatx16 v[1];
    float z = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float* q = reinterpret_cast<const float*>(smem) + (wave * 16 + r) * 64 + lane;
        v[0][r] = (q[0] + q[R * R]) + (q[2 * R * R] + q[3 * R * R]);
        const float t = v[0][r] * 0.0f;
        if (!EDGE || (row_of(r) < p.m && col < p.n)) z = z + t;
    }
    // (Each wave's own block, over the whole chunk.)
    if (__any(z != 0.0f)) b3_redo<AM, BMD, 1>(p, A, B, m0 + bm * 32, n0 + bn * 32, klen, lane, v);
    float* C = p.partial != nullptr ? p.partial + static_cast<int64_t>(plane) * p.m * p.n
                                    : p.c + static_cast<int64_t>(bi) * p.c_sb;
    const int64_t c_sm = p.partial != nullptr ? static_cast<int64_t>(p.n) : p.c_sm;
    const int64_t c_sn = p.partial != nullptr ? 1 : p.c_sn;
    const float beta = p.partial != nullptr ? 0.0f : p.beta;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (EDGE && (row_of(r) >= p.m || col >= p.n)) continue;
        float* q = C + row_of(r) * c_sm + col * c_sn;
        float x = v[0][r];
        if (beta != 0.0f) x = beta * *q + x;
        *q = x;
    }
}

// gemm_f32_b3sk<AM, BMD, TURNS>: gemm_f32_sk's runs, slots and tickets (gemm_pipe.h) over the three-piece
// sums of full 128x128 tiles: each run's part of a tile is checked, and summed again where it must be, before
// it meets the other run's. One workgroup per compute unit. 48^6 in rank 4 (2304^3): 185 -> 147 us, 166 TFLOP/s,
// with one wave per SIMD, the matrix cores 47 % busy at 2.0 GHz; 2048^3, the same wave on whole tiles, 126 -> 95 us.
template <int AM, int BMD, B3Turns TURNS>
__global__ __launch_bounds__(256, 1) void gemm_f32_b3sk(GemmArgs p) {
    constexpr int FM = 2, FN = 2, RA = 128, RB = 128, SLOT = 128 * 128, STEP = 128;
    constexpr int ST = B3Geo<RA>::BYTES + B3Geo<RB>::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[2 * ST + 16];
    uint32_t& ticket = *reinterpret_cast<uint32_t*>(smem + 2 * ST);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const uint32_t G = gridDim.x, bid = blockIdx.x;
    const uint32_t xcd = bid & 7u, slot_in = bid >> 3, q8 = G >> 3, r8 = G & 7u;
    const uint32_t r = xcd < r8 ? xcd * (q8 + 1) + slot_in : r8 * (q8 + 1) + (xcd - r8) * q8 + slot_in;
    const uint32_t per_plane = p.tiles_m * p.tiles_n;
    const uint64_t T = static_cast<uint64_t>(per_plane) * p.batch;
    const uint32_t S = p.k / STEP;
    const uint64_t steps = T * S;
    uint64_t x = static_cast<uint64_t>(r) * steps / G;
    const uint64_t end = static_cast<uint64_t>(r + 1) * steps / G;

    while (x < end) {
        const uint64_t t = x / S;
        const uint32_t s0 = static_cast<uint32_t>(x - t * S);
        const uint32_t s1 = static_cast<uint32_t>(min(static_cast<uint64_t>(S), s0 + (end - x)));
        const uint32_t len = s1 - s0;
        const bool whole = len == S;
        const bool first_part = s0 > 0;            // the run started inside this tile
        const uint32_t b = first_part ? r : r + 1;  // the run boundary splitting the tile
        const uint32_t k0 = whole || first_part ? 0 : S - len;
        const uint32_t bi = static_cast<uint32_t>(t / per_plane);
        const uint32_t tp = static_cast<uint32_t>(t - static_cast<uint64_t>(bi) * per_plane);
        const uint32_t group = tp / (8 * p.tiles_n), first_m = group * 8;
        const uint32_t gm = min(p.tiles_m - first_m, 8u), in_group = tp - group * 8 * p.tiles_n;
        const uint32_t m0 = (first_m + in_group % gm) * RA, n0 = (in_group / gm) * RB;
        const uint32_t kb = k0 * STEP;
        const float* A = p.a + static_cast<int64_t>(bi) * p.a_sb + static_cast<int64_t>(kb) * p.a_sk;
        const float* B = p.b + static_cast<int64_t>(bi) * p.b_sb + static_cast<int64_t>(kb) * p.b_sk;
        floatx16 acc[FM][FN];
        b3_zero(acc);
        const uint32_t bad = b3_sums<AM, BMD, 2, 2, FM, FN, false, TURNS>(p, smem, A, B, m0, n0, len * STEP, false, wave, lane, acc);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            if ((bad >> i & 1u) != 0) {
                b3_redo<AM, BMD, FN>(p, A, B, m0 + ((wave >> 1) * FM + i) * 32, n0 + (wave & 1) * FN * 32, len * STEP, lane, acc[i]);
            }
        }
        if (whole) {
            pl_store_c<FN>(p, acc, bi, m0, n0);
        } else {
            float* mine = p.partial + static_cast<int64_t>(2 * b + (first_part ? 1 : 0)) * SLOT + tid;
            const float* other = p.partial + static_cast<int64_t>(2 * b + (first_part ? 0 : 1)) * SLOT + tid;
            bool done = false;
            if (!first_part) {
                if (tid == 0) {
                    ticket = __hip_atomic_load(p.counters + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __syncthreads();
                done = ticket == 1;  // the first part's sum is complete
                __syncthreads();     // every thread has read `ticket` before it is reused
            }
            if (!done) {
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            __hip_atomic_store(mine + ((i * FN + j) * 16 + e) * 256, acc[i][j][e],
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                wait_vm<0>();  // every store of this thread acknowledged
                __syncthreads();
                if (tid == 0) {
                    ticket = __hip_atomic_fetch_add(p.counters + b, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
                }
                __syncthreads();
                done = ticket == 1;
            }
            if (done) {
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            acc[i][j][e] = acc[i][j][e] + __hip_atomic_load(other + ((i * FN + j) * 16 + e) * 256,
                                                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                pl_store_c<FN>(p, acc, bi, m0, n0);
                if (tid == 0) __hip_atomic_store(p.counters + b, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        x += len;
        // Every wave is done with the stages, and with `ticket`, before the next tile's writes.
        wait_lgkm0();
        __syncthreads();
    }
}

}  // namespace gemm_detail
}  // namespace lg
