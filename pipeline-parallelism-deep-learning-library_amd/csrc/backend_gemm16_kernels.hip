// gfx950 kernel of the Backend's 16-bit gemm (F16 / BF16 tensors): CpuBackend's arithmetic,
// bit for bit.
//
// crates/cpu/src/lib.rs:270-291 runs `accumulate` (:664-691) with loaders that widen each
// element exactly to f32 and a store that rounds to 16 bits, so every output is
//   acc = beta == 0 ? +0 : beta * widen(C)                        (C unread when beta is 0)
//   if alpha != 0: for k ascending: acc = acc + (alpha * widen(A[row, k])) * widen(B[k, col])
//   C = narrow(acc)
// with one f32 rounding per multiply and per add, and narrow = the half crate's (2.7.1)
// from_f32_const: round to nearest even on the f32 bits, NaN kept quiet with its sign and top
// payload bits. Here each output is one lane's private f32 accumulator that sees exactly these
// operations in this order; the file is compiled with -ffp-contract=off, so no multiply and add
// fuse. alpha * widen(a) does not depend on the column, so it is formed once per A element as
// the slice is staged: the same rounding the loop performs at every use. That leaves one
// multiply and one add per term: fused on the f32 matrix cores where the product needs no rounding
// (gemm16_chain, below), else separate on the VALU (gemm16_seq).
//
// gemm16_seq's tiling: 128x128 outputs per 256-thread workgroup, 8x8 per thread as two 4-row by two
// 4-column blocks 64 apart, so each k costs a thread four 128-bit LDS reads (a wave's reads
// are 4 broadcast addresses of A and 16 consecutive 16-byte words of B: no bank conflicts) for
// 128 VALU operations; 64x64 tiles (4x4 per thread, two reads for 32 operations) where the
// 128x128 grid would leave compute units idle. K advances in slices of 16 staged in LDS as f32, [k][row] and
// [k][col], double buffered; the next slice's 16-bit elements are in flight in registers while
// the current slice is consumed. The last slice runs only its valid k: a padded term would
// add +0 (turning a -0 sum into +0) or 0 * inf.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lg_internal.h"

namespace lg {
namespace {

constexpr int QT = 256;  // threads per workgroup, 16 x 16
constexpr int QK = 16;   // K slice
// Square tiles of QM = 16 * TM outputs a side, TM x TM per thread as (TM/4)^2 blocks of 4x4
// whose rows and columns are 64 apart: TM = 8 (128x128 tiles), or TM = 4 (64x64 tiles, for
// grids that would leave compute units idle).
template <int TM>
struct Geo16 {
    static constexpr int QM = 16 * TM;       // output tile edge
    static constexpr int QP = QM + 4;        // LDS row pitch in floats: 16-byte rows, k rows 4 banks apart
    static constexpr int QL = QM * QK / QT;  // elements per thread and operand per slice
    static constexpr int NB = TM / 4;        // 4x4 blocks per thread along each axis
    static_assert((TM == 4 || TM == 8) && QL * QT == QM * QK, "whole slices per thread");
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Exact widening (every finite 16-bit value is an f32).
template <int HK>
__device__ inline float widen(uint16_t h) {
    if constexpr (HK == 1) return __builtin_bit_cast(float, static_cast<uint32_t>(h) << 16);
    else return static_cast<float>(__builtin_bit_cast(_Float16, h));
}

// f32 -> f16 bits as the half crate's f16::from_f32_const: ties to even on the f32 bits,
// f16 subnormals kept, overflow to infinity, NaN quiet (0x0200) with the top ten payload bits.
__device__ inline uint16_t to_f16(float v) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const uint32_t sign = (x >> 16) & 0x8000u, exp = (x >> 23) & 0xffu, man = x & 0x7fffffu;
    if (exp == 0xffu) return static_cast<uint16_t>(sign | 0x7c00u | (man ? 0x0200u | (man >> 13) : 0u));
    const int e = static_cast<int>(exp) - 112;  // the f16 biased exponent
    if (e >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
    if (e > 0) {
        // Normal: drop 13 bits; a round-up carry may ripple into the exponent (up to infinity).
        const uint32_t kept = sign | (static_cast<uint32_t>(e) << 10) | (man >> 13);
        const uint32_t rest = man & 0x1fffu;
        return static_cast<uint16_t>(kept + ((rest > 0x1000u || (rest == 0x1000u && (kept & 1u))) ? 1u : 0u));
    }
    const int shift = 14 - e;  // f16 subnormal: units of 2^-24
    if (shift > 24) return static_cast<uint16_t>(sign);
    const uint32_t sig = man | 0x800000u;
    const uint32_t kept = sig >> shift, rest = sig & ((1u << shift) - 1u), half = 1u << (shift - 1);
    return static_cast<uint16_t>(sign | (kept + ((rest > half || (rest == half && (kept & 1u))) ? 1u : 0u)));
}

// f32 -> bf16 bits as bf16::from_f32_const: the high half rounded to nearest even, NaN | 0x40.
__device__ inline uint16_t to_bf16(float v) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    if ((x & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((x >> 16) | 0x40u);
    return static_cast<uint16_t>((x + 0x7fffu + ((x >> 16) & 1u)) >> 16);
}

template <int HK>
__device__ inline uint16_t narrow(float v) {
    if constexpr (HK == 1) return to_bf16(v);
    else return to_f16(v);
}

// One operand's slice [k0, k0+QK) x [r0, r0+QM) into registers: element e of the slice is
// (k = e % QK, row = e / QK) when the operand is contiguous along K, else (k = e / QM,
// row = e % QM), so consecutive lanes read consecutive addresses either way. Outside the
// operand: 0 (never summed: rows past the edge are not stored, k past the end not run).
template <int TM, typename G = Geo16<TM>>
__device__ inline void load_slice(uint16_t (&r)[G::QL], const uint16_t* __restrict__ p, int64_t s_row,
                                  int64_t s_k, uint32_t kfast, uint32_t rows_left, uint32_t k0,
                                  uint32_t k, int tid) {
#pragma unroll
    for (int it = 0; it < G::QL; ++it) {
        const int e = it * QT + tid;
        const uint32_t kk = kfast ? e % QK : e / G::QM, row = kfast ? e / QK : e % G::QM;
        r[it] = (row < rows_left && k0 + kk < k)
                    ? p[static_cast<int64_t>(row) * s_row + static_cast<int64_t>(k0 + kk) * s_k]
                    : uint16_t(0);
    }
}

// Registers -> LDS stage [k][row] as f32, each value times `scale` (alpha for A, so the stage
// holds alpha*a rounded to f32; 1 for B, an exact copy).
template <int HK, bool SCALE, int TM, typename G = Geo16<TM>>
__device__ inline void stage_slice(float* __restrict__ st, const uint16_t (&r)[G::QL], uint32_t kfast,
                                   float scale, int tid) {
#pragma unroll
    for (int it = 0; it < G::QL; ++it) {
        const int e = it * QT + tid;
        const int kk = kfast ? e % QK : e / G::QM, row = kfast ? e / QK : e % G::QM;
        const float v = widen<HK>(r[it]);
        st[kk * G::QP + row] = SCALE ? scale * v : v;
    }
}

template <int HK, int TM>
__global__ __launch_bounds__(QT) void gemm16_seq(Gemm16SeqArgs p) {
    using G = Geo16<TM>;
    constexpr int QM = G::QM, QP = G::QP, QL = G::QL, NB = G::NB;
    __shared__ __attribute__((aligned(16))) float As[2][QK * QP];
    __shared__ __attribute__((aligned(16))) float Bs[2][QK * QP];
    const uint32_t tm = blockIdx.x / p.tiles_n, tn = blockIdx.x - tm * p.tiles_n;
    const uint32_t m0 = tm * QM, n0 = tn * QM;
    const uint32_t mrem = p.m - m0, nrem = p.n - n0;
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;

    // Output (i, j) of this thread: row ty*4 + i%4 + 64*(i/4), column tx*4 + j%4 + 64*(j/4).
    float acc[TM][TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const uint32_t row = ty * 4 + (i & 3) + 64 * (i >> 2);
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const uint32_t col = tx * 4 + (j & 3) + 64 * (j >> 2);
            acc[i][j] = 0.0f;
            if (p.beta != 0.0f && row < mrem && col < nrem) {
                acc[i][j] = p.beta * widen<HK>(p.c[static_cast<int64_t>(m0 + row) * p.c_sm + (n0 + col)]);
            }
        }
    }

    if (p.alpha != 0.0f && p.k > 0) {
        const uint16_t* A = p.a + static_cast<int64_t>(m0) * p.a_sm;
        const uint16_t* B = p.b + static_cast<int64_t>(n0) * p.b_sn;
        uint16_t ra[QL], rb[QL];
        const uint32_t ktiles = (p.k + QK - 1) / QK;
        load_slice<TM>(ra, A, p.a_sm, p.a_sk, p.a_kfast, mrem, 0, p.k, tid);
        load_slice<TM>(rb, B, p.b_sn, p.b_sk, p.b_kfast, nrem, 0, p.k, tid);
        stage_slice<HK, true, TM>(As[0], ra, p.a_kfast, p.alpha, tid);
        stage_slice<HK, false, TM>(Bs[0], rb, p.b_kfast, 1.0f, tid);
        __syncthreads();
        for (uint32_t kt = 0; kt < ktiles; ++kt) {
            const int s = kt & 1;
            const bool more = kt + 1 < ktiles;
            if (more) {
                load_slice<TM>(ra, A, p.a_sm, p.a_sk, p.a_kfast, mrem, (kt + 1) * QK, p.k, tid);
                load_slice<TM>(rb, B, p.b_sn, p.b_sk, p.b_kfast, nrem, (kt + 1) * QK, p.k, tid);
            }
            const float* as = As[s];
            const float* bs = Bs[s];
            auto term = [&](int kk) {
                float av[TM], bv[TM];
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    const f32x4 a4 = *reinterpret_cast<const f32x4*>(as + kk * QP + 64 * q + ty * 4);
                    const f32x4 b4 = *reinterpret_cast<const f32x4*>(bs + kk * QP + 64 * q + tx * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        av[4 * q + e] = a4[e];
                        bv[4 * q + e] = b4[e];
                    }
                }
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        const float prod = av[i] * bv[j];
                        acc[i][j] = acc[i][j] + prod;
                    }
            };
            const uint32_t klen = more ? QK : p.k - kt * QK;
            if (klen == QK) {
#pragma unroll
                for (int kk = 0; kk < QK; ++kk) term(kk);
            } else {
                for (uint32_t kk = 0; kk < klen; ++kk) term(static_cast<int>(kk));
            }
            if (more) {
                stage_slice<HK, true, TM>(As[s ^ 1], ra, p.a_kfast, p.alpha, tid);
                stage_slice<HK, false, TM>(Bs[s ^ 1], rb, p.b_kfast, 1.0f, tid);
            }
            __syncthreads();
        }
    }

#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const uint32_t row = ty * 4 + (i & 3) + 64 * (i >> 2);
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const uint32_t col = tx * 4 + (j & 3) + 64 * (j >> 2);
            if (row < mrem && col < nrem) {
                p.c[static_cast<int64_t>(m0 + row) * p.c_sm + (n0 + col)] = narrow<HK>(acc[i][j]);
            }
        }
    }
}

// gemm16_chain<HK, NB, AV, BV>: the same chain on the f32 matrix cores. v_mfma_f32_16x16x4_f32
// adds its four products to an output one after another in k order, each as one fused
// multiply-add with f32 subnormals kept (checked bit for bit against fmaf over 400 random
// tiles, subnormal sums among them). A fused multiply-add rounds as the chain's multiply and add do
// wherever the product itself needs no rounding, and that is the rule here: f16 elements have 11
// significant bits and bf16 ones 8, so (alpha * a) * b has at most 24 when alpha has at most 2 or 8
// (1, -0.5, 0.75, ...; the host's chain_fuses), and f16 products cannot leave f32's range. bf16
// ones can, so a slice that holds an |alpha * a| or |b| outside [2^-55, 2^62) that is not zero takes separate
// multiplies and adds from the same stage (multiply_odd), at the VALU's rate: softmax weights and small gradients
// are there as a matter of course. us, one such element / some in every slice / gemm16_seq: 2048 x 4096 x 1024
// 158 / 362 / 420 (160 without any), 1501 x 1477 x 1023 73 / 171 / 174 (70), 128 x 1408 x 1024 17 / 51 / 128 (14.2); with
// whole tiles computed again from memory 763 / 642, 354 / 360 and 185 / 186.
// A last slice that is not full is padded with products (-0) * 1: adding -0 changes no sum.
//
// 32 NB x 32 NB outputs per 256-thread workgroup, four waves in 2 x 2 of NB x NB blocks of 16x16. All
// threads load: each 16 k of one row, so a slice is 2048 / (32 NB) deep. Stages hold f32,
// [16 k][k % 4][row][k / 4], so a lane's four steps are one 128-bit read, lanes on distinct banks. Two stages, the
// loads of a slice one slice ahead of its conversion, in registers. Bound: the f32 matrix rate, 157 TFLOP/s. 2048 x 4096 x
// 1024 against the VALU kernel gemm16_seq: bf16 411 -> 156 us, f16 411 -> 159 us; 128 x 1408 x 1024, a few
// workgroups whose chains alone set the time, 146 -> 15 us on 32x32 tiles; 1501 x 1477 x 1023 with odd rows
// 187 -> 127 us with 16-bit loads, 66 with 128-bit ones of any alignment.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 128 bits that are only known to be 2-byte aligned (a global load needs no more).
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2)));
template <bool VEC>
struct Raw16 {
    u32x4 v[2];
};
template <>
struct Raw16<false> {
    uint16_t v[16];
};

template <int HK, int NB, bool AV, bool BV>
__global__ __launch_bounds__(256, 2) void gemm16_chain(Gemm16SeqArgs p) {
    constexpr int R = 32 * NB, BK = 2048 / R, KG = BK / 16;
    constexpr int OP = R * BK;  // floats of one operand's stage
    __shared__ __attribute__((aligned(16))) float stage[2][2 * OP];
    __shared__ uint32_t odd_slice[2];  // of each stage: 1 + the last slice with an element whose products may round
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, lr = lane & 15, lk = lane >> 4;
    // Tiles in groups of eight rows, each XCD (workgroups go round the eight in turn) a run of them.
    const uint32_t total = gridDim.x, xcd = blockIdx.x & 7u, q8 = total >> 3, r8 = total & 7u;
    const uint32_t lin = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (blockIdx.x >> 3);
    const uint32_t group = lin / (8 * p.tiles_n), gm = min(p.tiles_m - group * 8, 8u), in = lin - group * 8 * p.tiles_n;
    const uint32_t m0 = (group * 8 + in % gm) * R, n0 = (in / gm) * R;

    f32x4 acc[NB][NB];
    // Output (i, j, r) of this lane.
    const uint32_t row0 = m0 + wm * NB * 16 + lk * 4, col0 = n0 + wn * NB * 16 + lr;
    auto row_of = [&](int i, int r) { return row0 + i * 16 + r; };
    auto col_of = [&](int j) { return col0 + j * 16; };
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[i][j][r] = 0.0f;
                if (p.beta != 0.0f && row_of(i, r) < p.m && col_of(j) < p.n) {
                    acc[i][j][r] = p.beta * widen<HK>(p.c[static_cast<int64_t>(row_of(i, r)) * p.c_sm + col_of(j)]);
                }
            }
    if constexpr (HK == 1) {
        if (tid < 2) odd_slice[tid] = 0;
        __syncthreads();
    }
    const uint32_t slices = (p.k + BK - 1) / BK;
    auto loop = [&](auto vec, const uint16_t* src, int64_t s_row, int64_t s_k, uint32_t rows, float scale,
                    float pad, float* to) __attribute__((always_inline)) {
        constexpr bool VEC = decltype(vec)::value;
        // This thread's row of the tile and 16-k group of the slice: consecutive lanes along the
        // operand's contiguous axis. Rows past the end repeat the last one. Addresses are the slice's
        // (uniform) first element and a 32-bit offset of the lane's.
        const uint32_t t = tid & 127;
        const uint32_t row = s_k == 1 ? t / KG : t % R, kg = s_k == 1 ? t % KG : t / R;
        const uint32_t off = static_cast<uint32_t>(min(row, rows - 1) * s_row + kg * 16 * s_k) * 2u;
        float* mine = to + kg * 16 * R + row * 4;
        Raw16<VEC> x;
        auto load = [&](uint32_t s) __attribute__((always_inline)) {
            const char* base = reinterpret_cast<const char*>(src + static_cast<int64_t>(s) * BK * s_k);
            if ((s + 1) * BK <= p.k) {
                if constexpr (VEC) {
                    x.v[0] = *reinterpret_cast<const u32x4u*>(base + off);
                    x.v[1] = *reinterpret_cast<const u32x4u*>(base + 16 + off);
                } else {
#pragma unroll
                    for (int j = 0; j < 16; ++j) x.v[j] = *reinterpret_cast<const uint16_t*>(base + j * s_k * 2 + off);
                }
            } else {
                const uint32_t k = s * BK + kg * 16;
                if constexpr (VEC) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        uint32_t lo = 0, hi = 0;
                        if (k + 2 * j < p.k) lo = *reinterpret_cast<const uint16_t*>(base + 4 * j + off);
                        if (k + 2 * j + 1 < p.k) hi = *reinterpret_cast<const uint16_t*>(base + 4 * j + 2 + off);
                        x.v[j >> 2][j & 3] = lo | hi << 16;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        x.v[j] = 0;
                        if (k + j < p.k) x.v[j] = *reinterpret_cast<const uint16_t*>(base + j * s_k * 2 + off);
                    }
                }
            }
        };
        auto put = [&](uint32_t s) __attribute__((always_inline)) {
            const uint32_t k = s * BK + kg * 16;
            float f[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                uint16_t h;
                if constexpr (VEC) h = static_cast<uint16_t>(x.v[j >> 3][(j >> 1) & 3] >> (16 * (j & 1)));
                else h = x.v[j];
                f[j] = scale * widen<HK>(h);
            }
            if constexpr (HK == 1) {
                // One instruction an element for the least and the largest magnitude (NaNs do not count, nor need
                // they); where zeros or small elements are among them, the least that is not zero: twice its bits less
                // one, which makes zero the largest. (Four instructions an element for all: 4096^3 1185 -> 1162 us.)
                constexpr float LEAST = 0x1p-55f, LARGEST = 0x1p62f;
                float least = LARGEST, most = 0.0f;
#pragma unroll
                for (int j = 0; j < 16; j += 2) {
                    __asm__("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(least) : "v"(f[j]), "v"(f[j + 1]));
                    __asm__("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(f[j]), "v"(f[j + 1]));
                }
                if (__any(least < LEAST || most >= LARGEST)) {
                    uint32_t low = 0xffffffffu;
#pragma unroll
                    for (int j = 0; j < 16; ++j) low = min(low, (__builtin_bit_cast(uint32_t, f[j]) << 1) - 1);
                    if (__any(low < (__builtin_bit_cast(uint32_t, LEAST) << 1) - 1 || most >= LARGEST)) odd_slice[s & 1] = s + 1;
                }
            }
            if (k + 16 > p.k) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (k + j >= p.k) f[j] = pad;
            }
            float* q = mine + (s & 1) * 2 * OP;
#pragma unroll
            for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(q + c * 4 * R) = f32x4{f[c], f[4 + c], f[8 + c], f[12 + c]};
        };
        // A slice's fragments, read before the conversions of the next one and multiplied behind them.
        f32x4 fa[KG][NB], fb[KG][NB];
        auto read = [&](uint32_t s) __attribute__((always_inline)) {
            const float* as = stage[s & 1] + lk * 4 * R + (wm * NB * 16 + lr) * 4;
            const float* bs = stage[s & 1] + OP + lk * 4 * R + (wn * NB * 16 + lr) * 4;
#pragma unroll
            for (int g = 0; g < KG; ++g) {
#pragma unroll
                for (int i = 0; i < NB; ++i) fa[g][i] = *reinterpret_cast<const f32x4*>(as + g * 16 * R + i * 64);
#pragma unroll
                for (int j = 0; j < NB; ++j) fb[g][j] = *reinterpret_cast<const f32x4*>(bs + g * 16 * R + j * 64);
            }
        };
        auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < KG; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[g][i][e], fb[g][j][e], acc[i][j], 0, 0, 0);
                        }
        };
        // The same slice as the chain is written: k by k, the next one's operands (past the last the first's
        // again) read behind its sums.
        auto multiply_odd = [&](uint32_t s) __attribute__((always_inline)) {
            const float* as = stage[s & 1] + (wm * NB * 16 + lk * 4) * 4;
            const float* bs = stage[s & 1] + OP + (wn * NB * 16 + lr) * 4;
            float a[2][NB * 4], b[2][NB];
            auto read = [&](int k, int to) __attribute__((always_inline)) {
                const int at = (k >> 4) * 16 * R + (k & 3) * 4 * R + ((k >> 2) & 3);
#pragma unroll
                for (int i = 0; i < NB * 4; ++i) a[to][i] = as[at + ((i >> 2) * 16 + (i & 3)) * 4];
#pragma unroll
                for (int j = 0; j < NB; ++j) b[to][j] = bs[at + j * 64];
            };
            read(0, 0);
#pragma unroll 1
            for (int k = 0; k < BK; k += 4) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    read((k + u + 1) % BK, (u + 1) & 1);
#pragma unroll
                    for (int i = 0; i < NB * 4; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            const float prod = a[u & 1][i] * b[u & 1][j];
                            acc[i >> 2][j][i & 3] = acc[i >> 2][j][i & 3] + prod;
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        load(0);
        put(0);
        if (slices > 1) load(1);
        __syncthreads();
        auto next = [&](uint32_t s) __attribute__((always_inline)) {
            if (s + 1 < slices) put(s + 1);
            if (s + 2 < slices) load(s + 2);
        };
        uint32_t s = 0;
        if constexpr (HK == 0) {
            for (; s < slices; ++s) {
                read(s);
                next(s);
                multiply();
                __syncthreads();
            }
        } else while (s < slices) {
            bool odd = false;
            for (; s < slices && !odd; ++s) {
                const uint32_t last = odd_slice[s & 1];
                read(s);
                next(s);
                odd = __builtin_amdgcn_readfirstlane(last) == s + 1;
                if (odd) {
                    multiply_odd(s);
                    // The MFMAs that follow add (-0) * 1, which changes no sum. (A branch around them takes 4 % of all
                    // other slices' time.)
#pragma unroll
                    for (int g = 0; g < KG; ++g)
#pragma unroll
                        for (int i = 0; i < NB; ++i) {
                            fa[g][i] = f32x4{-0.0f, -0.0f, -0.0f, -0.0f};
                            fb[g][i] = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
                        }
                }
                multiply();
                __syncthreads();
            }
            // Where one slice holds such elements the next ones mostly do too.
            for (; s < slices && __builtin_amdgcn_readfirstlane(odd_slice[s & 1]) == s + 1; ++s) {
                next(s);
                multiply_odd(s);
                __syncthreads();
            }
        }
    };
    if (wave < 2 && p.alpha == 1.0f) {
        // (One multiplication an element less: 4096^3 1220 -> 1200 us.)
        loop(std::integral_constant<bool, AV>{}, p.a + static_cast<int64_t>(m0) * p.a_sm, p.a_sm, p.a_sk, p.m - m0,
             1.0f, -0.0f, stage[0]);
    } else if (wave < 2) {
        loop(std::integral_constant<bool, AV>{}, p.a + static_cast<int64_t>(m0) * p.a_sm, p.a_sm, p.a_sk, p.m - m0,
             p.alpha, -0.0f, stage[0]);
    } else {
        loop(std::integral_constant<bool, BV>{}, p.b + static_cast<int64_t>(n0) * p.b_sn, p.b_sn, p.b_sk, p.n - n0,
             1.0f, 1.0f, stage[0] + OP);
    }

#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (row_of(i, r) < p.m && col_of(j) < p.n) {
                    p.c[static_cast<int64_t>(row_of(i, r)) * p.c_sm + col_of(j)] = narrow<HK>(acc[i][j][r]);
                }
            }
}

// Whether (alpha * a) * b never needs rounding (see gemm16_chain): alpha has at most 2 (f16) or 8 (bf16)
// significant bits and a moderate exponent.
bool chain_fuses(uint32_t kind, float alpha) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, alpha);
    const int e = static_cast<int>((bits >> 23) & 0xffu) - 127;
    const uint32_t below = kind == 1 ? 0xffffu : 0x3fffffu;  // mantissa bits past the first 8, past the first 2
    return e >= -10 && e <= 30 && (bits & below) == 0;
}

template <int HK, int NB>
void launch_chain_nb(hipStream_t s, const Gemm16SeqArgs& a, uint32_t groups) {
    const bool av = a.a_sk == 1, bv = a.b_sk == 1;
    const dim3 grid(groups);
    if (av && bv) hipLaunchKernelGGL((gemm16_chain<HK, NB, true, true>), grid, dim3(256), 0, s, a);
    else if (av) hipLaunchKernelGGL((gemm16_chain<HK, NB, true, false>), grid, dim3(256), 0, s, a);
    else if (bv) hipLaunchKernelGGL((gemm16_chain<HK, NB, false, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((gemm16_chain<HK, NB, false, false>), grid, dim3(256), 0, s, a);
}

// The kernel's 32-bit offsets within a tile's slice.
bool chain_near(const Gemm16SeqArgs& a) {
    auto near = [](int64_t s_row, int64_t s_k) {
        const uint64_t r = static_cast<uint64_t>(s_row), k = static_cast<uint64_t>(s_k);
        return r < (1u << 22) && k < (1u << 22);
    };
    return near(a.a_sm, a.a_sk) && near(a.b_sn, a.b_sk);
}

// Launches the chain kernel; returns its name for the launch log.
template <int HK>
const char* launch_chain(hipStream_t s, Gemm16SeqArgs a) {
    // The largest tiles whose grid still gives every compute unit two workgroups; the
    // smallest ones for anything less.
    uint32_t tile = 128;
    while (tile > 32 && gemm16_seq_workgroups(a.m, a.n, tile) < 2 * GEMM16_SEQ_CUS) tile /= 2;
    a.tile = tile;
    a.tiles_m = (a.m + tile - 1) / tile;
    a.tiles_n = (a.n + tile - 1) / tile;
    const uint64_t groups = gemm16_seq_workgroups(a.m, a.n, tile);
    if (groups == 0 || groups * 256 > 0xffffffffull) fail_invalid("16-bit gemm grid exceeds one launch");
    const uint32_t g = static_cast<uint32_t>(groups);
    if (tile == 128) {
        launch_chain_nb<HK, 4>(s, a, g);
        return HK == 1 ? "gemm_bf16_chain128" : "gemm_f16_chain128";
    }
    if (tile == 64) {
        launch_chain_nb<HK, 2>(s, a, g);
        return HK == 1 ? "gemm_bf16_chain64" : "gemm_f16_chain64";
    }
    launch_chain_nb<HK, 1>(s, a, g);
    return HK == 1 ? "gemm_bf16_chain32" : "gemm_f16_chain32";
}

}  // namespace

uint64_t gemm16_seq_workgroups(uint32_t m, uint32_t n, uint32_t tile) {
    return static_cast<uint64_t>((m + tile - 1) / tile) * ((n + tile - 1) / tile);
}

void launch_gemm16_seq(Context* ctx, hipStream_t s, const Gemm16SeqArgs& args) {
    const uint64_t groups = static_cast<uint64_t>(args.tiles_m) * args.tiles_n;
    if ((args.tile != 64 && args.tile != 128) || groups == 0 ||
        groups != gemm16_seq_workgroups(args.m, args.n, args.tile) || groups * QT > 0xffffffffull) {
        fail_invalid("16-bit gemm grid does not match its extents");
    }
    const dim3 grid(static_cast<uint32_t>(groups));
    const char* name = args.kind == 1 ? "gemm_bf16_seq" : "gemm_f16_seq";
    if (args.k > 0 && chain_fuses(args.kind, args.alpha) && chain_near(args)) {
        name = args.kind == 1 ? launch_chain<1>(s, args) : launch_chain<0>(s, args);
    } else if (args.kind == 1) {
        if (args.tile == 64) {
            hipLaunchKernelGGL((gemm16_seq<1, 4>), grid, dim3(QT), 0, s, args);
        } else {
            hipLaunchKernelGGL((gemm16_seq<1, 8>), grid, dim3(QT), 0, s, args);
        }
    } else {
        if (args.tile == 64) {
            hipLaunchKernelGGL((gemm16_seq<0, 4>), grid, dim3(QT), 0, s, args);
        } else {
            hipLaunchKernelGGL((gemm16_seq<0, 8>), grid, dim3(QT), 0, s, args);
        }
    }
    check_hip(hipGetLastError(), name);
    note_launch(ctx, name);
}

}  // namespace lg
