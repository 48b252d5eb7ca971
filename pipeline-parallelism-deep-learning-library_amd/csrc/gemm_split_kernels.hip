// Launches of the three-piece GEMM (gemm_split.h).
#include <hip/hip_runtime.h>

#include "gemm_split.h"

namespace lg {
namespace {

using namespace gemm_detail;

// How an operand's blocks are loaded. Only the unit stride counts: 128-bit loads need no more
// than the elements' own alignment.
int piece_mode(int64_t srow, int64_t sk) { return sk == 1 ? LOAD_K : srow == 1 ? LOAD_MN : LOAD_S; }

template <int AM, int BMD, int WM, int WN, int FM, int FN, bool EDGE>
void launch_tiles(hipStream_t s, const GemmArgs& a, uint32_t groups) {
    constexpr uint32_t TM = 32 * FM * WM, TN = 32 * FN * WN;
    if (a.tile != TM || a.tile_n != TN || (!EDGE && (a.m % TM != 0 || a.n % TN != 0 || a.k % B3_BK != 0)) ||
        (a.k_chunk % B3_BK != 0 && a.splits > 1)) {
        fail_invalid("three-piece GEMM launch does not match its tiles");
    }
    hipLaunchKernelGGL((gemm_f32_b3<AM, BMD, WM, WN, FM, FN, EDGE>), dim3(groups), dim3(64 * WM * WN), 0, s, a);
}

template <int AM, int BMD, bool EDGE>
void launch_kw(hipStream_t s, const GemmArgs& a, uint32_t groups) {
    if (a.tile != GEMM_SMALL_TILE || a.tile_n != GEMM_SMALL_TILE ||
        (!EDGE && (a.m % a.tile != 0 || a.n % a.tile_n != 0 || a.k % B3_BK != 0)) ||
        (a.k_chunk % B3_BK != 0 && a.splits > 1)) {
        fail_invalid("three-piece GEMM launch does not match its tiles");
    }
    hipLaunchKernelGGL((gemm_f32_b3kw<AM, BMD, EDGE>), dim3(groups), dim3(256), 0, s, a);
}

template <int AM, int BMD>
void launch_sk(hipStream_t s, const GemmArgs& a, uint32_t groups) {
    const uint64_t tiles = static_cast<uint64_t>(a.tiles_m) * a.tiles_n * a.batch;
    if (a.tile != GEMM_BM || a.tile_n != GEMM_BN || a.m % GEMM_BM != 0 || a.n % GEMM_BN != 0 || a.k % 128 != 0 ||
        a.splits != 1 || tiles < groups || groups != SK_RANGES || a.partial == nullptr || a.counters == nullptr) {
        fail_invalid("the stream-K GEMM needs full 128x128 tiles, at least one per range, K in whole steps "
                     "and its scratch");
    }
    if (a.k > B3_TURN_ALONE * B3_BK) {
        hipLaunchKernelGGL((gemm_f32_b3sk<AM, BMD, TURNS_AROUND>), dim3(groups), dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL((gemm_f32_b3sk<AM, BMD, TURNS_NONE>), dim3(groups), dim3(256), 0, s, a);
    }
}

}  // namespace

const char* launch_gemm_pieces(hipStream_t s, const GemmArgs& a, uint32_t groups) {
    const int am = piece_mode(a.a_sm, a.a_sk), bm = piece_mode(a.b_sn, a.b_sk);
    const bool full = a.m % a.tile == 0 && a.n % a.tile_n == 0 && a.k % B3_BK == 0;
#define LG_TILES(AMV, BMV, ...)                                \
    if (am == AMV && bm == BMV) {                               \
        launch_tiles<AMV, BMV, __VA_ARGS__>(s, a, groups);      \
    } else
    if (a.kernel == KERN_SK) {
#define LG_SK(AMV, BMV, NAME)                \
    if (am == AMV && bm == BMV) {             \
        launch_sk<AMV, BMV>(s, a, groups);    \
        return NAME;                          \
    }
        LG_SK(LOAD_K, LOAD_K, "gemm_f32_b3sk<K,K>")
        LG_SK(LOAD_K, LOAD_MN, "gemm_f32_b3sk<K,MN>")
        LG_SK(LOAD_MN, LOAD_K, "gemm_f32_b3sk<MN,K>")
        LG_SK(LOAD_MN, LOAD_MN, "gemm_f32_b3sk<MN,MN>")
#undef LG_SK
        fail_invalid("the stream-K GEMM needs a unit-stride axis in both operands");
    }
    if (a.tile == 256 && a.tile_n == 256) {
        LG_TILES(LOAD_K, LOAD_K, 2, 4, 4, 2, false)
        LG_TILES(LOAD_K, LOAD_MN, 2, 4, 4, 2, false) { fail_invalid("256x256 tiles need A contiguous along K"); }
        return bm == LOAD_K ? "gemm_f32_b3_256x256<K,K>" : "gemm_f32_b3_256x256<K,MN>";
    }
    if (a.tile == 256 && a.tile_n == 128) {
        LG_TILES(LOAD_K, LOAD_K, 4, 2, 2, 2, false)
        LG_TILES(LOAD_K, LOAD_MN, 4, 2, 2, 2, false) { fail_invalid("256x128 tiles need A contiguous along K"); }
        return bm == LOAD_K ? "gemm_f32_b3_256x128<K,K>" : "gemm_f32_b3_256x128<K,MN>";
    }
    static const char* const names[3][3] = {
        {"gemm_f32_b3<K,K>", "gemm_f32_b3<K,MN>", "gemm_f32_b3<K,S>"},
        {"gemm_f32_b3<MN,K>", "gemm_f32_b3<MN,MN>", "gemm_f32_b3<MN,S>"},
        {"gemm_f32_b3<S,K>", "gemm_f32_b3<S,MN>", "gemm_f32_b3<S,S>"}};
    static const char* const wide[2][2] = {{"gemm_f32_b3_128x256<K,K>", "gemm_f32_b3_128x256<K,MN>"},
                                           {"gemm_f32_b3_128x256<MN,K>", "gemm_f32_b3_128x256<MN,MN>"}};
    static const char* const kw[3][3] = {
        {"gemm_f32_b3kw<K,K>", "gemm_f32_b3kw<K,MN>", "gemm_f32_b3kw<K,S>"},
        {"gemm_f32_b3kw<MN,K>", "gemm_f32_b3kw<MN,MN>", "gemm_f32_b3kw<MN,S>"},
        {"gemm_f32_b3kw<S,K>", "gemm_f32_b3kw<S,MN>", "gemm_f32_b3kw<S,S>"}};
#define LG_KW(AMV, BMV, EDGEV)                      \
    if (am == AMV && bm == BMV) {                    \
        launch_kw<AMV, BMV, EDGEV>(s, a, groups);    \
    } else
    if (a.tile == GEMM_SMALL_TILE) {
        if (full && am != LOAD_S && bm != LOAD_S) {
            LG_KW(LOAD_K, LOAD_K, false)
            LG_KW(LOAD_K, LOAD_MN, false)
            LG_KW(LOAD_MN, LOAD_K, false)
            LG_KW(LOAD_MN, LOAD_MN, false) { fail_invalid("unknown operand load mode"); }
        } else {
            LG_KW(LOAD_K, LOAD_K, true)
            LG_KW(LOAD_K, LOAD_MN, true)
            LG_KW(LOAD_MN, LOAD_K, true)
            LG_KW(LOAD_MN, LOAD_MN, true)
            LG_KW(LOAD_K, LOAD_S, true)
            LG_KW(LOAD_MN, LOAD_S, true)
            LG_KW(LOAD_S, LOAD_K, true)
            LG_KW(LOAD_S, LOAD_MN, true)
            LG_KW(LOAD_S, LOAD_S, true) { fail_invalid("unknown operand load mode"); }
        }
        return kw[am][bm];
    }
#undef LG_KW
    if (a.tile_n == GEMM_WIDE_N) {
        LG_TILES(LOAD_K, LOAD_K, 2, 4, 2, 2, true)
        LG_TILES(LOAD_K, LOAD_MN, 2, 4, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_K, 2, 4, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_MN, 2, 4, 2, 2, true) { fail_invalid("128x256 tiles need unit-stride axes"); }
        return wide[am][bm];
    }
    if (full) {
        LG_TILES(LOAD_K, LOAD_K, 2, 2, 2, 2, false)
        LG_TILES(LOAD_K, LOAD_MN, 2, 2, 2, 2, false)
        LG_TILES(LOAD_MN, LOAD_K, 2, 2, 2, 2, false)
        LG_TILES(LOAD_MN, LOAD_MN, 2, 2, 2, 2, false)
        LG_TILES(LOAD_K, LOAD_S, 2, 2, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_S, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_K, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_MN, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_S, 2, 2, 2, 2, true) { fail_invalid("unknown operand load mode"); }
    } else {
        LG_TILES(LOAD_K, LOAD_K, 2, 2, 2, 2, true)
        LG_TILES(LOAD_K, LOAD_MN, 2, 2, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_K, 2, 2, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_MN, 2, 2, 2, 2, true)
        LG_TILES(LOAD_K, LOAD_S, 2, 2, 2, 2, true)
        LG_TILES(LOAD_MN, LOAD_S, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_K, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_MN, 2, 2, 2, 2, true)
        LG_TILES(LOAD_S, LOAD_S, 2, 2, 2, 2, true) { fail_invalid("unknown operand load mode"); }
    }
#undef LG_TILES
    return names[am][bm];
}

}  // namespace lg
