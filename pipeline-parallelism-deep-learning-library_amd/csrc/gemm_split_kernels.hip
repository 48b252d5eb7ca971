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

}  // namespace

const char* launch_gemm_pieces(hipStream_t s, const GemmArgs& a, uint32_t groups) {
    const int am = piece_mode(a.a_sm, a.a_sk), bm = piece_mode(a.b_sn, a.b_sk);
    const bool full = a.m % a.tile == 0 && a.n % a.tile_n == 0 && a.k % B3_BK == 0;
#define LG_TILES(AMV, BMV, ...)                                \
    if (am == AMV && bm == BMV) {                               \
        launch_tiles<AMV, BMV, __VA_ARGS__>(s, a, groups);      \
    } else
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
