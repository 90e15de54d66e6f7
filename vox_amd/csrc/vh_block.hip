// Launcher of k_block_tail.
#include "vh_block.hpp"
#include "vh_launch.hpp"

namespace vh {

// The LDS is that of one block per 16 rows: launches without ws take it at any length. No length is too long: against the
// separate launches the estimator's step gains 1.26x at 20 frames, 1.21x at 512, 1.17-1.20x up to 2048 and 1.04-1.11x from
// there to 5000, where blocks come in several rounds.
bool block_tail_ok(int64_t R, int C, int inner, int ff) {
    return C == kTailC && R > 0 && R <= INT32_MAX && inner > 0 && inner % 256 == 0 && ff > 0 && ff % 256 == 0 &&
           block_tail_smem(inner, ff) <= 160 * 1024;
}
// Blocks per 16 rows, each with a part of the FFN: as many as 256 CUs hold at once (one each: its 146 registers leave a SIMD
// three waves, and a block is two a SIMD), where ff gives each whole passes of 256. In the flow estimator's step 4 instead of 1: 1024 rows 18.2 -> 15.6 us a launch, 202 rows 18.8 ->
// 13.7 (the step 2737 -> 2547 and 2235 -> 1939 us). Every block repeats the out-projection and its norm.
static int block_tail_parts(int64_t R, int ff) {
    const int64_t tiles = (R + 127) / 128 * 8;
    for (int ns : {4, 2})
        if (tiles * ns <= 256 && ff % (256 * ns) == 0) return ns;
    return 1;
}
// Tiles times parts are at most 256, tiles at most 128.
int64_t block_tail_ws() { return 256 * 16 * kTailC; }
int64_t block_tail_counts() { return 128; }
template <int NS>
static hipError_t block_tail(const BlockTailArgs &a, hipStream_t s) {
    const size_t smem = block_tail_smem(a.inner, a.ff / NS);
    const hipError_t e = ensure_smem(reinterpret_cast<const void *>(&k_block_tail<NS>), smem);
    const unsigned grid = NS == 1 ? unsigned((a.R + 15) / 16) : unsigned((a.R + 127) / 128 * 8 * NS);
    return e != hipSuccess ? e : launch(k_block_tail<NS>, dim3(grid), dim3(512), smem, s, a);
}
hipError_t launch_block_tail(const BlockTailArgs &a0, hipStream_t s) {
    BlockTailArgs a = a0;
    a.status = status_word();
    if (!block_tail_ok(a.R, kTailC, a.inner, a.ff) || !a.a16 || !a.wo || !a.w1 || !a.w2 || !a.lw || !a.lb || !a.x ||
        (a.nw && (!a.nb || !a.out16)) || !(a.eps > 0.0))
        return hipErrorInvalidValue;
    const int ns = a.ws && a.count ? block_tail_parts(a.R, a.ff) : 1;
    return ns == 4 ? block_tail<4>(a, s) : ns == 2 ? block_tail<2>(a, s) : block_tail<1>(a, s);
}

}  // namespace vh
