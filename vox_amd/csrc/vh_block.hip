// Launcher of k_block_tail.
#include "vh_block.hpp"
#include "vh_launch.hpp"

namespace vh {

bool block_tail_ok(int64_t R, int C, int inner, int ff) {
    return C == kTailC && R > 0 && R <= INT32_MAX && inner > 0 && inner % 256 == 0 && ff > 0 && ff % 256 == 0 &&
           block_tail_smem(inner, ff) <= 160 * 1024;
}
hipError_t launch_block_tail(const BlockTailArgs &a0, hipStream_t s) {
    BlockTailArgs a = a0;
    a.status = status_word();
    if (!block_tail_ok(a.R, kTailC, a.inner, a.ff) || !a.a16 || !a.wo || !a.w1 || !a.w2 || !a.lw || !a.lb || !a.x ||
        (a.nw && (!a.nb || !a.out16)) || !(a.eps > 0.0))
        return hipErrorInvalidValue;
    const size_t smem = block_tail_smem(a.inner, a.ff);
    const hipError_t e = ensure_smem(reinterpret_cast<const void *>(&k_block_tail), smem);
    return e != hipSuccess ? e : launch(k_block_tail, dim3(unsigned((a.R + 15) / 16)), dim3(512), smem, s, a);
}

}  // namespace vh
