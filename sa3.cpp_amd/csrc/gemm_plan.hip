// The DMA-fed GEMM's instantiations for the planned bf16 products (gemm_dma.h: PLAIN).
#include "gemm_dma.h"

namespace sa3k {

namespace {

template <bool KN, int PLAIN>
void launch_plan(sa3k_ctx* ctx, const DmaParams& p, const TilePlan& t) {
    const int s = t.splits;
    switch (t.tile) {
        case T32x64: return launch_dma<32, 64, 1, 4, true, 2, KN, 0, false, PLAIN>(ctx, p, s);
        case T32x128: return launch_dma<32, 128, 1, 4, true, 4, KN, 0, false, PLAIN>(ctx, p, s);
        case T64x64: return launch_dma<64, 64, 2, 4, true, 4, KN, 0, false, PLAIN>(ctx, p, s);
        case T64x128: return launch_dma<64, 128, 2, 3, true, 8, KN, 0, false, PLAIN>(ctx, p, s);
        case T64x256:
            if constexpr (!KN && PLAIN == 1)
                if (p.hp.parts > 0) return launch_dma<64, 256, 1, 3, true, 8, false, 0, true, PLAIN>(ctx, p, s);
            return launch_dma<64, 256, 1, 3, true, 8, KN, 0, false, PLAIN>(ctx, p, s);
        case T128x128: return launch_dma<128, 128, 2, 3, true, 8, KN, 0, false, PLAIN>(ctx, p, s);
        case T256x256: return gemm_launch_big(ctx, p, s);
        default: return gemm_launch_wide(ctx, p, s);
    }
}

}  // namespace

void gemm_launch_plan(sa3k_ctx* ctx, const DmaParams& p, const TilePlan& t) {
    if (p.b_kn) launch_plan<true, 1>(ctx, p, t);
    else if (p.Nx > 0) launch_plan<false, 2>(ctx, p, t);
    else launch_plan<false, 1>(ctx, p, t);
}

}  // namespace sa3k
