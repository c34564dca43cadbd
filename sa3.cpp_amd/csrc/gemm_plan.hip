// The DMA-fed GEMM's instantiations for the planned bf16 products (gemm_dma.h: PLAIN).
#include "gemm_dma.h"

namespace sa3k {

namespace {

// one tile of the plan, with the stages it was planned with; WMW waves along its rows, NW in all
template <TileId T, int WMW, int NW, bool KN, int PLAIN, bool HP = false>
void launch_tile(sa3k_ctx* ctx, const DmaParams& p, int splits) {
    constexpr TileCost c = kTile[T];
    launch_dma<c.rows(), c.cols(), WMW, c.stages, true, NW, KN, 0, HP, PLAIN>(ctx, p, splits);
}

template <bool KN, int PLAIN>
void launch_plan(sa3k_ctx* ctx, const DmaParams& p, const TilePlan& t) {
    const int s = t.splits;
    switch (t.tile) {
        case T32x64: return launch_tile<T32x64, 1, 2, KN, PLAIN>(ctx, p, s);
        case T32x128: return launch_tile<T32x128, 1, 4, KN, PLAIN>(ctx, p, s);
        case T64x64: return launch_tile<T64x64, 2, 4, KN, PLAIN>(ctx, p, s);
        case T64x128: return launch_tile<T64x128, 2, 8, KN, PLAIN>(ctx, p, s);
        case T64x256:
            if constexpr (!KN)   // with extra columns too: an adapted QKV or cross-query product carries them
                if (p.hp.parts > 0) return launch_tile<T64x256, 1, 8, false, PLAIN, true>(ctx, p, s);
            return launch_tile<T64x256, 1, 8, KN, PLAIN>(ctx, p, s);
        case T128x128: return launch_tile<T128x128, 2, 8, KN, PLAIN>(ctx, p, s);
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
