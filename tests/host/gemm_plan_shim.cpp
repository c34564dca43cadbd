// C entry points over the host-only tile and split choice of the DMA-fed GEMM, for the CPU tests.
#include "gemm_plan.h"

extern "C" {

// out: tile rows, tile columns, LDS stages, splits; returns the estimate in us
double plan(int64_t M, int64_t N, int64_t K, int split, int big, int swiglu, int heads, int* out) {
    double est = 0.0;
    const sa3k::TilePlan p = sa3k::pick_plan(M, N, K, split != 0, big != 0, swiglu != 0, heads != 0, &est);
    const sa3k::TileCost& c = sa3k::kTile[p.tile];
    out[0] = c.rows();
    out[1] = c.cols();
    out[2] = c.stages;
    out[3] = p.splits;
    return est;
}

// whether cols extra columns ride on the product; *own: what they take in launches of their own, us
int cols_pay(int64_t M, int64_t N, int64_t K, int64_t cols, int swiglu, int heads, double* own) {
    *own = sa3k::rank_product_us(M, K);
    return sa3k::extra_cols_pay(M, N, K, cols, true, swiglu != 0, heads != 0);
}
}
