// The tile and split choice of bf16 products on the DMA-fed GEMM kernels: host arithmetic only, so
// that it compiles (and is checked) without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace sa3k {

// LDS of a workgroup of the DMA-fed kernels (a ring of `stages` K tiles, 128 bytes per operand row),
// and how many of them a CU's 160 KiB hold: the launchers' slots and the plan's both come from here
constexpr int kTileRowBytes = 128;
constexpr int dma_lds_bytes(int bm, int bn, int stages) { return stages * (bm + bn) * kTileRowBytes + 64; }
constexpr int dma_wg_per_cu(int bm, int bn, int stages) {
    return std::max(1, (160 * 1024) / dma_lds_bytes(bm, bn, stages));
}

// The tiles a bf16 product is cut into (gemm_dma.hip chooses, gemm_plan.hip launches)
enum TileId { T32x64, T32x128, T64x64, T64x128, T64x256, T128x128, T128x256, T256x256, kTiles };
struct TilePlan {
    TileId tile;
    int splits;
};

// What a bf16 launch is estimated to take, in us, from what its tiles measured on MI355X (f32
// output, K 768 to 12288, 77 to 4096 rows): per K tile of 64 a resident workgroup takes t1 alone on
// its CU and t2 beside a second one, and all of them together no less than their operand bytes at
// kOperandRate, the rate at which the caches feed the CUs' DMA. A round adds `fixed` for the launch,
// the first tile's latency and a lone epilogue.
// One workgroup per CU leaves the output stores of a round exposed (kStoreRate); two hide them behind
// each other's products. What the choice is about, K 1536: 343 x 1536 on 64 x 64 tiles 9.4 us, split
// in 6 on 128 x 128 with its reduction 16.9; 343 x 4608 on 64 x 128 12.2, 128 x 128 split in 2 21.7;
// 279 x 12288 on 64 x 256 or 128 x 256 20, 128 x 128 in two rounds 36; 2176 x 7680 on 128 x 256 64,
// 64 x 128 over 75; 2176 x 12288 on 256 x 256 104, 128 x 256 over 110. 64 x 128's t1 is what 132 to 144 of
// them took at K 6144 (31 to 32.5 us); at 0.28 they were preferred there to 128 x 128 split in 3 (2176 x
// 512, 700 x 1536, 343 x 3072: 26.7), and to 64 x 64 at 858 x 1024 x 1024 (9.9 against 8.0) or 128 x 7680 x
// 1536 (11.6 against 9.3).
struct TileCost {
    int lm, ln, stages;   // log2 of the tile's rows and columns, LDS stages
    double t1, t2, fixed;
    constexpr int rows() const { return 1 << lm; }
    constexpr int cols() const { return 1 << ln; }
    // resident workgroups per CU the estimate counts on: those that fit, of which more than two
    // gain nothing
    constexpr int per_cu() const { return std::min(2, dma_wg_per_cu(rows(), cols(), stages)); }
};
constexpr TileCost kTile[kTiles] = {
    {5, 6, 4, 0.200, 0.280, 3.0}, {5, 7, 4, 0.226, 0.226, 3.0}, {6, 6, 4, 0.207, 0.300, 3.5},
    {6, 7, 3, 0.300, 0.470, 3.0}, {6, 8, 3, 0.470, 0.470, 3.5}, {7, 7, 3, 0.470, 0.470, 4.0},
    {7, 8, 3, 0.580, 0.580, 6.0}, {8, 8, 2, 1.020, 1.020, 10.0}};
constexpr double kOperandRate = 14.2e6, kStoreRate = 5e6;   // bytes per us
// a separate kernel launch, and its rate over the bytes it moves
constexpr double kLaunch = 3.5, kPassRate = 5e6;

// (shifts and products by constants: a plan is worked out on the host for every launch)
inline double tile_us(const TileCost& c, int64_t tiles, int KT, int splits) {
    const int64_t n = tiles * splits;
    const int per_cu = c.per_cu(), ls = per_cu == 2 ? 9 : 8;   // log2 of the resident slots
    const int kt = splits == 1 ? KT : (int)((unsigned)(KT + splits - 1) / (unsigned)splits);
    const double bytes = (double)(c.rows() + c.cols()) * (128 / kOperandRate);
    const double out = per_cu == 1 ? (double)(1 << (c.lm + c.ln)) * (4 / kStoreRate) : 0.0;
    auto round = [&](int64_t w) {
        return kt * std::max(w > 256 ? c.t2 : c.t1, (double)w * bytes) + c.fixed + (double)w * out;
    };
    if (n <= (int64_t)1 << ls) return round(n);
    // two workgroups per CU drift apart, so a partly filled last round overlaps the one before it
    if (per_cu > 1) return round(512) * ((double)n * (1.0 / 512) + 0.3);
    const int64_t full = n >> ls, rest = n & 255;
    return (double)full * round(256) + (rest ? round(rest) : 0.0);
}

// The cheapest tile and split count of a bf16 Mt x Nt x K product under tile_us. A split pays for its
// partial sums and their reduction launch; tiles that cannot run an epilogue the caller asks for (the
// paired SwiGLU and the head preparation need 256 columns, the latter not 256 rows, and neither a
// split) pay for the separate kernel that replaces it. The layout of B has no say, so both layouts of
// one product sum alike. split: whether a split over K is allowed (then splits x tiles stays within
// the launch's resident workgroups); big: whether 256 x 256 tiles may be used.
inline TilePlan pick_plan(int64_t Mt, int64_t Nt, int64_t K, bool split, bool big, bool swiglu, bool heads,
                          double* est = nullptr) {
    const int KT = (int)(K / 64);
    const double out = (double)Mt * (double)Nt;
    TilePlan best{T128x256, 1};
    double best_us = 1e30;
    for (int i = 0; i < kTiles; ++i) {
        const TileCost& c = kTile[i];
        if (Mt <= 32 ? c.lm != 5 : c.lm == 5) continue;   // 32-row tiles where one holds every row
        if (i == T256x256 && !big) continue;
        const int64_t tiles = ((Mt + c.rows() - 1) >> c.lm) * ((Nt + c.cols() - 1) >> c.ln), slots = 256 * c.per_cu();
        const int most = split && KT >= 16 && tiles < slots
                             ? (int)std::min<int64_t>({(int64_t)16, KT / 4, slots / tiles}) : 1;
        // unsplit, split until the slots are full, and half of that
        const int counts[3] = {1, most / 2, most};
        for (int k = 0; k < (most > 1 ? 3 : 1); ++k) {
            const int s = counts[k];
            if (k && s < 2) continue;
            const bool fused = s == 1 && c.ln == 8;
            double us = tile_us(c, tiles, KT, s);
            if (s > 1) us += kLaunch + s * out * (8 / kPassRate);
            if (swiglu && !fused) us += kLaunch + out * (8 / kPassRate);
            if (heads && !(fused && c.lm != 8)) us += kLaunch + out * (10 / kPassRate);
            if (us < best_us) {
                best_us = us;
                best = TilePlan{(TileId)i, s};
            }
        }
    }
    if (est) *est = best_us;
    return best;
}

// What a bf16 product of M rows with at most 32 columns takes in launches of its own, in us: it streams
// its M x K operand at about 1 TB/s (measured on MI355X: 2176 x 32 x 1536 11.6, 2176 x 32 x 6144 42.7 with
// the reduction of its splits, which it needs past K 3072)
constexpr double kRankRate = 1e6;
inline double rank_product_us(int64_t M, int64_t K) {
    return kLaunch * (K > 3072 ? 2 : 1) + (double)M * (double)K * (2 / kRankRate);
}

// Whether Nx columns cost a bf16 M x N x K product less as extra output columns than as a product of
// their own, which runs beside it on the second stream at best, on the same CUs. Measured on MI355X
// against columns only where they cost at most 0.5 us: the DiT update (24 blocks of 1536, 2176 rows) 32.07
// -> 31.90 ms, 8 rank products a block instead of 11; the velocity of four such blocks, 1024 frames 1753
// -> 1679 us, 512 frames 1338 -> 1290. Charging a half or a fifth of the product measured the same.
inline bool extra_cols_pay(int64_t M, int64_t N, int64_t K, int64_t Nx, bool split, bool swiglu, bool heads) {
    double without = 0.0, with = 0.0;
    pick_plan(M, N, K, split, true, swiglu, heads, &without);
    pick_plan(M, N + Nx, K, split, true, swiglu, heads, &with);
    return with <= without + rank_product_us(M, K);
}

}  // namespace sa3k
