// The DMA-fed GEMM kernels' dispatch (gemm_dma.h has the kernel): the 256 x 256 kernel, the tile and
// split choice, and the instantiations with every load path.
#include "gemm_dma.h"

namespace sa3k {

namespace {

// 256 x 256 tiles for bf16 operands, one workgroup of 8 waves per CU (128 KiB of LDS in two
// stages). Per K tile of 64 a CU then moves 64 KiB from L2 for 8.4 MFLOP, half the bytes per flop
// of two 128 x 128 workgroups (which need the CU's whole 64 B/clk vector-memory path at the MFMA
// peak), and its waves own 64 x 128 blocks (2 x 4 MFMA blocks of 32 x 32), which cut LDS reads per
// flop by a quarter against 64 x 64.
//
// Every operand load goes through a buffer descriptor with a 32-bit per-lane offset (no 64-bit
// pointers, which would not leave room for the 128 accumulator registers): host-checked extents
// below 4 GiB. A (q, wave) DMA slot covers 8 consecutive rows, so with M % 8 == 0 its rows all come
// from A or all from the extra rows Ax, a choice made per slot on the scalar unit. Rows past the
// end are clamped to the last valid row of the same source. The rank segment (K2 <= 64) has its
// own descriptors; its chunks past K2 get an offset beyond the descriptor extent, which loads zeros.
struct BigSeg {
    uint32_t off[4];
};

template <bool KN, int NW = 8, bool XE = false>   // XE: as for gemm_dma_kernel
__global__ __launch_bounds__(NW * 64) void gemm_big_kernel(DmaParams p) {
    constexpr int BM = 256, BN = 256, NT = NW * 64, WMW = 4;
    constexpr int WTM = BM / WMW, WTN = BN / (NW / WMW);   // 64 x 128 (8 waves), 64 x 64 (16)
    constexpr int FM = WTM / 32, FN = WTN / 32;             // MFMA blocks per wave
    constexpr int NA = BM * 8 / NT, NB = BN * 8 / NT;       // DMA chunks per thread and tile
    constexpr int RPQ = NT / 8;                             // tile rows per DMA slot q
    constexpr int LPT = NA + NB;
    constexpr int STAGES = 2;
    constexpr int STAGE_BYTES = (BM + BN) * kRow;           // 64 KiB
    constexpr int EROW = BN + 8;
    constexpr int ER = 64;                                  // epilogue rows staged per pass
    static_assert(ER * EROW * 4 <= STAGES * STAGE_BYTES, "epilogue staging does not fit");
    __shared__ __attribute__((aligned(1024))) char lds[STAGES * STAGE_BYTES];

    const int64_t Mt = p.Mp + p.Mx;
    const int tiles_m = (int)((Mt + BM - 1) / BM), tiles_n = (int)((p.Nt + BN - 1) / BN);
    // This workgroup's item (split z, tile bid). Dispatch deals workgroups out to the 8 XCDs
    // round-robin in linear order (x fastest), so XCD c runs the linear ids L with L % 8 == c; it
    // takes the contiguous run [c T/8, (c+1) T/8) of the T items in (split, raster) order, so the
    // tiles of one split's K range that share A rows and B panels run on one XCD and share its L2.
    const int nwg = gridDim.x;   // tiles rounded up to a multiple of 8
    const int L = blockIdx.x + nwg * blockIdx.y;
    const int item = (L & 7) * ((nwg * (int)gridDim.y) >> 3) + (L >> 3);
    const int z = __builtin_amdgcn_readfirstlane(item / nwg);   // uniform: scalar operands derive from it
    const int bid = __builtin_amdgcn_readfirstlane(item - z * nwg);
    if (bid >= tiles_m * tiles_n) return;
    constexpr int G = 8;
    const int per_group = G * tiles_n;
    const int group = bid / per_group;
    const int first_m = group * G;
    const int gsz = min(tiles_m - first_m, G);
    const int in_g = bid - group * per_group;
    const int tm = first_m + in_g % gsz, tn = in_g / gsz;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave % WMW) * WTM, wn0 = (wave / WMW) * WTN;

    const int KT = (int)(p.K / 64);
    const int kt0 = z * p.kps;
    const int Tm = max(0, min(KT, kt0 + p.kps) - kt0);
    const bool ext = p.K2 > 0 && z == (int)gridDim.y - 1;
    const int T = Tm + (ext ? 1 : 0);
    const uint32_t k0b = (uint32_t)kt0 * 128u;   // byte offset of the split's first K tile

    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
    const u32x4 rs_a = buffer_rsrc(p.A, p.a_bytes), rs_ax = buffer_rsrc(p.Ax, p.ax_bytes);
    const u32x4 rs_b = buffer_rsrc(p.B, p.b_bytes), rs_bx = buffer_rsrc(p.Bx, p.bx_bytes);
    // the rank segment's descriptors: [rows][ld2] bf16, K2 valid columns
    const uint32_t a2_bytes = p.K2 > 0 ? (uint32_t)(((p.M - 1) * p.lda2 + p.K2) * 2) : 0u;
    const uint32_t a2x_bytes = p.K2 > 0 && p.Mx > 0 ? (uint32_t)(((p.Mx - 1) * p.lda2x + p.K2) * 2) : 0u;
    const uint32_t b2_bytes = p.K2 > 0 ? (uint32_t)(((p.N - 1) * p.ldb2 + p.K2) * 2) : 0u;
    const u32x4 rs_a2 = buffer_rsrc(p.A2, a2_bytes), rs_a2x = buffer_rsrc(p.A2x, a2x_bytes);
    const u32x4 rs_b2 = buffer_rsrc(p.B2, b2_bytes);
    constexpr uint32_t kNoData = 0xFFFFFFF0u;   // past every extent: loads zeros

    // per-thread DMA sources: slot s = q * NT + tid of the A (B) region, row s / 8, chunk kc. The 8
    // rows of slot (q, wave) start at m0 + (NT / 8) q + 8 wave, so their source is decided from
    // wave-uniform values (Mp % 8 == 0 when there are extra rows).
    BigSeg ao, a2o, bo, b2o;
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        const int s = q * NT + tid, row = s >> 3, kc = (s & 7) ^ swz(row);
        int64_t gm = m0 + row;
        if (gm >= Mt) gm = Mt - 1;
        const bool x = gm >= p.Mp;
        const int64_t lr = x ? gm - p.Mp : min(gm, p.M - 1);
        ao.off[q] = (uint32_t)((lr * (x ? p.ldax : p.lda) + kc * 8) * 2);
        a2o.off[q] = kc * 8 < p.K2 ? (uint32_t)((lr * (x ? p.lda2x : p.lda2) + kc * 8) * 2) : kNoData;
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int s = q * NT + tid, row = s >> 3, kc = (s & 7) ^ swz(row);
        int64_t gn = tile_col(p, n0, row);
        if (gn >= p.Nt) gn = p.Nt - 1;
        bo.off[q] = gn < p.N ? (uint32_t)((gn * p.ldb + kc * 8) * 2) : (uint32_t)(((gn - p.N) * p.ldbx + kc * 8) * 2);
        b2o.off[q] = kc * 8 < p.K2 && gn < p.N ? (uint32_t)((gn * p.ldb2 + kc * 8) * 2) : kNoData;
    }
    // wave-uniform, fixed over the K loop: bit q set when slot q's B rows are extra columns (N % 8
    // == 0), resp. its A rows extra rows (M % 8 == 0)
    unsigned bx_mask = 0, x_mask = 0;
#pragma unroll
    for (int q = 0; q < NB; ++q)
        if (min(tile_col(p, n0, RPQ * q + 8 * wave), p.Nt - 1) >= p.N) bx_mask |= 1u << q;
#pragma unroll
    for (int q = 0; q < NA; ++q)
        if (min(m0 + RPQ * q + 8 * wave, Mt - 1) >= p.Mp) x_mask |= 1u << q;
    auto slot_bx = [&](int q) { return ((bx_mask >> q) & 1u) != 0; };
    if constexpr (KN) {
        // [K][N] B: slot s of the B region is sub-tile s / 512 (64 columns), row k = (s % 512) / 8 of
        // the K tile, logical chunk (s % 8) ^ swz(k); columns past N read a valid column. A wave's
        // slot q lies in one sub-tile; with extra columns (N % 64 == 0) a sub-tile at or past N reads
        // them from Bx, [K][Nx] with row pitch ldbx.
        bx_mask = 0;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int s = q * NT + tid, t = s >> 9, k = (s & 511) >> 3, kc = (s & 7) ^ swz(k);
            const bool extra = p.Nx > 0 && n0 + 64 * ((q * NT + wave * 64) >> 9) >= p.N;   // wave-uniform
            int64_t gn = n0 + 64 * t + 8 * kc;
            if (extra) {
                bx_mask |= 1u << q;
                int64_t gx = gn - p.N;
                if (gx + 8 > p.Nx) gx = p.Nx - 8;
                bo.off[q] = (uint32_t)(((int64_t)k * p.ldbx + gx) * 2);
            } else {
                if (gn + 8 > p.N) gn = p.N - 8;
                bo.off[q] = (uint32_t)(((int64_t)k * p.ldb + gn) * 2);
            }
        }
    }
    auto slot_x = [&](int q) { return ((x_mask >> q) & 1u) != 0; };

    auto issue = [&](auto s_c, int t) {
        constexpr uint32_t so_lds = (uint32_t)((decltype(s_c)::value % STAGES) * STAGE_BYTES);
        const uint32_t dst0 = lds_base + wave * 64 * 16 + so_lds;
        if (t < Tm) {
            const uint32_t so = k0b + (uint32_t)t * 128u;
#pragma unroll
            for (int q = 0; q < NA; ++q) dma16b(slot_x(q) ? rs_ax : rs_a, ao.off[q], so, dst0 + q * NT * 16);
            if constexpr (KN) {   // the K tile is a row offset of the [K][N] operand
                const uint32_t sob = (uint32_t)(((int64_t)kt0 + t) * 64 * p.ldb * 2);
                const uint32_t sobx = (uint32_t)(((int64_t)kt0 + t) * 64 * p.ldbx * 2);
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    dma16b(pick_rsrc(slot_bx(q), rs_bx, rs_b), bo.off[q], slot_bx(q) ? sobx : sob,
                           dst0 + BM * kRow + q * NT * 16);
            } else {
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    dma16b(pick_rsrc(slot_bx(q), rs_bx, rs_b), bo.off[q], so, dst0 + BM * kRow + q * NT * 16);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NA; ++q) dma16b(slot_x(q) ? rs_a2x : rs_a2, a2o.off[q], 0u, dst0 + q * NT * 16);
#pragma unroll
            for (int q = 0; q < NB; ++q) dma16b(rs_b2, b2o.off[q], 0u, dst0 + BM * kRow + q * NT * 16);
        }
    };

    typedef float accv __attribute__((__vector_size__(16 * sizeof(float))));
    accv acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    auto frag = [&](const char* base, int row, int kc) { return base + row * kRow + ((kc ^ swz(row)) << 4); };
    // two K steps of fragments at a time: the reads of steps 2-3 go out while steps 0-1 compute
    auto compute = [&](const char* As) {
        const char* Bs = As + BM * kRow;
        const int r = lane & 31, g = lane >> 5;
        bf16x8 af[2][FM], bfr[2][FN];
        auto load = [&](int ks, int slot) {
            const int kc = 2 * ks + g;
#pragma unroll
            for (int i = 0; i < FM; ++i) af[slot][i] = *reinterpret_cast<const bf16x8*>(frag(As, wm0 + 32 * i + r, kc));
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (KN) {
                    const int nb = wn0 + 32 * j;
                    const char* sub = Bs + (nb >> 6) * (64 * kRow);
                    const int nl = (nb & 63) + 16 * ((lane >> 4) & 1), kb = 16 * ks + 8 * g;
                    bfr[slot][j] = cat44(ld_tr(sub, kb, nl, lane), ld_tr(sub, kb + 4, nl, lane));
                } else {
                    bfr[slot][j] = *reinterpret_cast<const bf16x8*>(frag(Bs, wn0 + 32 * j + r, kc));
                }
            }
        };
        auto mma = [&](int slot) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[slot][i], bfr[slot][j], acc[i][j], 0, 0, 0);
        };
        load(0, 0);
        load(1, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (p.prio) __builtin_amdgcn_s_setprio(1);
        mma(0);
        load(2, 0);
        __builtin_amdgcn_sched_barrier(0);
        mma(1);
        load(3, 1);
        __builtin_amdgcn_sched_barrier(0);
        mma(0);
        mma(1);
        if (p.prio) __builtin_amdgcn_s_setprio(0);
    };

    if (T > 0) issue(IC<0>{}, 0);
    for (int t0 = 0; t0 < T; t0 += STAGES) {
        static_for<STAGES>([&](auto s) {
            const int t = t0 + decltype(s)::value;
            if (t >= T) return;
            wait_vmcnt<0>();   // tile t landed (the only DMA group in flight)
            __asm__ volatile("s_barrier" ::: "memory");   // visible to all waves; tile t-1 consumed
            if (t + 1 < T) issue(IC<decltype(s)::value + 1>{}, t + 1);
            compute(lds + decltype(s)::value * STAGE_BYTES);
        });
    }

    // staged epilogue only (the host routes outputs that do not allow 16-byte stores elsewhere);
    // fixed chunk column per thread as in gemm_dma_kernel
    auto out_row = [&](int v) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); };
    constexpr int CPR = BN / 4;
    static_assert(NT % CPR == 0, "a thread's chunk column must not change between rows");
    const int cq = (tid % CPR) * 4;
    const int64_t nq = tile_col(p, n0, cq);
    const EpiCols kq = epi_cols(p, nq);
    const bool sw_tile = p.sw_half > 0 && n0 < 2 * p.sw_half;   // workgroup-uniform
    epi_cols_ready(kq);
    float* st = reinterpret_cast<float*>(lds);
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < BM; rb += ER) {
        if (wm0 == rb) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int c = wn0 + 32 * j + (lane & 31);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v) st[(32 * i + out_row(v)) * EROW + c] = acc[i][j][v];
            }
        }
        __syncthreads();
        staged_store<BN, NT, ER, EROW, false, XE>(p, st, m0, n0, rb, Mt, z, tid, cq, nq, kq, sw_tile, false,
                                              HeadPrepLane{}, nullptr);
        if (rb + ER < BM) __syncthreads();
    }
}

// Whether a bf16 product of Mt x Nt x K takes the 256 x 256 tiles (one workgroup per CU): where
// they fill the chip about as evenly as 128 x 128 tiles (two per CU) do, or with option gemm_big 3
// for K >= 8192 (they need no split over K there, or fewer), always with gemm_big 2. Measured on
// MI355X at 2176 rows: FFN up-projection 2176 x 12288 x 1536 107 vs 111 us, 2176 x 6144 x 1536 52
// vs 56 us, 8192^3 877 vs 1057 us; the 2176 x 7680 QKV projection (270 tiles) 98 vs 62 us.
bool use_big_tiles(const sa3k_ctx* ctx, int64_t Mt, int64_t Nt, int64_t K) {
    if (ctx->gemm_big == 0 || Mt <= 32 || Nt <= 64) return false;
    const int64_t t256 = ceil_div(Mt, 256) * ceil_div(Nt, 256), t128 = ceil_div(Mt, 128) * ceil_div(Nt, 128);
    const double q256 = (double)t256 / (double)(ceil_div(t256, 256) * 256);
    const double q128 = (double)t128 / (double)(ceil_div(t128, 512) * 512);
    return ctx->gemm_big == 2 || (t256 >= 200 && q256 >= q128 - 0.02) || (ctx->gemm_big == 3 && K >= 8192);
}

// Whether gemm_big_kernel can take this bf16 product: every extent addressable by a buffer
// descriptor, no in-kernel split reduction.
bool big_ok(const sa3k_ctx* ctx, const DmaParams& p) {
    auto extent = [&](int64_t rows, int64_t ld, int64_t k) -> int64_t { return rows > 0 ? ((rows - 1) * ld + k) * 2 : 0; };
    const int64_t lim = (int64_t)1 << 31;
    if (ctx->gemm_fixup != 0 || p.prescale) return false;
    if (extent(p.M, p.lda, p.K) >= lim || extent(p.N, p.ldb, p.K) >= lim) return false;
    if (p.b_kn && p.K * p.ldb * 2 >= lim) return false;
    if (p.Nx > 0 && (p.N % 8 != 0 || extent(p.Nx, p.ldbx, p.K) >= lim)) return false;
    if (p.b_kn && p.Nx > 0 && (p.N % 64 != 0 || p.Nx % 8 != 0 || (p.K - 1) * p.ldbx * 2 + p.Nx * 2 >= lim)) return false;
    if (p.Mx > 0 && extent(p.Mx, p.ldax, p.K) >= lim) return false;
    if (p.K2 > 0 && (extent(p.M, p.lda2, p.K2) >= lim || extent(p.N, p.ldb2, p.K2) >= lim ||
                     (p.Mx > 0 && extent(p.Mx, p.lda2x, p.K2) >= lim)))
        return false;
    return true;
}

// outputs allow the staged epilogue's 4-column stores: rows and vectors 16-byte (f32) / 8-byte
// (bf16) aligned
bool vec_epi_ok(const DmaParams& p) {
    auto ok = [](const void* q, int64_t ld, int align) {
        return q == nullptr || (ld % 4 == 0 && (uintptr_t)q % (uintptr_t)align == 0);
    };
    return p.N % 4 == 0 && p.Nt % 4 == 0 && ok(p.C, p.ldc, 16) && ok(p.U, p.ldu, 16) && ok(p.Ub, p.ldu, 8) &&
           ok(p.Cb, p.ldcb, 8) && ok(p.Cx, p.ldcx, 16) && ok(p.Cbx, p.ldcx, 8) && ok(p.colscale, 4, 16) &&
           ok(p.bias, 4, 16) && ok(p.Cbn, p.ldcn, 8);
}

}  // namespace

void gemm_launch_big(sa3k_ctx* ctx, DmaParams p, int chosen) {
    constexpr int BM = 256, BN = 256;
    const int64_t tiles = ceil_div(p.Mp + p.Mx, BM) * ceil_div(p.Nt, BN);
    const int64_t grid = ceil_div(tiles, 8) * 8;
    const int KT = (int)(p.K / 64);
    const int64_t slots = 256;   // one workgroup per CU (128 KiB of LDS)
    static_assert(kTile[T256x256].per_cu() == 1, "the plan's slots of the 256 x 256 tiles");
    static_assert((int64_t)256 * 256 * 256 <= kMaxSplitFloats, "256 x 256 split partials exceed kMaxSplitFloats");
    const int splits = split_count(ctx, tiles, slots, KT, &p.kps, chosen);
    p.ws = nullptr;
    p.counters = nullptr;
    auto extent = [&](int64_t rows, int64_t ld) -> uint32_t { return rows > 0 ? (uint32_t)(((rows - 1) * ld + p.K) * 2) : 0u; };
    p.a_bytes = extent(p.M, p.lda);
    p.ax_bytes = extent(p.Mx, p.ldax);
    p.b_bytes = extent(p.N, p.ldb);
    p.bx_bytes = extent(p.Nx, p.ldbx);
    if (p.b_kn) p.b_bytes = (uint32_t)(p.K * p.ldb * 2);   // the whole [K][ldb] operand (big_ok: < 2 GiB)
    if (p.b_kn && p.Nx > 0) {   // [K][Nx] extra columns (big_ok: N % 64 == 0, within reach)
        SA3K_REQUIRE(p.N % 64 == 0 && p.Nx % 8 == 0 && p.Nx <= p.ldbx, "[K][N] extra columns need N % 64 == 0");
        p.bx_bytes = (uint32_t)(((p.K - 1) * p.ldbx + p.Nx) * 2);
    }
    p.nt_store = ctx->gemm_nt_store;
    p.vec_epi = 1;
    settle_swiglu(p, BN, splits, p.b_kn != 0, 0);
    if (!p.b_kn) {   // the backward epilogues: [K][N] instantiations only, as in launch_dma
        p.ad.doh = nullptr;
        p.sb.du = nullptr;
    }
    settle_bwd_epilogues(p, splits, BN);
    const bool xe = p.ad.doh || p.sb.du;
    if (splits > 1) p.ws = gemm_workspace_bytes(ctx, (size_t)splits * (size_t)(p.Mp + p.Mx) * (size_t)p.Nt * sizeof(float));
    {
        KernelScope ks(ctx, p.b_kn ? "gemm_big<256,256,kn,bf16>" : "gemm_big<256,256,bf16>",
                       2.0 * (double)(p.M + p.Mx) * (double)p.Nt * (double)(p.K + p.K2));
        // 16 waves of 64 x 64 (four per SIMD); option gemm_cfg 4: 8 waves of 64 x 128 (the DiT update
        // 32.90 against 33.08 ms on one box)
        const dim3 g((unsigned)grid, (unsigned)splits);
        if (ctx->gemm_cfg == 4) {
            if (p.b_kn) launch_k(ctx, splits == 1, xe ? gemm_big_kernel<true, 8, true> : gemm_big_kernel<true, 8>, g,
                                 dim3(512), 0, p);
            else launch_k(ctx, splits == 1, gemm_big_kernel<false, 8>, g, dim3(512), 0, p);
        } else {
            if (p.b_kn) launch_k(ctx, splits == 1, xe ? gemm_big_kernel<true, 16, true> : gemm_big_kernel<true, 16>, g,
                                 dim3(1024), 0, p);
            else launch_k(ctx, splits == 1, gemm_big_kernel<false, 16>, g, dim3(1024), 0, p);
        }
        SA3K_LAUNCHED();
    }
    if (splits > 1) {
        KernelScope ks(ctx, "gemm_splitk_reduce");
        const int64_t items = p.vec_epi ? (p.Mp + p.Mx) * p.Nt / 4 : (p.Mp + p.Mx) * p.Nt;
        launch_k(ctx, true, gemm_dma_splitk_reduce, dim3((unsigned)ceil_div(items, kThreads)), dim3(kThreads), 0, p,
                 splits);
        SA3K_LAUNCHED();
    }
}

namespace {

// Whether a bf16 product can take the PLAIN instantiations: every operand within the 32-bit offsets
// of a buffer descriptor, extra rows, extra columns (beside a [N][K] B) and a second segment one at a
// time, as the default schedule has them, and none of the backward epilogues (off by default).
bool plain_ok(const DmaParams& p) {
    auto fits = [](int64_t rows, int64_t ld, int64_t k) { return ((rows - 1) * ld + k) * 2 < ((int64_t)1 << 32) - 256; };
    if (p.bq != 0 || (p.Nx != 0 && (p.b_kn || p.K2 > 0 || p.Mx > 0 || !fits(p.Nx, p.ldbx, p.K))) || p.ad.doh || p.sb.du || p.M <= 0 || p.K <= 0) return false;
    if (!fits(p.M, p.lda, p.K) || (p.Mx > 0 && (p.K2 > 0 || !fits(p.Mx, p.ldax, p.K)))) return false;
    if (p.b_kn ? !fits(p.K, p.ldb, p.ldb) : !fits(p.N, p.ldb, p.K)) return false;
    return p.K2 == 0 || (fits(p.M, p.lda2, p.K2) && fits(p.N, p.ldb2, p.K2));
}

// the plan applies where no option asks for a particular tile family
bool planned(const sa3k_ctx* ctx) {
    return ctx->gemm_small == 4 && (ctx->gemm_cfg == 0 || ctx->gemm_cfg == 4) && ctx->gemm_big == 3 && ctx->gemm_splits == 0 &&
           ctx->gemm_wg_per_cu == 0;
}

}  // namespace

void gemm_launch_wide(sa3k_ctx* ctx, const DmaParams& p, int chosen) {
    const bool eight = ctx->gemm_cfg == 4;   // 8 waves in place of 16
    if (p.b_kn) {
        if (eight) return launch_dma<128, 256, 2, 3, true, 8, true>(ctx, p, chosen);
        return launch_dma<128, 256, 2, 3, true, 16, true>(ctx, p, chosen);
    }
    if (p.hp.parts > 0) {   // falls back to the plain epilogue where headprep_ok refuses
        if (eight) return launch_dma<128, 256, 2, 3, true, 8, false, 0, true>(ctx, p, chosen);
        return launch_dma<128, 256, 2, 3, true, 16, false, 0, true>(ctx, p, chosen);
    }
    if (eight) return launch_dma<128, 256, 2, 3, true, 8>(ctx, p, chosen);
    return launch_dma<128, 256, 2, 3, true, 16>(ctx, p, chosen);
}

namespace {

// [K][N] B operands (bf16): the tiles of the default dispatch that have whole 64-column sub-tiles
void dispatch_dma_kn(sa3k_ctx* ctx, const DmaParams& p) {
    const int64_t Mt = p.Mp + p.Mx;
    if (planned(ctx) && p.N > 64 && plain_ok(p))
        return gemm_launch_plan(ctx, p, pick_plan(Mt, p.Nt, p.K, ctx->gemm_split, big_ok(ctx, p) && vec_epi_ok(p), false, false));
    if (use_big_tiles(ctx, Mt, p.N, p.K) && big_ok(ctx, p) && vec_epi_ok(p)) return gemm_launch_big(ctx, p, 0);
    if (Mt <= 32) return launch_dma<32, 128, 1, 4, true, 4, true>(ctx, p);
    if (p.N <= 64) return launch_dma<128, 64, 4, 4, true, 4, true>(ctx, p);
    const int64_t tiles128 = ceil_div(Mt, 128) * ceil_div(p.N, 128);
    if (tiles128 < 384 && p.K < 4096 && ctx->gemm_small == 2) return launch_dma<64, 128, 1, 3, true, 4, true>(ctx, p);
    if (tiles128 < 384 && ctx->gemm_small == 4) return launch_dma<128, 128, 2, 3, true, 8, true>(ctx, p);
    if (ctx->gemm_cfg == 1) return launch_dma<128, 128, 2, 2, true, 4, true>(ctx, p);
    return gemm_launch_wide(ctx, p, 0);
}

// B decoded from f16 / Q8_0 on its way into the MFMAs (bf16 A): the short-K small-grid tile of the
// bf16 dispatch, else 128 x 256 tiles with the 8 waves side by side along N (128 x 32 each), so
// every B fragment is decoded by one wave only (measured on MI355X, 2176 x 6144 x 1536 over Q8_0:
// 91.5 us against 107.5 us with 2 x 4 waves of 64 x 64, whose two wave rows decode each fragment);
// option gemm_dq 2 keeps the 2 x 4 layout. Both sum every output in the same order. These tiles split
// over K by their own rule (split_count): the planned count of the product over a bf16 copy belongs to
// smaller tiles and leaves these on few CUs (512 x 1536 x 6144 over Q8_0: 24 of 256, 165 us against 50
// split in 10; 2 x 7040 x 1728 37 against 20).
template <int BQ>
void dispatch_dma_dq(sa3k_ctx* ctx, const DmaParams& p) {
    const int64_t tiles128 = ceil_div(p.M, 128) * ceil_div(p.N, 128);
    // (decoded B: the 64 x 128 tile, whose four waves side by side along N decode each fragment once)
    if (tiles128 < 384 && p.K < 4096 && (ctx->gemm_small == 2 || ctx->gemm_small == 4))
        return launch_dma<64, 128, 1, 3, true, 4, false, BQ>(ctx, p);
    if (ctx->gemm_dq == 2) return launch_dma<128, 256, 2, 3, true, 8, false, BQ>(ctx, p);
    return launch_dma<128, 256, 1, 3, true, 8, false, BQ>(ctx, p);
}

template <bool BF16>
void dispatch_dma(sa3k_ctx* ctx, const DmaParams& p) {
    if constexpr (BF16) {
        if (planned(ctx) && p.bq == 0 && !p.b_kn && p.Nt > 64 && plain_ok(p))
            return gemm_launch_plan(ctx, p, pick_plan(p.Mp + p.Mx, p.Nt, p.K, ctx->gemm_split,
                                                        big_ok(ctx, p) && vec_epi_ok(p), p.sw_half > 0, p.hp.parts > 0));
        // per-head q/k preparation: 128 x 256 tiles
        if (p.hp.parts > 0 && p.bq == 0 && !p.b_kn) return gemm_launch_wide(ctx, p, 0);
        if (p.bq == 1) return dispatch_dma_dq<1>(ctx, p);
        if (p.bq == 2) return dispatch_dma_dq<2>(ctx, p);
        if (p.b_kn) return dispatch_dma_kn(ctx, p);
        if (use_big_tiles(ctx, p.Mp + p.Mx, p.Nt, p.K) && big_ok(ctx, p) && vec_epi_ok(p)) return gemm_launch_big(ctx, p, 0);
    }
    const int64_t Mt = p.Mp + p.Mx;
    if (Mt <= 32) return launch_dma<32, 128, 1, 4, BF16>(ctx, p);
    if (p.Nt <= 32) return launch_dma<128, 32, 4, 4, BF16>(ctx, p);
    if (p.Nt <= 64) return launch_dma<128, 64, 4, 4, BF16>(ctx, p);
    // bf16 from here on: what the plan does not take (an option that forces a tile family, a second
    // segment beside extra rows, operands past 4 GiB). Grids of 128x128 tiles that leave a quarter of
    // the two-per-CU slots idle: no split, on 128 x 128 tiles with eight waves in one workgroup per CU
    // (three stages, 96 KiB), at any K (measured on MI355X: 2176 x 1536 x 1536 21.4 us against 23.6 us on 64 x 128 tiles and 31.1 us
    // on the default tile split over K; 2176 x 1536 x 6144 67.7 against 71.1 us split over K; the
    // DiT update 34.56 against 35.16 ms with the short-K products alone, then 33.66 against 33.97 ms
    // with the long-K ones too). f32 with a short K: 64 x 128 tiles, no split.
    const int64_t tiles128 = ceil_div(Mt, 128) * ceil_div(p.Nt, 128);
    if constexpr (BF16)
        if (tiles128 < 384 && ctx->gemm_small == 4) return launch_dma<128, 128, 2, 3, true, 8>(ctx, p);
    // f32: bound by the f32 MFMA, so what counts is the busiest CU's share of the output. 64 x 64 tiles
    // where 64 x 128 ones fill the CUs unevenly (measured on MI355X, 2048 x 1536 x 1536: 768 tiles of 64 x
    // 64, three on each CU, 80 us; 384 of 64 x 128, two on half of them, 109 us; 1000 x 9216 x 6144 895
    // against 1214 on split 128 x 128 tiles; none of 120 shapes of 77 to 4096 rows, 512 to 9216 columns
    // and K 512 to 6144 slower by over 2%), and where the 128 x 128 ones, two to a CU, leave a last round
    // part empty: a CU that gets two of its tiles makes it a full round, so their share is 8 64 x 64 tiles
    // a round. An eighth less is asked for, and K 1024: 2048 x 9216 x 6144 (18 against 24) 1989 -> 1829
    // us, an f32 lora linear of 2048 tokens, 6144 to 9216, forward and backward 4497 -> 3819; 4096 x 9216 x
    // 1536 (36 against 40) would go 924 -> 949.
    if constexpr (!BF16) {
        const int64_t n128 = ceil_div(Mt, 64) * ceil_div(p.Nt, 128), n64 = ceil_div(Mt, 64) * ceil_div(p.Nt, 64);
        const int64_t share = ceil_div(n64, 256);
        const bool part_round = tiles128 >= 512 && p.K >= 1024 && 8 * share <= 7 * 8 * ceil_div(tiles128, 512);
        if (ctx->gemm_small == 4 && ctx->gemm_cfg == 0 && n128 >= 256 && (share < 2 * ceil_div(n128, 256) || part_round))
            return launch_dma<64, 64, 2, 3, false>(ctx, p);
    }
    if (tiles128 < 384 && p.K < (BF16 ? 4096 : 2048)) {
        switch (ctx->gemm_small) {
            case 1: return launch_dma<64, 128, 2, 2, BF16>(ctx, p);
            case 2: case 4: return launch_dma<64, 128, 1, 3, BF16>(ctx, p);
            case 3: return launch_dma<128, 64, 2, 2, BF16>(ctx, p);
            default: break;
        }
    }
    // bf16: 128 x 256 tiles (the plan's too), three stages in 144 KiB of LDS (one workgroup per CU), 16 waves of
    // 64 x 32 (four per SIMD, to hide the DMA and LDS latency behind each other's MFMAs). Against
    // two 128 x 128 workgroups per CU the tile moves a quarter fewer operand bytes per flop through
    // the CU's vector-memory path, which the MFMA rate otherwise saturates (measured on MI355X at
    // 2176 rows, 8 waves: QKV 2176 x 7680 x 1536 58.2 vs 64.7 us, 2176 x 3072 x 1536 27.4 vs
    // 31.0 us, the split-K products 2176 x 1536 x 6144 / 7680 / 12288 53.4 / 63.5 / 93.5 vs
    // 59.4 / 70.7 / 102.2 us); 16 waves against 8 (option gemm_cfg 4): 2176 x 7680 x 1536 with f32
    // output 76.7 vs 86.6 us, the DiT update 34.57 vs 35.00 ms.
    switch (ctx->gemm_cfg) {
        case 1: return launch_dma<128, 128, 2, 2, BF16>(ctx, p);    // 64 KiB LDS: two workgroups per CU
        case 4:
            if constexpr (BF16) return gemm_launch_wide(ctx, p, 0);
            else return launch_dma<128, 256, 2, 3, false, 8>(ctx, p);
        case 7: return launch_dma<128, 256, 2, 2, BF16, 8>(ctx, p);
        default:
            if constexpr (BF16) return gemm_launch_wide(ctx, p, 0);
            else return launch_dma<128, 128, 2, 2, false>(ctx, p);
    }
}

// Rounds of resident workgroups a bf16 DMA GEMM of Mt x Nt x K takes on the tile families of the
// dispatch above that do not go by estimated time (options that force one, a [K][N] B with extra
// columns), ignoring operand alignment: splits x tiles / slots, rounded up.
int64_t dma_rounds(const sa3k_ctx* ctx, int64_t Mt, int64_t Nt, int64_t K) {
    const int KT = (int)(K / 64);
    auto rounds = [&](int64_t tiles, int64_t slots) {
        return ceil_div(tiles * split_count(ctx, tiles, slots, KT, nullptr), slots);
    };
    if (use_big_tiles(ctx, Mt, Nt, K)) return rounds(ceil_div(Mt, 256) * ceil_div(Nt, 256), 256);
    if (Mt <= 32 || Nt <= 64) return 1;
    const int64_t tiles128 = ceil_div(Mt, 128) * ceil_div(Nt, 128);
    if (tiles128 < 384 && K < 4096 && ctx->gemm_small == 2) return rounds(ceil_div(Mt, 64) * ceil_div(Nt, 128), 512);
    if (tiles128 < 384 && ctx->gemm_small == 4) return rounds(tiles128, 256);
    if (ctx->gemm_cfg == 1) return rounds(tiles128, 512);
    return rounds(ceil_div(Mt, 128) * ceil_div(Nt, 256), 256);
}

}  // namespace

bool gemm_extra_cols_free(const sa3k_ctx* ctx, int64_t Mt, int64_t N, int64_t K, int64_t Nx, bool kn, bool swiglu,
                          bool heads) {
    if (planned(ctx) && !kn && N > 64) return extra_cols_pay(Mt, N, K, Nx, ctx->gemm_split, swiglu, heads);
    return dma_rounds(ctx, Mt, N + Nx, K) <= dma_rounds(ctx, Mt, N, K);
}

void gemm_run_dma(sa3k_ctx* ctx, const GemmDesc& d) {
    DmaParams p{d.A, d.lda, d.B, d.ldb, d.A2, d.lda2, d.B2, d.ldb2, d.K2, d.M, d.N, d.K, d.alpha,
                d.colscale, d.bias, d.C, d.ldc, d.accumulate, d.Cb, d.ldcb, d.U, d.Ub, d.ldu,
                d.Mx, d.Ax, d.ldax, d.A2x, d.lda2x, d.Cx, d.ldcx, d.accumulate_x, d.Cbx, nullptr, 0, ctx->zero_page};
    p.prescale = d.prescale;
    p.Mp = d.Mx > 0 ? ceil_div(d.M, 8) * 8 : d.M;
    p.Nx = d.Nx;
    p.Nt = d.N + d.Nx;
    p.Bx = d.Bx; p.ldbx = d.ldbx;
    p.alpha_x = d.alpha_x;
    p.Cbn = d.Cbn; p.ldcn = d.ldcn;
    p.bx_bytes = 0;
    p.b_kn = d.b_kn;
    p.bq = d.b_src == SRC_F16 ? 1 : d.b_src == SRC_Q8 ? 2 : 0;
    p.Bs = d.Bs; p.ldbs = d.ldbs;
    p.bs_bytes = 0;
    p.sw_half = d.sw_half; p.sw_g = d.sw_g; p.sw_ldg = d.sw_ldg; p.sw_done = d.sw_done;
    p.hp = d.hp; p.hp_done = d.hp_done; p.c_unfused_only = d.c_unfused_only;
    p.ad = d.ad; p.sb = d.sb; p.bwd_done = d.bwd_done;
    p.prio = ctx->gemm_prio;
    if (d.prec == SA3K_PREC_BF16) dispatch_dma<true>(ctx, p);
    else dispatch_dma<false>(ctx, p);
}

}  // namespace sa3k
