// Host-side launch planning of the MFMA tile engine, shared by
// libnnc_hip.so and the cost-model runtime (compiled without HIP there).
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define NNC_HD __host__ __device__
#else
#define NNC_HD
#endif

namespace nnc {

// ---------------------------------------------------------------------------
// stream-K bookkeeping. The stream-K region holds S = sk_tiles * iters slice
// iterations; workgroup g owns [lo(g), hi(g)) with lo(g) = g*S/G.
// ---------------------------------------------------------------------------
struct StreamK {
    int tiles, iters, G, sk_tiles;
    NNC_HD int64_t total() const { return (int64_t)sk_tiles * iters; }
    NNC_HD int64_t lo(int g) const { return total() * g / G; }
    NNC_HD int64_t hi(int g) const { return total() * (g + 1) / G; }
    // first workgroup whose range reaches into stream-K tile t
    NNC_HD int first_owner(int t) const {
        const int64_t start = (int64_t)t * iters;
        int g = (int)(start * G / total());
        while (g > 0 && hi(g - 1) > start) --g;
        while (hi(g) <= start) ++g;
        return g;
    }
    // true if some stream-K tile is shared (a range boundary inside a tile)
    bool needs_fixup() const {
        if (sk_tiles == 0 || iters == 1) return false;
        return !(total() % G == 0 && (total() / G) % iters == 0);
    }
};

// Host: choose the grid and the stream-K region for `tiles` tiles of
// `iters` slices on `slots` resident workgroups. `fixup_slices` is what
// finishing the shared tiles costs, in slice times of this tile shape (the
// fixup kernel's launch and partial traffic).
//  - few slices per tile (< 4): splitting costs more than the tail; plain
//    round-robin over min(tiles, slots) workgroups
//  - otherwise round-robin (every tile whole) unless stream-K's estimated
//    time, ceil(tiles * iters / G) + fixup_slices, is shorter than
//    round-robin's ceil(tiles / slots) * iters
//  - stream-K with tiles >= slots: all but the last full round plus the
//    partial round are split, so every workgroup ends at the same time
//  - stream-K with tiles < slots: everything is split, each workgroup
//    taking at least 4 slices (fewer workgroups for short problems)
inline StreamK plan_streamk(int tiles, int iters, int slots, int fixup_slices) {
    StreamK sk{};
    sk.tiles = tiles;
    sk.iters = iters;
    const int kMinSplitIters = 4, kMinRangeIters = 4;
    const int64_t total = (int64_t)tiles * iters;
    const int64_t dp_time = (int64_t)((tiles + slots - 1) / slots) * iters;
    if (iters < kMinSplitIters) {
        sk.G = tiles < slots ? tiles : slots;
        sk.sk_tiles = 0;
        return sk;
    }
    if (tiles >= slots) {
        const int rem = tiles % slots;
        sk.G = slots;
        const int64_t sk_time = (total + slots - 1) / slots + fixup_slices;
        sk.sk_tiles = (rem == 0 || sk_time >= dp_time) ? 0 : tiles - (tiles / slots - 1) * slots;
        return sk;
    }
    int64_t G = total / kMinRangeIters;
    if (G > slots) G = slots;
    if (G < tiles) G = tiles;
    const int64_t sk_time = (total + G - 1) / G + fixup_slices;
    if (sk_time >= dp_time) {
        sk.G = tiles;
        sk.sk_tiles = 0;
        return sk;
    }
    sk.G = (int)G;
    sk.sk_tiles = tiles;
    return sk;
}

// ---------------------------------------------------------------------------
// Short convolutions (conv.hip conv_ws_k): 32 x 32 output tiles, the four
// waves of a workgroup splitting each tile's K range, S workgroups sharing a
// tile (the last to arrive finishes it in the kernel), at most kWsMaxSlices
// slices of 32 k per wave held in registers (NS).
// Taken for convolutions with fewer 64 x 64 tiles than kWsMaxTiles64 and
// at most kWsMaxFlops of work (ResNet-18 at batch 1 and 2, and the stride-2
// convolutions at batch 4), where the 64 x 64 stream-K plan splits nearly
// every tile and needs a fixup launch. Bigger ones keep the LDS-shared
// tiles, whose waves share their operands: measured on ResNet-18, this
// kernel up to 0.5 GFLOP per convolution gives batch 1 0.262 -> 0.198 ms,
// batch 2 0.346 -> 0.286 ms, batch 4 0.436 -> 0.435 ms; up to 1 GFLOP batch
// 4 0.435 -> 0.466 ms and batch 8 0.570 -> 0.597 ms (its stride-2
// convolutions); and ResNet-18's layer 4 at batch 32 (7.4 GFLOP on 200
// tiles of 64 x 64) 25.8k -> 19.2k images/s.
// S: the smallest power of two that leaves a wave at most kWsMaxSlices
// slices; a split tile costs the finish's round trips (partial stores, the
// counter, partial loads: several slice times), so a tile that fits one
// workgroup stays whole, and a split one is split further while the grid
// stays within kWsGroups workgroups (one per CU) and each keeps at least 8
// slices.
// pieces: the waves multiply bf16 pieces (split_tile.h) where workgroups share
// CUs and have four or more slices a wave, so that the fp32 instruction, of
// 64 cycles for 2 k, is what they share: weights as stored, 23 slices on 276
// tiles 18.2 -> 15.0 us, 21 on 312 17.5 -> 14.2, 18 on 318 14.5 -> 14.0. A
// workgroup alone on its CU only waits for the cutting: 18 slices on 198
// tiles 10.4 -> 10.7, 8 on 214 5.6 -> 6.1, ResNet-18 at batch 1 191 -> 197.
// ---------------------------------------------------------------------------
constexpr int kWsMaxSlices = 6, kWsPieceSlices = 4;
constexpr int kWsMaxSplit = 16;
constexpr int kWsMaxTiles64 = 256;
constexpr double kWsMaxFlops = 5e8;
constexpr int kWsGroups = 256;

struct WsPlan {
    int64_t tiles;  // 32 x 32 tiles
    int iters;      // slices of 32 k
    int S, NS;
    bool pieces;
};

// false: no 32 x 32 tiles for this convolution
inline bool plan_ws_slices(int64_t Co, int64_t Npix, int64_t K, WsPlan& p) {
    if (K <= 0 || Co <= 0 || Npix <= 0) return false;
    if (((Co + 63) / 64) * ((Npix + 63) / 64) >= kWsMaxTiles64 || 2.0 * Co * (double)Npix * K > kWsMaxFlops)
        return false;
    p.tiles = ((Co + 31) / 32) * ((Npix + 31) / 32);
    p.iters = (int)((K + 31) / 32);
    int S = 1;
    while (S < kWsMaxSplit && (p.iters + S - 1) / S > 4 * kWsMaxSlices) S *= 2;
    if (S > 1)
        while (S < kWsMaxSplit && p.tiles * 2 * S <= kWsGroups && p.iters / (2 * S) >= 8) S *= 2;
    const int per = (p.iters + S - 1) / S;
    if (per > 4 * kWsMaxSlices) return false;
    p.S = S;
    p.NS = (per + 3) / 4;
    p.pieces = p.tiles * S > kWsGroups && p.NS >= kWsPieceSlices;
    return true;
}

// conv_ws_k (the tap-major layout is the caller's to check)
inline bool plan_ws(int64_t Co, int64_t Npix, int64_t K, WsPlan& p) {
    return K % 32 == 0 && plan_ws_slices(Co, Npix, K, p);
}

// conv_wss_k. Each of its workgroups first writes the table of its k's, so
// rounds of many short ones go to the 64 x 64 tiles: tiles more than 256
// times the smaller of the slices and three (one slice on 540 tiles 5.9 us
// here, 5.3 there; two on 630 6.9 and 6.4, on 402 5.4 and 6.2; six on 792 12.3
// and 10.8, on 582 11.3 and 14.5).
inline bool plan_ws_stored(int64_t Co, int64_t Npix, int64_t K, WsPlan& p) {
    if (!plan_ws_slices(Co, Npix, K, p)) return false;
    return p.S > 1 || (p.tiles + kWsGroups - 1) / kWsGroups <= (p.iters < 3 ? p.iters : 3);
}

// Short GEMMs (gemm.hip gemm_ws_k, the GEMM form of conv_ws_k): products of
// at most kGwsMaxFlops (a transformer encoder's projections and FFN2 at
// batch 8, sequence 128), on 32 x 32 tiles of every batch with the same
// split rule, while a wave holds at most kGwsMaxSlices slices (longer K
// splits over more workgroups) and the grid stays below kGwsMaxGroups.
// Measured on MI355X against the 64 x 64 direct-to-LDS tiles (rocprofv3,
// one kernel per product): 1024x256x256 5.8 vs 9.7 us, 512^3 7.0 vs 14.3,
// 1024x768x256 11.0 vs 11.5, 1024x256x1024 (split in two) 15.1 vs 16.1;
// the tile kernel ahead at 1024 workgroups (1024x1024x256: 12.2-12.8 vs
// 11.3-11.5 us) and with six slices per wave (768^3: 28.1 vs 22.4 us).
// `rows16`: every k-contiguous row is on a 16-byte boundary. Others load up
// to three more values per slice and stay on 64 x 64 tiles where many tiles
// have one slice per wave ([36,183,51] x [36,51,120] 6.2 vs 7.3 here;
// [59,3582] x [61,3582]^T 20.5 vs 8.5 here).
constexpr double kGwsMaxFlops = 1e9;
constexpr int kGwsMaxSlices = 4, kGwsMaxGroups = 1024;

inline bool plan_gemm_ws(int64_t M, int64_t N, int64_t K, int64_t batches, bool rows16, WsPlan& p) {
    if (M <= 0 || N <= 0 || K <= 0 || batches <= 0) return false;
    if (2.0 * M * (double)N * K * batches > kGwsMaxFlops) return false;
    p.tiles = ((M + 31) / 32) * ((N + 31) / 32) * batches;
    p.iters = (int)((K + 31) / 32);
    int S = 1;
    while (S < kWsMaxSplit && (p.iters + S - 1) / S > 4 * kGwsMaxSlices) S *= 2;
    if (S > 1)
        while (S < kWsMaxSplit && p.tiles * 2 * S <= kWsGroups && p.iters / (2 * S) >= 8) S *= 2;
    const int per = (p.iters + S - 1) / S;
    if (per > 4 * kGwsMaxSlices || p.tiles * S >= kGwsMaxGroups) return false;
    if (!rows16 && per <= 4 && p.tiles * S > kWsGroups) return false;
    p.S = S;
    p.NS = (per + 3) / 4;
    p.pieces = false;
    return true;
}

// Fixup cost in slice times of a BM x BN tile: about one slice for 128x128
// tiles, scaled by tile area for smaller tiles (shorter slices).
constexpr int fixup_slices_for(int bm, int bn) { return (128 * 128) / (bm * bn); }

// ---------------------------------------------------------------------------
// Tile and schedule of the split kernels (split_tile.h). The estimate of a
// launch is its start, its longest workgroup's slices of 32 k at a price that
// grows with the workgroups n that share a CU, an epilogue for each of that
// workgroup's whole tiles, and, where tiles are shared, what finishing them
// takes beside their partials' bytes. Prices in microseconds, fitted by least
// squares to every tile shape at every n, tiles whole and shared, of 95
// products and 43 convolutions on MI355X (the estimate's choice takes 1.03
// times the best one's time for aligned products, 1.02 for others, 1.01 for
// convolutions). What it decides, both sides measured: Gemm 2048^3 as 128x128
// tiles 101 us, as 64x64 134; 2048x1024x256 as 64x64 13.9, as 128x128 19.0;
// 1024x768x1024 64x64 at three per CU shared 24.3, whole 27; 3x3 convolutions
// at batch 32: 64 channels 56x56 as 64x256 whole 57, shared 68; 64 -> 128
// stride 2 as 128x128 whole 36, shared 40; 128 channels 28x28 shared 58, whole
// 61.
// ---------------------------------------------------------------------------
struct SplitTileCost {
    int bm, bn, max_per_cu;
    double start, tile;  // a launch; a workgroup's whole tile beside its slices
    double us[4];        // a slice, at 1..max_per_cu workgroups per CU
    double shared[4];    // more for shared tiles
    double per_mb, per_part;
};
constexpr SplitTileCost kGemm64 = {64, 64, 4, 3.7, 3.6, {0.68, 0.92, 1.38, 2.17}, {8.7, 8.1, 5.7, 6.5}, 0.40, 0};
constexpr SplitTileCost kGemm128 = {128, 128, 2, 3.8, 7.1, {1.27, 2.54, 0, 0}, {10.6, 5.4, 0, 0}, 0.40, 0};
// rows off 16-byte boundaries, or K or N no multiple of 4
constexpr SplitTileCost kGemm64u = {64, 64, 4, 2.2, 4.1, {0.84, 1.15, 1.56, 2.46}, {12.1, 12.9, 14.2, 16.6}, 0.05, 0};
constexpr SplitTileCost kGemm128x64u = {128, 64, 3, 3.7, 5.3, {1.15, 1.71, 3.58, 0}, {16.9, 15.8, 14.0, 0}, 0.05, 0};
// the fp32 instruction on 64x64 tiles (gemm_dma_k), one workgroup per CU
constexpr SplitTileCost kGemmFp32 = {64, 64, 1, 3.9, 2.8, {0.61, 0, 0, 0}, {6.5, 0, 0, 0}, 0.40, 0};
constexpr SplitTileCost kConv64 = {64, 64, 4, 4.6, 2.3, {0.79, 1.06, 1.38, 2.37}, {5.5, 3.7, 3.9, 0.9}, 0.37, 0.16};
constexpr SplitTileCost kConv128 = {128, 128, 2, 4.1, 5.4, {1.39, 2.51, 0, 0}, {5.8, 1.6, 0, 0}, 0.37, 0.16};
constexpr SplitTileCost kConv64x256 = {64, 256, 2, 4.9, 5.1, {1.85, 2.97, 0, 0}, {4.9, 1.9, 0, 0}, 0.37, 0.16};

struct SplitPlan {
    StreamK sk;
    double us;
};

// Shared product tiles with at most this many partials are finished in the
// split kernel: a second launch costs more than the last workgroup's reads.
constexpr int kSplitInKernelParts = 8;

// parts of a shared tile at most
inline int64_t split_parts(const StreamK& sk) {
    const int64_t per = sk.total() / sk.G;
    return per > 0 ? (sk.iters + per - 1) / per + 1 : sk.iters;
}

inline double split_estimate(const SplitTileCost& c, const StreamK& sk, int cus) {
    auto at = [&](int64_t groups) {
        const int64_t n = (groups + cus - 1) / cus;
        return (n < 1 ? 1 : n > c.max_per_cu ? c.max_per_cu : n) - 1;
    };
    const int64_t whole = sk.tiles - sk.sk_tiles;
    const int64_t full = whole / sk.G, rem = whole % sk.G;
    double us = c.start + c.tile * (double)(full + (rem != 0));
    us += (double)full * sk.iters * c.us[at(sk.G)] + (rem ? sk.iters * c.us[at(rem)] : 0.0);
    if (sk.sk_tiles) us += (double)((sk.total() + sk.G - 1) / sk.G) * c.us[at(sk.G)];
    if (sk.needs_fixup())
        us += c.shared[at(sk.G)] + c.per_part * (double)split_parts(sk) +
              c.per_mb * ((double)sk.G + sk.sk_tiles) * c.bm * c.bn * 4e-6;
    return us;
}

// The cheapest schedule of `tiles` tiles of `iters` slices on 1 to max_per_cu
// workgroups per CU, tiles whole or shared.
inline SplitPlan plan_split(const SplitTileCost& c, int64_t tiles, int iters, int cus) {
    SplitPlan best{};
    best.us = 1e30;
    for (int n = 1; n <= c.max_per_cu; ++n)
        for (int whole = 0; whole < 2; ++whole) {
            const StreamK sk = plan_streamk((int)tiles, iters, n * cus, whole ? 1 << 20 : 0);
            if (sk.G < 1) continue;
            const double us = split_estimate(c, sk, cus);
            if (us < best.us) best = SplitPlan{sk, us};
        }
    return best;
}

// Tile shape and schedule of a tap-major convolution (K a multiple of 32).
struct ConvSplitPlan {
    SplitTileCost tile;
    StreamK sk;
    double us;
};
inline ConvSplitPlan plan_conv_split(int64_t Co, int64_t Npix, int64_t K, int cus) {
    auto plan = [&](const SplitTileCost& c) {
        return plan_split(c, ((Co + c.bm - 1) / c.bm) * ((Npix + c.bn - 1) / c.bn), (int)(K / 32), cus);
    };
    const SplitTileCost& large = Co <= 64 ? kConv64x256 : kConv128;
    const SplitPlan a = plan(kConv64), b = plan(large);
    return a.us <= b.us ? ConvSplitPlan{kConv64, a.sk, a.us} : ConvSplitPlan{large, b.sk, b.us};
}

// Products that stay on the fp32 matrix instruction whatever the estimate:
// one round of 64x64 tiles over a few slices. The kernel's start, not its
// products, is what takes the time there, and cutting the operands lengthens
// it ([64,128,64] x [64,64,128] 6.9 us, split 7.0; unaligned [30,71,71] x
// [71,32] 7.3 and 7.7; beyond: unaligned 1001x999x333 24 and 15). Over one or
// two slices a few rounds more do ([24,247,25] x [24,25,242] 6.4 and 7.9;
// 1862x2348x41 16.8 and 17.5).
inline bool gemm_stays_fp32(int64_t tiles64, int64_t iters, bool aligned, int cus) {
    return tiles64 <= cus ? iters <= (aligned ? 8 : 4) : iters <= 2 && tiles64 <= (aligned ? 4 : 5) * cus;
}

// Tiles of a product that no other kernel takes. `aligned`: 16-byte rows on
// both sides. Unaligned rows keep a second-level sum (they were summed that
// way before), for which 64x64 and 128x64 tiles have registers.
struct GemmTilePlan {
    SplitTileCost tile;
    bool fp32;     // gemm_dma_k (aligned) or gemm_streamk_k
    bool one_per_cu;  // gemm_dma_k on one workgroup per CU, else all resident ones
    StreamK sk;    // of the split kernels
    double us;
};
inline GemmTilePlan plan_gemm_tiles(int64_t M, int64_t N, int64_t K, int64_t batches, bool aligned, int cus) {
    const int iters = (int)((K + 31) / 32);
    auto tiles = [&](const SplitTileCost& c) { return ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * batches; };
    if (gemm_stays_fp32(tiles(kGemmFp32), iters, aligned, cus)) return GemmTilePlan{kGemmFp32, true, false, StreamK{}, 0.0};
    const SplitTileCost &s = aligned ? kGemm64 : kGemm64u, &l = aligned ? kGemm128 : kGemm128x64u;
    const SplitPlan a = plan_split(s, tiles(s), iters, cus), b = plan_split(l, tiles(l), iters, cus);
    GemmTilePlan p = a.us <= b.us ? GemmTilePlan{s, false, false, a.sk, a.us} : GemmTilePlan{l, false, false, b.sk, b.us};
    if (aligned && tiles(kGemmFp32) <= cus) {
        // within one round the fp32 tiles need no cutting: 495x320x3072 22.0
        // us, split 25.0; 355x2592x1152 27.7 and 29.9; but 478x928x2496 35 and 28
        const StreamK sk = plan_streamk((int)tiles(kGemmFp32), iters, cus, fixup_slices_for(64, 64));
        const double us = split_estimate(kGemmFp32, sk, cus);
        if (us < p.us) p = GemmTilePlan{kGemmFp32, true, true, sk, us};
    }
    return p;
}

}  // namespace nnc
