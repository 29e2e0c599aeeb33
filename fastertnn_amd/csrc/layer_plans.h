// How layers are cut into launches: rules on sizes alone (the host side of the kernels; plain C++).
#pragma once
#include <stdint.h>

#include <algorithm>

#include "pair_walk.h"

namespace ftnn {

constexpr int kTNN = 0, kTBN = 1, kBTN = 2, kBNN = 3;

inline int cpack_of(int C) { return (int)(((int64_t)C + 63) / 64); }

inline bool ranges_meet(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}

// The grid of k_dense_rows: blocks of 32 rows along x and, past 2^23 of them, z (a grid dimension holds fewer than 2^32 threads), groups
// of four words along y.  Workgroups enough: each makes all the words of its rows, the input then comes through one L2 only (32 x 16 x 64 x 64,
// 5 x 5, BNN: 26.5 -> 24.4 us as a layer).
constexpr uint32_t kDenseBlocksX = 1u << 23;
struct DenseGrid {
    uint32_t x, y, z;
};
inline DenseGrid dense_rows_grid(int64_t M /* rows, below 2^31 */, int groups) {
    const int64_t blocks = (M + 31) / 32;
    DenseGrid g;
    g.x = (uint32_t)std::min<int64_t>(blocks, kDenseBlocksX);
    g.y = M >= 65536 ? 1u : (uint32_t)std::min(groups, 65535);
    g.z = (uint32_t)((blocks + kDenseBlocksX - 1) / kDenseBlocksX);
    return g;
}

// Dense rows straight from the fp32 input (k_dense_rows), or from its bit planes in two launches (k_dense_rows_planes).  The first reads a tap as
// `loads` values of 4 bytes, again for every window that holds it; the second quantises each pixel once and reads a tap as 8 or 16 bytes, for
// a launch more.  us of either side in a graph, but for what both have, fitted to 1050 layers of 1 to 32 channels, windows of 3 x 1 to 17 x 17 and 16 to
// 1200000 pixels; 0.6 is taken off the launch, so that a tie keeps the planes.  The choice is 0.3 % from the better form in the mean (the planes
// alone 13 %, the input alone 12 %), and 13 of the 1050 are 3 to 23 % slower than from the planes.  Layers, us, from the planes / the input:
// 22 x 9 x 209 x 209 -> 10, 3 x 3, BNN 79.8 / 66.1; 52 x 11 x 45 x 45 -> 25, 9 x 1, TNN 24.3 / 18.4; 61 x 19 x 186 x 186 -> 12, 9 x 9 stride 2, BNN 152 / 493;
// 26 x 17 x 70 x 70 -> 6, 11 x 11 stride 2, TNN 24.4 / 53.2.  Eight taps at most of 23 channels and more are one trip of a workgroup, which then
// waits longer than it works: 25 x 30 x 29 x 151 -> 39, 5 x 1, TNN 19.6 / 24.6, but on 6762 pixels, 7 x 1, 10.5 / 9.6.  Inputs of 4 GiB and
// more go by the planes: offsets within the input are 32 bits wide.
inline int dense_loads(int C) { return C <= 8 ? 8 : C <= 12 ? 12 : C <= 16 ? 16 : C <= 24 ? 24 : 32; }
inline bool dense_rows_from_input(bool ternary, int64_t pixels /* of the input */, int C, int64_t M, int taps, int W_stride) {
    if (pixels * C >= (1LL << 30) || (C > 22 && taps <= 8 && M > 20000)) return false;
    const double in = 1e-6 * (double)pixels, read = 1e-6 * (double)M * taps;   // pixels and taps, in millions
    if (C <= 8) return read * (W_stride > 1 ? 2.60 : 1.02) < 2.6 + 23.3 * in;
    return read * dense_loads(C) * (W_stride > 1 ? 0.473 : 0.223) < 0.9 + 15.5 * in + read * (ternary ? 1.49 : 1.94);
}

// Few kernels leave the tiles of k_rows mostly empty, so that such a layer's dense rows stay on the vector ALU: up to 15 on one group of words
// (256 x 16 x 16 x 16 -> 8 BTN 10.9 us on the vector ALU / 12.5), up to eight on some more (7 x 14 x 94 x 94 -> 8, 5 x 5, TBN 17.4 / 19.9; 57024 pixels -> 3,
// 28 words, TBN 32.6 / 37.6), but 212064 -> 3, 32 words, BTN 118 / 70 and 10000 -> 10, 60 words, TNN 24.6 / 19.3.  Of 400 layers of 1 to 24 kernels 4 are 6 to
// 9 % slower than on the vector ALU (15 by the first line alone).
inline bool few_kernels(int64_t M, int KN, int Kw) { return (KN < 16 && Kw == 4) || (KN <= 8 && Kw <= 44 && M <= 100000); }

// How k_conv_f4 cuts a layer of M pixels, KN kernels and rows of K words.
//
// K split: enough wavefronts to occupy the chip's 1024 SIMDs, but no exchange where the tiles alone do that (a tile = 64
// kernels x 64 pixels).  Where a wavefront's run of K is long, a second round of a few tiles costs more than the exchange.
// Lines of the fp32 results: fits to 920 layers (every split and the small tile measured; the mean layer is 0.5 % from its
// best); e.g. us on splits 1 / 2 / 4 / small tiles: 944 tiles x 135 words 36 / 29 / 30 / 37, 724 x 36 23 / 17 / 17 / 19, 320 x 200
// 37 / 25 / 22 / 25, 216 x 18 10.2 / 8.9 / 8.0 / 7.7, 1568 x 144 54 / 57 / 57 / 70.  Hand-overs, which keep wavefronts shorter at the
// end, have the lines of a sweep of their own (90 chains: 0.5 % from their best).
//
// Few 64 x 64 tiles: tiles of 32 x 32, four times the workgroups.  fp32 results of fewer than 120 words up to 300 tiles; but where 190 to
// 256 tiles give most of the 256 compute units one workgroup each and a row is long (72 words), those are ahead unless the last
// kernel tile is half empty.  Layer and quantiser in a graph, us, 64 x 64 split four ways / 32 x 32: 216 tiles x 108 words 9.8 / 10.4,
// 240 x 99 11.2 / 11.7, 208 x 117 12.5 / 13.5 (20 such layers 3 % ahead in the mean); 160 x 99 10.8 / 10.2, 280 x 90 11.3 / 10.9, 196 x 36 7.3 / 7.2.
//
// Small tiles that do not fill the compute units and long rows: eight wavefronts split K.  A run of K words is a chain of loads, two pairs in
// flight, and the exchange grows by 0.2 us.  Layer and quantiser in a graph, us, on four / eight wavefronts: 24 tiles x 392 words 12.1 / 10.1,
// 99 x 525 19.2 / 15.0, 189 x 425 16.8 / 12.9, 158 x 196 9.5 / 8.4, 96 x 75 7.6 / 7.0; the other way 100 x 18 6.0 / 6.2, 976 x 18 7.6 / 9.2,
// 305 x 72 8.8 / 9.4.  Of 213 layers the 86 within these lines take 0.75 - 1.0 of the time; hand-overs are of chains whose rows are shorter.
struct LayerCut {
    bool small, deep;   // tiles of 32 x 32; K split over eight wavefronts (of small tiles)
    int split;          // over 1, 2 or 4 of a workgroup's wavefronts
};
// force_split: 0, or the split to take; small_below: -1, or the count of 64 x 64 tiles below which tiles are small (tuning aids)
inline LayerCut layer_cut(int64_t M, int KN, int K, bool hand_over, int force_split, int64_t small_below) {
    LayerCut c;
    const int64_t tiles = ((M + 63) / 64) * ((KN + 63) / 64);
    const bool long_run = !hand_over && K >= 40;
    const int64_t from1 = hand_over ? 600 : long_run ? 1500 : 1024, from2 = hand_over ? 450 : long_run ? 800 : 520;
    c.split = force_split ? force_split : tiles >= from1 ? 1 : tiles >= from2 ? 2 : 4;
    while (c.split > 1 && (K + 1) / 2 < c.split) c.split /= 2;   // no wavefront without K words of its own, forced or not
    const bool one_round = K >= 72 && tiles >= 190 && tiles <= 256 && (KN + 31) / 32 % 2 == 0;
    c.small = tiles < (small_below >= 0 ? small_below : !hand_over && K < 120 && !one_round ? 300 : 150);
    c.deep = c.small && !force_split && !hand_over && K >= 75 && ((M + 31) / 32) * ((KN + 31) / 32) <= 256;
    return c;
}

// A small layer in one launch (k_direct_f4): eight wavefronts per workgroup, on a tile of 32 pixels or images.
constexpr int kDirectLgWaves = 3;   // (four wavefronts: slower from two pieces of input on)
constexpr uint32_t kDirectNowhere = 0x80000000u;   // an offset that, with a few planes added to it, lies beyond every image taken here
struct DirectPlan {
    bool fc;
    int H, W, OH, OW;         // as the kernel sees the image: one row for 1 x 1 windows without a stride
    int lgTW, OHt, OWt;       // a tile is 2^lgTW pixels wide; rows and columns of outputs that its region of the input serves
    int RW, RP;               // the region: pixels of a row, in all
    int rstep, cstep, lrow, lcol;
    uint32_t tiles_x, image_tiles;
    int lgS, groups;          // 2^lgS wavefronts split K; workgroups per tile
    int64_t tiles, pieces, lds_bytes;
};
// Which layers run there, and how.  A workgroup's time grows with the pieces of input it fetches (512 dwords of records of 16 values at a
// time; 2048 quads for a fully connected one), and a second workgroup per compute unit costs as much as the first.  Lines from 230
// layers, both forms in a graph, us (two launches / here): 21 x 128 x 9 x 21 -> 256, 3 x 3 6.4 / 6.9 (300 workgroups), 20 x 128 x 20 x 20 ->
// 128, 3 x 3 6.8 / 8.5 (300); two pieces of input with a window 19 x 256 x 10 x 10 -> 128, 3 x 3 stride 2 5.7 / 5.9, without one
// 14 x 512 x 12 x 12 -> 64 5.4 / 4.8; all eight wavefronts on kernels of their own and nearly a whole piece 2 x 128 x 53 x 53 -> 256, 3 x 3
// 7.7 / 8.2, half a piece 24 x 64 x 14 x 14 -> 256, 3 x 3 7.0 / 6.2; fully connected 9 x 2081 -> 3584 (4752 quads) 5.1 / 5.8,
// 15 x 812 -> 6673 (3120) 5.0 / 5.3, 8 x 1337 -> 1121 (2688) 5.1 / 4.8.
inline bool direct_plan(int type, const ConvGeom& cg, int C, int N, int KN, DirectPlan* out) {
    constexpr int kWaves = 1 << kDirectLgWaves;
    DirectPlan& a = *out;
    a = DirectPlan();
    const int KB = (KN + 31) / 32, KH = cg.K / (cg.CP * cg.KW), NP = (cg.K + 1) / 2;
    const int64_t M = (int64_t)N * cg.OH * cg.OW;
    const bool fc = a.fc = cg.H == 1 && cg.W == 1 && KH == 1 && cg.KW == 1 && cg.H_pad == 0 && cg.W_pad == 0;
    const int most = fc ? 400 : 256;   // workgroups
    if ((M + 31) / 32 * ((KB + kWaves - 1) / kWaves) > most) return false;
    if (((int64_t)cg.CP * 64 + 64) * cg.H * cg.W * 4 > kDirectNowhere) return false;   // offsets within an image
    a.H = cg.H, a.W = cg.W, a.OH = cg.OH, a.OW = cg.OW;
    a.tiles_x = a.image_tiles = 1;
    int64_t U;   // pieces of work in fetching a tile's input
    if (fc) {
        a.RP = a.RW = 32;
        a.tiles = (N + 31) / 32;
        U = (int64_t)std::min(32, N) * cg.CP * 16;
        if (U > 3072) return false;
        // binary weights take half the bytes as rows: 4 x 2312 -> 9837 (5.8 MB of records) 6.1 / 6.0, 3 x 2750 -> 12499 (8.6) 6.0 / 5.4 with the
        // weights within the Infinity Cache, which larger ones need not be
        if ((type == kTBN || type == kBNN) && (int64_t)KN * cg.CP * 16 > (8 << 20)) return false;
    } else {
        if (KH == 1 && cg.KW == 1 && cg.H_pad == 0 && cg.W_pad == 0 && cg.H_stride == 1 && cg.W_stride == 1) {
            a.W = a.OW = cg.H * cg.W;
            a.H = a.OH = 1;
        }
        a.rstep = KH == 1 ? cg.H_stride : 1, a.cstep = cg.KW == 1 ? cg.W_stride : 1;
        a.lrow = KH == 1 ? 1 : cg.H_stride, a.lcol = cg.KW == 1 ? 1 : cg.W_stride;
        int64_t best = INT64_MAX, RPbest = 0;
        for (int lg = 5; lg >= 2; lg--) {
            const int TW = 1 << lg, TH = 32 >> lg;
            const int OWt = std::min(TW, a.OW), OHt = std::min(TH, a.OH);
            const int64_t RW = (int64_t)(OWt - 1) * a.lcol + cg.KW, RH = (int64_t)(OHt - 1) * a.lrow + KH;
            if (RW > 4096 || RH > 4096) continue;
            const int64_t tx = (a.OW + TW - 1) / TW, ty = (a.OH + TH - 1) / TH;
            const int64_t cost = tx * ty * (RW * RH + 16);
            if (cost < best) {
                best = cost, RPbest = RW * RH;
                a.lgTW = lg, a.OWt = OWt, a.OHt = OHt, a.RW = (int)RW;
                a.tiles_x = (uint32_t)tx, a.image_tiles = (uint32_t)(tx * ty);
            }
        }
        U = RPbest * cg.CP * 4;
        if (best == INT64_MAX || U > (cg.K == cg.CP && a.cstep == 1 && a.rstep == 1 ? 1024 : 512)) return false;
        a.RP = (int)RPbest;
        a.tiles = (int64_t)N * a.image_tiles;
    }
    a.pieces = U;
    // K split: eight ways on long rows, and on the shortest, where a workgroup's time goes with the blocks it stores; else four; less where that
    // takes more than 256 workgroups.  us at 8 / 4 / 2 / 1: 10 x 128 x 8 x 8 -> 64, 5 x 5 4.4 / 4.9 / 5.6 / 7.3, 5 x 64 x 2 x 5 -> 512, 1 x 1 4.0 / 4.0 / 4.2 / 4.5,
    // 10 x 256 x 9 x 9 -> 256, 1 x 1 4.7 / 4.6 / 4.7 / 5.1.
    a.lgS = NP >= 16 || (NP <= 2 && a.tiles * KB <= 192) ? kDirectLgWaves : 2;
    auto groups_at = [&](int lg) { return (KB + (kWaves >> lg) - 1) >> (kDirectLgWaves - lg); };
    while (a.lgS > 0 && a.tiles * groups_at(a.lgS) > 256) a.lgS--;
    a.groups = groups_at(a.lgS);
    if (a.tiles * a.groups > most || (!fc && a.lgS == 0 && U > 384 && cg.K > cg.CP)) return false;
    // Fewer than four wavefronts on a K: a wavefront's run of pairs becomes what a workgroup takes longest for, a workgroup of many for one tile
    // sooner than the only one, and tiles of a pixel or two are all store.  Of 1000 layers this leaves 801, which take 0.84 of the two launches' time in
    // the mean, two of them up to 5 % more; without it 86 took more than 3 % more, up to 1.86 times as long.  us, two launches / here: 26 x 224 x 3 x 6 -> 1429, 3 x 5 stride 2 (runs
    // of 30) 6.8 / 12.0, 17 x 95 x 5 x 5 -> 1045, 3 x 3 (9, two workgroups per tile) 6.5 / 7.5, 26 x 40 x 3 x 3 -> 1810, 3 x 3 to one pixel 5.8 / 7.2,
    // but 8 x 128 x 28 x 28 -> 128, 3 x 3 (5, the only one) 6.6 / 6.2.
    const int run = (NP + (1 << a.lgS) - 1) >> a.lgS;
    if (!fc && a.lgS <= 1 && (run > (a.groups == 1 ? 9 : 4) || 20 * M <= 3 * 32 * a.tiles)) return false;
    a.lds_bytes = std::max<int64_t>((int64_t)cg.CP * a.RP * 16 + 16 + 8LL * NP, (64 << kDirectLgWaves) * 64);
    return a.lds_bytes <= (64 << 10);
}

}  // namespace ftnn
