// Which form of a matrix-core product runs (the host side of rows_kernels.hip; plain C++).
#pragma once
#include <stdint.h>

namespace ftnn {

// A grid dimension holds fewer than 2^32 threads: tiles, rounded up to whole eighths, times the 256 of a workgroup.  It also
// keeps row numbers below 2^31 in the last tile.
constexpr int64_t kMaxRowsTiles = (1 << 24) - 8;
inline int64_t rows_tiles(int64_t prow, int64_t qrow, int edge) { return ((prow + edge - 1) / edge) * ((qrow + edge - 1) / edge); }

// How a product is cut: blocks of 32 x 32 per wavefront, and the wavefronts that split K (1: four of them on tiles of their own).  Small
// tiles fill the chip with little work, large ones spend fewer instructions and bytes per multiply; wavefronts on tiles of their own need no
// meeting, which is most of the time where rows are short.  The choice goes by estimates in us, a + b (n - 1) + w (c + d (n - 1)) + e r for n
// rounds of 256 workgroups, w words (pairs of words) per wavefront and r million results.  Eight wavefronts are for tiles that leave compute
// units idle: from a second round on four are ahead (8 x 16384 -> 16384, weights from memory, 13.9 / 14.9).
struct ProductForm {
    int p, q, ks;
    double a, b, c, d, e;
};
// The least estimate among the first `count` forms; a larger tile that splits K over four wavefronts is taken below `tie` times the least before it.
inline int form_of(const ProductForm* forms, int count, double tie, int64_t prow, int64_t qrow, int words) {
    const int64_t pb = (prow + 31) / 32, qb = (qrow + 31) / 32;
    int best = -1;
    double least = 1e300;
    for (int i = 0; i < count; i++) {
        const ProductForm& f = forms[i];
        const int own = f.ks == 1 ? 2 : 1;   // 2 x 2 tiles per workgroup
        const int64_t tiles = ((pb + f.p * own - 1) / (f.p * own)) * ((qb + f.q * own - 1) / (f.q * own));
        // (fitted, and measured, on up to 256 tiles only: eight wavefronts on one)
        if (tiles > kMaxRowsTiles || (f.ks == 8 && tiles > 256)) continue;
        const double n1 = (double)((tiles + 255) / 256 - 1), w = (double)words / f.ks;
        const double t = f.a + f.b * n1 + w * (f.c + f.d * n1) + f.e * 1e-6 * (double)prow * (double)qrow;
        if (t < (f.ks == 4 && f.p > 1 ? tie : 1.0) * least) least = t, best = i;
    }
    return best;
}

// Fits to 995 products, 32 x 32 x 256 to 8192 x 8192 x 131072 below 160 tiles of 256 x 256 and up to 1.5e8 results above, all types, row-major and
// NCHW, every form measured; the last one is both operands packed by a launch and then multiplied in their best form (below).  The
// choice is 0.9 % from the best form in the mean.  us, four wavefronts that split K / now: 332 x 8180 x 256 BTN 8.2 / 5.3, 534 x 4978 x 768
// 9.1 / 6.5, 2506 x 1365 x 512 BNN 9.3 / 6.5, 190 x 5514 x 26368 37.5 / 27.3, 1446 x 725 x 20736 TBN 24.8 / 21.3.  From 160 tiles on, packed first / now: 3328 x
// 3328 x 1024 TNN 31 / 16, 6016 x 6016 x 256 56 / 31, 137912 x 157 x 512 68 / 27, 12014 x 1415 x 2816 TBN 68 / 39, 14694 x 2992 x 1792 90 / 60.
constexpr ProductForm kRowsForms[] = {{1, 1, 4, 3.43, 0.04, 0.0621, 0.0497, 0.72}, {2, 2, 4, 3.88, 0.71, 0.1107, 0.1156, 0.66},
                                      {3, 3, 4, 5.74, 3.18, 0.1986, 0.2273, 0.81}, {4, 4, 4, 7.79, 3.66, 0.2677, 0.3204, 0.69},
                                      {1, 1, 1, 3.54, 0.00, 0.0502, 0.0455, 0.47}, {1, 1, 8, 3.75, 0.09, 0.0858, 0.1057, 0.82},
                                      {2, 2, 1, 4.62, 0.00, 0.1076, 0.1139, 0.56}, {4, 4, 1, 18.69, 10.44, 0.3071, 0.2606, 0.51}};
constexpr int kRowsFormsOfRows = (int)(sizeof(kRowsForms) / sizeof(kRowsForms[0])) - 1;   // without the last
// Where a larger tile that splits K is less than 1 % ahead by the estimates it is 6 % behind by measurement (80 products; between the other forms
// such a tie is one), and long rows of binary operands lose most: us, by the least estimate / now: 752 x 459 x 98048 TBN 48.1 / 41.0, 334 x 811 x 97792
// BNN 48.4 / 41.8, 186 x 2684 x 113152 TBN 58.4 / 50.9.  A term for binary operands makes the estimates no better.
constexpr double kRowsTie = 0.99;
inline int rows_form(int64_t prow, int64_t qrow, int Kw) { return form_of(kRowsForms, kRowsFormsOfRows, kRowsTie, prow, qrow, Kw); }

inline bool mm_rows_within_limits(int64_t M, int KN, int Kw) {
    return 64LL * Kw < (1LL << 24) && M <= 0x7fffffffLL && rows_tiles(M, KN, 128) <= kMaxRowsTiles;   // (more rows are more tiles, or overflow)
}
// whether the product of the rows as they are is ahead of both operands packed by a launch and multiplied then
inline bool mm_rows_ahead_of_packing(int64_t M, int64_t OHW, int KN, int Kw) {
    if (!mm_rows_within_limits(M, KN, Kw)) return false;
    return form_of(kRowsForms, kRowsFormsOfRows + 1, kRowsTie, OHW > 1 ? KN : M, OHW > 1 ? M : KN, Kw) != kRowsFormsOfRows;
}

// Operands kept: the forms above, or workgroup tiles of 256 x 256 through LDS (k_mfma_p4, the last).  Fits to the same products; the
// choice is 1 % from the best form in the mean.  us, on k_mfma_p4 alone (tiles of 128 x 128 below 160 of 256 x 256) / now: 256 x 256 x 4096
// 11.5 / 4.3, 36 x 246 x 15616 30.5 / 6.2, 182 x 1444 x 26624 48.6 / 12.3, 1024 x 1024 x 8192 20.3 / 7.2, 2048 x 2048 x 16384 37.0 / 27, 534 x 4978 x 768
// 9.3 / 6.9; 3328 x 3328 x 1024 22 / 15, 6016 x 6016 x 1024 58 / 38, 8192 x 8192 x 1536 98 / 68, 20021 x 2017 x 256 BNN 53 / 38, 42190 x 2443 x 256 157 / 96, 8396 x 1216 x
// 3072 31 / 21.  Tiles of 32 x 32 and 64 x 64 that split K are bound by the L1 (46 bytes per cycle and compute unit), 128 x 128 by the matrix pipe
// (1040 cycles per pair of words for 1024 of multiplies); short rows with many results by the stores (3.5 - 5.5 TB/s).
constexpr ProductForm kPackedForms[] = {{1, 1, 4, 3.51, 0.14, 0.0976, 0.0756, 0.75}, {1, 1, 8, 3.95, 0.53, 0.1324, 0.1691, 1.32},
                                        {1, 2, 4, 4.54, 0.17, 0.1246, 0.1200, 0.57}, {2, 1, 4, 3.79, 0.36, 0.0982, 0.1142, 0.62},
                                        {2, 2, 4, 4.43, 0.58, 0.1742, 0.1811, 0.69}, {3, 3, 4, 6.36, 3.52, 0.3449, 0.3770, 0.44},
                                        {4, 4, 4, 8.44, 4.48, 0.5230, 0.5731, 0.28}, {1, 1, 1, 3.67, 0.02, 0.0740, 0.0585, 0.71},
                                        {2, 2, 1, 4.39, 0.25, 0.1764, 0.1700, 0.62}, {4, 4, 1, 14.28, 7.83, 0.5053, 0.5027, 0.42}};
inline int packed_form(int64_t prow, int64_t qrow, int pairs) {
    return form_of(kPackedForms, (int)(sizeof(kPackedForms) / sizeof(kPackedForms[0])), 1.0, prow, qrow, pairs);
}

}  // namespace ftnn
