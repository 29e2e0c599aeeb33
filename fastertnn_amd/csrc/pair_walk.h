// How the layer kernel walks the K words of a tile (host and device; the host side is plain C++).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define FTNN_HD __host__ __device__ __forceinline__
#else
#define FTNN_HD inline
#endif

namespace ftnn {

// Division of a 32-bit unsigned n by a fixed d without the ~25-instruction expansion of "/":
// m = floor(2^32 / d) (saturated for d = 1) under-estimates the quotient by at most one, which one
// compare fixes.  Exact for every n < 2^32, d >= 1.
struct FastDiv {
    uint32_t d, m;
};
inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f;
    f.d = d;
    f.m = d <= 1 ? 0xffffffffu : (uint32_t)((1ull << 32) / d);
    return f;
}
FTNN_HD uint32_t fastdiv(uint32_t n, const FastDiv& f) {
    uint32_t q = (uint32_t)(((uint64_t)n * f.m) >> 32);
    if (n - q * f.d >= f.d) q++;
    return q;
}

// geometry of one conv layer as the implicit-im2row GEMM needs it
struct ConvGeom {
    int H, W, CP, OH, OW, KW, K;   // K = C_pack*KH*KW words per plane before rounding
    int H_pad, W_pad, H_stride, W_stride;
    FastDiv dOW, dCP, dKW;
};

// How a lane's word moves on when its run of pairs ends.  C_pack even: a run is the C_pack / 2 pairs of a tap, two planes
// apart, then the next tap.  C_pack odd: every pair is a run, and both halves move on by two words = (kh, kw, ic).
struct PairWalk {
    int even, run, NP;       // NP: pairs per row, ceil(K / 2)
    int dkh, dkw, dic, KH;
    FastDiv dRun;            // C_pack / 2
};
inline PairWalk make_pair_walk(const ConvGeom& cg) {
    PairWalk p;
    p.even = cg.CP % 2 == 0;
    p.run = p.even ? cg.CP / 2 : 1;
    p.NP = (cg.K + 1) / 2;
    const int taps = p.even ? 1 : 2 / cg.CP;
    p.dic = p.even ? 0 : 2 % cg.CP;
    p.dkh = taps / cg.KW;
    p.dkw = taps % cg.KW;
    p.KH = cg.K / (cg.CP * cg.KW);
    p.dRun = make_fastdiv((uint32_t)p.run);
    return p;
}

// A lane's word of pair p, 2 p + h = (kh, kw, ic) of the reference's K order, and where its record lies: off() records from the
// record of tap (0, 0) in plane 0, computed when a run starts, plus the scalar soff, in units of UNIT per record.  UNIT 16 (bytes)
// is for operands below 4 GiB only: a call's operand has up to 2^31 records, 32 GiB, and within one image soff reaches
// C_pack - 2 planes of them.
template <uint32_t UNIT>
struct PairPos {
    int kh, kw, ic, left;    // left: pairs left in the run
    uint32_t soff, step;

    template <bool FIRST>    // FIRST: p is 0
    FTNN_HD void start(const PairWalk& pw, const ConvGeom& cg, int p, int h) {
        left = pw.run;
        soff = 0;
        step = (uint32_t)(cg.H * cg.W) * (2u * UNIT);
        if (pw.even) {
            int tap = 0;
            if constexpr (!FIRST) {
                tap = (int)fastdiv((uint32_t)p, pw.dRun);
                const int j = p - tap * pw.run;
                left -= j;
                soff = (uint32_t)j * step;
            }
            kh = FIRST ? 0 : (int)fastdiv((uint32_t)tap, cg.dKW);
            kw = tap - kh * cg.KW;
            ic = h;
        } else {
            const uint32_t w = (uint32_t)(2 * p + h);
            const int tap = (int)fastdiv(w, cg.dCP);
            ic = (int)w - tap * cg.CP;
            kh = (int)fastdiv((uint32_t)tap, cg.dKW);
            kw = tap - kh * cg.KW;
        }
    }
    FTNN_HD uint32_t off(const ConvGeom& cg) const { return (uint32_t)ic * (uint32_t)(cg.H * cg.W) + (uint32_t)(kh * cg.W + kw); }
    FTNN_HD bool next(const PairWalk& pw, const ConvGeom& cg) {   // on to the next pair; true: a new run, off() has changed
        soff += step;
        if (--left != 0) return false;
        left = pw.run;
        soff = 0;
        ic += pw.dic;
        const bool c = ic >= cg.CP;
        ic -= c ? cg.CP : 0;
        kw += pw.dkw + (c ? 1 : 0);
        const bool d = kw >= cg.KW;
        kw -= d ? cg.KW : 0;
        kh += pw.dkh + (d ? 1 : 0);
        return true;
    }
};

}  // namespace ftnn
