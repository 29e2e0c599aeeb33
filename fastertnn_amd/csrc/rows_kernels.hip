// The fp4 matrix-core GEMM straight from packed rows: one launch, no expansion pass, no scratch.
//
// k_mfma and k_mfma_p4 (mfma_kernels.hip) read operands that a launch of their own has brought into matrix-core form.  For
// products below a few hundred 256 x 256 tiles that launch and its round trip through memory cost as much as the product
// itself, and from there on they still do where rows are short.  Here a wavefront fetches the bit planes as they lie, 16 bytes of
// signs and zeros per lane, and makes the E2M1 nibbles in registers beside the multiplies: 10 vector instructions per 32 rows x 64 lanes, so that a wavefront
// tile of 4 x 4 blocks of 32 x 32 spends 6 issue slots per multiply of 8 slots.
//
//   * The wavefronts of a workgroup work on ONE output tile and split K: wavefront w takes the groups of four words
//     w, w + KS, ...  Nothing is shared in the K loop, so it has no barrier; the partial tiles meet in LDS at the end.  Where rows are
//     short and results many, that end is most of the time: four wavefronts work on tiles of their own then, on all of K.
//   * A group travels global -> LDS by LDS-direct loads into a ring of the wavefront's own, four lanes on the 64 contiguous
//     bytes of a ternary row (two on the 32 of a binary one), and from there to registers in the operand's order.
//     Loaded straight into that order, 64 lanes touch 64 pieces of cache lines per instruction and the L1 delivers
//     16 bytes per cycle; in row order it delivers 64 (both measured on operands that lie in the L2).  The pieces of a row
//     are permuted by its number on the way, so that the 16-byte LDS reads spread over all banks.
//   * Neighbouring wavefronts take neighbouring groups: two groups of a row share a 128-byte line.
//   * Signed nibbles (0x2, 0x0, 0xA): a lane flagged zero becomes +-0 whatever its sign bit, which adds nothing, and no
//     row sums are needed; sums are exact while 64 Kw < 2^24.
//
// What bounds it: a lone wavefront per SIMD issues about 2550 cycles of instructions per group on 4 x 4 blocks for 2048
// cycles of matrix pipe (the LDS-direct loads and LDS reads of a group add 14 cycles each to a slot's multiply), at the
// clock that sustained multiplies of mixed signs allow (1.9 GHz on all compute units).  Device time of a whole call from
// packed rows, before (expansion launch + k_mfma, or the vector ALU) and now: 256 x 256 x 4096 4.8 -> 3.6 us,
// 512 x 512 x 4096 10.2 -> 3.8, 1024 x 1024 x 8192 17.8 -> 7.6, 1500 x 1500 x 12032 32.6 -> 17.5, 2048 x 2048 x 16384 44.1 ->
// 31, 8 x 16384 x 16384 57.8 -> 12.3.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "ftnn_internal.h"

namespace ftnn {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// fn(0), ..., fn(N - 1) with compile-time indices
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& fn, std::integer_sequence<int, I...>) {
    (fn(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& fn) {
    static_for_impl(fn, std::make_integer_sequence<int, N>{});
}

// a lane's share of one group of a row: the 128 lanes of its half, as planes
template <bool TERN>
struct RawRow {
    v4u s, z;
};
template <>
struct RawRow<false> {
    v4u s;
};

__device__ __forceinline__ void mfma_f4(v16f& c, const v4u& a, const v4u& b) {
    const v8i va = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
    const v8i vb = {(int)b.x, (int)b.y, (int)b.z, (int)b.w, 0, 0, 0, 0};
    // cbsz = blgp = 4: both operands E2M1, unscaled
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(va, vb, c, 4, 4, 0, 0, 0, 0);
}

// Half of a lane's operand for one K word from 32 lanes of its row: HALF 0 the nibble dwords 0 and 1, HALF 1 the dwords 2
// and 3.  Nibble j of dword k is lane 4 j + k: both operands take their lanes in the same order, so any order serves.
template <bool TERN, int HALF>
__device__ __forceinline__ void unpack_half(const RawRow<TERN>& r, int i, v4u& e) {
    if constexpr (TERN) {
        const uint32_t s = r.s[i], z = r.z[i];
        // nibble bits 0, 1: nonzero, bits 2, 3: sign, of two lanes: (~z & 0x3) | (s & 0xC) as one three-input operation
        // (f = (~a & c) | (b & ~c): table 0x4E; written with operators, the compiler folds the masks below into it twice)
        const uint32_t w = HALF == 0 ? __builtin_amdgcn_bitop3_b32(z, s << 2, 0x33333333u, 0x4E)
                                     : __builtin_amdgcn_bitop3_b32(z >> 2, s, 0x33333333u, 0x4E);
        e[2 * HALF] = (w << 1) & 0xAAAAAAAAu;
        e[2 * HALF + 1] = w & 0xAAAAAAAAu;
    } else {
        const uint32_t s = r.s[i];
        e[2 * HALF] = ((HALF == 0 ? s << 3 : s << 1) & 0x88888888u) | 0x22222222u;
        e[2 * HALF + 1] = ((HALF == 0 ? s << 2 : s) & 0x88888888u) | 0x22222222u;
    }
}

// LDS-direct loads: 16 bytes per lane from base + voff (base uniform); the 64 lanes land contiguously.  M0 holds the LDS
// address (one wait state after writing it); the instruction's immediate offset moves the source and the LDS address
// alike, so two loads into adjacent KiB share one M0 (v1 is then the source less 1024).  Inline asm, so that the compiler does
// not order its own LDS reads against the loads; the kernel counts them by hand.  M0 is an operand, which the compiler sets in
// front of the statement: single loads, pairs and runs of four measured the same within 2 % from 256 x 256 to 3072 x 3072.
template <bool TWO>
__device__ __forceinline__ void dma16(uint32_t lds_byte_addr, const char* b0, uint32_t v0, const char* b1, uint32_t v1) {
    if constexpr (TWO)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %3, %4 offset:1024"
                     :
                     : "{m0}"(lds_byte_addr), "v"(v0), "s"(b0), "v"(v1), "s"(b1)
                     : "memory");
    else
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(lds_byte_addr), "v"(v0), "s"(b0) : "memory");
}

// Which tile a workgroup works on.  Workgroups go to the eight XCDs round-robin by number; XCD x takes the x-th eighth of the
// tiles, in bands of four P tiles walked along Q, so that the 32 tiles an XCD works on at a time are about 4 x 8 and its
// L2 fetches 12 panels of rows for them instead of up to 33 (3072 x 3072 x 24576 on 4 x 4 blocks: 119 -> 115 us).
struct RowsOrder {
    uint32_t tiles, per_xcd, px;   // tiles in all, per XCD (rounded up), along P
    FastDiv band, last;            // tiles of a whole band; P tiles of the last band (px % 4, or 4)
    __device__ __forceinline__ bool tile(uint32_t wg, int* tx, int* ty) const {
        const uint32_t t = (wg & 7u) * per_xcd + (wg >> 3);
        if (t >= tiles) return false;
        const uint32_t b = fastdiv(t, band), r = t - b * band.d;
        uint32_t y = r >> 2, x = r & 3u;
        if (b * 4u + 4u > px) {   // the last, narrower band
            y = fastdiv(r, last);
            x = r - y * last.d;
        }
        *tx = (int)(b * 4u + x);
        *ty = (int)y;
        return true;
    }
};

// where a result goes: element q_img * img_stride + q_pix + p * p_stride for P row p and Q row q = (q_img, q_pix).  A row-major
// result (P = activation rows, Q = weight rows: lanes along the columns) has one image; an NCHW result (P = weights, Q =
// activations: lanes along the pixels) splits q by OH * OW.
struct RowsOut {
    float* y;
    int64_t img_stride;
    uint32_t p_stride;
    FastDiv img;
    float bias, lim, alpha;   // r = sum - bias; PReLU scales r < lim by alpha
    bool past_caches;         // (host) how results leave, by stores_past_caches; the kernels' NT
};

// Blocks that meet in LDS at a time
constexpr int meeting_blocks(int nm, int ks) { return nm * ks * 4 > 144 ? nm / 2 : nm; }

// The quads that wavefront ks of a workgroup finishes: block and quad of the block.  KS > 1: in rounds of R blocks, of each the quads
// ks, ks + KS, ...
template <int NM, int KS>
struct QuadOf {
    static constexpr int R = meeting_blocks(NM, KS), PER_ROUND = KS == 1 ? 4 * NM : R * 4 < KS ? 1 : R * 4 / KS, ROUNDS = KS == 1 ? 1 : NM / R,
                         N = PER_ROUND * ROUNDS;
    static_assert(KS == 1 || (KS % 4 == 0 && (R * 4 < KS || R * 4 % KS == 0) && NM % R == 0), "whole quads per wavefront");
    static __device__ __forceinline__ int block(int i, int ks) {
        return KS == 1 ? i / 4 : i / PER_ROUND * R + i % PER_ROUND * (KS / 4) + (KS == 4 ? 0 : ks >> 2);
    }
    static __device__ __forceinline__ int sub(int i, int ks) { return KS == 1 ? i % 4 : KS == 4 ? ks : ks & 3; }
};

// Where a product's results go.  Accumulator e of block (a, b): P row 32 (prb0 + a) + 8 (e / 4) + 4 h + e % 4, Q row 32 (qrb0 + b) + lr; four
// of them are a quad.  result(quad of sums, i) is what is stored, for quad i of the wavefront (QuadOf).
// PReLU in the reference's two forms, "f <= 0 -> f *= alpha" (mm_p2_final_tnn_avx2.c:204-208) and "r >= 0 ? r : alpha * r"
// (mm_p2_final_tbn_avx2.c:73): results are integers below 2^24, so both are one compare, against 0.5 or 0.
template <bool WHOLE, bool NT>
__device__ __forceinline__ void put_quad(const float4& t, int p0, int qrb, const RowsOut& ro, int prow, int qrow, int lane) {
    const int lr = lane & 31, h = lane >> 5;   // P rows p0 + 4 h .. + 3 (p0 uniform) of Q block qrb
    const size_t stride = ro.p_stride;
    const uint32_t q = (uint32_t)(qrb * 32 + lr), img = fastdiv(q, ro.img);
    float* const d = ro.y + (size_t)p0 * stride;
    const size_t lo = (size_t)img * (size_t)ro.img_stride + (q - img * ro.img.d) + (size_t)(4 * h) * stride;
    auto put = [](float v, float* at) {
        if constexpr (NT) __builtin_nontemporal_store(v, at);
        else *at = v;
    };
    const int p = p0 + 4 * h;
    if (WHOLE || (q < (uint32_t)qrow && p < prow)) {
        put(t.x, d + lo);
        if (WHOLE || p + 1 < prow) put(t.y, d + stride + lo);
        if (WHOLE || p + 2 < prow) put(t.z, d + 2 * stride + lo);
        if (WHOLE || p + 3 < prow) put(t.w, d + 3 * stride + lo);
    }
}
// fn(whether all of a tile of P blocks prb0 .. and Q blocks qrb0 .. lies inside) (uniform)
template <int WTP, int WTQ, typename F>
__device__ __forceinline__ void by_wholeness(int prb0, int qrb0, int prow, int qrow, F&& fn) {
    if ((prb0 + WTP) * 32 <= prow && (qrb0 + WTQ) * 32 <= qrow) fn(std::true_type{});
    else fn(std::false_type{});
}

// The end of a product whose wavefronts split K: the partial tiles meet in LDS, wavefront ks sums the quads ks, ks + KS, ... over all
// wavefronts and stores them.
template <int WTP, int WTQ, int KS, bool NT, typename F>
__device__ __forceinline__ void meet_and_store(v16f (&acc)[WTP][WTQ], float4* lds, const RowsOut& ro, int prb0, int qrb0, int prow, int qrow,
                                               int ks, int lane, F&& result) {
    typedef QuadOf<WTP * WTQ, KS> QO;
    constexpr int R = QO::R, QUADS = QO::PER_ROUND;
#pragma unroll
    for (int round = 0; round < QO::ROUNDS; round++) {
        __syncthreads();   // every wavefront is done with its ring, or with the round before
#pragma unroll
        for (int j = 0; j < R; j++) {
            const v16f& c = acc[(round * R + j) / WTQ][(round * R + j) % WTQ];
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++)
                lds[((ks * R + j) * 4 + e4) * 64 + lane] = make_float4(c[4 * e4], c[4 * e4 + 1], c[4 * e4 + 2], c[4 * e4 + 3]);
        }
        __syncthreads();
        if (R * 4 < KS && ks >= R * 4) continue;   // no quad of its own (and no further round)
        float4 t[QUADS];   // all sums before the first store: the branch around the stores would hold the reads back
#pragma unroll
        for (int i = 0; i < QUADS; i++) {
            const int quad = i * KS + ks;
            t[i] = lds[quad * 64 + lane];
#pragma unroll
            for (int v = 1; v < KS; v++) {
                const float4 u = lds[(v * R * 4 + quad) * 64 + lane];
                t[i].x += u.x;
                t[i].y += u.y;
                t[i].z += u.z;
                t[i].w += u.w;
            }
            t[i] = result(t[i], round * QUADS + i);
        }
        by_wholeness<WTP, WTQ>(prb0, qrb0, prow, qrow, [&](auto whole) {
#pragma unroll
            for (int i = 0; i < QUADS; i++) {
                const int blk = QO::block(round * QUADS + i, ks);
                put_quad<decltype(whole)::value, NT>(t[i], (prb0 + blk / WTQ) * 32 + 8 * QO::sub(i, ks), qrb0 + blk % WTQ, ro, prow, qrow, lane);
            }
        });
    }
}

// the same for a wavefront with whole sums
template <int WTP, int WTQ, bool NT, typename F>
__device__ __forceinline__ void store_whole_sums(v16f (&acc)[WTP][WTQ], const RowsOut& ro, int prb0, int qrb0, int prow, int qrow, int lane, F&& result) {
    float4 t[WTP * WTQ * 4];
#pragma unroll
    for (int i = 0; i < WTP * WTQ * 4; i++) {
        const v16f& c = acc[i / 4 / WTQ][i / 4 % WTQ];
        const int e = 4 * (i % 4);
        t[i] = result(make_float4(c[e], c[e + 1], c[e + 2], c[e + 3]), i);
    }
    by_wholeness<WTP, WTQ>(prb0, qrb0, prow, qrow, [&](auto whole) {
#pragma unroll
        for (int i = 0; i < WTP * WTQ * 4; i++)
            put_quad<decltype(whole)::value, NT>(t[i], (prb0 + i / 4 / WTQ) * 32 + 8 * (i % 4), qrb0 + i / 4 % WTQ, ro, prow, qrow, lane);
    });
}

// A wavefront's tile is WTP x WTQ blocks of 32 x 32, a workgroup's the same tile: its KS wavefronts split K.  KS = 1: four wavefronts, 2 x 2
// of these tiles, each on all of K.
template <bool TP, bool TQ, int WTP, int WTQ, int KS>
struct RowsTile {
    static constexpr int WV = KS == 1 ? 2 : 1, NW = KS == 1 ? 4 : KS;   // tiles per side of a workgroup, wavefronts
    static constexpr int NS = 2;                             // ring slots: deeper rings (where they fit) measured no faster
    static constexpr int NM = WTP * WTQ, NB = WTP + WTQ;
    static constexpr int LP = TP ? 2 : 1, LQ = TQ ? 2 : 1;   // KiB (and loads) per row block and group
    static constexpr int LPG = WTP * LP + WTQ * LQ;          // per wavefront and group
    static constexpr int R = meeting_blocks(NM, KS);
    static constexpr size_t ring = (size_t)NW * NS * LPG * 1024, red = KS == 1 ? 0 : (size_t)R * KS * 4096;
    static constexpr size_t lds = ring > red ? ring : red;
    static_assert(lds <= (160u << 10), "LDS of a compute unit");
};

template <bool TP, bool TQ, int WTP, int WTQ, int KS, bool NT>
__global__ __launch_bounds__(64 * (KS == 1 ? 4 : KS)) void k_rows(const char* __restrict__ P, const char* __restrict__ Q, int prow, int qrow, int G,
                                                  RowsOrder od, RowsOut ro) {
    extern __shared__ float4 lds[];
    typedef RowsTile<TP, TQ, WTP, WTQ, KS> TL;
    constexpr int NM = TL::NM, NB = TL::NB, NS = TL::NS, LP = TL::LP, LQ = TL::LQ, LPG = TL::LPG;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, h = lane >> 5;
    constexpr int WV = TL::WV;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ks = KS == 1 ? 0 : wave;
    int tx, ty;
    if (!od.tile(blockIdx.x, &tx, &ty)) return;   // past the last tile (the whole workgroup)
    // first row blocks: within the operands
    const int prb0 = (tx * WV + (KS == 1 ? wave >> 1 : 0)) * WTP, qrb0 = (ty * WV + (KS == 1 ? wave & 1 : 0)) * WTQ;
    if (KS == 1 && (prb0 * 32 >= prow || qrb0 * 32 >= qrow)) return;   // no such tile (these wavefronts never wait for each other)
    constexpr uint32_t GP = TP ? 64u : 32u, GQ = TQ ? 64u : 32u;   // bytes of a group of 4 words
    const uint32_t rbp = (uint32_t)G * GP, rbq = (uint32_t)G * GQ;  // bytes of a row

    // Sources of the LDS-direct loads: a ternary row block and group is two loads of 16 rows x 64 bytes, four lanes per
    // row, a binary one a single load of 32 rows x 32 bytes, two lanes per row; rows past the operand are clamped (their
    // results are never stored).  One base per side, advanced by GP or GQ per group; row block, row, piece and the
    // immediate offset a load carries are in its 32-bit lane offset.
    constexpr uint32_t SPAN = 1024;   // the largest immediate offset
    const char* const pbase = P + (size_t)prb0 * 32 * rbp - SPAN;
    const char* const qbase = Q + (size_t)qrb0 * 32 * rbq - SPAN;
    auto src_row = [&](int j, bool tern) { return tern ? j * 16 + (lane >> 2) : lane >> 1; };
    auto src_piece = [&](bool tern) { return (uint32_t)(tern ? (lane & 3) ^ ((lane >> 4) & 3) : (lane & 1) ^ ((lane >> 4) & 1)) * 16u; };
    uint32_t pv[WTP][LP], qv[WTQ][LQ];
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int j = 0; j < LP; j++)
            pv[a][j] = (uint32_t)min(a * 32 + src_row(j, TP), prow - 1 - prb0 * 32) * rbp + src_piece(TP) + SPAN -
                       (uint32_t)((a * LP + j) & 1) * 1024u;
#pragma unroll
    for (int b = 0; b < WTQ; b++)
#pragma unroll
        for (int j = 0; j < LQ; j++)
            qv[b][j] = (uint32_t)min(b * 32 + src_row(j, TQ), qrow - 1 - qrb0 * 32) * rbq + src_piece(TQ) + SPAN -
                       (uint32_t)((WTP * LP + b * LQ + j) & 1) * 1024u;
    // this lane's pieces of a row block in LDS: the signs and the zeros of its half
    auto piece_at = [&](bool tern, int piece) {
        return (uint32_t)(tern ? lr * 64 + (piece ^ ((lr >> 2) & 3)) * 16 : lr * 32 + (piece ^ ((lr >> 3) & 1)) * 16);
    };
    const uint32_t rd_ts = piece_at(true, h), rd_tz = piece_at(true, 2 + h), rd_b = piece_at(false, h);
    const uint32_t ring0 = (uint32_t)wave * (NS * LPG * 1024);
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
    const char* const ring = reinterpret_cast<const char*>(lds) + ring0;

    // load number i of group gg into KiB i of the ring slot and, if i is even and below `end`, load i + 1 with it
    auto issue = [&](auto itag, auto end, int gg, int slot) {
        constexpr int i = decltype(itag)::value;
        constexpr bool two = (i & 1) == 0 && i + 1 < decltype(end)::value;
        const char *pg = pbase + (size_t)gg * GP, *qg = qbase + (size_t)gg * GQ;
        auto base = [&](int k) { return k < WTP * LP ? pg : qg; };
        auto voff = [&](int k) { return k < WTP * LP ? pv[k / LP][k % LP] : qv[(k - WTP * LP) / LQ][(k - WTP * LP) % LQ]; };
        // (an odd load by itself carries no immediate offset: its source is whole again)
        const uint32_t kib = lds0 + ring0 + (uint32_t)(slot * LPG + i) * 1024u;
        dma16<two>(kib, base(i), voff(i) + ((i & 1) ? 1024u : 0u), base(i + two), voff(i + two));
    };
    // planes of operand f (P blocks, then Q blocks) of the group in registers; its nibbles for two K words
    RawRow<TP> rp[WTP];
    RawRow<TQ> rq[WTQ];
    v4u ep[2][WTP], eq[2][WTQ];
    auto read_plane = [&](int slot, int f, bool zeros) {
        const char* L = ring + (size_t)slot * LPG * 1024 + (f < WTP ? f * LP : WTP * LP + (f - WTP) * LQ) * 1024;
        if (f < WTP) {
            if (!zeros) rp[f].s = *reinterpret_cast<const v4u*>(L + (TP ? rd_ts : rd_b));
            if constexpr (TP) {
                if (zeros) rp[f].z = *reinterpret_cast<const v4u*>(L + rd_tz);
            }
        } else {
            if (!zeros) rq[f - WTP].s = *reinterpret_cast<const v4u*>(L + (TQ ? rd_ts : rd_b));
            if constexpr (TQ) {
                if (zeros) rq[f - WTP].z = *reinterpret_cast<const v4u*>(L + rd_tz);
            }
        }
    };
    auto unpack = [&](auto half, int i, int set, int f) {
        constexpr int H = decltype(half)::value;
        if (f < WTP) unpack_half<TP, H>(rp[f], i, ep[set][f]);
        else unpack_half<TQ, H>(rq[f - WTP], i, eq[set][f - WTP]);
    };
    v16f acc[WTP][WTQ];
    // One K word of the group in `slot`: multiply operand set I & 1 and unpack the next word's operands, half an operand at a
    // time between the multiplies.  Words 0 and 1 also issue the loads of group gl into this slot (whose contents are in
    // registers), word 2 reads the next group, each operand's planes right behind its last unpacking.
    constexpr int NW = 2 * NB;
    auto step = [&](auto itag, int slot, int next_slot, int gl) {
        constexpr int I = decltype(itag)::value;
        if constexpr (I == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPG * (NS - 1)) : "memory");   // the next group has landed
        static_for<NM>([&](auto mtag) {
            constexpr int m = decltype(mtag)::value;
            mfma_f4(acc[m / WTQ][m % WTQ], ep[I & 1][m / WTQ], eq[I & 1][m % WTQ]);
            static_for<(m + 1) * NW / NM - m * NW / NM>([&](auto ktag) {
                constexpr int j = m * NW / NM + decltype(ktag)::value, i = (I + 1) & 3;
                if constexpr (I == 2 && (j & 1) == 0 && j > 0) read_plane(next_slot, (j >> 1) - 1, true);
                unpack(std::integral_constant<int, j & 1>{}, i, (I + 1) & 1, j >> 1);
                if constexpr (I == 2 && (j & 1) == 1) read_plane(next_slot, j >> 1, false);
                if constexpr (I == 2 && j == NW - 1) read_plane(next_slot, j >> 1, true);
            });
            if constexpr (I < 2) {
                constexpr int lo = I == 0 ? 0 : LPG / 2, n = I == 0 ? LPG / 2 : LPG - LPG / 2;
                static_for<(m + 1) * n / NM - m * n / NM>([&](auto ktag) {
                    constexpr int i = lo + m * n / NM + decltype(ktag)::value;
                    if constexpr ((i & 1) == 0 || i == lo) issue(std::integral_constant<int, i>{}, std::integral_constant<int, lo + n>{}, gl, slot);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    int g = ks, gl = ks;   // this wavefront's groups are ks, ks + KS, ...; gl: the next one to be loaded (past the end: the last one again)
    if (g < G) {
#pragma unroll
        for (int t = 0; t < NS; t++) {
            static_for<LPG>([&](auto itag) {
                constexpr int i = decltype(itag)::value;
                if constexpr ((i & 1) == 0) issue(itag, std::integral_constant<int, LPG>{}, min(gl, G - 1), t);
            });
            gl += KS;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int b = 0; b < WTQ; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[a][b][e] = 0.0f;
    if (g < G) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPG * (NS - 1)) : "memory");
#pragma unroll
        for (int f = 0; f < NB; f++) {
            read_plane(0, f, false);
            read_plane(0, f, true);
        }
#pragma unroll
        for (int f = 0; f < NB; f++) {
            unpack(std::integral_constant<int, 0>{}, 0, 0, f);
            unpack(std::integral_constant<int, 1>{}, 0, 0, f);
        }
        int slot = 0;
        while (g < G) {
            const int next_slot = slot + 1 == NS ? 0 : slot + 1;
            const int gc = min(gl, G - 1);
            step(std::integral_constant<int, 0>{}, slot, next_slot, gc);
            step(std::integral_constant<int, 1>{}, slot, next_slot, gc);
            step(std::integral_constant<int, 2>{}, slot, next_slot, gc);
            step(std::integral_constant<int, 3>{}, slot, next_slot, gc);
            slot = next_slot;
            g += KS;
            gl += KS;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in the LDS that the partial tiles take now

    auto result = [&](const float4& t, int) {
        auto prelu = [&](float v) {
            const float r = v - ro.bias;
            return r < ro.lim ? r * ro.alpha : r;
        };
        return make_float4(prelu(t.x), prelu(t.y), prelu(t.z), prelu(t.w));
    };
    if constexpr (KS == 1) store_whole_sums<WTP, WTQ, NT>(acc, ro, prb0, qrb0, prow, qrow, lane, result);
    else meet_and_store<WTP, WTQ, KS, NT>(acc, lds, ro, prb0, qrb0, prow, qrow, ks, lane, result);
}

// The same product of operands kept in packed4 form (mfma_kernels.hip: 1 KiB blocks of 32 rows x two K words, lane l's 16 bytes
// the words' nibbles at two bits per lane in offset codes; sP, sQ: the rows' sums).
//
// A block is one contiguous load of a wavefront and a word's operand six vector instructions beside WTP x WTQ multiplies, so the
// wavefronts read registers straight from memory: a ring of NB sets of blocks, each asked for NB - 1 pairs of words ahead (ordinary
// loads, counted by the compiler, held in place by scheduling fences).  While one word's operands are multiplied the next one's are
// unpacked, between the multiplies.
template <int WTP, int WTQ, int KS, int NB, bool NT>
__global__ __launch_bounds__(64 * (KS == 1 ? 4 : KS)) void k_packed(const uint4* __restrict__ Pc, const uint4* __restrict__ Qc, int prow, int qrow, int KP,
                                                    const int* __restrict__ sP, const int* __restrict__ sQ, int off, RowsOrder od, RowsOut ro) {
    extern __shared__ float4 lds[];
    constexpr int NM = WTP * WTQ, NO = WTP + WTQ;
    const int tid = threadIdx.x, lane = tid & 63;
    constexpr int WV = KS == 1 ? 2 : 1;   // as k_rows
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ks = KS == 1 ? 0 : wave;
    int tx, ty;
    if (!od.tile(blockIdx.x, &tx, &ty)) return;   // past the last tile (the whole workgroup)
    const int prb0 = (tx * WV + (KS == 1 ? wave >> 1 : 0)) * WTP, qrb0 = (ty * WV + (KS == 1 ? wave & 1 : 0)) * WTQ;
    if (KS == 1 && (prb0 * 32 >= prow || qrb0 * 32 >= qrow)) return;
    const int prbmax = (prow + 31) / 32 - 1, qrbmax = (qrow + 31) / 32 - 1;
    // row blocks past the operand are clamped (their results are never stored)
    const uint4* src[NO];   // uniform
#pragma unroll
    for (int f = 0; f < NO; f++)
        src[f] = f < WTP ? Pc + (size_t)min(prb0 + f, prbmax) * KP * 64 : Qc + (size_t)min(qrb0 + (f - WTP), qrbmax) * KP * 64;
    v4u raw[NB][NO];
    v4u e[2][NO];   // a word's operands: P blocks, then Q blocks
    auto load = [&](int set, int pair) {   // (past the end: the last pair, not used)
        const size_t at = (size_t)min(pair, KP - 1) * 64;
#pragma unroll
        for (int f = 0; f < NO; f++) raw[set][f] = *reinterpret_cast<const v4u*>(src[f] + at + lane);
    };
    auto unpack = [&](int set, int word, int f) {
        constexpr uint32_t m = 0x33333333u;
        const uint32_t a = raw[set][f][2 * word], b = raw[set][f][2 * word + 1];
        e[word][f] = v4u{a & m, (a >> 2) & m, b & m, (b >> 2) & m};
    };
    v16f acc[WTP][WTQ];
    // word `word` of the pair in the operand set multiplied, and word `nword` of the pair in set `nset` unpacked
    auto step = [&](auto word, int nset) {
        constexpr int W = decltype(word)::value;
        static_for<NM>([&](auto mtag) {
            constexpr int m = decltype(mtag)::value;
            mfma_f4(acc[m / WTQ][m % WTQ], e[W][m / WTQ], e[W][WTP + m % WTQ]);
            static_for<(m + 1) * NO / NM - m * NO / NM>([&](auto ktag) { unpack(nset, 1 - W, m * NO / NM + decltype(ktag)::value); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    const int n = (KP - ks + KS - 1) / KS;   // pairs ks, ks + KS, ... of this wavefront (0 or less: none)
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int b = 0; b < WTQ; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[a][b][i] = 0.0f;
    if (n > 0) {
#pragma unroll
        for (int j = 0; j < NB; j++) load(j, ks + j * KS);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 0; f < NO; f++) unpack(0, 0, f);
        int pair = ks + NB * KS;   // the next one to ask for
        for (int i = 0; i < n; i += NB) {
            static_for<NB>([&](auto jtag) {
                constexpr int j = decltype(jtag)::value;
                if (j == 0 || i + j < n) {
                    step(std::integral_constant<int, 0>{}, j);
                    load(j, pair);
                    pair += KS;
                    __builtin_amdgcn_sched_barrier(0);
                    step(std::integral_constant<int, 1>{}, (j + 1) % NB);
                }
            });
        }
    }
    // dot = 4 sum - sum of the P row - sum of the Q row - lanes (off: with BNN's constant), all of it below 2^24; the sums are there for
    // whole blocks of rows.  All of them are read before the first store, which they would wait for (loads and stores are counted together and in
    // order): 123056 x 635 x 3328 225 -> 204 us, 9660 x 10247 x 256 118 -> 98.  Ahead of the operands they gain nothing more.
    typedef QuadOf<NM, KS> QO;
    auto result = [&](const float4& t, int i) {
        const int blk = QO::block(i, ks);
        const int4 s = *reinterpret_cast<const int4*>(sP + min(prb0 + blk / WTQ, prbmax) * 32 + 8 * QO::sub(i, ks) + 4 * (lane >> 5));
        const int o = sQ[min(qrb0 + blk % WTQ, qrbmax) * 32 + (lane & 31)] + off;
        auto prelu = [&](float v, int sp) {
            const float r = (float)((int)(v * 4.0f) - sp - o);
            return r < ro.lim ? r * ro.alpha : r;
        };
        return make_float4(prelu(t.x, s.x), prelu(t.y, s.y), prelu(t.z, s.z), prelu(t.w, s.w));
    };
    if constexpr (KS == 1) store_whole_sums<WTP, WTQ, NT>(acc, ro, prb0, qrb0, prow, qrow, lane, result);
    else meet_and_store<WTP, WTQ, KS, NT>(acc, lds, ro, prb0, qrb0, prow, qrow, ks, lane, result);
}

template <bool TP, bool TQ, int WT, int KS, bool NT>
hipError_t launch_rows_kernel(const char* P, const char* Q, int64_t prow, int64_t qrow, int G, const RowsOut& ro, hipStream_t st) {
    typedef RowsTile<TP, TQ, WT, WT, KS> TL;
    auto kern = k_rows<TP, TQ, WT, WT, KS, NT>;
    // the loads are counted by hand (s_waitcnt vmcnt(N)): a build with scratch accesses is refused; the opt-in to more than
    // 64 KiB of dynamic LDS is per kernel
    static const hipError_t configured = []() {
        const void* k = reinterpret_cast<const void*>(&k_rows<TP, TQ, WT, WT, KS, NT>);
        hipFuncAttributes attr;
        hipError_t e = hipFuncGetAttributes(&attr, k);
        if (e == hipSuccess && attr.localSizeBytes != 0) e = hipErrorLaunchFailure;
        if (e != hipSuccess) return e;
        return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)TL::lds);
    }();
    if (configured != hipSuccess) return configured;
    constexpr int edge = 32 * WT * TL::WV;
    const int64_t px = (prow + edge - 1) / edge, qy = (qrow + edge - 1) / edge;
    if (px * qy > kMaxRowsTiles) return hipErrorInvalidValue;
    RowsOrder od;
    od.tiles = (uint32_t)(px * qy);
    od.per_xcd = (od.tiles + 7) / 8;
    od.px = (uint32_t)px;
    od.band = make_fastdiv((uint32_t)(4 * qy));
    od.last = make_fastdiv((uint32_t)(px % 4 ? px % 4 : 4));
    hipLaunchKernelGGL(kern, dim3(8 * od.per_xcd), dim3(64 * TL::NW), TL::lds, st, P, Q, (int)prow, (int)qrow, G, od, ro);
    return hipGetLastError();
}
// A kernel per kind of store: deciding in the kernel costs a workgroup's end 0.1 us.  Whole calls from packed rows, us, past the caches only / by
// stores_past_caches: TBN 22240 x 1537 x 256 79 / 25, BNN 20021 x 2017 x 256 87 / 29, 12309 x 5416 x 512 142 / 55.
template <bool TP, bool TQ, int WT, int KS>
hipError_t launch_rows_tile(const char* P, const char* Q, int64_t prow, int64_t qrow, int G, const RowsOut& ro, hipStream_t st) {
    if constexpr (KS != 8)   // (256 tiles at most: small results)
        if (!ro.past_caches) return launch_rows_kernel<TP, TQ, WT, KS, false>(P, Q, prow, qrow, G, ro, st);
    return launch_rows_kernel<TP, TQ, WT, KS, true>(P, Q, prow, qrow, G, ro, st);
}

template <bool TP, bool TQ>
hipError_t launch_rows_types(const char* P, const char* Q, int64_t prow, int64_t qrow, int Kw, const RowsOut& ro, hipStream_t st) {
    switch (rows_form(prow, qrow, Kw)) {
        case 0: return launch_rows_tile<TP, TQ, 1, 4>(P, Q, prow, qrow, Kw / 4, ro, st);
        case 1: return launch_rows_tile<TP, TQ, 2, 4>(P, Q, prow, qrow, Kw / 4, ro, st);
        case 2: return launch_rows_tile<TP, TQ, 3, 4>(P, Q, prow, qrow, Kw / 4, ro, st);
        case 4: return launch_rows_tile<TP, TQ, 1, 1>(P, Q, prow, qrow, Kw / 4, ro, st);
        case 5: return launch_rows_tile<TP, TQ, 1, 8>(P, Q, prow, qrow, Kw / 4, ro, st);
        case 6: return launch_rows_tile<TP, TQ, 2, 1>(P, Q, prow, qrow, Kw / 4, ro, st);
        default: return launch_rows_tile<TP, TQ, 4, 4>(P, Q, prow, qrow, Kw / 4, ro, st);
    }
}

template <int WTP, int WTQ, int KS, int NB, bool NT>
hipError_t launch_packed_kernel(const uint4* P, const uint4* Q, int64_t prow, int64_t qrow, int KP, const int* sP, const int* sQ, int off,
                              const RowsOut& ro, hipStream_t st) {
    constexpr int WV = KS == 1 ? 2 : 1, EP = 32 * WTP * WV, EQ = 32 * WTQ * WV;
    constexpr int lds_bytes = KS == 1 ? 0 : meeting_blocks(WTP * WTQ, KS) * KS * 4096;
    static_assert(lds_bytes <= (160 << 10), "LDS of a compute unit");
    static const hipError_t configured =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_packed<WTP, WTQ, KS, NB, NT>), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (configured != hipSuccess) return configured;
    const int64_t px = (prow + EP - 1) / EP, qy = (qrow + EQ - 1) / EQ;
    if (px * qy > kMaxRowsTiles) return hipErrorInvalidValue;
    RowsOrder od;
    od.tiles = (uint32_t)(px * qy);
    od.per_xcd = (od.tiles + 7) / 8;
    od.px = (uint32_t)px;
    od.band = make_fastdiv((uint32_t)(4 * qy));
    od.last = make_fastdiv((uint32_t)(px % 4 ? px % 4 : 4));
    hipLaunchKernelGGL((k_packed<WTP, WTQ, KS, NB, NT>), dim3(8 * od.per_xcd), dim3(64 * (KS == 1 ? 4 : KS)), lds_bytes, st, P, Q, (int)prow, (int)qrow, KP, sP, sQ,
                       off, od, ro);
    return hipGetLastError();
}
template <int WTP, int WTQ, int KS, int NB>
hipError_t launch_packed_tile(const uint4* P, const uint4* Q, int64_t prow, int64_t qrow, int KP, const int* sP, const int* sQ, int off,
                              const RowsOut& ro, hipStream_t st) {
    if constexpr (KS != 8)
        if (!ro.past_caches) return launch_packed_kernel<WTP, WTQ, KS, NB, false>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st);
    return launch_packed_kernel<WTP, WTQ, KS, NB, true>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st);
}

}  // namespace

hipError_t launch_mm_rows(int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                          float alpha, float* d_y, hipStream_t st) {
    const bool at = type == kTNN || type == kTBN, wt = type == kTNN || type == kBTN;
    const bool nchw = OHW > 1;
    RowsOut ro;
    ro.y = d_y;
    ro.img_stride = (int64_t)KN * OHW;
    ro.p_stride = (uint32_t)(nchw ? OHW : KN);
    ro.img = make_fastdiv(nchw ? (uint32_t)OHW : 0xffffffffu);
    // BNN: the lanes past K_unpack are +1 in both operands and add 64 Kw - K_unpack (mm_p2_final_bnn_avx2.c:55-58)
    ro.bias = type == kBNN ? (float)(64 * Kw - K_unpack) : 0.0f;
    ro.lim = type == kTNN ? 0.5f : 0.0f;
    ro.alpha = alpha;
    ro.past_caches = stores_past_caches(nchw ? OHW : KN, M, KN);
    const char* P = reinterpret_cast<const char*>(nchw ? d_b : d_a);
    const char* Q = reinterpret_cast<const char*>(nchw ? d_a : d_b);
    const int64_t prow = nchw ? KN : M, qrow = nchw ? M : KN;
    const bool tp = nchw ? wt : at, tq = nchw ? at : wt;
    if (tp && tq) return launch_rows_types<true, true>(P, Q, prow, qrow, Kw, ro, st);
    if (tp) return launch_rows_types<true, false>(P, Q, prow, qrow, Kw, ro, st);
    if (tq) return launch_rows_types<false, true>(P, Q, prow, qrow, Kw, ro, st);
    return launch_rows_types<false, false>(P, Q, prow, qrow, Kw, ro, st);
}

bool launch_mm_packed(int type, const void* d_ac, const void* d_bc, const int* sA, const int* sB, int64_t M, int OHW, int KN, int Kw,
                      int K_unpack, float alpha, float* d_y, hipStream_t st, hipError_t* err) {
    const bool nchw = OHW > 1;
    RowsOut ro;
    ro.y = d_y;
    ro.img_stride = (int64_t)KN * OHW;
    ro.p_stride = (uint32_t)(nchw ? OHW : KN);
    ro.img = make_fastdiv(nchw ? (uint32_t)OHW : 0xffffffffu);
    ro.bias = 0.0f;
    ro.lim = type == kTNN ? 0.5f : 0.0f;
    ro.alpha = alpha;
    ro.past_caches = stores_past_caches(nchw ? OHW : KN, M, KN);
    const int off = 64 * Kw + (type == kBNN ? 64 * Kw - K_unpack : 0);   // the lanes of a row pair, padding included, and BNN's constant
    const uint4 *P = static_cast<const uint4*>(nchw ? d_bc : d_ac), *Q = static_cast<const uint4*>(nchw ? d_ac : d_bc);
    const int *sP = nchw ? sB : sA, *sQ = nchw ? sA : sB;
    const int64_t prow = nchw ? KN : M, qrow = nchw ? M : KN;
    const int KP = Kw / 2;
    auto go = [&](hipError_t e) {
        *err = e;
        return true;
    };
    switch (packed_form(prow, qrow, KP)) {
        case 0: return go(launch_packed_tile<1, 1, 4, 8>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 1: return go(launch_packed_tile<1, 1, 8, 8>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 2: return go(launch_packed_tile<1, 2, 4, 6>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 3: return go(launch_packed_tile<2, 1, 4, 6>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 4: return go(launch_packed_tile<2, 2, 4, 6>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 5: return go(launch_packed_tile<3, 3, 4, 4>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 6: return go(launch_packed_tile<4, 4, 4, 3>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 7: return go(launch_packed_tile<1, 1, 1, 6>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        case 8: return go(launch_packed_tile<2, 2, 1, 4>(P, Q, prow, qrow, KP, sP, sQ, off, ro, st));
        default: return false;
    }
}

}  // namespace ftnn
