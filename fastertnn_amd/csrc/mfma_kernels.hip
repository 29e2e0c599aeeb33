// Matrix-core formulation of the same GEMMs (gfx950): the comparison path to the
// vector-ALU popcount kernel of mm_kernels.hip, selected where it measures faster.
//
// Semantics are unchanged (src/tnns/mm_p2_final_{tnn,tbn,btn,bnn}_avx2.c): every
// accumulator is the integer dot product of the decoded {-1,0,+1} / {-1,+1} lanes,
// which is what the popcount formulas compute, so results stay bit-exact:
//   * MFMA int8  (v_mfma_i32_32x32x32_i8): lanes become bytes 0x01 / 0x00 / 0xFF, int32
//     accumulate;
//   * MFMA fp4   (v_mfma_f32_32x32x64_f8f6f4, E2M1): lanes become nibbles 0x2 / 0x0 / 0xA
//     (+1.0 / 0 / -1.0), fp32 accumulate -- exact while 64*Kw < 2^24, which the host
//     checks.  Twice the matrix rate of int8.  The conv layers keep both operands at two bits
//     per lane (records, see P2) and split them in registers; the fp4 GEMM engine itself
//     (k_pack4, k_mfma_p4 further down) codes a lane a as (a + 1) / 2, also at two bits.
//
// The kernels of the int8 engine:
//   k_expand  Packing-2 (or single-plane binary) rows -> "fragments": 1 KiB blocks
//             holding 32 rows x 32 lanes in exactly the register
//             layout of an MFMA operand (lane l = (k half l/32, row l%32), 16 bytes).
//             HBM-bound, one pass per operand.
//   k_mfma    256 x 256 output tile per workgroup (4 wavefronts, 128 x 128 each, 256
//             accumulator registers per lane).  Fragments travel global -> LDS with
//             LDS-direct loads (no VGPRs, and a fragment lands contiguously, so the
//             later 128-bit LDS reads are conflict-free without padding), through a
//             4-stage ring; one barrier per step.  LDS reads of the next fragment and
//             the DMA issue are interleaved with the MFMAs of the current one.
#include <type_traits>

#include "ftnn_internal.h"

namespace ftnn {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Ring of NS LDS buffers, each holding KF fragments per row-block: one barrier per KF fragments.
// A workgroup of 2 x 2 wavefronts computes (64 WTP) x (64 WTQ) results, a wavefront WTP x WTQ blocks of 32 x 32:
// 4 x 4 for problems with enough 256 x 256 tiles to fill the chip, 2 x 2 (128 x 128) below that.
template <int WTP, int WTQ, int KF, int NS>
struct Tile {
    static constexpr int RBP = 2 * WTP, RBQ = 2 * WTQ;   // row-blocks per operand side
    static constexpr int FR = (RBP + RBQ) * KF;          // fragments per step: the P row-blocks' first, then the Q ones'
    static constexpr int FW = FR / 4;                    // fragments staged by one wavefront per step
    static constexpr int NL = WTP + WTQ;                 // LDS reads per wavefront and k fragment
    static constexpr int NM = WTP * WTQ;                 // multiplies per wavefront and k fragment
    static constexpr int DPI = FW / NL;                  // fragments a wavefront stages per LDS read of the last fragment
    static constexpr size_t lds_bytes = (size_t)NS * FR * 1024;
    static_assert(FR % 4 == 0 && FW % NL == 0, "whole staged fragments per wavefront and per LDS read");
    static_assert(NS >= 2 && KF % 2 == 0, "register sets alternate per fragment");
};

// ------------------------------------------------------------------ expansion
// grid (row-blocks, groups / 4), block 256: thread = (row r = t%32, dword pair dq = t/32).
// A group is 4 words (256 lanes) of a packed row: 16 dwords (8 sign, 8 zero) for ternary
// rows, 8 dwords for binary rows.  Rows past `rows` expand to zeros.
// FORM: int8 fragments, or records of two bits per lane (see P2) as blocks [row block][pair of K words][lane l = (word of the
// pair l / 32, row l % 32)][16 bytes], in the layers' lane order or in natural order.
enum { FORM_I8, FORM_REC, FORM_REC_NATURAL };

// four lanes per byte, bit i of a byte -> the lanes' places in a record byte (1, 0, 5, 4); shifted by two for the signs
__device__ __forceinline__ uint32_t spread_lanes(uint32_t v) {
    v &= 0x0F0F0F0Fu;
    return ((v & 0x09090909u) << 1) | ((v >> 1) & 0x01010101u) | ((v << 3) & 0x20202020u);
}

template <int FORM, bool TERN>
__device__ __forceinline__ void expand_block(const uint32_t* __restrict__ P, int rows, int G, uint4* __restrict__ out, int rb,
                                             int gy, uint32_t* stage, uint32_t* __restrict__ kept = nullptr) {
    // A workgroup expands kGPB adjacent groups of its 32 rows: 256 contiguous bytes of each ternary row (128 of a
    // binary one).  They are fetched row-wise, 16 bytes per thread with neighbouring threads on neighbouring bytes,
    // and turned through LDS into the (row, dword) order the expansion works in: fetched in that order directly,
    // every load instruction would touch 32 cache lines for 256 bytes.
    constexpr int kGPB = 4;
    constexpr int DPG = TERN ? 16 : 8;        // dwords per group and row
    constexpr int RD = kGPB * DPG;            // dwords per row in the block: 64 / 32
    constexpr int RS = RD + 1;                // LDS row stride: odd, the 32 rows of a read hit 32 banks
    const int g0 = gy * kGPB, t = threadIdx.x;
    {
        constexpr int PPR = RD / 4;           // 16-byte pieces per row: 16 / 8
        const int gmax = min(kGPB, G - g0) * (DPG / 4);   // pieces of a row that exist
#pragma unroll
        for (int k = 0; k < (32 * PPR) / 256; k++) {
            const int idx = t + 256 * k, rr = idx / PPR, pc = idx - rr * PPR;
            const int srow = min(rb * 32 + rr, rows - 1);
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (pc < gmax) v = *reinterpret_cast<const uint4*>(P + ((size_t)srow * G + g0) * DPG + pc * 4);
            if (kept && pc < gmax && rb * 32 + rr < rows) *reinterpret_cast<uint4*>(kept + ((size_t)srow * G + g0) * DPG + pc * 4) = v;
            uint32_t* d = stage + rr * RS + pc * 4;
            d[0] = v.x;
            d[1] = v.y;
            d[2] = v.z;
            d[3] = v.w;
        }
    }
    __syncthreads();
    const int r = t & 31, dq = t >> 5;
    const bool live = rb * 32 + r < rows;
    uint32_t sv[kGPB], zv[kGPB];
#pragma unroll
    for (int i = 0; i < kGPB; i++) {
        sv[i] = stage[r * RS + i * DPG + dq];
        zv[i] = TERN ? stage[r * RS + i * DPG + 8 + dq] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kGPB; i++) {
        const int g = g0 + i;
        if (g >= G) break;
        const uint32_t nz = live ? ~zv[i] : 0u;
        const uint32_t s = sv[i] & nz;   // a lane flagged zero is zero whatever its sign bit says
        if constexpr (FORM != FORM_I8) {
            const int w = g * 4 + (dq >> 1), half = dq & 1;   // this thread: 32 lanes of word w
            uint2* rec = reinterpret_cast<uint2*>(out + ((size_t)rb * (G * 2) + (w >> 1)) * 64 + (w & 1) * 32 + r) + half;
            if constexpr (FORM == FORM_REC) {
                // dwords `half` and 2 + `half` of the record; the threads of the two halves of a word are lanes l and l + 32:
                // the swap gives the lower one dwords 0 and 1, the upper one 2 and 3
                const uint32_t d0 = spread_lanes(nz) | spread_lanes(s) << 2, d1 = spread_lanes(nz >> 4) | spread_lanes(s >> 4) << 2;
                const auto d = __builtin_amdgcn_permlane32_swap(d0, d1, false, false);
                *rec = make_uint2(d[0], d[1]);
            } else {
                uint32_t o[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {   // eight lanes -> eight nibbles, sign << 3 | nonzero << 1
                    uint32_t a = (s >> (8 * q)) & 0xffu, b = (nz >> (8 * q)) & 0xffu;
                    a = (a | (a << 12)) & 0x000F000Fu;
                    a = (a | (a << 6)) & 0x03030303u;
                    a = (a | (a << 3)) & 0x11111111u;
                    b = (b | (b << 12)) & 0x000F000Fu;
                    b = (b | (b << 6)) & 0x03030303u;
                    b = (b | (b << 3)) & 0x11111111u;
                    o[q] = (a << 3) | (b << 1);
                }
                *rec = make_uint2(p2_join(o[0], o[1]), p2_join(o[2], o[3]));
            }
        } else {
            // fragment = one 32-lane dword: its two 16-lane halves are the k halves
            uint4* frag = out + ((size_t)rb * (G * 8) + (g * 8 + dq)) * 64;
#pragma unroll
            for (int half = 0; half < 2; half++) {
                const uint32_t sh = (s >> (16 * half)) & 0xffffu, nh = (nz >> (16 * half)) & 0xffffu;
                uint32_t o[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    // 4 bits -> 4 byte LSBs: bit i lands on bit 8i, no carries
                    const uint32_t sb = (((sh >> (4 * q)) & 15u) * 0x204081u) & 0x01010101u;
                    const uint32_t nb = (((nh >> (4 * q)) & 15u) * 0x204081u) & 0x01010101u;
                    o[q] = nb | (sb * 0xffu);
                }
                frag[half * 32 + r] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
    }
}

// kept: where the packed rows themselves are copied to on the way (a copy of its own costs the caller 20 us), or null
template <int FORM, bool TERN>
__global__ __launch_bounds__(256) void k_expand(const uint32_t* __restrict__ P, int rows, int G, uint4* __restrict__ out,
                                                uint32_t* __restrict__ kept) {
    __shared__ uint32_t stage[32 * 65];
    expand_block<FORM, TERN>(P, rows, G, out, blockIdx.x, blockIdx.y, stage, kept);
}

// both int8 operands of a GEMM in one launch (the same K): the first ceil(rows_a / 32) workgroup columns expand A, the others B
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_expand2(const uint32_t* __restrict__ Pa, int rows_a, uint4* __restrict__ out_a,
                                                 const uint32_t* __restrict__ Pb, int rows_b, uint4* __restrict__ out_b, int G) {
    __shared__ uint32_t stage[32 * 65];
    const int rba = (rows_a + 31) / 32;
    if ((int)blockIdx.x < rba) expand_block<FORM_I8, TA>(Pa, rows_a, G, out_a, blockIdx.x, blockIdx.y, stage);
    else expand_block<FORM_I8, TB>(Pb, rows_b, G, out_b, (int)blockIdx.x - rba, blockIdx.y, stage);
}

// ----------------------------------------------------------------------- GEMM
template <bool F4>
struct Acc {
    typedef v16i type;
};
template <>
struct Acc<true> {
    typedef v16f type;
};

template <bool F4>
__device__ __forceinline__ void mfma(typename Acc<F4>::type& c, const uint4& a, const uint4& b) {
    if constexpr (F4) {
        const v8i va = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
        const v8i vb = {(int)b.x, (int)b.y, (int)b.z, (int)b.w, 0, 0, 0, 0};
        // cbsz = blgp = 4: both operands E2M1; scale operands 0 select the unscaled instruction
        c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(va, vb, c, 4, 4, 0, 0, 0, 0);
    } else {
        const v4i va = {(int)a.x, (int)a.y, (int)a.z, (int)a.w};
        const v4i vb = {(int)b.x, (int)b.y, (int)b.z, (int)b.w};
        c = __builtin_amdgcn_mfma_i32_32x32x32_i8(va, vb, c, 0, 0, 0);
    }
}

// LDS-direct load of 16 bytes per lane: the 64 lanes land contiguously at lds_byte_addr.
// Issued through inline asm so that the compiler does not order its own LDS reads against
// it; the kernel waits for it by hand (s_waitcnt vmcnt before the barrier that publishes
// the buffer).  M0 carries the LDS address; one wait state is required after writing M0.
__device__ __forceinline__ void dma16(const uint4* gsrc, uint32_t lds_byte_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gsrc), "{m0}"(lds_byte_addr) : "memory");
}

// Epilogue of the GEMM kernels: r = acc - bias, then PReLU in the reference's form for the type (form 0 "f = r; if
// (f <= 0) f *= alpha", mm_p2_final_tnn_avx2.c:204-208; form 1 "r >= 0 ? r : alpha * r", mm_p2_final_tbn_avx2.c:73), stored
// row-major (SWAP = false, OHW == 1) or in NCHW order.  Accumulator e of block (a, b): P row = 32 * (prb + a) + 8 * (e / 4)
// + 4 * (lane / 32) + e % 4, Q row = 32 * (qrb + b) + lane % 32.
template <bool F4, bool SWAP, bool NT, int WTP, int WTQ>
__device__ __forceinline__ void store_tile(const typename Acc<F4>::type (&acc)[WTP][WTQ], float* __restrict__ Y, int M, int KN,
                                           int OHW, int prb, int qrb, int lane, int bias, int form, float alpha) {
    const bool le_form = form == 0;
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int b = 0; b < WTQ; b++) {
            const int q = (qrb + b) * 32 + (lane & 31);
            const int pbase = (prb + a) * 32 + 4 * (lane >> 5);
            size_t qoff;
            if (SWAP) {   // q = i is fixed per block: split it into (image, pixel) once
                const int img = q / OHW;
                qoff = (size_t)img * KN * OHW + (q - img * OHW);
            } else {
                qoff = (size_t)q;
            }
            const bool qok = q < (SWAP ? M : KN);
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int p = pbase + 8 * (e >> 2) + (e & 3);
                const int r = (int)acc[a][b][e] - bias;
                const float fr = (float)r;
                // form 0: scale when f <= 0 (a zero becomes 0 * alpha); form 1: scale when r < 0
                const bool scale = le_form ? (fr <= 0.0f) : (r < 0);
                const float f = scale ? fr * alpha : fr;
                const size_t o = SWAP ? qoff + (size_t)p * OHW : (size_t)p * KN + qoff;
                if (qok && p < (SWAP ? KN : M)) {
                    if (NT) __builtin_nontemporal_store(f, &Y[o]);
                    else Y[o] = f;
                }
            }
        }
}

// P operand = MFMA A side (its rows index the accumulator registers), Q operand = MFMA B
// side (its rows run along the lanes).  SWAP = false: P = activation rows i, Q = weight
// rows j (lanes along j: contiguous for a row-major m x n result).  SWAP = true: P =
// weights, Q = activations (lanes along i: contiguous for an NCHW result with OHW > 1).
// The epilogue computes r = acc - bias, then PReLU in the reference's form for the type:
// form 0 "f = r; if (f <= 0) f *= alpha" (mm_p2_final_tnn_avx2.c:204-208), form 1
// "r >= 0 ? r : alpha * r" (mm_p2_final_tbn_avx2.c:73).
template <bool SWAP, bool NT, int WTP, int WTQ, int kKF, int kNS>
__global__ __launch_bounds__(256) void k_mfma(const uint4* __restrict__ Pf, const uint4* __restrict__ Qf,
                                              float* __restrict__ Y, int M, int KN, int OHW, int KB,
                                              int bias, int form, float alpha) {
    extern __shared__ uint4 lds[];   // kNS buffers of kFR KiB
    typedef Acc<false>::type acc_t;
    typedef Tile<WTP, WTQ, kKF, kNS> TL;
    constexpr int RBP = TL::RBP, RBQ = TL::RBQ, kFR = TL::FR, kFW = TL::FW, NL = TL::NL, NM = TL::NM, DPI = TL::DPI;
    constexpr int kPF = RBP * kKF;   // fragments of the P side per step
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wy = wave >> 1, wx = wave & 1;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
    const int prb0 = blockIdx.x * RBP, qrb0 = blockIdx.y * RBQ;
    const int prbmax = (prow + 31) / 32 - 1, qrbmax = (qrow + 31) / 32 - 1;
    acc_t acc[WTP][WTQ];
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int b = 0; b < WTQ; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[a][b][e] = 0;

    // fragment f of a step: the P side's kPF fragments first (row-block f / kKF, k fragment f % kKF), then the Q
    // side's; row-blocks past the operand are clamped (their results are never stored)
    const uint4* src[kFW];
#pragma unroll
    for (int i = 0; i < kFW; i++) {
        const int f = wave * kFW + i;
        const bool qside = f >= kPF;
        const int g = qside ? f - kPF : f, rbi = g / kKF, kbi = g % kKF;
        const uint4* base = !qside ? Pf + ((size_t)min(prb0 + rbi, prbmax) * KB + kbi) * 64
                                   : Qf + ((size_t)min(qrb0 + rbi, qrbmax) * KB + kbi) * 64;
        src[i] = base + lane;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
    const int nstep = KB / kKF;
    uint4 fa[2][WTP], fb[2][WTQ];
    // one LDS read of fragment k of buffer `buf` into register set `set`, in the order the MFMAs
    // consume them: i = 0: fa0, 1..WTQ: fb0..fb(WTQ-1), then fa1..fa(WTP-1)
    auto ldone = [&](int buf, int k, int set, int i) {
        const uint4* L = lds + (size_t)buf * kFR * 64;
        if (i == 0) fa[set][0] = L[((wy * WTP + 0) * kKF + k) * 64 + lane];
        else if (i <= WTQ) fb[set][i - 1] = L[((RBP + wx * WTQ + (i - 1)) * kKF + k) * 64 + lane];
        else fa[set][i - WTQ] = L[((wy * WTP + (i - WTQ)) * kKF + k) * 64 + lane];
    };
    // the multiplies that go with LDS read i: the NM of a k fragment spread evenly over its NL reads (WT / 2 each on a
    // square tile), in the order (a, b) = (m / WTQ, m % WTQ)
    auto mfma2 = [&](int set, int i) {
#pragma unroll
        for (int m = i * NM / NL; m < (i + 1) * NM / NL; m++) mfma<false>(acc[m / WTQ][m % WTQ], fa[set][m / WTQ], fb[set][m % WTQ]);
    };
    auto stage = [&](int step) {
        const uint32_t dst = lds0 + (uint32_t)(step % kNS) * (kFR * 1024);
#pragma unroll
        for (int i = 0; i < kFW; i++) dma16(src[i] + (size_t)step * kKF * 64, dst + (uint32_t)(wave * kFW + i) * 1024);
    };
    // prologue: the first kNS stages in flight, wait for stage 0 only
#pragma unroll
    for (int p = 0; p < kNS; p++)
        if (p < nstep) stage(p);
    if (nstep >= kNS) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFW * (kNS - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NL; i++) ldone(0, 0, 0, i);

    auto step_body = [&](int s, auto full_tag) {
        constexpr bool FULL = decltype(full_tag)::value;   // FULL: s + kNS < nstep
#pragma unroll
        for (int k = 0; k < kKF; k++) {
            const int set = k & 1;
            if (k + 1 < kKF) {
#pragma unroll
                for (int i = 0; i < NL; i++) {
                    ldone(s % kNS, k + 1, set ^ 1, i);
                    mfma2(set, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // Last fragment of the step: all of this step is in registers.  Stage s+1 must
                // have landed (stages s+2 .. s+kNS-1 may still be in flight); after the barrier
                // buffer s % kNS is free for stage s+kNS.
                if (FULL || s + kNS - 1 < nstep) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFW * (kNS - 2)) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                const bool do_ld = FULL || s + 1 < nstep;
                const uint32_t dst = lds0 + (uint32_t)(s % kNS) * (kFR * 1024);
#pragma unroll
                for (int i = 0; i < NL; i++) {
                    if (FULL) {
#pragma unroll
                        for (int j = 0; j < DPI; j++)
                            dma16(src[i * DPI + j] + (size_t)(s + kNS) * kKF * 64, dst + (uint32_t)(wave * kFW + i * DPI + j) * 1024);
                    }
                    if (do_ld) ldone((s + 1) % kNS, 0, set ^ 1, i);
                    mfma2(set, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    int s = 0;
    for (; s + kNS < nstep; s++) step_body(s, std::true_type{});
    for (; s < nstep; s++) step_body(s, std::false_type{});

    store_tile<false, SWAP, NT, WTP, WTQ>(acc, Y, M, KN, OHW, prb0 + wy * WTP, qrb0 + wx * WTQ, lane, bias, form, alpha);
}

// ------------------------------------------------- fp4 operands at two bits per lane, offset codes
// The fp4 GEMM is bound by power, not by its schedule.  The same instruction stream runs a quarter faster on
// operands that are all zero, and a chain of nothing but these MFMAs on registers holds 2.39 GHz on zeros, 2.25 GHz on
// lanes of {0, 0.5, 1} and 1.97 GHz on lanes of {-1, 0, +1}: it is the mixed signs in the adder trees and the operand
// bytes on the move (L2 -> LDS -> registers) that hold the clock down.  The GEMM's own operand form answers both:
//
//   offset codes   a lane a in {-1, 0, +1} travels as a' = (a + 1) / 2 in {0, 0.5, 1}, E2M1 codes 0, 1, 2: no negative
//                  product anywhere.  With S = sum a' b' over all L = 64 Kw lanes of a row pair (padding lanes are
//                  a = b = 0 or +-1 like any other and enter the sums below the same way)
//                      sum a b = 4 S - sum a - sum b - L,
//                  exact in fp32 while 4 L <= 2^24 (S is a multiple of 1/4 below L).  The row sums are counted when
//                  the operand is packed and sit behind its blocks; the epilogue undoes the offset.
//   two bits       codes 0, 1, 2 use bits 0 and 1 of a nibble, so two dwords of nibbles D0, D1 share one dword,
//                  P = D0 | D1 << 2, and come apart with D0 = P & 0x33333333, D1 = (P >> 2) & 0x33333333: 1.5 vector
//                  instructions per dword, issued beside the MFMAs.  Half the bytes in HBM, through L2 -> LDS and
//                  through the LDS reads.
//
// Layout ("packed4"): 1 KiB blocks [row block of 32][pair of K words][lane l = (k half l / 32, row l % 32)][16 bytes], the
// 16 bytes of a lane being (P0, P1) of the even K word and (P0, P1) of the odd one, P0 = D0 | D1 << 2, P1 = D2 | D3 << 2
// with D0 .. D3 the 32 lanes of the lane's k half as nibbles in offset codes, eight to a dword.  One LDS-direct load of 16 bytes
// per lane moves a row block's two K words.  Behind the blocks: one int32 per row (rows rounded up to 32), sum of the
// row's lanes.

// zeroes p[0 .. n) and q[0 .. m) (m may be 0)
__global__ void k_zero_i32(int* __restrict__ p, int n, int* __restrict__ q, int m) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
    else if (i - n < m) q[i - n] = 0;
}

// grid (row blocks, groups / 4), block 256: as k_expand, writing the packed4 layout (Kw words per row) and
// adding the lanes of its rows into sums (zeroed before the launch)
template <bool TERN>
__device__ __forceinline__ void pack4_block(const uint32_t* __restrict__ P, int rows, int G, uint2* __restrict__ out,
                                            int* __restrict__ sums, int rb, int gy, uint32_t* stage, int* rowsum) {
    constexpr int kGPB = 4;
    constexpr int DPG = TERN ? 16 : 8;        // dwords per group and row
    constexpr int RD = kGPB * DPG;            // dwords per row in the block
    constexpr int RS = RD + 1;                // LDS row stride: odd, the 32 rows of a read hit 32 banks
    const int g0 = gy * kGPB, t = threadIdx.x;
    if (t < 32) rowsum[t] = 0;
    {
        constexpr int PPR = RD / 4;           // 16-byte pieces per row
        const int gmax = min(kGPB, G - g0) * (DPG / 4);
#pragma unroll
        for (int k = 0; k < (32 * PPR) / 256; k++) {
            const int idx = t + 256 * k, rr = idx / PPR, pc = idx - rr * PPR;
            const int srow = min(rb * 32 + rr, rows - 1);
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (pc < gmax) v = *reinterpret_cast<const uint4*>(P + ((size_t)srow * G + g0) * DPG + pc * 4);
            uint32_t* d = stage + rr * RS + pc * 4;
            d[0] = v.x;
            d[1] = v.y;
            d[2] = v.z;
            d[3] = v.w;
        }
    }
    __syncthreads();
    const int r = t & 31, dq = t >> 5;        // dq: dword of the group = (K word dq / 2, k half dq % 2)
    int lanesum = 0;
#pragma unroll
    for (int i = 0; i < kGPB; i++) {
        const int g = g0 + i;
        if (g >= G) break;
        const uint32_t sv = stage[r * RS + i * DPG + dq];
        const uint32_t zero = TERN ? stage[r * RS + i * DPG + 8 + dq] : 0u;
        const uint32_t plus = ~(sv | zero), minus = sv & ~zero;
        lanesum += __popc(plus) - __popc(minus);
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {   // 8 lanes -> 8 nibbles: bit i lands on bit 4 i
            uint32_t a = (plus >> (8 * q)) & 0xffu, b = (zero >> (8 * q)) & 0xffu;
            a = (a | (a << 12)) & 0x000F000Fu;
            a = (a | (a << 6)) & 0x03030303u;
            a = (a | (a << 3)) & 0x11111111u;
            b = (b | (b << 12)) & 0x000F000Fu;
            b = (b | (b << 6)) & 0x03030303u;
            b = (b | (b << 3)) & 0x11111111u;
            o[q] = (a << 1) | b;        // +1 -> 2 (1.0), 0 -> 1 (0.5), -1 -> 0
        }
        const int w = g * 4 + (dq >> 1), h = dq & 1;   // K word and k half of this thread's 32 lanes
        const size_t block = (size_t)rb * (G * 2) + (w >> 1);
        out[(block * 64 + h * 32 + r) * 2 + (w & 1)] = make_uint2(o[0] | (o[1] << 2), o[2] | (o[3] << 2));
    }
    atomicAdd(&rowsum[r], lanesum);
    __syncthreads();
    if (t < 32 && rb * 32 + t < rows) atomicAdd(&sums[rb * 32 + t], rowsum[t]);
}

template <bool TERN>
__global__ __launch_bounds__(256) void k_pack4(const uint32_t* __restrict__ P, int rows, int G, uint2* __restrict__ out,
                                               int* __restrict__ sums) {
    __shared__ uint32_t stage[32 * 65];
    __shared__ int rowsum[32];
    pack4_block<TERN>(P, rows, G, out, sums, blockIdx.x, blockIdx.y, stage, rowsum);
}

// both operands of a GEMM in one launch, as k_expand2
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_pack4_2(const uint32_t* __restrict__ Pa, int rows_a, uint2* __restrict__ out_a,
                                                 int* __restrict__ sums_a, const uint32_t* __restrict__ Pb, int rows_b,
                                                 uint2* __restrict__ out_b, int* __restrict__ sums_b, int G) {
    __shared__ uint32_t stage[32 * 65];
    __shared__ int rowsum[32];
    const int rba = (rows_a + 31) / 32;
    if ((int)blockIdx.x < rba) pack4_block<TA>(Pa, rows_a, G, out_a, sums_a, blockIdx.x, blockIdx.y, stage, rowsum);
    else pack4_block<TB>(Pb, rows_b, G, out_b, sums_b, (int)blockIdx.x - rba, blockIdx.y, stage, rowsum);
}

// (P0, P1) of one K word -> the lane's 16 bytes of nibbles
__device__ __forceinline__ uint4 unpack4(uint32_t p0, uint32_t p1) {
    constexpr uint32_t m = 0x33333333u;
    return make_uint4(p0 & m, (p0 >> 2) & m, p1 & m, (p1 >> 2) & m);
}

// The epilogue of the offset form: dot = 4 acc - sum of the P row - sum of the Q row - lanes, then as store_tile
// (off = lanes + the BNN bias).  sums: the tile's row sums in LDS, RB * 32 of the P side, then RB * 32 of the Q side
// (zero for rows past the operand, which store nothing).
template <bool SWAP, bool NT, int WT>
__device__ __forceinline__ void store_tile_offset(const Acc<true>::type (&acc)[WT][WT], float* __restrict__ Y, int M, int KN, int OHW,
                                                  int prb, int qrb, int lane, const int* sums, int wy, int wx, int off, int form,
                                                  float alpha) {
    constexpr int RB = 2 * WT;
    const bool le_form = form == 0;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
#pragma unroll
    for (int a = 0; a < WT; a++) {
        int4 sp[4];   // the lane's 16 P rows of this block: rows 4 * (lane / 32) + 8 * j + (0..3)
#pragma unroll
        for (int j = 0; j < 4; j++) sp[j] = *reinterpret_cast<const int4*>(sums + (wy * WT + a) * 32 + 4 * (lane >> 5) + 8 * j);
        const int pbase = (prb + a) * 32 + 4 * (lane >> 5);
#pragma unroll
        for (int b = 0; b < WT; b++) {
            const int q = (qrb + b) * 32 + (lane & 31);
            const bool qok = q < qrow;
            const int sq = sums[RB * 32 + (wx * WT + b) * 32 + (lane & 31)] + off;
            size_t qoff;
            if (SWAP) {   // q = i is fixed per block: split it into (image, pixel) once
                const int img = q / OHW;
                qoff = (size_t)img * KN * OHW + (q - img * OHW);
            } else {
                qoff = (size_t)q;
            }
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int p = pbase + 8 * (e >> 2) + (e & 3);
                const int4& s4 = sp[e >> 2];
                const int spv = (e & 3) == 0 ? s4.x : (e & 3) == 1 ? s4.y : (e & 3) == 2 ? s4.z : s4.w;
                const int r = (int)(acc[a][b][e] * 4.0f) - spv - sq;
                const float fr = (float)r;
                const bool scale = le_form ? (fr <= 0.0f) : (r < 0);
                const float f = scale ? fr * alpha : fr;
                const size_t o = SWAP ? qoff + (size_t)p * OHW : (size_t)p * KN + qoff;
                if (qok && p < prow) {
                    if (NT) __builtin_nontemporal_store(f, &Y[o]);
                    else Y[o] = f;
                }
            }
        }
    }
}

// The fp4 GEMM on packed4 operands.  Same tiling as k_mfma<true, ...> (2 x 2 wavefronts, 4 x 4 blocks of 32 x 32 each,
// steps of two K words, ring of four stages filled by LDS-direct loads that the kernel counts by hand), with one 1 KiB block
// per row block and step.  A step: the first K word's 16 multiplies run while the second one's operands are unpacked;
// then the barrier; the second K word's multiplies run beside the loads of stage s + kNS and the LDS reads of stage
// s + 1, one read per slot of two multiplies (a 16-byte LDS read holds the wavefront's issue for 16 cycles), each block
// unpacked LAG slots after its read -- the last LAG blocks in the first slots of the next step.
struct TileP4 {
    static constexpr int WT = 4, NS = 4;
    static constexpr size_t lds_bytes = (size_t)NS * 4 * WT * 1024;
};
template <bool SWAP, bool NT>
__global__ __launch_bounds__(256) void k_mfma_p4(const uint4* __restrict__ Pc, const uint4* __restrict__ Qc, float* __restrict__ Y,
                                                 int M, int KN, int OHW, int KP, const int* __restrict__ sP,
                                                 const int* __restrict__ sQ, int off, int form, float alpha) {
    extern __shared__ uint4 lds[];   // kNS stages of kFR KiB
    typedef typename Acc<true>::type acc_t;
    constexpr int WT = TileP4::WT, kNS = TileP4::NS, RB = 2 * WT, kFR = 2 * RB, kFW = kFR / 4, NL = 2 * WT;   // kFW = WT blocks staged per wavefront and step
    static_assert(NL % kFW == 0 && (NL / 2) % 2 == 0, "loads and reads spread evenly over the slots");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wy = wave >> 1, wx = wave & 1;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
    const int prb0 = blockIdx.x * RB, qrb0 = blockIdx.y * RB;
    const int prbmax = (prow + 31) / 32 - 1, qrbmax = (qrow + 31) / 32 - 1;
    acc_t acc[WT][WT];
#pragma unroll
    for (int a = 0; a < WT; a++)
#pragma unroll
        for (int b = 0; b < WT; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[a][b][e] = 0;

    // block f of a stage: side f / RB (0 = P, 1 = Q), row block f % RB; row blocks past the operand are clamped
    const uint4* src[kFW];
#pragma unroll
    for (int i = 0; i < kFW; i++) {
        const int f = wave * kFW + i;
        const int side = f / RB, rbi = f % RB;
        const uint4* base = side == 0 ? Pc + (size_t)min(prb0 + rbi, prbmax) * KP * 64 : Qc + (size_t)min(qrb0 + rbi, qrbmax) * KP * 64;
        src[i] = base + lane;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
    const int nstep = KP;
    auto stage = [&](int step) {
        const uint32_t dst = lds0 + (uint32_t)(step % kNS) * (kFR * 1024) + wave * (kFW * 1024);
#pragma unroll
        for (int i = 0; i < kFW; i++) dma16(src[i] + (size_t)step * 64, dst + i * 1024);
    };
    // raw: the packed blocks of the stage being consumed; e[k]: the unpacked operands of its K word k.  Slots in the
    // order the multiplies take them: 0: P block 0, 1..WT: Q blocks, then P blocks 1..WT-1.
    uint4 ra[WT], rq[WT], ea[2][WT], eq[2][WT];
    auto read_raw = [&](int buf, int i) {
        const uint4* L = lds + (size_t)buf * kFR * 64;
        if (i == 0) ra[0] = L[(wy * WT + 0) * 64 + lane];
        else if (i <= WT) rq[i - 1] = L[(RB + wx * WT + (i - 1)) * 64 + lane];
        else ra[i - WT] = L[(wy * WT + (i - WT)) * 64 + lane];
    };
    auto unpack = [&](int k, int i) {
        const uint4& r = i == 0 ? ra[0] : (i <= WT ? rq[i - 1] : ra[i - WT]);
        const uint4 v = k == 0 ? unpack4(r.x, r.y) : unpack4(r.z, r.w);
        if (i == 0) ea[k][0] = v;
        else if (i <= WT) eq[k][i - 1] = v;
        else ea[k][i - WT] = v;
    };
    auto mfma2 = [&](int k, int i) {
#pragma unroll
        for (int j = 0; j < WT / 2; j++) {
            const int m = (WT / 2) * i + j;
            mfma<true>(acc[m / WT][m % WT], ea[k][m / WT], eq[k][m % WT]);
        }
    };

    // prologue: the first kNS stages in flight, wait for stage 0 only
#pragma unroll
    for (int p = 0; p < kNS; p++)
        if (p < nstep) stage(p);
    if (nstep >= kNS) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFW * (kNS - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NL; i++) read_raw(0, i);
#pragma unroll
    for (int i = 0; i < NL; i++) unpack(0, i);

    // slots between the LDS read of a block and its unpacking: far enough for the read to have landed, near enough for
    // every block to be unpacked by the slot that multiplies it first (block b: slot 0 for P block 0, (b - 1) / (WT / 2)
    // for Q block b - 1, 2 (b - WT) for P block b - WT)
    constexpr int LAG = 4;
    static_assert(LAG <= NL - 1 && LAG <= NL - WT + (WT - 1) / (WT / 2) && LAG <= WT + 1, "a block is unpacked before its first multiply");
    auto step_body = [&](int s, auto full_tag) {
        constexpr bool FULL = decltype(full_tag)::value;   // FULL: s + kNS < nstep
        // first K word: multiply, and unpack the second one's operands (their packed blocks arrived a phase ago); the
        // first LAG slots also unpack the last LAG blocks of this stage's first K word, read at the end of the step before
#pragma unroll
        for (int i = 0; i < NL; i++) {
            if (i < LAG && s > 0) unpack(0, NL - LAG + i);
            unpack(1, i);
            mfma2(0, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Everything of this stage is in registers.  Stage s + 1 must have landed (stages s + 2 .. s + kNS - 1 may
        // still be in flight); after the barrier buffer s % kNS is free for stage s + kNS.
        if (FULL || s + kNS - 1 < nstep) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFW * (kNS - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const bool do_ld = FULL || s + 1 < nstep;
        const uint32_t dst = lds0 + (uint32_t)(s % kNS) * (kFR * 1024) + wave * (kFW * 1024);
        // second K word: every slot issues one LDS read of the next stage and unpacks the block read LAG slots before;
        // the first kFW slots also issue the loads of stage s + kNS
#pragma unroll
        for (int i = 0; i < NL; i++) {
            if (do_ld) read_raw((s + 1) % kNS, i);
            if (FULL && i < kFW) dma16(src[i] + (size_t)(s + kNS) * 64, dst + i * 1024);
            if (do_ld && i >= LAG) unpack(0, i - LAG);
            mfma2(1, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + kNS < nstep; s++) step_body(s, std::true_type{});
    for (; s < nstep; s++) step_body(s, std::false_type{});

    // the tile's row sums through LDS (every load of the ring has landed and been read: the last steps wait for all)
    __syncthreads();
    int* sums = reinterpret_cast<int*>(lds);
    if (tid < RB * 32) {
        const int pr = prb0 * 32 + tid, qr = qrb0 * 32 + tid;
        sums[tid] = pr < prow ? sP[pr] : 0;
        sums[RB * 32 + tid] = qr < qrow ? sQ[qr] : 0;
    }
    __syncthreads();
    store_tile_offset<SWAP, NT, WT>(acc, Y, M, KN, OHW, prb0 + wy * WT, qrb0 + wx * WT, lane, sums, wy, wx, off, form, alpha);
}

// ------------------------------------------------------------ conv layers as workgroup tiles (fp4, records)
// Large layers.  2 x 2 wavefronts per workgroup, WTP x WTQ blocks of 32 x 32 each: (64 WTP) x (64 WTQ) results.  P side:
// weights, Q side: pixels (SWAP; without it, for one-pixel images, P = rows of the activations and Q = weights, row-major).
// Both operands are blocks of records: 1 KiB = 32 rows x two K words, lane l = (word of the pair l / 32, row l % 32).  A stage
// of the LDS ring holds one pair of every row block, filled by LDS-direct loads that the kernel counts by hand; a block is one
// 16-byte read per lane, split into the nibbles of two multiplies (lanes of both words of a pair enter both, see P2).  The
// schedule is k_mfma_p4's: the first word's multiplies run while the second one's operands are split; then, behind the barrier, the
// second word's multiplies run beside the LDS reads of the next pair, each block split LAG slots
// after its read.  At four bits per lane a step of two K words moved 72 KiB through the LDS for 512 cycles of matrix pipe (256 x 128
// tile) and took 1080 cycles, bound by that; at two it moves 36 KiB.  What bounds it now is one wavefront per SIMD: counters of
// 8 x 1024 x 56 x 56 -> 1024, 3 x 3 stride 2 (76400 cycles per wavefront, 72 steps, matrix pipe busy for 48 %): per step 16 multiplies, 110 other
// vector, 20 scalar, 7 LDS and 3 load instructions, about 700 cycles of issue, and 27 % of the time in waits; no bank conflict.
//
// IMPL: a conv layer with implicit im2row.  Qc is then the layer's quantised input in the form T2[n][C_pack][row][column % s]
// [column / s][16 bytes] (k_quantize_f4 with TILED): lane l of a block of K words 2 i, 2 i + 1 loads the record of its pixel at
// the tap of word w = 2 i + l / 32 = (kh KW + kw) C_pack + ic, from input pixel (oh s + kh - p, ow s + kw - p) of plane ic, or
// the fill record behind the planes (zeros, or +1 for binary activations: the reference's fill,
// src/tnns/ternarize2row_avx2.c:748-755, src/tnns/binarize2row_avx2.c:151) where that pixel lies outside the image or w is a
// padding word.  In T2 the 32 pixels are consecutive records within an output row whatever the stride.  Every wavefront stages
// a quarter of each side, so that none holds the others up at the barrier.  A wavefront issues one instruction every few
// cycles, so what the gather adds per block must stay a handful of instructions:
//   * a table behind the ring, one entry per K word, holds what does not depend on the pixel: the bit of the word's tap (0
//     for a padding word), and the word's part of the record index (plane, tap row, column class and slot offset);
//   * per row block a lane keeps the mask of the taps that fall inside the image for its pixel, and its pixel's part of the index;
// a block's source is then one AND, one add, one select and the address.
template <int WTP, int WTQ, int NS>
struct TileRec {
    static constexpr int RBP = 2 * WTP, RBQ = 2 * WTQ;         // row blocks per operand side
    static constexpr int FR = RBP + RBQ;                       // blocks per stage: the P side's, then the Q side's
    static constexpr int PW = RBP / 4, QW = RBQ / 4, FW = PW + QW;   // blocks a wavefront stages
    static constexpr int NL = WTP + WTQ, NM = WTP * WTQ;       // LDS reads per pair of words, multiplies per word
    static constexpr int LAG = NL >= 8 ? 4 : 3;
    static constexpr size_t lds_bytes = (size_t)NS * FR * 1024;
    static_assert(RBP % 4 == 0 && RBQ % 4 == 0 && FW <= NL, "a quarter of each side per wavefront, one load per slot");
};

template <bool SWAP, bool NT, int WTP, int WTQ, int NS, bool IMPL>
__global__ __launch_bounds__(256) void k_mfma_s2(const uint4* __restrict__ Pc, const uint4* __restrict__ Qc, float* __restrict__ Y,
                                                 int M, int KN, int OHW, int KP /* pairs of words per row */, int nstep, int bias,
                                                 int form, float alpha, ConvGeom cg, FastDiv dOHW, int Ws, FastDiv dSW) {
    static_assert(!IMPL || SWAP, "implicit im2row: the pixels along the lanes");
    extern __shared__ uint4 lds[];   // NS stages of FR KiB, then the table
    typedef Acc<true>::type acc_t;
    typedef TileRec<WTP, WTQ, NS> TL;
    constexpr int RBP = TL::RBP, RBQ = TL::RBQ, FR = TL::FR, PW = TL::PW, QW = TL::QW, FW = TL::FW;
    constexpr int NL = TL::NL, NM = TL::NM, LAG = TL::LAG;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wy = wave >> 1, wx = wave & 1;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
    // Tile of this workgroup.  Under IMPL the kernel tiles of one pixel tile read the same part of T2; workgroups are dealt
    // to the eight XCDs round-robin by their linear number, so the tiles are renumbered to keep those on one XCD (its L2
    // then fetches that part once, not once per kernel tile): XCD x takes the pixel tiles x, x + 8, ...; the pixel
    // tiles beyond the last multiple of eight keep the plain order.
    uint32_t bx = blockIdx.x, by = blockIdx.y;
    if constexpr (IMPL) {
        const uint32_t kt = gridDim.x, pt8 = gridDim.y / 8 * 8, lin = bx + kt * by;
        if (lin < kt * pt8) {
            const uint32_t xcd = lin & 7u, slot = lin >> 3;
            by = xcd + 8u * (slot / kt);
            bx = slot % kt;
        }
    }
    const int prb0 = bx * RBP, qrb0 = by * RBQ;
    const int prbmax = (prow + 31) / 32 - 1, qrbmax = (qrow + 31) / 32 - 1;
    acc_t acc[WTP][WTQ];
#pragma unroll
    for (int a = 0; a < WTP; a++)
#pragma unroll
        for (int b = 0; b < WTQ; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[a][b][e] = 0;

    // Wavefront w stages row blocks w PW .. of the P side and w QW .. of the Q side; row blocks past the operand are clamped (their results are never stored).
    const uint4* psrc[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) psrc[i] = Pc + (size_t)min(prb0 + wave * PW + i, prbmax) * KP * 64 + lane;
    const uint4* qsrc[IMPL ? 1 : QW];
    uint32_t tapmask[IMPL ? QW : 1], qbase[IMPL ? QW : 1];
    const uint32_t row16 = (uint32_t)(cg.W_stride * Ws);            // records per input row
    const uint32_t plane16 = (uint32_t)cg.H * row16;                // per plane of 64 channels
    const uint32_t fill_rec = (uint32_t)cg.CP * plane16 * (uint32_t)((M - 1) / OHW + 1);   // right behind the planes
    uint2* const wtab = reinterpret_cast<uint2*>(lds + (size_t)NS * FR * 64);
    const int words = 2 * nstep;
    if constexpr (IMPL) {
        for (int w = tid; w < words; w += 256) {
            const int tap = (int)fastdiv((uint32_t)w, cg.dCP), ic = w - tap * cg.CP;
            const int kh = (int)fastdiv((uint32_t)tap, cg.dKW), kw = tap - kh * cg.KW;
            // column ow s + d with d = kw - pad: class d mod s, slot ow + floor(d / s) (d made non-negative by a
            // multiple of s first: the host keeps the padding below 4096 s)
            const uint32_t dd = (uint32_t)(kw - cg.W_pad + 4096 * cg.W_stride);
            const uint32_t dq = fastdiv(dd, dSW), cls = dd - dq * (uint32_t)cg.W_stride;
            wtab[w] = make_uint2(w < cg.K ? 1u << tap : 0u,
                                 (uint32_t)ic * plane16 + (uint32_t)kh * row16 + cls * (uint32_t)Ws + dq - 4096u);
        }
#pragma unroll
        for (int j = 0; j < QW; j++) {
            const int rb = wave * QW + j;
            const uint32_t q = (uint32_t)min((qrb0 + rb) * 32 + (lane & 31), M - 1);
            const uint32_t img = fastdiv(q, dOHW);
            const uint32_t pix = q - img * (uint32_t)OHW;
            const int oh = (int)fastdiv(pix, cg.dOW), ow = (int)pix - oh * cg.OW;
            const int ih0 = oh * cg.H_stride - cg.H_pad, iw0 = ow * cg.W_stride - cg.W_pad;
            // (image, plane 0, row ih0, class 0, slot ow): wraps for a negative ih0, and the word's part brings it back
            // whenever the tap is inside
            qbase[j] = img * (uint32_t)cg.CP * plane16 + (uint32_t)ih0 * row16 + (uint32_t)ow;
            uint32_t m = 0u;
            for (int kh = 0, tap = 0; kh < cg.K / (cg.CP * cg.KW); kh++)
                for (int kw = 0; kw < cg.KW; kw++, tap++)
                    m |= ((unsigned)(ih0 + kh) < (unsigned)cg.H && (unsigned)(iw0 + kw) < (unsigned)cg.W ? 1u : 0u) << tap;
            tapmask[j] = m;
        }
        __syncthreads();   // the table is complete before the first stage is issued
    } else {
#pragma unroll
        for (int i = 0; i < QW; i++) qsrc[i] = Qc + (size_t)min(qrb0 + wave * QW + i, qrbmax) * KP * 64 + lane;
    }
    // this lane's word of the pair that its wavefront gathers of the stage about to be issued (stages are issued strictly in
    // order); its table entry is read one stage ahead of its use
    int g_w = lane >> 5;
    uint2 wt = make_uint2(0u, 0u), wt_ahead = make_uint2(0u, 0u);
    if constexpr (IMPL) wt_ahead = wtab[g_w];
    auto next_words = [&]() {
        wt = wt_ahead;
        g_w = min(g_w + 2, words - 1);   // (past the last stage: any entry)
        wt_ahead = wtab[g_w];
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
    auto load = [&](int i, int step) {   // slot i of the wavefront's loads for stage `step`
        const uint32_t dst = lds0 + (uint32_t)(step % NS) * (FR * 1024);
        if (i < PW) {
            dma16(psrc[i] + (size_t)step * 64, dst + (uint32_t)(wave * PW + i) * 1024);
        } else {
            const int j = i - PW;
            const uint32_t d = dst + (uint32_t)(RBP + wave * QW + j) * 1024;
            if constexpr (IMPL) dma16(Qc + ((tapmask[j] & wt.x) != 0u ? qbase[j] + wt.y : fill_rec), d);   // a select on the index: no branch
            else dma16(qsrc[j] + (size_t)step * 64, d);
        }
    };
    auto stage = [&](int step) {
        if constexpr (IMPL) next_words();
#pragma unroll
        for (int i = 0; i < FW; i++) load(i, step);
    };
    // raw: the records of the pair being consumed; e[k]: its nibbles for multiply k.  Slots in the order the multiplies take
    // them: 0: P block 0, 1 .. WTQ: Q blocks, then P blocks 1 .. WTP - 1.
    uint4 rp[WTP], rq[WTQ], ep[2][WTP], eq[2][WTQ];
    auto read_raw = [&](int buf, int i) {
        const uint4* L = lds + (size_t)buf * FR * 64 + lane;
        if (i == 0) rp[0] = L[(wy * WTP + 0) * 64];
        else if (i <= WTQ) rq[i - 1] = L[(RBP + wx * WTQ + (i - 1)) * 64];
        else rp[i - WTQ] = L[(wy * WTP + (i - WTQ)) * 64];
    };
    auto split = [&](int k, int i) {
        const uint4& r = i == 0 ? rp[0] : (i <= WTQ ? rq[i - 1] : rp[i - WTQ]);
        const uint32_t d0 = k == 0 ? r.x : r.z, d1 = k == 0 ? r.y : r.w;
        const uint4 v = make_uint4(d0 & kP2Mask, (d0 << 1) & kP2Mask, d1 & kP2Mask, (d1 << 1) & kP2Mask);
        if (i == 0) ep[k][0] = v;
        else if (i <= WTQ) eq[k][i - 1] = v;
        else ep[k][i - WTQ] = v;
    };
    // the multiplies of slot i: the NM of a word spread evenly over the NL slots, in the order (a, b) = (m / WTQ, m % WTQ)
    auto multiply = [&](int k, int i) {
#pragma unroll
        for (int m = i * NM / NL; m < (i + 1) * NM / NL; m++) mfma<true>(acc[m / WTQ][m % WTQ], ep[k][m / WTQ], eq[k][m % WTQ]);
    };

    // prologue: the first NS stages in flight, wait for stage 0 only
#pragma unroll
    for (int p = 0; p < NS; p++)
        if (p < nstep) stage(p);
    if (nstep >= NS) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FW * (NS - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NL; i++) read_raw(0, i);
#pragma unroll
    for (int i = 0; i < NL; i++) split(0, i);

    // A block read in slot i is split in slot i + LAG, the last LAG ones in the first slots of the next pair, ahead of their
    // first multiply (block b: P block 0 and Q block 0 in the slot of m = 0, Q block j of m = j, P block a of m = a WTQ).
    auto step_body = [&](int s, auto full_tag) {
        constexpr bool FULL = decltype(full_tag)::value;   // FULL: s + NS < nstep
#pragma unroll
        for (int i = 0; i < NL; i++) {
            if (i < LAG && s > 0) split(0, NL - LAG + i);
            split(1, i);
            multiply(0, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Everything of this stage is in registers.  Stage s + 1 must have landed (stages s + 2 .. s + NS - 1 may still be in
        // flight); after the barrier buffer s % NS is free for stage s + NS.
        if (FULL || s + NS - 1 < nstep) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FW * (NS - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if constexpr (FULL && IMPL) next_words();
        const bool do_ld = FULL || s + 1 < nstep;
#pragma unroll
        for (int i = 0; i < NL; i++) {
            if (do_ld) read_raw((s + 1) % NS, i);
            if (FULL && i < FW) load(i, s + NS);
            if (do_ld && i >= LAG) split(0, i - LAG);
            multiply(1, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + NS < nstep; s++) step_body(s, std::true_type{});
    for (; s < nstep; s++) step_body(s, std::false_type{});

    store_tile<true, SWAP, NT, WTP, WTQ>(acc, Y, M, KN, OHW, prb0 + wy * WTP, qrb0 + wx * WTQ, lane, bias, form, alpha);
}

// ------------------------------------------------------------ conv layer (fp4)
// Layer-sized problems (a few GMAC, 10^3..10^5 output pixels) are latency-, not throughput-bound,
// and their im2row operand does not exist in memory.  This kernel therefore works on small tiles
// with many wavefronts in flight and gathers its activation fragments itself:
//   * a wavefront owns 64 kernels x 64 output pixels (2 x 2 MFMA blocks, 64 accumulator
//     registers).  A workgroup is 4 wavefronts: S of them split the K loop of one tile (each takes a
//     run of pairs of words in the reference's K order (kh*KW + kw)*C_pack + ic; words dealt out in turn cost layers
//     0.2-0.6 us more, as every step then changes the tap), so it covers 4/S pixel tiles.  S = 1 where there are tiles enough (no exchange at all), 2 or
//     4 where they alone would leave most of the chip idle (launch_conv_f4 has the lines); the partial tiles then meet in
//     LDS and each wavefront finishes 4/S of the tile's four blocks;
//   * weights are the MFMA A side (rows = accumulator registers), pixels the B side (rows =
//     lanes), so a store instruction writes 32 consecutive pixels of one NCHW plane;
//   * both operands come as records of two bits per lane (P2): lane (row or pixel, hw) loads the 16 bytes of word 2 i + hw of its
//     row, which hold the operands of two multiplies; a load instruction moves two K words of 32 rows.  What bounds the
//     K loop is the return path of vector memory, 64 bytes per cycle and compute unit over all its wavefronts: at four
//     bits per lane a K word of a 64 x 64 tile took a wavefront 540-620 cycles, for 128 of matrix pipe;
//   * the two words of a pair are two planes of one tap where C_pack is even (the tap is then the same for all lanes and
//     changes every C_pack / 2 pairs), else any two neighbouring words: each lane half walks its own taps;
//   * a tap outside the image contributes zeros for ternary inputs, +1 lanes for binary ones (the reference's fill,
//     src/tnns/ternarize2row_avx2.c:748-755, src/tnns/binarize2row_avx2.c:151);
//   * the words that round K up to a multiple of 4 are skipped, but for the one that makes up the last pair of an odd K: its
//     activation lanes are zeros (BNN's epilogue constant counts the real words only).
// ABIN: binary activations (padding value +1).  FORM0: the TNN form of PReLU, "f <= 0 -> f *= alpha"
// (mm_p2_final_tnn_avx2.c:204-208), else "r >= 0 ? r : alpha * r" (mm_p2_final_tbn_avx2.c:73).
// QMODE: 0 = fp32 NCHW result, 1 / 2 = ternary / binary hand-over to the next layer (QuantOut).
// All three are compile-time so that the per-element epilogue carries no selects for them.
// TA x TB: blocks of 32 kernels x 32 pixels per wavefront.  2 x 2, or 1 x 1 with S = 4, or S = 8 on a workgroup of eight, for layers with few tiles: a
// wavefront moves a bounded number of bytes per cycle from a cold L2 whatever its prefetch depth, so a small layer gets faster
// only with more wavefronts, on more compute units.  Kernel tiles of 32 come in pairs under the hand-over (a pixel's
// record is written by two workgroups, 8 bytes each; a tile past KN writes padding lanes).
// The unsplit hand-over variants are the ones launched with several thousand wavefronts (stems,
// first stages): they are asked to fit three wavefronts per SIMD, which they do without scratch.
// BUF: fragments arrive through buffer loads.  Their offsets are 32-bit, the place of a word within the operand is a
// scalar offset, and an offset beyond the buffer returns zeros, which is what a tap outside the image must contribute for
// ternary activations (binary ones or the +1 lanes in while splitting the record).
// Needs both operands below 4 GiB (p2_bytes, wf_bytes: the sizes the descriptors announce).  fp32 results leave through buffer
// stores too, relative to the tile's first image and kernel: y_span bounds what a tile reaches from there, whatever the size
// of the result.
template <bool ABIN, bool FORM0, int QMODE, int TA, int TB, int S, bool BUF>
__global__ __launch_bounds__(S == 8 ? 512 : 256) __attribute__((amdgpu_waves_per_eu((S == 1 && QMODE != 0) ? 3 : 1, 8))) void k_conv_f4(
    const uint4* __restrict__ P2, const uint4* __restrict__ Wf, float* __restrict__ Y, int M, int KN, int OHW, int KP /* pairs a weight row is stored at */,
    int bias, float alpha, FastDiv dOHW, ConvGeom cg, PairWalk pw, QuantOut qo, uint32_t p2_bytes, uint32_t wf_bytes, uint32_t y_span, XcdOrder xo, uint32_t launched_x, uint32_t kernel_tiles) {
    constexpr int WPB = S == 8 ? 8 : 4;   // wavefronts per workgroup (single-wavefront workgroups for S = 1
                                          // measured slower: neighbours no longer share weight fragments in L1)
    constexpr int NB = 3;                 // register sets of records: NB - 1 pairs of loads in flight; four and six measured slower
    constexpr int NBLK = TA * TB;
    constexpr int PUB = NBLK == 1 ? 1 : 4 - 4 / S;   // blocks a wavefront hands to the others of its tile
    __shared__ float4 red[S > 1 ? WPB * PUB * 4 * 64 : 1];   // [wavefront][slot][e / 4][lane]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave % S, pt = wave / S;   // K share and pixel tile of this wavefront
    const int h = lane >> 5, lr = lane & 31;
    uint32_t bx, by;   // pixel tiles, kernel tile
    xo.tile<QMODE == 0>(blockIdx.x + launched_x * blockIdx.y, bx, by);   // (gridDim would bring 256 bytes of hidden arguments: 0.1 us a launch)
    if (QMODE == 0 && xo.mask == 0) {   // plain: pixel tiles are the inner index
        const uint32_t t = bx;
        bx = by;
        by = t;
    }
    const int px0 = ((int)bx * (WPB / S) + pt) * 32 * TB, kn0 = (int)by * 32 * TA;

    int ih0[TB], iw0[TB];
    uint32_t img[TB], pix[TB], xrec[TB];   // xrec: record of (image, plane 0, pixel (ih0, iw0)) in P2[n][C_pack][pixel]
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const uint32_t q = (uint32_t)min(px0 + 32 * b + lr, M - 1);
        img[b] = fastdiv(q, dOHW);
        pix[b] = q - img[b] * (uint32_t)OHW;
        const int oh = (int)fastdiv(pix[b], cg.dOW), ow = (int)pix[b] - oh * cg.OW;
        ih0[b] = oh * cg.H_stride - cg.H_pad;
        iw0[b] = ow * cg.W_stride - cg.W_pad;
        xrec[b] = img[b] * (uint32_t)(cg.CP * cg.H * cg.W) + (uint32_t)(ih0[b] * cg.W + iw0[b]);
    }
    const int rbmax = (KN + 31) / 32 - 1;

    // The pairs of this wavefront, [p, p1).  A lane's word is 2 p + h = (kh, kw, ic) of the reference's K order; addresses and
    // borders are computed when a run of pairs ends (PairWalk), within one everything is scalar.
    int p = S == 1 ? 0 : (int)((uint32_t)(pw.NP * ks) / S);
    const int p1 = S == 1 ? pw.NP : (int)((uint32_t)(pw.NP * (ks + 1)) / S);
    const int pairs = p1 - p;
    // (the scalar part of its place in bytes for buffer loads, whose operand is below 3.75 GiB, and in records for any operand)
    PairPos<BUF ? 16u : 1u> pos;
    pos.template start<S == 1>(pw, cg, p, h);
    struct Rec {
        v4i w[TA], x[TB];
        uint32_t fill[TB];   // ABIN: the nibbles that a tap outside the image is replaced by (0: none)
        bool in[TB];         // (without BUF) x[b] holds a real input pixel
    };
    uint32_t vx[TB], fill[TB];   // the lane's record (BUF: byte offset) at its present word
    bool in[TB];
    auto tap = [&]() {
        const bool real = pos.kh < pw.KH;   // the word that makes up the last pair of an odd K is none
        const uint32_t off = pos.off(cg);
#pragma unroll
        for (int b = 0; b < TB; b++) {
            const bool inside = (unsigned)(ih0[b] + pos.kh) < (unsigned)cg.H && (unsigned)(iw0[b] + pos.kw) < (unsigned)cg.W;
            const bool valid = inside && real;
            if constexpr (ABIN) fill[b] = real && !inside ? 0x22222222u : 0u;   // (vx last, as in the other branch below: no register behind a pointer)
            const uint32_t rec = xrec[b] + off;   // wraps to the right value whenever the tap is inside
            if constexpr (BUF) {
                vx[b] = valid ? rec * 16u : 0xffffff00u;   // an offset beyond the buffer returns zeros
            } else {
                vx[b] = valid ? rec : 0u;
                in[b] = valid;
            }
        }
    };
    tap();
    // buffer descriptors (base; stride 0; bytes; raw 32-bit data format)
    const __amdgpu_buffer_rsrc_t brs_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(P2), 0, (int)p2_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t brs_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(Wf), 0, (int)wf_bytes, 0x00020000);
    // All loads of a pair are unconditional and are issued two pairs ahead of the one being multiplied.  They are ordinary
    // loads (plain, or buffer-load builtins), so the compiler owns the dependency between a load and the use of its
    // registers and places every s_waitcnt vmcnt itself; what keeps a load where the code issues it -- and not next to
    // its use, where the scheduler would sink it -- is the scheduling fence after each pair's loads.
    uint32_t vw = (uint32_t)lane * 16u;
    auto load = [&](Rec& f) {   // pair p, then on to the next one
#pragma unroll
        for (int a = 0; a < TA; a++) {
            const uint32_t block = (uint32_t)min(kn0 / 32 + a, rbmax) * (uint32_t)KP + (uint32_t)p;
            if constexpr (BUF) {
                const v4u v = __builtin_amdgcn_raw_buffer_load_b128(brs_w, (int)vw, (int)(block * 1024u), 0);
                f.w[a] = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
            } else {
                f.w[a] = *reinterpret_cast<const v4i*>(Wf + (size_t)block * 64 + lane);
            }
        }
#pragma unroll
        for (int b = 0; b < TB; b++) {
            if constexpr (BUF) {
                const v4u v = __builtin_amdgcn_raw_buffer_load_b128(brs_x, (int)vx[b], (int)pos.soff, 0);
                f.x[b] = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
            } else {
                f.x[b] = *reinterpret_cast<const v4i*>(P2 + ((size_t)vx[b] + (in[b] ? pos.soff : 0u)));
            }
            if constexpr (!BUF) f.in[b] = in[b];
        }
#pragma unroll
        for (int b = 0; b < TB; b++)
            if constexpr (ABIN) f.fill[b] = fill[b];
        if (p + 1 < p1) {
            p++;
            if (pos.next(pw, cg)) tap();
        } else if (BUF) {   // past the end: offsets beyond the buffers, which move no data (else the last pair is read again)
            vw = 0xffffff00u;
#pragma unroll
            for (int b = 0; b < TB; b++) vx[b] = 0xffffff00u;
        }
        __builtin_amdgcn_sched_barrier(0);   // these loads stay in front of the multiplies that follow
    };
    v16f acc[TA][TB];
    auto compute = [&](const Rec& f) {
#pragma unroll
        for (int k = 0; k < 2; k++) {   // dwords 0 and 1 of the records, then 2 and 3
            v8i x[TB], wv[TA];
#pragma unroll
            for (int b = 0; b < TB; b++) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t d = BUF || f.in[b] ? (uint32_t)f.x[b][2 * k + i] : 0u;
                    const uint32_t fl = ABIN ? f.fill[b] : 0u;
                    x[b][2 * i] = (int)((d & kP2Mask) | fl);
                    x[b][2 * i + 1] = (int)(((d << 1) & kP2Mask) | fl);
                }
#pragma unroll
                for (int i = 4; i < 8; i++) x[b][i] = 0;
            }
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const uint32_t d0 = (uint32_t)f.w[a][2 * k], d1 = (uint32_t)f.w[a][2 * k + 1];
                wv[a] = v8i{(int)(d0 & kP2Mask), (int)((d0 << 1) & kP2Mask), (int)(d1 & kP2Mask), (int)((d1 << 1) & kP2Mask), 0, 0, 0, 0};
            }
            // cbsz = blgp = 4: both operands E2M1, unscaled (see mfma<true>)
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int b = 0; b < TB; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv[a], x[b], acc[a][b], 4, 4, 0, 0, 0, 0);
        }
    };

    // The register sets rotate by name (the loop is unrolled by NB); loads past the last pair are not multiplied.
    Rec f[NB];
#pragma unroll
    for (int j = 0; j < NB - 1; j++) load(f[j]);
    {   // the accumulators are cleared while the first loads are on their way
        const float init = ks == 0 ? acc_init<QMODE>(qo, FORM0 ? 0.0f : (float)bias) : 0.0f;   // only BNN has a bias
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[a][b][e] = init;
    }
    for (int i = 0; i < pairs; i += NB) {   // (a share of K is empty where there are fewer pairs than S)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            load(f[(j + NB - 1) % NB]);
            if (j == 0 || i + j < pairs) compute(f[j]);
        }
    }

    // Block id = TB * a + b; wavefront ks of a tile finishes the blocks with id % S == ks and hands
    // the others over through LDS.  Every copy below names its accumulator registers statically,
    // under a wave-uniform branch, so that no register array is indexed at run time.
    auto for_blocks = [&](auto&& fn) {
        fn(std::integral_constant<int, 0>{});
        if constexpr (NBLK == 4) {
            fn(std::integral_constant<int, 1>{});
            fn(std::integral_constant<int, 2>{});
            fn(std::integral_constant<int, 3>{});
        }
    };
    auto slot_of = [](int blk, int v) {   // slot of blk among the blocks that wavefront v does not own
        return NBLK == 1 ? 0 : (S == 4 ? (blk < v ? blk : blk - 1) : blk / 2);
    };
    if constexpr (S > 1) {
        for_blocks([&](auto blk_tag) {
            constexpr int BLK = decltype(blk_tag)::value;
            if (BLK % S != ks) {
                float4* dst = red + (size_t)((wave * PUB + slot_of(BLK, ks)) * 4) * 64 + lane;
                const v16f& c = acc[BLK / TB][BLK % TB];
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++)
                    dst[e4 * 64] = make_float4(c[4 * e4], c[4 * e4 + 1], c[4 * e4 + 2], c[4 * e4 + 3]);
            }
        });
        __syncthreads();
    }
    // whole sum of a block that this wavefront finishes, in ordinary registers (accumulated in place it would go back into
    // the accumulator registers and out again)
    auto total = [&](auto blk_tag) {
        constexpr int BLK = decltype(blk_tag)::value;
        v16f c = acc[BLK / TB][BLK % TB];
        if constexpr (S > 1) {
#pragma unroll
            for (int v = 0; v < S; v++) {
                if (v != BLK % S) {   // source wavefront pt * S + v
                    const float4* src = red + (size_t)(((pt * S + v) * PUB + slot_of(BLK, v)) * 4) * 64 + lane;
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) {
                        const float4 t = src[e4 * 64];
                        c[4 * e4] += t.x;
                        c[4 * e4 + 1] += t.y;
                        c[4 * e4 + 2] += t.z;
                        c[4 * e4 + 3] += t.w;
                    }
                }
            }
        }
        return c;
    };
    // accumulator e of block (a, b): kernel = kn0 + 32 a + 8 (e / 4) + 4 h + e % 4, pixel = px0 + 32 b + lr
    if constexpr (QMODE == 0) {
        const uint32_t img0 = __builtin_amdgcn_readfirstlane(img[0]);
        const __amdgpu_buffer_rsrc_t brs_y =
            __builtin_amdgcn_make_buffer_rsrc(Y + ((size_t)img0 * KN + kn0) * OHW, 0, (int)y_span, 0x00020000);
        // slopes from +0 to 1: PReLU is then max(r, r * alpha), bit for bit (with -0 a zero TNN sum becomes -0, which no maximum gives)
        const bool as_max = __float_as_uint(alpha) <= __float_as_uint(1.0f);
        for_blocks([&](auto blk_tag) {
            constexpr int BLK = decltype(blk_tag)::value, a = BLK / TB, b = BLK % TB;
            if (BLK % S == ks) {
                const v16f c = total(blk_tag);
                float r[16];
                if (as_max) {
#pragma unroll
                    for (int e = 0; e < 16; e++) r[e] = __builtin_fmaxf(c[e], c[e] * alpha);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; e++) r[e] = prelu_ref<FORM0>(c[e], alpha);
                }
                const bool live = px0 + 32 * b + lr < M;
                const int p0 = kn0 + 32 * a + 4 * h;
                auto put = [&](auto whole, auto nt) {
                    constexpr bool NT = decltype(nt)::value;
                    if constexpr (BUF) {
                        // a lane's part, and the kernel's row as a scalar; lanes past the pixels store beyond the buffer: nothing
                        const uint32_t vy =
                            live ? (((img[b] - img0) * (uint32_t)KN + (uint32_t)(32 * a + 4 * h)) * (uint32_t)OHW + pix[b]) * 4u : 0xffffff00u;
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const int row = 8 * (e >> 2) + (e & 3);
                            if (decltype(whole)::value || p0 + row < KN)
                                __builtin_amdgcn_raw_buffer_store_b32((unsigned)__float_as_uint(r[e]), brs_y, (int)vy, (int)((uint32_t)(row * 4) * (uint32_t)OHW), NT ? 2 : 0);
                        }
                    } else if (live) {
                        float* yq = Y + ((size_t)img[b] * KN + p0) * OHW + pix[b];
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const int row = 8 * (e >> 2) + (e & 3);
                            if (decltype(whole)::value || p0 + row < KN) {
                                if (NT) __builtin_nontemporal_store(r[e], yq + (size_t)row * OHW);
                                else yq[(size_t)row * OHW] = r[e];
                            }
                        }
                    }
                };
                // A whole block stores in a straight line.  With the check of the row beside the uniform one in a single
                // condition, every store is a branch of its own: 0.3-0.8 us of a 4-12 us layer (1 x 64 x 56 x 56, 3 x 3:
                // 5.5 against 4.9 us with the quantiser; 8 x 256 x 56 x 56 -> 128, 1 x 1: 12.2 against 11.4).
                const bool inside = kn0 + 32 * a + 32 <= KN;
                // A result beyond the Infinity Cache (see XcdOrder) is stored past the caches: 8 x 1024 x 1024 -> 130 behind a first
                // layer, 3 x 3 1605 -> 1207 us, 1 x 1 1240 -> 1125; 40 x 128 x 128 -> 2048 the same within its spread (870-970).
                // Only whole sectors, as in stores_past_caches.
                if (xo.mask == 0 && stores_past_caches(OHW, M, KN)) {
                    if (inside) put(std::true_type{}, std::true_type{});
                    else put(std::false_type{}, std::true_type{});
                } else {
                    if (inside) put(std::true_type{}, std::false_type{});
                    else put(std::false_type{}, std::false_type{});
                }
            }
        });
    } else {
        // Hand-over to an fp4 layer: dwords 2 h and 2 h + 1 of a pixel's record are lane half h of its two 32-kernel blocks
        const uint32_t KT = TA == 2 ? kernel_tiles : kernel_tiles >> 1, kt = TA == 2 ? by : by >> 1;
        auto out_rec = [&](int b) {
            return static_cast<unsigned char*>(qo.p2) + (((size_t)img[b] * KT + kt) * (uint32_t)OHW + pix[b]) * 16 + 8 * h;
        };
        if constexpr (NBLK == 4 && S < 4) {   // the wavefront finishes both kernel blocks of a pixel block
            auto pixel_block = [&](auto b_tag) {
                constexpr int b = decltype(b_tag)::value;
                if (b % S == ks) {
                    const uint32_t d0 = hand_over_block<FORM0, QMODE>(total(b_tag), alpha, qo, kn0, h, KN);
                    const uint32_t d1 = hand_over_block<FORM0, QMODE>(total(std::integral_constant<int, TB + b>{}), alpha, qo, kn0 + 32, h, KN);
                    if (px0 + 32 * b + lr < M) *reinterpret_cast<uint2*>(out_rec(b)) = make_uint2(d0, d1);
                }
            };
            pixel_block(std::integral_constant<int, 0>{});
            pixel_block(std::integral_constant<int, 1>{});
        } else {   // one block
            for_blocks([&](auto blk_tag) {
                constexpr int BLK = decltype(blk_tag)::value, a = BLK / TB, b = BLK % TB;
                if (BLK % S == ks) {
                    const uint32_t d = hand_over_block<FORM0, QMODE>(total(blk_tag), alpha, qo, kn0 + 32 * a, h, KN);
                    const int part = TA == 2 ? a : (int)(by & 1u);
                    if (px0 + 32 * b + lr < M) *reinterpret_cast<uint32_t*>(out_rec(b) + 4 * part) = d;
                }
            });
        }
    }
}

// tiles of 256 x 256 below which the 128 x 128 tiles of k_mfma and of the record blocks' product are used (FTNN_MFMA_SMALL_BELOW: tuning aid)
inline int64_t mfma_small_tile_below() {
    static const int64_t v = []() {
        const char* e = getenv("FTNN_MFMA_SMALL_BELOW");
        return e ? (int64_t)atoll(e) : (int64_t)160;
    }();
    return v;
}

// Two workgroups of the smaller tiles share a compute unit: where rows are long, one's stores go on beside the other's multiplies,
// and only the write-back at the end of a launch through the caches is left (stores_past_caches).  us past / through the caches, on fp4
// tiles of 128 x 128: 30000 x 150 x 4096 (64 words) 23.2 / 19.9, x 16384 55.3 / 55.2, 5905 x 1474 x 27904 121 / 129.
inline bool tile_hides_stores(int WT, int Kw) { return WT < 4 && Kw > 128; }

template <bool SWAP, bool NT, int WTP, int WTQ, int KF, int NS>
hipError_t launch_gemm_tile_as(const uint4* Pf, const uint4* Qf, float* Y, int M, int KN, int OHW, int KB,
                            int bias, int form, float alpha, hipStream_t st) {
    auto kern = k_mfma<SWAP, NT, WTP, WTQ, KF, NS>;
    constexpr size_t lds_bytes = Tile<WTP, WTQ, KF, NS>::lds_bytes;
    // the opt-in to more than 64 KiB of dynamic LDS is per kernel; done once, thread-safe
    // The kernel counts its LDS-direct loads by hand (s_waitcnt vmcnt(N)); a scratch access would be one more
    // vector-memory operation inside those windows, so a build of it that spills is refused (once per variant).
    static const hipError_t configured = []() {
        const void* kern = reinterpret_cast<const void*>(&k_mfma<SWAP, NT, WTP, WTQ, KF, NS>);
        hipFuncAttributes attr;
        hipError_t e = hipFuncGetAttributes(&attr, kern);
        if (e == hipSuccess && attr.localSizeBytes != 0) e = hipErrorLaunchFailure;
        if (e != hipSuccess) return e;
        return hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Tile<WTP, WTQ, KF, NS>::lds_bytes);
    }();
    if (configured != hipSuccess) return configured;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
    dim3 grid((prow + 64 * WTP - 1) / (64 * WTP), (qrow + 64 * WTQ - 1) / (64 * WTQ));
    if (grid.y > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, grid, dim3(256), lds_bytes, st, Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha);
    return hipGetLastError();
}

template <bool SWAP, int WTP, int WTQ, int KF, int NS>
hipError_t launch_gemm_tile(const uint4* Pf, const uint4* Qf, float* Y, int M, int KN, int OHW, int KB,
                            int bias, int form, float alpha, hipStream_t st) {
    return stores_past_caches(SWAP ? OHW : KN, M, KN) || tile_hides_stores(WTP, KB / 2)
               ? launch_gemm_tile_as<SWAP, true, WTP, WTQ, KF, NS>(Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha, st)
               : launch_gemm_tile_as<SWAP, false, WTP, WTQ, KF, NS>(Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha, st);
}

template <bool SWAP>
hipError_t launch_gemm(const uint4* Pf, const uint4* Qf, float* Y, int M, int KN, int OHW, int KB,
                       int bias, int form, float alpha, hipStream_t st) {
    // 256 x 256 tiles re-read the operands least, but a problem must have enough of them for the chip's
    // 256 compute units; below that, 128 x 128 tiles (two workgroups fit a compute unit)
    const int64_t big = (((int64_t)M + 255) / 256) * ((KN + 255) / 256);
    bool small = big < mfma_small_tile_below();
    // Fewer than 112 tiles of 128 x 128 leave most compute units idle: tiles of 64 x 64 then, four fragments per step
    // (from 144 tiles on the larger tile is faster; tiles of 128 x 64 lose everywhere).
    // FTNN_MFMA_TINY_BELOW = n moves the threshold (tuning aid).
    static const int tiny_below = getenv("FTNN_MFMA_TINY_BELOW") ? atoi(getenv("FTNN_MFMA_TINY_BELOW")) : 112;
    const int64_t mid = (((int64_t)M + 127) / 128) * ((KN + 127) / 128);
    if (small && mid < tiny_below) return launch_gemm_tile<SWAP, 1, 1, 4, 4>(Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha, st);
    return small ? launch_gemm_tile<SWAP, 2, 2, 2, 4>(Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha, st)
                 : launch_gemm_tile<SWAP, 4, 4, 2, 4>(Pf, Qf, Y, M, KN, OHW, KB, bias, form, alpha, st);
}

template <int FORM>
hipError_t launch_expand(bool tern, const uint32_t* rows_ptr, int rows, int G, uint4* out, uint32_t* kept, hipStream_t st) {
    dim3 grid((rows + 31) / 32, (G + 3) / 4);   // 4 groups per workgroup (kGPB in the kernel)
    if (grid.y > 65535) return hipErrorInvalidValue;
    if (tern) hipLaunchKernelGGL((k_expand<FORM, true>), grid, dim3(256), 0, st, rows_ptr, rows, G, out, kept);
    else hipLaunchKernelGGL((k_expand<FORM, false>), grid, dim3(256), 0, st, rows_ptr, rows, G, out, kept);
    return hipGetLastError();
}

template <bool SWAP, bool NT>
hipError_t launch_gemm_p4_as(const uint4* Pc, const uint4* Qc, float* Y, int M, int KN, int OHW, int KP, const int* sP,
                               const int* sQ, int off, int form, float alpha, hipStream_t st) {
    auto kern = k_mfma_p4<SWAP, NT>;
    // hand-counted LDS-direct loads: no scratch (see launch_gemm_tile); the opt-in to more than 64 KiB of LDS is per kernel
    static const hipError_t configured = []() {
        const void* k = reinterpret_cast<const void*>(&k_mfma_p4<SWAP, NT>);
        hipFuncAttributes attr;
        hipError_t e = hipFuncGetAttributes(&attr, k);
        if (e == hipSuccess && attr.localSizeBytes != 0) e = hipErrorLaunchFailure;
        if (e != hipSuccess) return e;
        return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)TileP4::lds_bytes);
    }();
    if (configured != hipSuccess) return configured;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN, edge = 64 * TileP4::WT;
    dim3 grid((prow + edge - 1) / edge, (qrow + edge - 1) / edge);
    if (grid.y > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, grid, dim3(256), TileP4::lds_bytes, st, Pc, Qc, Y, M, KN, OHW, KP, sP, sQ, off, form, alpha);
    return hipGetLastError();
}

template <bool SWAP>
hipError_t launch_gemm_p4(const uint4* Pc, const uint4* Qc, float* Y, int M, int KN, int OHW, int KP, const int* sP, const int* sQ,
                          int off, int form, float alpha, hipStream_t st) {
    return stores_past_caches(SWAP ? OHW : KN, M, KN)
               ? launch_gemm_p4_as<SWAP, true>(Pc, Qc, Y, M, KN, OHW, KP, sP, sQ, off, form, alpha, st)
               : launch_gemm_p4_as<SWAP, false>(Pc, Qc, Y, M, KN, OHW, KP, sP, sQ, off, form, alpha, st);
}

}  // namespace

int64_t mfma_fragment_bytes(bool f4, int64_t rows, int Kw) {
    // 1 KiB fragments: 32 rows x one word (fp4) or half a word (int8)
    return ((rows + 31) / 32) * (int64_t)(f4 ? Kw : 2 * Kw) * 1024;
}

hipError_t launch_mfma_expand(bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st) {
    return launch_expand<FORM_I8>(ternary, reinterpret_cast<const uint32_t*>(d_rows), rows, Kw / 4, static_cast<uint4*>(d_out), nullptr, st);
}

int64_t record_block_bytes(int64_t rows, int Kw) { return ((rows + 31) / 32) * (int64_t)(Kw / 2) * 1024; }

hipError_t launch_expand_records(bool ternary, bool natural, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st,
                                 int64_t* d_kept) {
    const uint32_t* R = reinterpret_cast<const uint32_t*>(d_rows);
    uint4* out = static_cast<uint4*>(d_out);
    uint32_t* kept = reinterpret_cast<uint32_t*>(d_kept);
    return natural ? launch_expand<FORM_REC_NATURAL>(ternary, R, rows, Kw / 4, out, kept, st)
                   : launch_expand<FORM_REC>(ternary, R, rows, Kw / 4, out, kept, st);
}

hipError_t launch_mfma_gemm(int type, const void* d_af, const void* d_bf, int64_t M, int OHW, int KN,
                            int Kw, int K_unpack, float alpha, float* d_y, hipStream_t st) {
    const uint4* Af = static_cast<const uint4*>(d_af);
    const uint4* Bf = static_cast<const uint4*>(d_bf);
    // BNN: the lanes past K_unpack are +1 in both operands and add 64*Kw - K_unpack to the dot
    // product; the reference's K_unpack - 2*popc(a^b) leaves them out (mm_p2_final_bnn_avx2.c:55-58)
    const int bias = type == kBNN ? 64 * Kw - K_unpack : 0;
    const int form = type == kTNN ? 0 : 1;
    return OHW > 1 ? launch_gemm<true>(Bf, Af, d_y, (int)M, KN, OHW, 2 * Kw, bias, form, alpha, st)
                   : launch_gemm<false>(Af, Bf, d_y, (int)M, KN, OHW, 2 * Kw, bias, form, alpha, st);
}

// ---- packed4: the fp4 GEMM's operands at two bits per lane in offset codes (Kw a multiple of 4, as everywhere) ----
namespace {
inline int64_t packed4_block_bytes(int64_t rows, int Kw) { return ((rows + 31) / 32) * (int64_t)(Kw / 2) * 1024; }
}  // namespace

// the blocks, then one int32 per row of the row blocks (a multiple of 128 bytes)
int64_t mfma_packed4_bytes(int64_t rows, int Kw) { return packed4_block_bytes(rows, Kw) + ((rows + 31) / 32) * 128; }

namespace {
inline int* packed4_sums(void* d_out, int64_t rows, int Kw) {
    return reinterpret_cast<int*>(static_cast<char*>(d_out) + packed4_block_bytes(rows, Kw));
}

// zero_sums = false: the caller has zeroed the row sums on the stream already
hipError_t launch_pack4(bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out, bool zero_sums, hipStream_t st) {
    dim3 grid((rows + 31) / 32, (Kw / 4 + 3) / 4);   // 4 groups of 4 words per workgroup
    if (grid.y > 65535) return hipErrorInvalidValue;
    const uint32_t* R = reinterpret_cast<const uint32_t*>(d_rows);
    int* sums = packed4_sums(d_out, rows, Kw);
    if (grid.x > 0x7fffff00u / 32) return hipErrorInvalidValue;
    const int nsum = (int)grid.x * 32;
    if (zero_sums) hipLaunchKernelGGL(k_zero_i32, dim3((nsum + 255) / 256), dim3(256), 0, st, sums, nsum, nullptr, 0);
    if (ternary) hipLaunchKernelGGL((k_pack4<true>), grid, dim3(256), 0, st, R, rows, Kw / 4, static_cast<uint2*>(d_out), sums);
    else hipLaunchKernelGGL((k_pack4<false>), grid, dim3(256), 0, st, R, rows, Kw / 4, static_cast<uint2*>(d_out), sums);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_mfma_pack4(bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st) {
    return launch_pack4(ternary, d_rows, rows, Kw, d_out, true, st);
}

hipError_t launch_mfma_gemm_packed4(int type, const void* d_ac, const void* d_bc, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                                    float alpha, float* d_y, hipStream_t st) {
    const uint4* Ac = static_cast<const uint4*>(d_ac);
    const uint4* Bc = static_cast<const uint4*>(d_bc);
    const int* sA = reinterpret_cast<const int*>(static_cast<const char*>(d_ac) + packed4_block_bytes(M, Kw));
    const int* sB = reinterpret_cast<const int*>(static_cast<const char*>(d_bc) + packed4_block_bytes(KN, Kw));
    const int bias = type == kBNN ? 64 * Kw - K_unpack : 0;   // as launch_mfma_gemm
    const int off = 64 * Kw + bias;                           // the lanes of a row pair, padding included
    const int form = type == kTNN ? 0 : 1;
    hipError_t e;
    if (launch_mm_packed(type, d_ac, d_bc, sA, sB, M, OHW, KN, Kw, K_unpack, alpha, d_y, st, &e)) return e;
    return OHW > 1 ? launch_gemm_p4<true>(Bc, Ac, d_y, (int)M, KN, OHW, Kw / 2, sB, sA, off, form, alpha, st)
                   : launch_gemm_p4<false>(Ac, Bc, d_y, (int)M, KN, OHW, Kw / 2, sA, sB, off, form, alpha, st);
}

namespace {
constexpr int kMaxTileRouteWords = 2040;   // K words per row the tile kernel keeps a table entry for (16 KiB of LDS)
template <bool SWAP, bool NT, int WTP, int WTQ, int NS, bool IMPL>
hipError_t launch_records_tile_as(const uint4* Pc, const uint4* Qc, float* Y, int M, int KN, int OHW, int KP, int nstep, int bnn_k, int form,
                               float alpha, const ConvGeom& cg, hipStream_t st) {
    auto kern = k_mfma_s2<SWAP, NT, WTP, WTQ, NS, IMPL>;
    typedef TileRec<WTP, WTQ, NS> TL;
    constexpr size_t kLdsMax = 160u << 10;   // LDS of a compute unit
    const size_t lds_bytes = TL::lds_bytes + (IMPL ? (size_t)nstep * 2 * 8 : 0);   // the ring, then the table of K words
    if (lds_bytes > kLdsMax) return hipErrorInvalidValue;
    // as launch_gemm_tile: hand-counted LDS-direct loads, so no scratch; the LDS opt-in is per kernel
    static const hipError_t configured = []() {
        const void* k = reinterpret_cast<const void*>(&k_mfma_s2<SWAP, NT, WTP, WTQ, NS, IMPL>);
        hipFuncAttributes attr;
        hipError_t e = hipFuncGetAttributes(&attr, k);
        if (e == hipSuccess && attr.localSizeBytes != 0) e = hipErrorLaunchFailure;
        if (e != hipSuccess) return e;
        return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax);
    }();
    if (configured != hipSuccess) return configured;
    const int prow = SWAP ? KN : M, qrow = SWAP ? M : KN;
    dim3 grid((prow + 64 * WTP - 1) / (64 * WTP), (qrow + 64 * WTQ - 1) / (64 * WTQ));
    if (grid.y > 65535) return hipErrorInvalidValue;
    // BNN: every lane that is no real (channel, tap) is +1 x +1 in both operands, padding words included
    const int bias = bnn_k ? 128 * nstep - bnn_k : 0;
    hipLaunchKernelGGL(kern, grid, dim3(256), lds_bytes, st, Pc, Qc, Y, M, KN, OHW, KP, nstep, bias, form, alpha, cg,
                       make_fastdiv((uint32_t)OHW), IMPL ? (cg.W + cg.W_stride - 1) / cg.W_stride : 0, make_fastdiv(IMPL ? (uint32_t)cg.W_stride : 1u));
    return hipGetLastError();
}

// The larger tiles store as those of the GEMM do (stores_past_caches).  Strided layers on 256 x 128, under sustained load, us, past / through
// the caches: whole sectors 50.2 / 52.3 (8 x 1024 x 56 x 56 -> 1024), 137 / 142, 114 / 118; other rows 65.3 / 57.5 (34 x 1024 x 28 x 28 -> 1024),
// 118 / 112, 95.9 / 90.5, 192 / 185.  Of 128 x 128 two workgroups share a compute unit, one's stores go on beside the other's
// multiplies: past the caches 0.94 to 1.08 of the time through them on other rows, 0.87 to 0.99 on whole sectors.
template <bool SWAP, int WTP, int WTQ, int NS, bool IMPL>
hipError_t launch_records_tile(const uint4* Pc, const uint4* Qc, float* Y, int M, int KN, int OHW, int KP, int nstep, int bnn_k, int form,
                               float alpha, const ConvGeom& cg, hipStream_t st) {
    if constexpr (WTP >= 4) {
        if (!stores_past_caches(SWAP ? OHW : KN, M, KN))
            return launch_records_tile_as<SWAP, false, WTP, WTQ, NS, IMPL>(Pc, Qc, Y, M, KN, OHW, KP, nstep, bnn_k, form, alpha, cg, st);
    }
    return launch_records_tile_as<SWAP, true, WTP, WTQ, NS, IMPL>(Pc, Qc, Y, M, KN, OHW, KP, nstep, bnn_k, form, alpha, cg, st);
}

template <bool SWAP>
hipError_t launch_records(const uint4* Pc, const uint4* Qc, float* Y, int M, int KN, int OHW, int Kw, int bnn_k, int form, float alpha,
                          hipStream_t st) {
    const int64_t big = (((int64_t)M + 255) / 256) * ((KN + 255) / 256);
    return big < mfma_small_tile_below()
               ? launch_records_tile<SWAP, 2, 2, 4, false>(Pc, Qc, Y, M, KN, OHW, Kw / 2, Kw / 2, bnn_k, form, alpha, ConvGeom(), st)
               : launch_records_tile<SWAP, 4, 4, 4, false>(Pc, Qc, Y, M, KN, OHW, Kw / 2, Kw / 2, bnn_k, form, alpha, ConvGeom(), st);
}
}  // namespace

hipError_t launch_records_gemm(int type, const void* d_a, const void* d_b, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                               float alpha, float* d_y, hipStream_t st) {
    const uint4 *A = static_cast<const uint4*>(d_a), *B = static_cast<const uint4*>(d_b);
    const int bnn_k = type == kBNN ? K_unpack : 0, form = type == kTNN ? 0 : 1;
    return OHW > 1 ? launch_records<true>(B, A, d_y, (int)M, KN, OHW, Kw, bnn_k, form, alpha, st)
                   : launch_records<false>(A, B, d_y, (int)M, KN, OHW, Kw, bnn_k, form, alpha, st);
}

// Large layers with a stride and long rows go to the tile kernel with implicit im2row: the layer kernel gathers records a stride
// apart, so it moves twice the cache lines per record and its L1 is what bounds it; T2 keeps them side by side.  90 random layers of
// 900 to 6000 tiles of 64 x 64 and 60 to 400 words with strides of 2 to 4, both kernels under sustained load in turn, quantiser included: from
// 1500 tiles and 100 words on the tile kernel takes 0.93 of the layer kernel's time in the mean (0.78 to 1.11, ahead on 34 of 38; us, tiles /
// layer kernel: 2032 tiles x 243 words 109 / 119, 2760 x 153 at stride 4 126 / 161, 2688 x 125 at stride 3 91 / 104, 3056 x 225 109 / 119; 3488 x 126
// 95 / 86), with shorter rows 1.06 (2496 x 63 56 / 42, 4875 x 72 80 / 70), with fewer tiles 1.02 (1104 x 144 54 / 47, 1056 x 92 487 / 486, 1088 x 369
// at stride 3 118 / 127).  At stride 1 the layer kernel is ahead by 5 to 50 %.  FTNN_CONV_TILES_FROM = n: tuning aid; it sets the tile
// count and drops the other conditions.
namespace {
// the tile kernel's limits: a tap mask of 32 bits per pixel, a table entry per K word, 32-bit record indices into T2,
// its tiles of 128 pixels in y of a launch, which takes 65535, and its way of keeping kw - pad non-negative
bool conv_tiles_within_limits(int64_t M, int CP, int taps, int64_t t2_bytes, int W_pad, int W_stride) {
    const int64_t K = (int64_t)CP * taps;
    return taps <= 32 && (K + 3) / 4 * 4 <= kMaxTileRouteWords && (M + 127) / 128 <= 65535 && t2_bytes / 16 <= 0x7fffffffLL &&
           W_pad < 4096 * (int64_t)W_stride;
}
}  // namespace

bool conv_f4_tile_route(int64_t M, int KN, int CP, int taps, int64_t t2_bytes, int W_pad, int W_stride) {
    static const char* tune = getenv("FTNN_CONV_TILES_FROM");
    static const int64_t from = tune ? atoll(tune) : 1500;
    const int64_t tiles = ((M + 63) / 64) * ((KN + 63) / 64);
    return tiles >= from && (tune || (W_stride > 1 && (int64_t)CP * taps >= 100 && M >= 512)) &&
           conv_tiles_within_limits(M, CP, taps, t2_bytes, W_pad, W_stride);
}

// A large conv layer as workgroup tiles staged through LDS, the activation records gathered from T2
// (launch_quantize_f4_tiled; k_mfma_s2 with IMPL): fp32 NCHW result only.  d_wf: the weights as record blocks
// (round4(cg.K) words per row).
hipError_t launch_conv_f4_tiles(int type, const void* d_t2, const void* d_wf, const ConvGeom& cg, int N, int KN, int K_unpack,
                                float alpha, float* d_y, hipStream_t st) {
    const int OHW = cg.OH * cg.OW;
    const int64_t M = (int64_t)N * OHW;
    const int KP = round4(cg.K) / 2, pairs = (cg.K + 1) / 2;
    if (!conv_tiles_within_limits(M, cg.CP, cg.K / cg.CP, quantize_f4_tiled_bytes(N, cg.CP * 64, cg.H, cg.W, cg.W_stride), cg.W_pad, cg.W_stride))
        return hipErrorInvalidValue;
    const int bnn_k = type == kBNN ? K_unpack : 0, form = type == kTNN ? 0 : 1;
    const uint4* Wf = static_cast<const uint4*>(d_wf);
    const uint4* T2 = static_cast<const uint4*>(d_t2);
    // Tiles of 256 kernels x 128 pixels where those fill most of the chip in one round, else 128 x 128.  Ten layers of 1500 tiles of
    // 64 x 64 and more with 196 to 252 of them, under sustained load, 128 x 128 / 256 x 128: 8 x 1024 x 56 x 56 -> 1024 (196) 51.4 / 50.2 us,
    // 34 x 1024 x 28 x 28 -> 1024 (212) 59.6 / 57.5, 6 x 2105 x 56 x 87 -> 1024 (232) 120 / 114, the others 0.94 to 0.99; from 258 on 217 / 193
    // and up to 1.4.  FTNN_CONV_TILE_SHAPE = 22 | 42 forces one (tuning aid)
    static const int tune = getenv("FTNN_CONV_TILE_SHAPE") ? atoi(getenv("FTNN_CONV_TILE_SHAPE")) : 0;
    const int64_t mid = ((M + 127) / 128) * ((KN + 255) / 256);
    int shape = mid >= 180 && mid <= 256 ? 42 : 22;
    if (tune == 22 || tune == 42) shape = tune;
    if (shape == 42) return launch_records_tile<true, 4, 2, 4, true>(Wf, T2, d_y, (int)M, KN, OHW, KP, pairs, bnn_k, form, alpha, cg, st);
    return launch_records_tile<true, 2, 2, 4, true>(Wf, T2, d_y, (int)M, KN, OHW, KP, pairs, bnn_k, form, alpha, cg, st);
}

hipError_t launch_conv_f4(int type, const void* d_p2, const void* d_wf, const ConvGeom& cg, int N, int KN,
                          int K_unpack, float alpha, float* d_y, hipStream_t st, const QuantOut& qo) {
    const int OHW = cg.OH * cg.OW;
    const int64_t M = (int64_t)N * OHW;
    const int KP = round4(cg.K) / 2;
    const PairWalk pw = make_pair_walk(cg);
    // BNN: the channel lanes past C are +1 in both operands (see launch_mfma_gemm); padding words are skipped
    const int bias = type == kBNN ? 64 * cg.K - K_unpack : 0;
    static const int tune = []() {   // tuning aid: force the K split (1, 2 or 4; anything else is ignored)
        const char* e = getenv("FTNN_CONV_SPLIT");
        const int v = e ? atoi(e) : 0;
        return (v == 1 || v == 2 || v == 4) ? v : 0;
    }();
    static const int64_t tune_small = getenv("FTNN_CONV_SMALL_BELOW") ? atoi(getenv("FTNN_CONV_SMALL_BELOW")) : -1;
    const LayerCut cut = layer_cut(M, KN, cg.K, qo.mode != 0, tune, tune_small);
    const int split = cut.split, tpb = 4 / split;   // pixel tiles per workgroup (see the kernel)
    const bool small = cut.small, deep = cut.deep;
    dim3 grid((unsigned)(((M + 63) / 64 + tpb - 1) / tpb), (unsigned)((KN + 63) / 64));
    if (small) grid = dim3((unsigned)((M + 31) / 32), (unsigned)(qo.mode != 0 ? 2 * ((KN + 63) / 64) : (KN + 31) / 32));
    if (M > 0x7fffff00LL) return hipErrorInvalidValue;   // pixel indices stay below 2^31
    // A launch takes 65535 workgroups in y: from 65536 kernel tiles on they go in x.  The kernel goes by the linear number.
    const dim3 launched = grid.y > 65535 ? dim3(grid.y, grid.x) : grid;
    if (launched.y > 65535) return hipErrorInvalidValue;
    const uint4* P2 = static_cast<const uint4*>(d_p2);
    const uint4* Wf = static_cast<const uint4*>(d_wf);
    const FastDiv dOHW = make_fastdiv((uint32_t)OHW);
    // operand sizes: the buffer-load variants announce them in their descriptors
    const int64_t p2_bytes = (int64_t)N * cg.CP * cg.H * cg.W * 16, wf_bytes = (int64_t)((KN + 31) / 32) * KP * 1024;
    static const bool no_buf = getenv("FTNN_CONV_NO_BUFFER_LOADS") != nullptr;   // tuning aid
    // an fp32 tile reaches over 64 kernels of its first image and as many more images as 64 pixels may touch, within the result
    const int64_t y_span = std::min(((int64_t)std::min(N - 1, 63 / OHW + 1) * KN + 64) * OHW, M * KN) * 4;
    const bool buf = !no_buf && p2_bytes <= 0xf0000000LL && wf_bytes <= 0xf0000000LL && (qo.mode != 0 || y_span <= 0xf0000000LL);
    auto clip = [](int64_t v) { return (uint32_t)std::min<int64_t>(v, 0xffffffffLL); };
    const uint64_t wgs = (uint64_t)grid.x * grid.y;
    if (wgs > 0xffffffffull) return hipErrorInvalidValue;   // (no such result fits in memory)
    const bool plain = qo.mode == 0 && M * KN * 4 > kXcdOrderResultBytes;
    const XcdOrder xo = plain ? make_xcd_order(grid.y, grid.x, true) : make_xcd_order(grid.x, grid.y, false);
    // kernel variant: activation kind and PReLU form follow the type, then hand-over mode, tile and split, loads
    auto launch = [&](auto abin, auto form0, auto qmode, auto blocks, auto sp) -> hipError_t {
        constexpr bool A = decltype(abin)::value, F = decltype(form0)::value;
        constexpr int Q = decltype(qmode)::value, T = decltype(blocks)::value, SP = decltype(sp)::value;
        auto go = [&](auto kern) -> hipError_t {
            hipLaunchKernelGGL(kern, launched, dim3(SP == 8 ? 512 : 256), 0, st, P2, Wf, d_y, (int)M, KN, OHW, KP, bias, alpha, dOHW, cg, pw, qo,
                               clip(p2_bytes), clip(wf_bytes), clip(y_span), xo, launched.x, grid.y);
            return hipGetLastError();
        };
        return buf ? go(k_conv_f4<A, F, Q, T, T, SP, true>) : go(k_conv_f4<A, F, Q, T, T, SP, false>);
    };
    auto by_split = [&](auto abin, auto form0, auto qmode) -> hipError_t {
        typedef std::integral_constant<int, 1> one;
        typedef std::integral_constant<int, 2> two;
        typedef std::integral_constant<int, 4> four;
        if constexpr (decltype(qmode)::value == 0)
            if (deep) return launch(abin, form0, qmode, one{}, std::integral_constant<int, 8>{});
        if (small) return launch(abin, form0, qmode, one{}, four{});
        if (split == 1) return launch(abin, form0, qmode, two{}, one{});
        if (split == 2) return launch(abin, form0, qmode, two{}, two{});
        if (split == 4) return launch(abin, form0, qmode, two{}, four{});
        return hipErrorInvalidValue;
    };
    auto by_mode = [&](auto abin, auto form0) -> hipError_t {
        if (qo.mode == 0) return by_split(abin, form0, std::integral_constant<int, 0>{});
        if (qo.mode == 1) return by_split(abin, form0, std::integral_constant<int, 1>{});
        if (qo.mode == 2) return by_split(abin, form0, std::integral_constant<int, 2>{});
        return hipErrorInvalidValue;
    };
    if (type == kTNN) return by_mode(std::false_type{}, std::true_type{});
    if (type == kTBN) return by_mode(std::false_type{}, std::false_type{});
    return by_mode(std::true_type{}, std::false_type{});   // BTN, BNN
}

// A whole call from packed rows below 160 tiles of 256 x 256 multiplies the rows as they are (k_rows) and needs no scratch: packing both operands
// first costs such a product more than the packed4 kernel gains.  Device time of the two, us (rows / packed4 or, before
// k_rows, fragments): 2048 x 2048 x 16384 (64 tiles) 31.5 / 44, 3072 x 3072 x 24576 (144) 107 / 136.  Products narrower than 128 would leave
// more than half of such a tile empty.  From 160 tiles on scratch is asked for, and the estimates decide (mm_rows_ahead_of_packing: short
// rows stay as they are; 4096 x 4096 x 32768 218 / 190, x 2048 36 / 42, x 256 16 / 26).
static bool few_big_tiles(int64_t M, int KN) { return ((M + 255) / 256) * ((KN + 255) / 256) < mfma_small_tile_below(); }
bool mm_from_rows(int64_t M, int KN, int Kw) {
    return mm_rows_within_limits(M, KN, Kw) && (few_big_tiles(M, KN) || KN < 128 || M < 128);
}

// What the explicit engine asks its callers for: both operands as fragments below 160 tiles, in packed4 form from there on.
// A product from the rows touches none of it; AUTO asks for none below 160 tiles.
int64_t mfma_f4_mm_scratch_bytes(int64_t M, int KN, int Kw) {
    return few_big_tiles(M, KN) ? mfma_fragment_bytes(true, M, Kw) + mfma_fragment_bytes(true, KN, Kw)
                                : mfma_packed4_bytes(M, Kw) + mfma_packed4_bytes(KN, Kw);
}

hipError_t launch_mm_mfma(bool f4, int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW,
                          int KN, int Kw, int K_unpack, float alpha, float* d_y, void* d_scratch,
                          hipStream_t st) {
    const bool a_tern = (type == kTNN || type == kTBN), b_tern = (type == kTNN || type == kBTN);
    // a product that packs its operands first may have its result over them, whatever the estimates say (asked within mm_rows_within_limits only)
    auto over = [&]() {
        const int64_t y_bytes = 4 * M * KN;
        return ranges_meet(d_y, y_bytes, d_a, M * Kw * (a_tern ? 16 : 8)) || ranges_meet(d_y, y_bytes, d_b, (int64_t)KN * Kw * (b_tern ? 16 : 8));
    };
    if (f4 && (mm_from_rows(M, KN, Kw) || (mm_rows_ahead_of_packing(M, OHW, KN, Kw) && !over())))
        return launch_mm_rows(type, d_a, d_b, M, OHW, KN, Kw, K_unpack, alpha, d_y, st);
    if (f4) {   // the fp4 GEMM takes its operands at two bits per lane
        void* Ac = d_scratch;
        void* Bc = static_cast<char*>(d_scratch) + mfma_packed4_bytes(M, Kw);
        const int64_t na64 = (M + 31) / 32 * 32, nb64 = ((int64_t)KN + 31) / 32 * 32;
        if (na64 + nb64 > 0x7fffff00LL) return hipErrorInvalidValue;
        const int na = (int)na64, nb = (int)nb64;   // one launch zeroes both operands' row sums
        hipLaunchKernelGGL(k_zero_i32, dim3((na + nb + 255) / 256), dim3(256), 0, st, packed4_sums(Ac, M, Kw), na,
                           packed4_sums(Bc, KN, Kw), nb);
        // both operands packed by one launch
        const dim3 grid((unsigned)(na / 32 + nb / 32), (unsigned)((Kw / 4 + 3) / 4));
        if (grid.y > 65535) return hipErrorInvalidValue;
        const uint32_t *Ra = reinterpret_cast<const uint32_t*>(d_a), *Rb = reinterpret_cast<const uint32_t*>(d_b);
        uint2 *Oa = static_cast<uint2*>(Ac), *Ob = static_cast<uint2*>(Bc);
        int *Sa = packed4_sums(Ac, M, Kw), *Sb = packed4_sums(Bc, KN, Kw);
#define FTNN_PACK2(TA_, TB_) hipLaunchKernelGGL((k_pack4_2<TA_, TB_>), grid, dim3(256), 0, st, Ra, (int)M, Oa, Sa, Rb, KN, Ob, Sb, Kw / 4)
        if (a_tern && b_tern) FTNN_PACK2(true, true);
        else if (a_tern) FTNN_PACK2(true, false);
        else if (b_tern) FTNN_PACK2(false, true);
        else FTNN_PACK2(false, false);
#undef FTNN_PACK2
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        return launch_mfma_gemm_packed4(type, Ac, Bc, M, OHW, KN, Kw, K_unpack, alpha, d_y, st);
    }
    void* Af = d_scratch;
    void* Bf = static_cast<char*>(d_scratch) + mfma_fragment_bytes(false, M, Kw);
    {   // both operands expanded by one launch
        const dim3 grid((unsigned)((M + 31) / 32 + (KN + 31) / 32), (unsigned)((Kw / 4 + 3) / 4));
        if (grid.y > 65535) return hipErrorInvalidValue;
        const uint32_t *Ra = reinterpret_cast<const uint32_t*>(d_a), *Rb = reinterpret_cast<const uint32_t*>(d_b);
        uint4 *Oa = static_cast<uint4*>(Af), *Ob = static_cast<uint4*>(Bf);
#define FTNN_EXP2(TA_, TB_) hipLaunchKernelGGL((k_expand2<TA_, TB_>), grid, dim3(256), 0, st, Ra, (int)M, Oa, Rb, KN, Ob, Kw / 4)
        if (a_tern && b_tern) FTNN_EXP2(true, true);
        else if (a_tern) FTNN_EXP2(true, false);
        else if (b_tern) FTNN_EXP2(false, true);
        else FTNN_EXP2(false, false);
#undef FTNN_EXP2
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return launch_mfma_gemm(type, Af, Bf, M, OHW, KN, Kw, K_unpack, alpha, d_y, st);
}

}  // namespace ftnn
