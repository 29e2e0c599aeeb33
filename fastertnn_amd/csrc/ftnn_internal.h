// Internal declarations shared by the kernel files and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_plans.h"
#include "pair_walk.h"
#include "product_forms.h"

namespace ftnn {

typedef float v16f __attribute__((ext_vector_type(16)));

inline int round4(int k) { return 4 * ((k + 3) / 4); }
inline int out_dim(int in, int pad, int k, int stride) { return (in + 2 * pad - k) / stride + 1; }

// Which tile of outer x inner ones a workgroup of the layer kernels takes.  Workgroups go to the eight XCDs round-robin by
// their linear number; XCD x takes the x-th eighth of the tiles, walked inner index first.  With the pixels as the outer
// index every layer of a chain gives an image to the same XCD, whose L2 then still holds what that XCD wrote in the layer
// before, and the kernel tiles of a pixel tile and the halo of neighbouring ones are fetched once
// (152-layer chain at batch 8: 1103 -> 980 us; in plain order every XCD fetches nearly all of the input from beyond its L2).
// Weights as the outer index (an XCD then reads an eighth of them and all pixels): 1134 us.
//
// fp32 results beyond the 256 MiB of the Infinity Cache keep the plain order (`plain`): such a layer is bound by its
// stores, and neighbouring workgroups then fill neighbouring pages of HBM instead of eight regions at a time.  First layers,
// plain / XCD order: 32 x 3 x 224 x 224 -> 64, 3 x 3 (392 MiB) 120 / 131 us, 8 x 3 x 1024 x 1024 -> 130 (4 GiB) 1405 / 1495; last layers of
// a chain: 40 x 256 x 112 x 112 -> 256, 1 x 1 (490 MiB) 147 / 155, 40 x 64 x 128 x 128 -> 2048 (5 GiB) 933 / 1078 (some sizes go the other
// way by up to 6 %).  Up to 245 MiB the XCD order is ahead: 40 x 64 x 112 x 112 -> 128, 3 x 3 66 / 57.
// The plain order is the same arithmetic on one share (mask 0), so that a launch takes no branch before its arguments.
struct XcdOrder {
    uint32_t per, rem;   // tiles of an XCD; the first `rem` XCDs take one more
    uint32_t mask;       // 7, or 0: plain
    FastDiv inner;
    template <bool MAYBE_PLAIN>
    __device__ __forceinline__ void tile(uint32_t wg, uint32_t& o, uint32_t& i) const {
        const uint32_t x = wg & (MAYBE_PLAIN ? mask : 7u), t = x * per + min(x, rem) + (wg >> (MAYBE_PLAIN ? mask & 3u : 3u));
        o = fastdiv(t, inner);
        i = t - o * inner.d;
    }
};
constexpr int64_t kXcdOrderResultBytes = 256LL << 20;
inline XcdOrder make_xcd_order(uint64_t outer, uint32_t inner, bool plain) {   // outer * inner below 2^32
    XcdOrder x;
    x.per = (uint32_t)(outer * inner / 8);
    x.rem = (uint32_t)(outer * inner % 8);
    x.mask = plain ? 0u : 7u;
    x.inner = make_fastdiv(inner);
    return x;
}

// The GEMM tiles (k_mfma, k_mfma_p4) and layers with results beyond the Infinity Cache (k_conv_f4) store rows of 32 results, `row`
// values apart: past the caches (non-temporal) where those are whole sectors of 64 bytes, and where the result is small;
// through the caches a launch ends with their write-back.  Large results of other rows go through the caches, which put the parts
// of a sector together; past them each part is a read and a write of memory.  Whole calls, us, past / through the caches: TNN
// 4096 x 4096 x 4096 44 / 52, x 4112 columns 65 / 72, x 4111 92 / 68; 6016 x 6016 x 512 58 / 72, 6001 x 6001 124 / 60; operands kept,
// 30000 x 150 x 512 (17 MiB) 14.1 / 10.2.
inline __host__ __device__ bool stores_past_caches(int row, int64_t M, int KN) { return row % 16 == 0 || M * KN <= (4 << 20); }

// Quantised layer operands: two bits per lane, a record of 16 bytes per 64 lanes ("P2").
//
// A lane in {-1, 0, +1} is an E2M1 nibble 0xA / 0x0 / 0x2, which uses bits 1 (not zero) and 3 (sign) only, so two dwords of
// nibbles D0, D1 share one dword P = D0 | D1 >> 1 and come apart as D0 = P & 0xAAAAAAAA, D1 = (P << 1) & 0xAAAAAAAA: 1.5 vector
// instructions per dword beside the multiplies, for half the bytes through memory, L1 and LDS and half the loads.  The
// layer kernels are bound by those bytes (64 per cycle and compute unit come back from the L1) and not by instructions.
// Against nibbles at four bits: see the layer kernels.
//
// Lane c = 32 a + 8 q + 4 h + i of a record sits in dword 2 h + a, byte q, nibble i / 2; even i in bits 1 and 3, odd i in bits
// 0 and 2.  That is the order in which an accumulator tile holds its kernels (a: block, h: lane half, 4 q + i: register), so
// an epilogue hands its results over without exchanging lanes.  Dwords 0, 1 feed one multiply, dwords 2, 3 the next.
// Few-channel first layers keep their lanes in plain order (`natural`: dword j holds lanes 16 j .. 16 j + 7 as D0 and the
// next eight as D1) in both operands: any order serves as long as both have it.
constexpr uint32_t kP2Mask = 0xAAAAAAAAu;   // D0 of a dword
constexpr uint32_t kP2Plus = 0x33333333u;   // +1 in every lane: the padding of binary activations
__device__ __forceinline__ uint32_t p2_join(uint32_t d0, uint32_t d1) { return d0 | d1 >> 1; }

// Fused hand-over to a following fp4 layer: instead of the fp32 result, a GEMM kernel writes the
// next layer's quantised input, P2[n][ceil(KN/64)][pixel][16 bytes] (see launch_quantize_f4), from
// the same fp32 values: mode 1 = ternary with threshold t (strict compares), 2 = binary, 0 = off.
// Kernels past KN in the last 64-channel word get the padding lane.
//
// cut = true: the thresholds as cuts on the integer r in front of PReLU, found on the host (make_quant_out).  PReLU does
// not fall for a slope >= 0, so r -> sign is a staircase:
//   ternary  -1 for r < lo, +1 for r > lo + width, 0 between
//   binary   -1 (bit set) for r < lo, else +1
// An accumulator that starts at `init` ends at a = r - lo (binary: r - lo + 1/2), and a value takes two vector
// instructions, clamp(a - width, 0, 1) = p and med3(a, -1, p) (binary: one, med3(a, -1/2, 1/2)), before two of them
// become two nibbles in one conversion (v_cvt_scalef32_pk_fp4_f32).  Other slopes and thresholds run PReLU and compare.
struct QuantOut {
    void* p2 = nullptr;
    float t = 0.0f;       // the next layer's threshold
    int mode = 0;
    bool cut = false;
    float lo = 0.0f, width = 0.0f;
};
constexpr int kMaxCutSum = 1 << 22;   // largest |r| the cuts are made for: r - lo and its half steps stay exact in fp32

// alpha, form0: the producing layer's PReLU; max_sum: bound of |r|
QuantOut make_quant_out(void* p2, int mode, float t, float alpha, int64_t max_sum);

// the E2M1 nibble of one value under QuantOut mode 1 / 2 (src/tnns/ternarize2row_avx2.c:443-449,
// src/tnns/binarize2row_avx2.c:19-21); `live` = false gives the padding lane of that mode
__device__ __forceinline__ uint32_t quant_nibble(float v, float t, bool ternary, bool live) {
    // selects only: a branch per element costs more than the whole computation
    uint32_t r;
    if (ternary) {
        r = v > t ? 0x2u : 0x0u;
        r = v < -t ? 0xAu : r;
        r = live ? r : 0x0u;
    } else {
        r = v < t ? 0xAu : 0x2u;
        r = live ? r : 0x2u;
    }
    return r;
}

// eight values -> one dword of E2M1 nibbles, value k in nibble k: ternary out of {+1, -1, 0}, binary out of {+1/2, -1/2}
// (the conversion divides by its scale)
template <int QMODE>
__device__ __forceinline__ uint32_t pack_fp4x8(const float* z) {
    constexpr float scale = QMODE == 1 ? 1.0f : 0.5f;
    uint32_t d = 0u;
    d = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(d, z[0], z[1], scale, 0);
    d = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(d, z[2], z[3], scale, 1);
    d = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(d, z[4], z[5], scale, 2);
    d = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(d, z[6], z[7], scale, 3);
    return d;
}

// PReLU in the reference's two forms: "f <= 0 -> f *= alpha" (TNN, src/tnns/mm_p2_final_tnn_avx2.c:204-208; a zero
// becomes 0 * alpha) and "r >= 0 ? r : alpha * r" (the others, src/tnns/mm_p2_final_tbn_avx2.c:73)
template <bool FORM0>
__device__ __forceinline__ float prelu_ref(float r, float alpha) {
    const bool scale = FORM0 ? (r <= 0.0f) : (r < 0.0f);
    return scale ? r * alpha : r;
}

// what an accumulator starts at: r = sum - bias with the hand-over's cut taken off, see QuantOut (wave-uniform)
template <int QMODE>
__device__ __forceinline__ float acc_init(const QuantOut& qo, float bias) {
    if (QMODE == 0 || !qo.cut) return 0.0f - bias;
    return 0.0f - qo.lo - bias + (QMODE == 2 ? 0.5f : 0.0f);
}

// One 32-kernel block of a pixel under the hand-over.  v[e] = this lane's 16 accumulators (started at acc_init), kernel
// kbase + 8 (e / 4) + 4 h + e % 4 (h = lane half).  Returns dword 2 h + a of the pixel's record (a: the block's number in its word).
template <bool FORM0, int QMODE>
__device__ __forceinline__ uint32_t hand_over_block(const v16f& v, float alpha, const QuantOut& qo, int kbase, int h, int KN) {
    const bool whole = kbase + 32 <= KN;   // wave-uniform: the block holds real kernels only
    if (qo.cut) {
        float z[16];   // even registers, then odd ones
#pragma unroll
        for (int e = 0; e < 16; e++) {
            float& d = z[(e >> 1) + 8 * (e & 1)];
            if (QMODE == 1) d = __builtin_amdgcn_fmed3f(v[e], -1.0f, __builtin_amdgcn_fmed3f(v[e] - qo.width, 0.0f, 1.0f));
            else d = __builtin_amdgcn_fmed3f(v[e], -0.5f, 0.5f);
        }
        if (!whole) {   // kernels past KN hold the padding lane
#pragma unroll
            for (int e = 0; e < 16; e++) {
                float& d = z[(e >> 1) + 8 * (e & 1)];
                d = kbase + 8 * (e >> 2) + 4 * h + (e & 3) < KN ? d : (QMODE == 1 ? 0.0f : 0.5f);
            }
        }
        return p2_join(pack_fp4x8<QMODE>(z), pack_fp4x8<QMODE>(z + 8));
    }
    uint32_t d[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 16; e++)
        d[e & 1] |= quant_nibble(prelu_ref<FORM0>(v[e], alpha), qo.t, QMODE == 1, kbase + 8 * (e >> 2) + 4 * h + (e & 3) < KN) << (4 * (e >> 1));
    return p2_join(d[0], d[1]);
}

// record a failure text for ftnn_last_error(); returns `code`
int fail(int code, const char* fmt, ...);

// shape and size-limit validation shared by every layer entry point; fills OH / OW; FTNN_OK or a recorded failure
int check_conv_shape(int N, int C, int H, int W, int H_pad, int W_pad, int kH, int kW, int H_stride, int W_stride,
                     int* OH, int* OW);

// ---- pack_kernels.hip: launchers (arguments already validated) ----
hipError_t launch_quantize_im2row(bool ternary, const float* d_x, const float* d_thr, int N, int C,
                                  int H, int W, int H_pad, int W_pad, int kH, int kW, int H_stride,
                                  int W_stride, int64_t* d_out, void* d_scratch, hipStream_t st);
hipError_t launch_pack_weights(bool ternary, const float* d_w, const float* d_thr, int KN, int C,
                               int KH, int KW, int64_t* d_out, hipStream_t st);
hipError_t launch_pack_gemm_operand(const float* d_x, int I, int J, int64_t* d_out, hipStream_t st);

// ---- mm_kernels.hip ----
hipError_t launch_mm(int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW, int KN,
                     int Kw /* words per plane, multiple of 4 */, int K_unpack, float alpha,
                     float* d_y, hipStream_t st, const QuantOut& qo = QuantOut());

// GEMM straight from the channel-packed input P (no im2row matrix in memory)
hipError_t launch_mm_implicit(int type, const void* d_p, const int64_t* d_b, const ConvGeom& cg, int N,
                              int KN, int K_unpack, float alpha, float* d_y, hipStream_t st,
                              const QuantOut& qo = QuantOut());
// quantise only: fp32 NCHW -> P
hipError_t launch_quantize(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                           void* d_p, hipStream_t st);

// quantise only, into two-bit records: fp32 NCHW -> P2[n][C_pack][pixel][16 bytes] (operand of launch_conv_f4)
hipError_t launch_quantize_f4(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                              void* d_p2, hipStream_t st);
// quantise only, into Packing-2 rows: fp32 [N][C] -> N rows (activations of a fully connected layer as launch_mm_rows reads them)
hipError_t launch_quantize_rows(bool ternary, const float* d_x, const float* d_thr, int N, int C, int64_t* d_out, hipStream_t st);

// dense re-packing of both operands for layers with C <= 32 (several taps per 64-lane word), the activations from fp32
bool dense_applies(int C, int KH, int KW, int* T_out, int* Kd_out);
hipError_t launch_dense_rows(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W, int H_pad, int W_pad,
                             int kH, int kW, int H_stride, int W_stride, void* d_p /* room for launch_quantize's planes */, int64_t* d_out, hipStream_t st);
hipError_t launch_dense_weights(bool ternary, const int64_t* d_qw, int KN, int C, int kH, int kW,
                                int64_t* d_out, hipStream_t st);

// the same for the fp4 layer kernel (C <= 8): quantise to one nibble dword per pixel (d_pq,
// dense_f4_pq_bytes), then string T taps per 64-lane word into A2[n][Kd][output pixel][16 bytes] (d_a2, natural lane
// order), the operand of launch_conv_f4 for a 1x1 layer with C_pack = Kd over the OH x OW output pixels
bool dense_f4_applies(int C, int KH, int KW);
// stem_kernels.hip: the same layer in one kernel (fp32 input -> result, the rows never stored) where its input
// patch fits the LDS: bytes of LDS it needs, 0 = does not apply
int64_t stem_f4_lds_bytes(int C, int KH, int KW, int H_stride, int W_stride);
hipError_t launch_stem_f4(int type, const float* d_x, const float* d_thr, const void* d_wf, int N, int C, int H,
                          int W, int KN, int KH, int KW, int H_pad, int W_pad, int H_stride, int W_stride,
                          float alpha, float* d_y, hipStream_t st, const QuantOut& qo);
int64_t dense_f4_pq_bytes(int N, int H, int W);
hipError_t launch_dense_rows_f4(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                                int H_pad, int W_pad, int kH, int kW, int H_stride, int W_stride, void* d_pq,
                                void* d_a2, hipStream_t st);

// ---- mfma_kernels.hip: matrix-core formulation ----
// Bytes of an operand brought into engine form: int8 fragments (1 KiB per 32 rows and half word), or what a layer's weights are
// given (1 KiB per 32 rows and word; their records take half of it)
int64_t mfma_fragment_bytes(bool f4, int64_t rows, int Kw);
// packed rows -> int8 fragments
hipError_t launch_mfma_expand(bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st);
// packed rows -> record blocks, 1 KiB [row block of 32][pair of K words][lane l = (word of the pair l / 32, row l % 32)][16 bytes]:
// weights of the fp4 layer kernels, and im2row rows of the layers' GEMM route.  natural: lane order of few-channel first layers;
// d_kept: also copies the rows there
int64_t record_block_bytes(int64_t rows, int Kw);
hipError_t launch_expand_records(bool ternary, bool natural, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st,
                                 int64_t* d_kept = nullptr);
hipError_t launch_mfma_gemm(int type, const void* d_af, const void* d_bf, int64_t M, int OHW, int KN,
                            int Kw, int K_unpack, float alpha, float* d_y, hipStream_t st);
// the layers' GEMM route: both operands as record blocks
hipError_t launch_records_gemm(int type, const void* d_a, const void* d_b, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                               float alpha, float* d_y, hipStream_t st);
// the fp4 GEMM's own operand form, two bits per lane ("packed4"): what ftnn_expand_rows / ftnn_mm_expanded /
// ftnn_mm_engine use for FTNN_ENGINE_MFMA_F4
int64_t mfma_packed4_bytes(int64_t rows, int Kw);
hipError_t launch_mfma_pack4(bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out, hipStream_t st);
hipError_t launch_mfma_gemm_packed4(int type, const void* d_ac, const void* d_bc, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                                    float alpha, float* d_y, hipStream_t st);
// whether launch_mm_mfma runs an fp4 product straight from the packed rows (launch_mm_rows): by shape
bool mm_from_rows(int64_t M, int KN, int Kw);
// scratch that the explicit fp4 engine asks for
int64_t mfma_f4_mm_scratch_bytes(int64_t M, int KN, int Kw);
hipError_t launch_mm_mfma(bool f4, int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW,
                          int KN, int Kw, int K_unpack, float alpha, float* d_y, void* d_scratch,
                          hipStream_t st);

// ---- rows_kernels.hip: the fp4 matrix-core product of packed rows as they are, one launch, no scratch ----
// (where mm_rows_within_limits: fp32 sums of +-1 products stay exact, and the grid holds the product)
hipError_t launch_mm_rows(int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                          float alpha, float* d_y, hipStream_t st);

// The same for operands in packed4 form (launch_mfma_pack4) with their rows' sums.  False where workgroup tiles through LDS (k_mfma_p4) are
// ahead: nothing has been done then.
bool launch_mm_packed(int type, const void* d_ac, const void* d_bc, const int* sA, const int* sB, int64_t M, int OHW, int KN, int Kw,
                      int K_unpack, float alpha, float* d_y, hipStream_t st, hipError_t* err);

// conv layer on the fp4 matrix cores: activations from launch_quantize_f4, weights as the record blocks
// launch_expand_records makes of the packed weight rows (Kw = round4(cg.K) words per row)
hipError_t launch_conv_f4(int type, const void* d_p2, const void* d_wf, const ConvGeom& cg, int N, int KN,
                          int K_unpack, float alpha, float* d_y, hipStream_t st, const QuantOut& qo = QuantOut());


// the same layer as workgroup tiles of 128 x 128 or 256 x 128 staged through LDS (the activation records gathered from T2, the
// quantised input in the layout of launch_quantize_f4_tiled): for layers with conv_f4_tile_route() and an fp32 result
int64_t quantize_f4_tiled_bytes(int N, int C, int H, int W, int W_stride);
hipError_t launch_quantize_f4_tiled(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                                    int W_stride, void* d_t2, hipStream_t st);
bool conv_f4_tile_route(int64_t M, int KN, int CP, int taps, int64_t t2_bytes, int W_pad, int W_stride);
hipError_t launch_conv_f4_tiles(int type, const void* d_t2, const void* d_wf, const ConvGeom& cg, int N, int KN,
                                int K_unpack, float alpha, float* d_y, hipStream_t st);

// ---- direct_kernels.hip ----
// A small layer from its fp32 input in one launch, no scratch; d_wf: its weights as record blocks.  False where the layer is none of
// those it is meant for: nothing has been done then.
bool launch_direct_f4(int type, const float* d_x, const float* d_thr, const void* d_wf, const ConvGeom& cg, int C, int N, int KN,
                      int K_unpack, float alpha, float* d_y, hipStream_t st, hipError_t* err);

// ---- ftnn_api.hip ----  (arguments already validated)
// The fp4 layer with weights expanded beforehand (d_wf: launch_expand_records of the packed rows).
// d_x != null: the input is quantised into d_p2 (N*H*W*C_pack*16 bytes) first; d_x == null: d_p2 already
// holds it (written by the previous layer through its QuantOut).  qo.mode != 0: d_y is not written.
int conv_f4_expanded(int type, const float* d_x, const float* d_thr, const void* d_wf, int N, int C, int H,
                     int W, int KN, int KH, int KW, int H_pad, int W_pad, int H_stride, int W_stride,
                     float prelu_alpha, void* d_p2, float* d_y, hipStream_t st, const QuantOut& qo);
// the vector-ALU layer; d_scratch as for ftnn_conv
// (weights_prepared: for a few-channel layer d_qw already holds the re-packed rows of launch_dense_weights; any_engine: their product
// may run on the matrix cores)
int conv_valu(int type, const float* d_x, const float* d_thr, const int64_t* d_qw, int N, int C, int H, int W,
              int KN, int KH, int KW, int H_pad, int W_pad, int H_stride, int W_stride, float prelu_alpha,
              void* d_scratch, float* d_y, hipStream_t st, const QuantOut& qo, bool weights_prepared, bool any_engine);
// bytes of the fp4 layer's operand region (d_p2 above) for this shape, rounded up to 256: P2, or for a
// few-channel layer the nibble pixels and dense rows
int64_t conv_f4_operand_bytes(int N, int C, int H, int W, int KH, int KW, int OH, int OW, int KN, int W_stride);
// words per row of the weights as the fp4 layer reads them (the dense re-packing shortens them)
int conv_f4_weight_words(int C, int KH, int KW);

}  // namespace ftnn
