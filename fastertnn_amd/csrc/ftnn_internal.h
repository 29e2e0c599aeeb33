// Internal declarations shared by the kernel files and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ftnn {

constexpr int kTNN = 0, kTBN = 1, kBTN = 2, kBNN = 3;

typedef float v16f __attribute__((ext_vector_type(16)));

inline int cpack_of(int C) { return (int)(((int64_t)C + 63) / 64); }
inline int round4(int k) { return 4 * ((k + 3) / 4); }
inline int out_dim(int in, int pad, int k, int stride) { return (in + 2 * pad - k) / stride + 1; }

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
__device__ __forceinline__ uint32_t fastdiv(uint32_t n, const FastDiv& f) {
    uint32_t q = __umulhi(n, f.m);
    if (n - q * f.d >= f.d) q++;
    return q;
}

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

// geometry of one conv layer as the implicit-im2row GEMM needs it
struct ConvGeom {
    int H, W, CP, OH, OW, KW, K;   // K = C_pack*KH*KW words per plane before rounding
    int H_pad, W_pad, H_stride, W_stride;
    FastDiv dOW, dCP, dKW;
};

// Fused hand-over to a following fp4 layer: instead of the fp32 result, a GEMM kernel writes the
// next layer's quantised input, P4[n][ceil(KN/64)][pixel][32 bytes] (see launch_quantize_f4), from
// the same fp32 values: mode 1 = ternary with threshold t (strict compares), 2 = binary, 0 = off.
// Kernels past KN in the last 64-channel word get the padding nibble.
//
// cut = true: the thresholds as cuts on the integer r in front of PReLU, found on the host (make_quant_out).  PReLU does
// not fall for a slope >= 0, so r -> sign is a staircase:
//   ternary  -1 for r < lo, +1 for r > lo + width, 0 between
//   binary   -1 (bit set) for r < lo, else +1
// An accumulator that starts at `init` ends at a = r - lo (binary: r - lo + 1/2), and a value takes two vector
// instructions, clamp(a - width, 0, 1) = p and med3(a, -1, p) (binary: one, med3(a, -1/2, 1/2)), before two of them
// become two nibbles in one conversion (v_cvt_scalef32_pk_fp4_f32).  Other slopes and thresholds run PReLU and compare.
struct QuantOut {
    void* p4 = nullptr;
    float t = 0.0f;       // the next layer's threshold
    int mode = 0;
    bool cut = false;
    float lo = 0.0f, width = 0.0f;
};
constexpr int kMaxCutSum = 1 << 22;   // largest |r| the cuts are made for: r - lo and its half steps stay exact in fp32

// alpha, form0: the producing layer's PReLU; max_sum: bound of |r|
QuantOut make_quant_out(void* p4, int mode, float t, float alpha, int64_t max_sum);

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

// Lanes l and l ^ 32 hold the nibbles of one pixel for a 32-kernel block, lane half h those of kernels 8 q + 4 h + {0..3},
// as d.x (q = 0, 1) and d.y (q = 2, 3), 16 bits per q; the block's dword q is the pair's 16 bits side by side.
// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second.
//
// one block: lane half h returns dwords 2 h and 2 h + 1
__device__ __forceinline__ uint2 exchange_halves(const uint2& d) {
    const auto r = __builtin_amdgcn_permlane32_swap(d.x, d.y, false, false);
    // lanes 0..31: r[0] = own d.x, r[1] = d.x of lane + 32; lanes 32..63: r[0] = d.y of lane - 32, r[1] = own d.y
    return make_uint2((r[0] & 0xffffu) | (r[1] << 16), (r[0] >> 16) | (r[1] & 0xffff0000u));
}
// two blocks (the pixel's 64 kernels): lane half h returns the 16 bytes of block h
__device__ __forceinline__ uint4 exchange_blocks(const uint2& b0, const uint2& b1) {
    const auto r = __builtin_amdgcn_permlane32_swap(b0.x, b1.x, false, false);
    const auto s = __builtin_amdgcn_permlane32_swap(b0.y, b1.y, false, false);
    return make_uint4((r[0] & 0xffffu) | (r[1] << 16), (r[0] >> 16) | (r[1] & 0xffff0000u),
                      (s[0] & 0xffffu) | (s[1] << 16), (s[0] >> 16) | (s[1] & 0xffff0000u));
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
// kbase + 8 (e / 4) + 4 h + e % 4 (h = lane half).  Returns the nibbles as exchange_halves / exchange_blocks take them.
template <bool FORM0, int QMODE>
__device__ __forceinline__ uint2 hand_over_block(const v16f& v, float alpha, const QuantOut& qo, int kbase, int h, int KN) {
    const bool whole = kbase + 32 <= KN;   // wave-uniform: the block holds real kernels only
    if (qo.cut) {
        float z[16];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            if (QMODE == 1) z[e] = __builtin_amdgcn_fmed3f(v[e], -1.0f, __builtin_amdgcn_fmed3f(v[e] - qo.width, 0.0f, 1.0f));
            else z[e] = __builtin_amdgcn_fmed3f(v[e], -0.5f, 0.5f);
        }
        if (!whole) {   // kernels past KN hold the padding lane
#pragma unroll
            for (int e = 0; e < 16; e++)
                z[e] = kbase + 8 * (e >> 2) + 4 * h + (e & 3) < KN ? z[e] : (QMODE == 1 ? 0.0f : 0.5f);
        }
        return make_uint2(pack_fp4x8<QMODE>(z), pack_fp4x8<QMODE>(z + 8));
    }
    uint32_t half[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
        half[g] = 0u;
#pragma unroll
        for (int i = 0; i < 4; i++)
            half[g] |= quant_nibble(prelu_ref<FORM0>(v[4 * g + i], alpha), qo.t, QMODE == 1, kbase + 8 * g + 4 * h + i < KN) << (4 * i);
    }
    return make_uint2(half[0] | (half[1] << 16), half[2] | (half[3] << 16));
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

// quantise only, into fp4 nibbles: fp32 NCHW -> P4[n][C_pack][pixel][32 bytes] (operand of launch_conv_f4)
hipError_t launch_quantize_f4(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                              void* d_p4, hipStream_t st);
// quantise only, into Packing-2 rows: fp32 [N][C] -> N rows (activations of a fully connected layer as launch_mm_rows reads them)
hipError_t launch_quantize_rows(bool ternary, const float* d_x, const float* d_thr, int N, int C, int64_t* d_out, hipStream_t st);

// dense re-packing of both operands for layers with C <= 32 (several taps per 64-lane word)
bool dense_applies(int C, int KH, int KW, int* T_out, int* Kd_out);
hipError_t launch_dense_rows(bool ternary, const void* d_p, int N, int C, int H, int W, int H_pad, int W_pad,
                             int kH, int kW, int H_stride, int W_stride, int64_t* d_out, hipStream_t st);
hipError_t launch_dense_weights(bool ternary, const int64_t* d_qw, int KN, int C, int kH, int kW,
                                int64_t* d_out, hipStream_t st);

// the same for the fp4 layer kernel (C <= 8): quantise to one nibble dword per pixel (d_pq,
// dense_f4_pq_bytes), then string T taps per 64-lane word into A4[n][Kd][output pixel][32 bytes] (d_a4), the
// operand of launch_conv_f4 for a 1x1 layer with C_pack = Kd over the OH x OW output pixels
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
                                void* d_a4, hipStream_t st);

// ---- mfma_kernels.hip: matrix-core formulation (int8 or fp4 operands expanded into d_scratch) ----
int64_t mfma_fragment_bytes(bool f4, int64_t rows, int Kw);
hipError_t launch_mfma_expand(bool f4, bool ternary, const int64_t* d_rows, int rows, int Kw, void* d_out,
                              hipStream_t st, int64_t* d_kept = nullptr /* also copies the rows there */);
hipError_t launch_mfma_gemm(bool f4, int type, const void* d_af, const void* d_bf, int64_t M, int OHW, int KN,
                            int Kw, int K_unpack, float alpha, float* d_y, hipStream_t st);
// the fp4 GEMM's own operand form, two bits per lane ("packed4"): what ftnn_expand_rows / ftnn_mm_expanded /
// ftnn_mm_engine use for FTNN_ENGINE_MFMA_F4 (the layer kernels keep the plain fragments above)
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
// fp32 sums of +-1 products stay exact, and the grid holds the product
bool mm_rows_within_limits(int64_t M, int KN, int Kw);
hipError_t launch_mm_rows(int type, const int64_t* d_a, const int64_t* d_b, int64_t M, int OHW, int KN, int Kw, int K_unpack,
                          float alpha, float* d_y, hipStream_t st);

// conv layer on the fp4 matrix cores: activations from launch_quantize_f4, weights as the fp4 fragments
// launch_mfma_expand(true, ...) makes of the packed weight rows (Kw = round4(cg.K) words per row)
hipError_t launch_conv_f4(int type, const void* d_p4, const void* d_wf, const ConvGeom& cg, int N, int KN,
                          int K_unpack, float alpha, float* d_y, hipStream_t st, const QuantOut& qo = QuantOut());


// the same layer as workgroup tiles of 128 x 128 or 256 x 256 staged through LDS (the GEMM kernel with its activation
// fragments gathered from T4, the quantised input in the layout of launch_quantize_f4_tiled): for layers with
// conv_f4_tile_route() and an fp32 result
int64_t quantize_f4_tiled_bytes(int N, int C, int H, int W, int W_stride);
hipError_t launch_quantize_f4_tiled(bool ternary, const float* d_x, const float* d_thr, int N, int C, int H, int W,
                                    int W_stride, void* d_t4, hipStream_t st);
bool conv_f4_tile_route(int64_t M, int KN, int CP, int taps, int64_t t4_bytes, int W_pad, int W_stride);
hipError_t launch_conv_f4_tiles(int type, const void* d_p4, const void* d_wf, const ConvGeom& cg, int N, int KN,
                                int K_unpack, float alpha, float* d_y, hipStream_t st);

// ---- ftnn_api.hip ----  (arguments already validated)
// The fp4 layer with weights expanded beforehand (d_wf: launch_mfma_expand(true, ...) of the packed rows).
// d_x != null: the input is quantised into d_p4 (N*H*W*C_pack*32 bytes) first; d_x == null: d_p4 already
// holds it (written by the previous layer through its QuantOut).  qo.mode != 0: d_y is not written.
int conv_f4_expanded(int type, const float* d_x, const float* d_thr, const void* d_wf, int N, int C, int H,
                     int W, int KN, int KH, int KW, int H_pad, int W_pad, int H_stride, int W_stride,
                     float prelu_alpha, void* d_p4, float* d_y, hipStream_t st, const QuantOut& qo);
// the vector-ALU layer; d_scratch as for ftnn_conv
// (weights_prepared: for a few-channel layer d_qw already holds the re-packed rows of launch_dense_weights)
int conv_valu(int type, const float* d_x, const float* d_thr, const int64_t* d_qw, int N, int C, int H, int W,
              int KN, int KH, int KW, int H_pad, int W_pad, int H_stride, int W_stride, float prelu_alpha,
              void* d_scratch, float* d_y, hipStream_t st, const QuantOut& qo, bool weights_prepared);
// bytes of the fp4 layer's operand region (d_p4 above) for this shape, rounded up to 256: P4, or for a
// few-channel layer the nibble pixels and dense rows
int64_t conv_f4_operand_bytes(int N, int C, int H, int W, int KH, int KW, int OH, int OW, int KN, int W_stride);
// words per row of the weights as the fp4 layer reads them (the dense re-packing shortens them)
int conv_f4_weight_words(int C, int KH, int KW);

}  // namespace ftnn
