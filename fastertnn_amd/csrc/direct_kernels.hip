// A small layer from fp32 input to fp32 result in one launch.
//
// A layer of a few thousand pixels takes the layer kernel 1 us beyond its launch, and the quantiser in front of it 0.6: most of
// the call is two launches (1.7 us each in a graph, 2.2 us of host time each).  Here a workgroup fetches the piece of the input
// that a tile of 32 output pixels reads (all channels, the window's halo included), quantises it into the records of the layer
// kernels in LDS, and multiplies it with the record blocks of the layer's prepared weights.  Nothing is stored in between.
//
//   * A workgroup is eight wavefronts.  2^lgS of them split the K words of one block of 32 kernels x 32 pixels, so that a workgroup
//     covers 8 / 2^lgS blocks of kernels of its tile; the shares meet in LDS.
//   * A tile is 2^lgTW x 32 / 2^lgTW pixels of one image, whichever reads the least input; 1 x 1 windows without a stride see the image
//     as one row.  Region pixels outside the image hold the reference's fill, so that a tap is an LDS offset, the same for all lanes
//     of a half, from a table with an entry per K word (words past K point at a record of zeros).
//   * Quantising takes five vector instructions per value: signs and compares are pushed one after the other into a dword whose
//     bits then lie as the record wants them.
//   * Fully connected layers (FC): a tile is 32 images, their rows read as they lie, and the operands change sides, so that lanes run
//     along the kernels and the result's rows.
//
// What bounds it: the chain launch -> arguments -> input -> LDS -> multiplies -> LDS -> result, 2.5 to 3 us beside the launch, and
// the L1, which delivers the pieces of the input's rows a cache line at a time.  Every tile reads its halo and every workgroup
// all channels, so this is for small layers only (direct_plan).  Device time in a graph, us, quantiser + layer kernel / here:
// 8 x 128 x 28 x 28 -> 128, 3 x 3 6.5 / 6.2; 1 x 64 x 16 x 16 -> 256, 3 x 3 5.1 / 4.4; 3 x 64 x 39 x 39 -> 256, 1 x 1 6.5 / 5.3; 8 x 512 -> 1000
// fully connected 4.9 / 4.3; 1 x 7660 -> 413 6.1 / 4.9: 0.84 in the mean of 800 layers with a window.  Queued from Python, where a launch is also 2.2 us of the
// host's, the same five 7.6 / 6.1, 7.6 / 4.3, 7.6 / 5.1, 7.8 / 4.2, 7.7 / 4.8.
#include "ftnn_internal.h"

namespace ftnn {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kLgW = kDirectLgWaves, kThreads = 64 << kLgW;
constexpr int G = 4;   // pairs of K words in flight

struct DirectArgs {
    const float* x;
    const float* thr;
    const uint4* Wf;
    float* Y;
    int N, C, CP, H, W, KN, OH, OW;
    int K, NP, KP;            // words of a row, pairs of them, pairs a weight row is stored at
    int RW, RP;               // the region of the input that a tile reads: pixels of a row, in all
    int rstep, cstep;         // input rows / columns between neighbouring region pixels
    int lrow, lcol;           // region rows / columns between neighbouring output pixels
    int H_stride, W_stride, H_pad, W_pad, KW;
    int lgTW, lgS;
    int OHt, OWt;             // rows and columns of outputs that a tile's region serves
    int vec4;
    FastDiv dRP, dRW, dTX, dTI, dCP, dKW;
    float bias, lim, alpha;
    XcdOrder xo;
};

__device__ __forceinline__ uint32_t push(uint32_t acc, bool bit) { return acc + acc + (bit ? 1u : 0u); }
__device__ __forceinline__ uint32_t push_sign(uint32_t acc, float v) { return __builtin_amdgcn_alignbit(acc, __float_as_uint(v), 31); }

// Four lanes (channels 4 q .. 4 q + 3 of a record's 64) as one byte of their record, pushed into acc from the right
template <bool ABIN>
__device__ __forceinline__ uint32_t push4(uint32_t acc, const float* v, float t) {
    if constexpr (ABIN) {   // src/tnns/binarize2row_avx2.c:19-21
        acc = push(push(acc, v[2] < t), v[3] < t);
        acc = acc << 2 | 3u;
        acc = push(push(acc, v[0] < t), v[1] < t);
        acc = acc << 2 | 3u;
    } else {   // strict compares, src/tnns/ternarize2row_avx2.c:443-449, for t >= 0; the sign of a zero lane is of no account
        acc = push_sign(push_sign(acc, v[2]), v[3]);
        acc = push(push(acc, __builtin_fabsf(v[2]) > t), __builtin_fabsf(v[3]) > t);
        acc = push_sign(push_sign(acc, v[0]), v[1]);
        acc = push(push(acc, __builtin_fabsf(v[0]) > t), __builtin_fabsf(v[1]) > t);
    }
    return acc;
}
// the same for a negative threshold: below -t comes first
__device__ __forceinline__ uint32_t push4_any(uint32_t acc, const float* v, float t) {
    uint32_t b = 0u;
#pragma unroll
    for (int i = 0; i < 4; i++) b |= (v[i] < -t ? 5u : v[i] > t ? 1u : 0u) << (4 * (i >> 1) + 1 - (i & 1));
    return acc << 8 | b;
}
// the bits of four lanes of which the first `real` are channels of the input
__device__ __forceinline__ uint32_t real_mask4(int real) { return (uint32_t)(0xffaf0f0a00ull >> (8 * min(max(real, 0), 4))) & 0xffu; }

template <bool ABIN, bool FC>
__global__ __launch_bounds__(kThreads) void k_direct_f4(DirectArgs a) {
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, lr = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t tile, grp;
    a.xo.tile<false>(blockIdx.x, tile, grp);
    const int ks = wave & ((1 << a.lgS) - 1), kb = (int)(grp << (kLgW - a.lgS)) + (wave >> a.lgS);   // K share, block of 32 kernels
    const int p0 = (a.NP * ks) >> a.lgS, p1 = (a.NP * (ks + 1)) >> a.lgS;
    const bool idle = kb * 32 >= a.KN;   // wave-uniform: no such kernels

    const uint32_t rec_bytes = (uint32_t)(a.CP * a.RP) * 16u;   // records, then a record of zeros, then the table
    uint32_t* const words = reinterpret_cast<uint32_t*>(lds);
    uint32_t* const tab = words + rec_bytes / 4 + 4;
    const int rbmax = (a.KN + 31) / 32 - 1;
    const uint4* const wp = a.Wf + (size_t)min(kb, rbmax) * a.KP * 64 + lane;
    v4i w[G];
    auto weights = [&](v4i* to, int p) {   // pairs p, p + 1, ... of this wavefront's share
#pragma unroll
        for (int d = 0; d < G; d++)
            if (p + d < p1) to[d] = *reinterpret_cast<const v4i*>(wp + (size_t)(p + d) * 64);
    };
    // what else there is to do while the first piece of the input is on its way
    auto meanwhile = [&]() {
#pragma unroll
        for (int d = 0; d < G; d++) w[d] = v4i{0, 0, 0, 0};
        weights(w, p0);
        // where a K word's records lie, from the record of the lane's output pixel at tap (0, 0), plane 0
        for (int i = tid; i < 2 * a.NP; i += kThreads) {
            uint32_t off;
            if constexpr (FC) {
                off = (uint32_t)i * 512u;
            } else {
                const int tap = (int)fastdiv((uint32_t)i, a.dCP), ic = i - tap * a.CP;
                const int kh = (int)fastdiv((uint32_t)tap, a.dKW), kw = tap - kh * a.KW;
                off = (uint32_t)(ic * a.RP + kh * a.RW + kw) * 16u;
            }
            tab[i] = i < a.K ? off : ~0u;
        }
        if (tid < 4) words[rec_bytes / 4 + tid] = 0u;
    };

    int n, oh = 0, ow = 0;
    if constexpr (FC) {
        n = (int)tile * 32;
        const int rows = min(32, a.N - n), quads = a.CP * 16, U = rows * quads;
        const float* const xt = a.x + (size_t)n * a.C;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(xt), 0, rows * a.C * 4, 0x00020000);
        constexpr int UN = 4;
        float v[UN][4], t[UN];
        int row[UN], c[UN];
        auto fetch = [&](int u0) {
#pragma unroll
            for (int k = 0; k < UN; k++) {
                const int u = min(u0 + k * kThreads, U - 1);   // (past the end: the last one again, the same bytes)
                row[k] = (int)fastdiv((uint32_t)u, a.dRP);
                c[k] = (u - row[k] * quads) * 4;
                const uint32_t o = ((uint32_t)row[k] * (uint32_t)a.C + (uint32_t)c[k]) * 4u;   // (lanes past the row's end are masked below)
                if (a.vec4) {
                    const v4u q = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)o, 0, 0);
                    v[k][0] = __uint_as_float(q.x), v[k][1] = __uint_as_float(q.y), v[k][2] = __uint_as_float(q.z), v[k][3] = __uint_as_float(q.w);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) v[k][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(o + 4u * i), 0, 0));
                }
                t[k] = a.thr[n + row[k]];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        int u0 = wave * 64;
        do {   // (a wavefront with nothing of its own repeats the last piece)
            fetch(u0 + lane);
            if (u0 == wave * 64) meanwhile();
#pragma unroll
            for (int k = 0; k < UN; k++) {
                uint32_t b = ABIN ? push4<true>(0u, v[k], t[k]) : t[k] >= 0.0f ? push4<false>(0u, v[k], t[k]) : push4_any(0u, v[k], t[k]);
                const uint32_t m = real_mask4(a.C - c[k]);
                b = (b & m) | (ABIN ? 0x33u & ~m : 0u);
                const int pl = c[k] >> 6, cc = c[k] & 63;   // dword 2 h + a, byte q of the record
                reinterpret_cast<unsigned char*>(lds)[(pl * 32 + row[k]) * 16 + (2 * ((cc >> 2) & 1) + (cc >> 5)) * 4 + ((cc >> 3) & 3)] = (unsigned char)b;
            }
            u0 += UN * kThreads;
        } while (u0 < U);
    } else {
        n = (int)fastdiv(tile, a.dTI);
        const uint32_t r = tile - (uint32_t)n * a.dTI.d;
        const int tyi = (int)fastdiv(r, a.dTX), txi = (int)(r - (uint32_t)tyi * a.dTX.d);
        const int oh0 = tyi * (32 >> a.lgTW), ow0 = txi << a.lgTW;
        oh = oh0 + (lr >> a.lgTW), ow = ow0 + (lr & ((1 << a.lgTW) - 1));
        const int ih0 = oh0 * a.H_stride - a.H_pad, iw0 = ow0 * a.W_stride - a.W_pad;
        const float t = a.thr[n];
        const uint32_t HW = (uint32_t)(a.H * a.W), plane = HW * 4u;
        // offsets past the image's last channel return zeros
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x + (size_t)n * a.C * HW), 0, (int)((uint32_t)a.C * plane), 0x00020000);
        const int U = a.RP * 4 * a.CP;
        struct Unit {
            float v[16];
            uint32_t at;   // dword of its record
            int c0;
            bool inside;
        };
        auto fetch = [&](Unit& f, int u) {
            const uint32_t q = fastdiv((uint32_t)u, a.dRP), px = (uint32_t)u - q * (uint32_t)a.RP;
            const uint32_t ry = fastdiv(px, a.dRW), rx = px - ry * (uint32_t)a.RW;
            const int ih = ih0 + (int)ry * a.rstep, iw = iw0 + (int)rx * a.cstep;
            f.inside = (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
            const uint32_t pl = q >> 2, j = q & 3u;   // dword j of the record: channels c0 + 8 q + i
            f.c0 = (int)(pl * 64u + 32u * (j & 1u) + 4u * (j >> 1));
            f.at = (pl * (uint32_t)a.RP + px) * 4u + j;
            const uint32_t o = f.inside ? (uint32_t)f.c0 * plane + (uint32_t)(ih * a.W + iw) * 4u : kDirectNowhere;
#pragma unroll
            for (int e = 0; e < 16; e++)
                f.v[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(o + (uint32_t)(8 * (e >> 2) + (e & 3)) * plane), 0, 0));
            __builtin_amdgcn_sched_barrier(0);
        };
        Unit f;
        int u = tid;
        if (u < U) fetch(f, u);
        meanwhile();
        while (u < U) {
            Unit next = f;
            if (u + kThreads < U) fetch(next, u + kThreads);
            uint32_t dw = 0u;
            if (ABIN || t >= 0.0f) {
#pragma unroll
                for (int q = 3; q >= 0; q--) dw = push4<ABIN>(dw, f.v + 4 * q, t);
            } else {
#pragma unroll 1
                for (int q = 3; q >= 0; q--) {
                    float z[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) z[i] = q == 0 ? f.v[i] : q == 1 ? f.v[4 + i] : q == 2 ? f.v[8 + i] : f.v[12 + i];
                    dw = push4_any(dw, z, t);
                }
            }
            if (a.C & 63) {
                uint32_t m = 0u;
#pragma unroll
                for (int q = 3; q >= 0; q--) m = m << 8 | real_mask4(a.C - f.c0 - 8 * q);
                dw = (dw & m) | (ABIN ? kP2Plus & ~m : 0u);
            }
            words[f.at] = f.inside ? dw : (ABIN ? kP2Plus : 0u);
            f = next;
            u += kThreads;
        }
    }
    __syncthreads();

    const uint32_t base = FC ? (uint32_t)lr * 16u : (uint32_t)(min(lr >> a.lgTW, a.OHt - 1) * a.lrow * a.RW + min(lr & ((1 << a.lgTW) - 1), a.OWt - 1) * a.lcol) * 16u;
    v16f acc;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.0f;
    if (!idle) {
        // G pairs at a time, all their records asked for first; pairs past the share read the record of zeros
        for (int p = p0; p < p1; p += G) {
            uint32_t at[G];
            v4i x[G], wn[G];
#pragma unroll
            for (int d = 0; d < G; d++) at[d] = tab[2 * min(p + d, a.NP - 1) + h], wn[d] = w[d];
            weights(wn, p + G);
#pragma unroll
            for (int d = 0; d < G; d++) {
                const bool zero = at[d] == ~0u || p + d >= p1;
                x[d] = *reinterpret_cast<const v4i*>(reinterpret_cast<const char*>(lds) + (zero ? rec_bytes : base + at[d]));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < G; d++) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const uint32_t x0 = (uint32_t)x[d][2 * k], x1 = (uint32_t)x[d][2 * k + 1], w0 = (uint32_t)w[d][2 * k], w1 = (uint32_t)w[d][2 * k + 1];
                    const v8i xv = {(int)(x0 & kP2Mask), (int)((x0 << 1) & kP2Mask), (int)(x1 & kP2Mask), (int)((x1 << 1) & kP2Mask), 0, 0, 0, 0};
                    const v8i wv = {(int)(w0 & kP2Mask), (int)((w0 << 1) & kP2Mask), (int)(w1 & kP2Mask), (int)((w1 << 1) & kP2Mask), 0, 0, 0, 0};
                    // cbsz = blgp = 4: both operands E2M1, unscaled; result rows run along the first one
                    acc = FC ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(xv, wv, acc, 4, 4, 0, 0, 0, 0)
                             : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, xv, acc, 4, 4, 0, 0, 0, 0);
                }
            }
#pragma unroll
            for (int d = 0; d < G; d++) w[d] = wn[d];
        }
    }

    // The shares of a block meet in LDS, where the records are no longer needed: [wave][quad of elements][lane].  Element
    // e of a block is its row 8 (e / 4) + 4 h + e % 4.
    __syncthreads();
    float4* const red = reinterpret_cast<float4*>(lds);
#pragma unroll
    for (int q = 0; q < 4; q++) red[(wave * 4 + q) * 64 + lane] = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    __syncthreads();
    const int kn0 = kb * 32;
    float* y;
    size_t ystep;
    int last;          // rows of the block from this one on do not exist
    bool live = !idle;
    if constexpr (FC) {
        y = a.Y + (size_t)n * a.KN + kn0 + lr;
        ystep = (size_t)a.KN;
        last = a.N - n;
        live = live && kn0 + lr < a.KN;
    } else {
        const size_t OHW = (size_t)a.OH * a.OW;
        y = a.Y + ((size_t)n * a.KN + kn0) * OHW + (uint32_t)(oh * a.OW + ow);
        ystep = OHW;
        last = a.KN - kn0;
        live = live && oh < a.OH && ow < a.OW;
    }
    if (live) {
        const int S = 1 << a.lgS;
        const float4* const src = red + (wave - ks) * 256 + lane;
        for (int q = ks; q < 4; q += S) {
            float4 s = src[q * 64];
            for (int v = 1; v < S; v++) {
                const float4 o = src[v * 256 + q * 64];
                s.x += o.x, s.y += o.y, s.z += o.z, s.w += o.w;
            }
            const int row = 8 * q + 4 * h;
            float* const d = y + (size_t)row * ystep;
            const float r[4] = {s.x - a.bias, s.y - a.bias, s.z - a.bias, s.w - a.bias};
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (row + i < last) d[(size_t)i * ystep] = r[i] < a.lim ? r[i] * a.alpha : r[i];
        }
    }
}

// the kernel's arguments for a plan, but for the pointers and the type's constants
DirectArgs direct_args(const DirectPlan& p, const ConvGeom& cg, int C, int N, int KN) {
    DirectArgs a = {};
    a.N = N, a.C = C, a.CP = cg.CP, a.H = p.H, a.W = p.W, a.KN = KN, a.OH = p.OH, a.OW = p.OW;
    a.K = cg.K, a.NP = (cg.K + 1) / 2, a.KP = round4(cg.K) / 2;
    a.H_stride = cg.H_stride, a.W_stride = cg.W_stride, a.H_pad = cg.H_pad, a.W_pad = cg.W_pad, a.KW = cg.KW;
    a.dCP = cg.dCP, a.dKW = cg.dKW;
    a.RW = p.RW, a.RP = p.RP;
    a.rstep = p.rstep, a.cstep = p.cstep, a.lrow = p.lrow, a.lcol = p.lcol;
    a.lgTW = p.lgTW, a.OWt = p.OWt, a.OHt = p.OHt, a.lgS = p.lgS;
    a.dRP = make_fastdiv(p.fc ? (uint32_t)cg.CP * 16u : (uint32_t)p.RP);
    a.dRW = make_fastdiv((uint32_t)p.RW), a.dTX = make_fastdiv(p.tiles_x), a.dTI = make_fastdiv(p.image_tiles);
    a.xo = make_xcd_order((uint64_t)p.tiles, (uint32_t)p.groups, false);
    return a;
}

}  // namespace

bool launch_direct_f4(int type, const float* d_x, const float* d_thr, const void* d_wf, const ConvGeom& cg, int C, int N, int KN,
                      int K_unpack, float alpha, float* d_y, hipStream_t st, hipError_t* err) {
    // tuning aid, and off where another one forces a form of the layer kernels
    static const bool off = getenv("FTNN_NO_DIRECT_LAYERS") || getenv("FTNN_CONV_SPLIT") || getenv("FTNN_CONV_NO_BUFFER_LOADS") ||
                            getenv("FTNN_CONV_SMALL_BELOW") || getenv("FTNN_CONV_TILES_FROM");
    DirectPlan p;
    if (off || !direct_plan(type, cg, C, N, KN, &p)) return false;
    // One launch reads the input while it stores the result; a result that lies over its input (or the thresholds) needs the input
    // quantised before the first store.
    const int64_t y_bytes = 4LL * N * KN * cg.OH * cg.OW;
    if (ranges_meet(d_y, y_bytes, d_x, 4LL * N * C * cg.H * cg.W) || ranges_meet(d_y, y_bytes, d_thr, 4LL * N)) return false;
    DirectArgs a = direct_args(p, cg, C, N, KN);
    a.vec4 = C % 4 == 0 && reinterpret_cast<uintptr_t>(d_x) % 16 == 0;
    a.x = d_x, a.thr = d_thr, a.Wf = static_cast<const uint4*>(d_wf), a.Y = d_y;
    // BNN: the channel lanes past C are +1 in both operands; padding words are skipped
    a.bias = type == kBNN ? (float)(64 * cg.K - K_unpack) : 0.0f;
    // results are integers below 2^24, so the reference's two forms of PReLU are one compare, against 0.5 or 0
    a.lim = type == kTNN ? 0.5f : 0.0f;
    a.alpha = alpha;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles * p.groups)), dim3(kThreads), (size_t)p.lds_bytes, st, a);
        *err = hipGetLastError();
        return true;
    };
    if (type == kBTN || type == kBNN) return p.fc ? go(k_direct_f4<true, true>) : go(k_direct_f4<true, false>);
    return p.fc ? go(k_direct_f4<false, true>) : go(k_direct_f4<false, false>);
}

}  // namespace ftnn
