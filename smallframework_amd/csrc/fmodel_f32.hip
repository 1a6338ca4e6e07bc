// Whole-model forward pass of a small float32 CNN in ONE launch for gfx950 (small_hip_fmodel_*).
//
// A keyword-spotting DS-CNN (49x10x1 input, 25x5x64 activations = 32 KB, 87 KB of weights) run layer by layer is
// eleven dependent launches that each sit at the launch-latency floor.  Here one workgroup of 1024 threads owns one
// image from input to logits: the activation tensors stay in the compute unit's LDS, each layer's weights are
// brought into LDS one layer ahead (double buffered, global memory to LDS directly), only the image and the model's output touch global memory and
// the layers are separated by workgroup barriers instead of kernel boundaries.  A depthwise-separable chain (what a DS-CNN is) has a
// kernel of its own further down, whose images may be cut into bands for several compute units; any other model runs on the general one.
//
// Layers (the functions of include/small/interface_abstract.hpp on float buffers, fused as Conv2DLayer /
// DepthwiseConv2DLayer::compute_output issue them: bias, convolution, ReLU or LeakyReLU):
//   convolution, input channels % 16 == 0   v_mfma_f32_16x16x4_f32, rows = 16 output channels, columns = 16 pixels
//   convolution, 1..3 input channels        the same instruction on a gathered patch (model input only)
//   depthwise convolution                   vector ALU, a lane = 4 channels of one output pixel
//   depthwise 3x3 -> 1x1 convolution        one layer: a lane's depthwise results ARE its MFMA operand of the 1x1
//                                           convolution (the same pixel, the same four channels), so the depthwise
//                                           tensor is never stored and its arithmetic issues between the MFMAs
//   whole-image average / max pooling       a wave per channel quad: lanes fold pixels, then xor-shuffles (deterministic)
// A fully connected layer is the 1x1 convolution on the 1x1 image pooling leaves.
//
// LDS layout of an activation tensor: [C/16][P][16] floats, the four channel quads of pixel p stored in the order
// q ^ ((p >> 1) & 3).  An MFMA operand read is one 16-byte read per lane at a 64-byte pixel pitch; with that swizzle
// eight neighbouring pixels cover all 32 banks, without it they would share two.  One such read feeds four MFMAs:
// lane (pixel, kq) holds channels 4kq .. 4kq+3, MFMA j of the step contracts channels {j, 4+j, 8+j, 12+j}, and the
// filter is re-ordered once, when the model is created, so that the matching four weights are one 16-byte read too:
//   Wt[co block][tap][ci block][kq][co % 16][j] = F[co][ci = 16 * block + 4 kq + j][tap].
// Numerics: float32 MFMA accumulation, bias added and activation applied on the accumulators.
#include "common.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

using namespace shp;

namespace
{

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int NT = 1024;                 // 16 waves, 4 per SIMD; one workgroup per compute unit (LDS)
constexpr int NW = NT / WAVE;
constexpr int MAX_LAYERS = 32;
constexpr int MAX_TENSORS = 8;
constexpr int NPRE = 3;                  // 16-byte pieces of the next layer's weights a thread carries: 48 KB per layer
constexpr int LDS_LIMIT = 160 * 1024;

enum { K_STEM = 0, K_CONV = 1, K_DW = 2, K_POOL_AVG = 3, K_POOL_MAX = 4, K_DWPW = 5 };

struct FMLayer
{
    int kind;
    int src_off, dst_off;                // float offsets in LDS; dst_off < 0: the model output in global memory
    int Ci, Co, H, W, Ho, Wo, kh, kw, stride, pt, pl;
    int K, chunks;                       // first layer: reduction length kh*kw*Ci and its chunks of 16 (four MFMA steps)
    int blob_off, blob16;                // the layer's weights in the blob (float offset) and their size in 16-byte pieces
    int next_blob_off, next_blob16;      // the same of the layer after this one (0 pieces after the last): read with this record
    int bias_off, ktab_off;              // float offsets inside the layer's weights
    float nscale;                        // what a negative result is multiplied by: 1 none, 0 ReLU, slope LeakyReLU
    float r_wo, r_cob, r_p, norm;        // 1 / Wo, 1 / (Co / 16), 1 / (Ho * Wo), pooling scale
    // K_DWPW: a 3x3 depthwise convolution whose result feeds the 1x1 convolution that follows without leaving registers
    int Co2, w2_off, bias2_off;          // the 1x1 convolution: output channels, weights and bias inside the layer's weights
    float nscale2, r_cob2;               // ... and 1 / (Co2 / 16)
};

struct FMHeader
{
    int n_layers;
    int in_C, in_H, in_W, in_off;        // the model input and the LDS float offset it is staged at
    int w_lds, w_floats;                 // weights: two buffers of w_floats floats at float offset w_lds
    int pool_off;                        // 4096 + 512 floats of pooling partials
    int zero_off;                        // 16 bytes of zeros: what a tap outside the image reads
    int in_elems, out_elems;             // floats per image in global memory
    int lds_bytes;
    FMLayer layer[MAX_LAYERS];
};
typedef const __attribute__((address_space(4))) FMHeader *HeaderPtr;

__device__ __forceinline__ FMLayer load_layer(HeaderPtr hdr, int li)
{
    FMLayer L;
    __builtin_memcpy(&L, &hdr->layer[li], sizeof(FMLayer));
    return L;
}

// float offset of channel quad q of pixel p in a [C/16][P][16] tensor
__device__ __forceinline__ int apos(int cb, int P, int p, int q) { return ((cb * P + p) * 4 + (q ^ ((p >> 1) & 3))) * 4; }

__device__ __forceinline__ float act_bf(float v, float neg_scale)
{
    const float n = fmaf(v, neg_scale, 0.f);      // "+ 0": the -0 of x * 0 becomes the +0 ReLU gives
    return v > 0.f ? v : n;
}

// Values that another workgroup of the same launch reads: written through to where every XCD sees them and read from there,
// eight bytes at a time (a fence of the whole device instead writes back and drops an L2 per wave: 3 us a band).
__device__ __forceinline__ void store_shared(float *g, float4 v)
{
    unsigned long long *d = reinterpret_cast<unsigned long long *>(g);
    const uint4 u = __builtin_bit_cast(uint4, v);
    __hip_atomic_store(d, u.x | (unsigned long long)u.y << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(d + 1, u.z | (unsigned long long)u.w << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float4 load_shared(const float *g)
{
    const unsigned long long *d = reinterpret_cast<const unsigned long long *>(g);
    const unsigned long long a = __hip_atomic_load(d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long b = __hip_atomic_load(d + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(float4, make_uint4((unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32)));
}
// The compiler moves no memory access across (a builtin wait alone does not keep it from that).
__device__ __forceinline__ void keep_order() { asm volatile("" ::: "memory"); }

// ---- model creation: weights into operand order ---------------------------------------------------------------
// kind K_CONV: packed filter [Co/16][Ci/16][taps][16 ci][16 co] -> Wt[Co/16][taps][Ci/16][kq][co16][j]
// kind K_STEM: packed filter [Co/16][K][16 co] -> Wt[Co/16][chunk][kq][co16][j] = F[k = 16 chunk + 4 j + kq], zero from K on
// kind K_DW:   packed filter [C/16][taps][16] unchanged
// followed by the bias (zeros without one)
__global__ __launch_bounds__(256) void fm_prep_kernel(int kind, const float *__restrict__ f, const float *__restrict__ bias,
                                                      float *__restrict__ dst, int Co, int Ci, int taps, int K, int chunks,
                                                      int w_floats)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < w_floats)
    {
        float v = 0.f;
        if (kind == K_CONV)
        {
            const int CiB = Ci / CB;
            const int j = i & 3, co16 = (i >> 2) & 15, kq = (i >> 6) & 3;
            int r = i >> 8;
            const int cib = r % CiB; r /= CiB;
            const int tap = r % taps, cob = r / taps;
            v = f[((((size_t)cob * CiB + cib) * taps + tap) * CB + 4 * kq + j) * CB + co16];
        }
        else if (kind == K_STEM)
        {
            const int j = i & 3, co16 = (i >> 2) & 15, kq = (i >> 6) & 3, r = i >> 8;
            const int chunk = r % chunks, cob = r / chunks, k = 16 * chunk + 4 * j + kq;
            if (k < K) v = f[((size_t)cob * K + k) * CB + co16];
        }
        else
            v = f[i];
        dst[i] = v;
    }
    if (i < Co) dst[w_floats + i] = bias ? bias[i] : 0.f;
}

// ---- device: layers --------------------------------------------------------------------------------------------
// Convolution on MFMA; TP pixel tiles of one channel block per wave step share the filter operand.  The K-steps
// (tap, input channel block) are taken four at a time: all twelve (TP = 2) operand reads of a chunk are issued before
// its first MFMA, so a chunk pays the LDS latency once; a tap outside the image reads the block of zeros.
template <int TP>
__device__ __forceinline__ void conv_layer(const FMLayer &L, float *lds, const float *wl, const float *zero, float *gout,
                                           int wave, int lane)
{
    const int col = lane & 15, kq = lane >> 4;
    const int CoB = L.Co / CB, CiB = L.Ci / CB, S = L.kh * L.kw * CiB;
    const int Pin = L.H * L.W, P = L.Ho * L.Wo;
    const int n_pt = (P + 15) >> 4, n_grp = (n_pt + TP - 1) / TP, n_work = n_grp * CoB;
    const float *src = lds + L.src_off;
    for (int work = wave; work < n_work; work += NW)
    {
        const int pg = (int)(((float)work + 0.5f) * L.r_cob);
        const int cob = work - pg * CoB;
        int ih0[TP], iw0[TP], p[TP];
        bool pv[TP];
#pragma unroll
        for (int t = 0; t < TP; ++t)
        {
            p[t] = (pg * TP + t) * 16 + col;
            pv[t] = p[t] < P;
            const int pc = pv[t] ? p[t] : 0;
            const int oh = (int)(((float)pc + 0.5f) * L.r_wo), ow = pc - oh * L.Wo;
            ih0[t] = oh * L.stride - L.pt;
            iw0[t] = ow * L.stride - L.pl;
        }
        floatx4 acc[TP];
#pragma unroll
        for (int t = 0; t < TP; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
        const float *wrow = wl + ((cob * S * 4 + kq) * 16 + col) * 4;
        int a = 0, b = 0, cib = 0;                       // the next step to load (uniform)
        for (int s0 = 0; s0 < S; s0 += 4)
        {
            float4 A[4], B[TP][4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const bool live = s0 + u < S;            // uniform
                A[u] = *reinterpret_cast<const float4 *>(live ? wrow + (s0 + u) * 256 : zero);
#pragma unroll
                for (int t = 0; t < TP; ++t)
                {
                    const int ih = ih0[t] + a, iw = iw0[t] + b;
                    const bool ok = live && pv[t] && (unsigned)ih < (unsigned)L.H && (unsigned)iw < (unsigned)L.W;
                    B[t][u] = *reinterpret_cast<const float4 *>(ok ? src + apos(cib, Pin, ih * L.W + iw, kq) : zero);
                }
                // channel block fastest, then the window column, then the row
                const bool w1 = cib + 1 == CiB;
                cib = w1 ? 0 : cib + 1;
                const bool w2 = w1 && b + 1 == L.kw;
                b = w2 ? 0 : b + (w1 ? 1 : 0);
                a += w2 ? 1 : 0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const float Av[4] = {A[u].x, A[u].y, A[u].z, A[u].w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < TP; ++t)
                    {
                        const float Bv[4] = {B[t][u].x, B[t][u].y, B[t][u].z, B[t][u].w};
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Av[j], Bv[j], acc[t], 0, 0, 0);
                    }
            }
        }
        const float4 bias = *reinterpret_cast<const float4 *>(wl + L.bias_off + cob * CB + 4 * kq);
#pragma unroll
        for (int t = 0; t < TP; ++t)
        {
            if (!pv[t]) continue;
            const float4 v = make_float4(act_bf(acc[t][0] + bias.x, L.nscale), act_bf(acc[t][1] + bias.y, L.nscale),
                                         act_bf(acc[t][2] + bias.z, L.nscale), act_bf(acc[t][3] + bias.w, L.nscale));
            if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + apos(cob, P, p[t], kq)) = v;
            else *reinterpret_cast<float4 *>(gout + ((size_t)cob * P + p[t]) * CB + 4 * kq) = v;
        }
    }
}

// first layer, 1..3 input channels: the image lies in LDS as it does in memory, [H][W][Ci]; reduction element
// k = (a * kw + b) * Ci + ci.  In MFMA step 4 * chunk + j lane (pixel, kq) supplies element k = 16 chunk + 4 j + kq of
// its pixel's patch; where that element lies comes from a table written with the weights (one 16-byte read per
// chunk), and the gathered operand serves TC output-channel blocks.
template <int TC>
__device__ __forceinline__ void stem_layer(const FMLayer &L, float *lds, const float *wl, const float *zero, float *gout,
                                           int wave, int lane)
{
    const int col = lane & 15, kq = lane >> 4;
    const int CoB = L.Co / CB, P = L.Ho * L.Wo;
    const int n_pt = (P + 15) >> 4, n_cg = CoB / TC, n_work = n_pt * n_cg;
    const float r_ncg = L.r_cob * (float)TC;                 // 1 / n_cg
    const float *src = lds + L.src_off;
    const int4 *ktab = reinterpret_cast<const int4 *>(wl + L.ktab_off);
    for (int work = wave; work < n_work; work += NW)
    {
        const int pt = (int)(((float)work + 0.5f) * r_ncg), cg = work - pt * n_cg;
        const int p = pt * 16 + col;
        const bool pv = p < P;
        const int pc = pv ? p : 0;
        const int oh = (int)(((float)pc + 0.5f) * L.r_wo), ow = pc - oh * L.Wo;
        const int ih0 = oh * L.stride - L.pt, iw0 = ow * L.stride - L.pl;
        floatx4 acc[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        // the operands of chunk ch: where its four patch elements lie (table), the elements, the filter quads
        auto gather = [&](int ch, float4 (&A)[TC], float (&bv)[4]) {
            const int4 e4 = ktab[ch * 4 + kq];               // a | b << 8 | ci << 16 per step; -1 past the end
            const int ev[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
            for (int c = 0; c < TC; ++c)
                A[c] = *reinterpret_cast<const float4 *>(wl + ((((cg * TC + c) * L.chunks + ch) * 4 + kq) * 16 + col) * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int e = ev[j];
                const int ih = ih0 + (e & 255), iw = iw0 + ((e >> 8) & 255);
                const bool ok = pv && e >= 0 && (unsigned)ih < (unsigned)L.H && (unsigned)iw < (unsigned)L.W;
                bv[j] = *(ok ? src + (ih * L.W + iw) * L.Ci + (e >> 16) : zero);
            }
        };
        auto multiply = [&](const float4 (&A)[TC], const float (&bv)[4]) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < TC; ++c)
                {
                    const float Av[4] = {A[c].x, A[c].y, A[c].z, A[c].w};
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(Av[j], bv[j], acc[c], 0, 0, 0);
                }
        };
        // chunk ch + 1 is gathered between the MFMAs of chunk ch (a wave issues in order: see dwpw_layer)
        float4 Ac[TC], An[TC];
        float bc[4], bn[4];
        gather(0, Ac, bc);
        for (int ch = 0; ch + 1 < L.chunks; ++ch)
        {
            gather(ch + 1, An, bn);
            multiply(Ac, bc);
#pragma unroll
            for (int c = 0; c < TC; ++c) Ac[c] = An[c];
#pragma unroll
            for (int j = 0; j < 4; ++j) bc[j] = bn[j];
#pragma unroll
            for (int g = 0; g < 4 * TC; ++g)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            }
        }
        multiply(Ac, bc);
        if (!pv) continue;
#pragma unroll
        for (int c = 0; c < TC; ++c)
        {
            const int cob = cg * TC + c;
            const float4 bias = *reinterpret_cast<const float4 *>(wl + L.bias_off + cob * CB + 4 * kq);
            const float4 v = make_float4(act_bf(acc[c][0] + bias.x, L.nscale), act_bf(acc[c][1] + bias.y, L.nscale),
                                         act_bf(acc[c][2] + bias.z, L.nscale), act_bf(acc[c][3] + bias.w, L.nscale));
            if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + apos(cob, P, p, kq)) = v;
            else *reinterpret_cast<float4 *>(gout + ((size_t)cob * P + p) * CB + 4 * kq) = v;
        }
    }
}

// Depthwise convolution with a compile-time window: a lane owns 4 channels of one output pixel and walks over a
// share of the channel blocks.  The window's nine positions (offsets into the block, the zeros for taps outside the
// image) are worked out once per lane; per channel block a tap costs two 16-byte LDS reads and four multiply-adds.
template <int KH, int KW>
__device__ __forceinline__ void dw_layer_win(const FMLayer &L, float *lds, const float *wl, const float *zero, float *gout, int tid)
{
    constexpr int T = KH * KW;
    const int CiB = L.Ci / CB;
    const int Pin = L.H * L.W, P = L.Ho * L.Wo, n_lane = P * 4;
    int G = NT / n_lane;                                   // lane groups along the channel blocks
    G = G < 1 ? 1 : (G > CiB ? CiB : G);
    const int per = (CiB + G - 1) / G;                     // channel blocks per group
    const float *src = lds + L.src_off;
    for (int i = tid; i < n_lane * G; i += NT)
    {
        const int g = (int)(((float)i + 0.5f) * L.r_p * 0.25f);      // i / n_lane
        const int r = i - g * n_lane;
        const int q = r & 3, p = r >> 2;
        const int oh = (int)(((float)p + 0.5f) * L.r_wo), ow = p - oh * L.Wo;
        const int ih0 = oh * L.stride - L.pt, iw0 = ow * L.stride - L.pl;
        const int cb0 = g * per, cb1 = cb0 + per < CiB ? cb0 + per : CiB;
        const float *xp[T];
        int xstep[T];
#pragma unroll
        for (int a = 0; a < KH; ++a)
#pragma unroll
            for (int b = 0; b < KW; ++b)
            {
                const int ih = ih0 + a, iw = iw0 + b;
                const bool ok = (unsigned)ih < (unsigned)L.H && (unsigned)iw < (unsigned)L.W;
                xp[a * KW + b] = ok ? src + apos(cb0, Pin, ih * L.W + iw, q) : zero;
                xstep[a * KW + b] = ok ? Pin * CB : 0;
            }
        const float *w = wl + cb0 * T * CB + 4 * q;
        const float *bp = wl + L.bias_off + cb0 * CB + 4 * q;
        int dpos = apos(cb0, P, p, q);
        for (int cb = cb0; cb < cb1; ++cb)
        {
            float4 x[T], k[T];
#pragma unroll
            for (int t = 0; t < T; ++t)
            {
                x[t] = *reinterpret_cast<const float4 *>(xp[t]);
                k[t] = *reinterpret_cast<const float4 *>(w + t * CB);
                xp[t] += xstep[t];
            }
            float4 acc = *reinterpret_cast<const float4 *>(bp);
#pragma unroll
            for (int t = 0; t < T; ++t)
            {
                acc.x = fmaf(x[t].x, k[t].x, acc.x); acc.y = fmaf(x[t].y, k[t].y, acc.y);
                acc.z = fmaf(x[t].z, k[t].z, acc.z); acc.w = fmaf(x[t].w, k[t].w, acc.w);
            }
            acc.x = act_bf(acc.x, L.nscale); acc.y = act_bf(acc.y, L.nscale);
            acc.z = act_bf(acc.z, L.nscale); acc.w = act_bf(acc.w, L.nscale);
            if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + dpos) = acc;
            else *reinterpret_cast<float4 *>(gout + ((size_t)cb * P + p) * CB + 4 * q) = acc;
            w += T * CB; bp += CB; dpos += P * CB;
        }
    }
}

// Depthwise 3x3 + activation feeding a 1x1 convolution + activation.  In the MFMA operand layout lane (pixel, kq) supplies
// channels 4kq .. 4kq+3 of its pixel for each input-channel block: exactly one depthwise result quad.  So the wave
// computes the block's depthwise quad on the vector ALU (nine 16-byte reads of the input, nine of the taps, 36
// multiply-adds) while the MFMAs of the previous block run, and hands it to the MFMAs of all TC output-channel blocks.
// The depthwise tensor never exists in memory, and a layer boundary (barrier, LDS round trip) disappears.
template <int TC>
__device__ __forceinline__ void dwpw_layer(const FMLayer &L, float *lds, const float *wl, const float *zero, float *gout,
                                           int wave, int lane)
{
    constexpr int T = 9;
    const int col = lane & 15, kq = lane >> 4;
    const int CiB = L.Ci / CB, CoB = L.Co2 / CB;
    const int Pin = L.H * L.W, P = L.Ho * L.Wo;
    const int n_pt = (P + 15) >> 4, n_cg = CoB / TC, n_work = n_pt * n_cg;
    const float r_ncg = L.r_cob2 * (float)TC;                // 1 / n_cg
    const float *src = lds + L.src_off;
    for (int work = wave; work < n_work; work += NW)
    {
        const int pt = (int)(((float)work + 0.5f) * r_ncg), cg = work - pt * n_cg;
        const int p = pt * 16 + col;
        const bool pv = p < P;
        const int pc = pv ? p : 0;
        const int oh = (int)(((float)pc + 0.5f) * L.r_wo), ow = pc - oh * L.Wo;
        const int ih0 = oh * L.stride - L.pt, iw0 = ow * L.stride - L.pl;
        const float *xp[T];
        int xstep[T];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b)
            {
                const int ih = ih0 + a, iw = iw0 + b;
                const bool ok = pv && (unsigned)ih < (unsigned)L.H && (unsigned)iw < (unsigned)L.W;
                xp[a * 3 + b] = ok ? src + apos(0, Pin, ih * L.W + iw, kq) : zero;
                xstep[a * 3 + b] = ok ? Pin * CB : 0;
            }
        const float *wk = wl + 4 * kq;                       // depthwise taps [ci block][tap][16]
        const float *bk = wl + L.bias_off + 4 * kq;
        // the depthwise quad of the next input-channel block (advances the pointers)
        auto depthwise = [&]() -> float4 {
            float4 acc = *reinterpret_cast<const float4 *>(bk);
#pragma unroll
            for (int t = 0; t < T; ++t)
            {
                const float4 x = *reinterpret_cast<const float4 *>(xp[t]);
                const float4 k = *reinterpret_cast<const float4 *>(wk + t * CB);
                acc.x = fmaf(x.x, k.x, acc.x); acc.y = fmaf(x.y, k.y, acc.y);
                acc.z = fmaf(x.z, k.z, acc.z); acc.w = fmaf(x.w, k.w, acc.w);
                xp[t] += xstep[t];
            }
            wk += T * CB; bk += CB;
            return make_float4(act_bf(acc.x, L.nscale), act_bf(acc.y, L.nscale), act_bf(acc.z, L.nscale), act_bf(acc.w, L.nscale));
        };
        floatx4 acc[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        const float *arow = wl + L.w2_off + ((cg * TC * CiB * 4 + kq) * 16 + col) * 4;      // + (c * CiB + cib) * 256
        auto filter = [&](int cib, float4 (&A)[TC]) {
#pragma unroll
            for (int c = 0; c < TC; ++c) A[c] = *reinterpret_cast<const float4 *>(arow + (c * CiB + cib) * 256);
        };
        auto multiply = [&](const float4 (&A)[TC], const float4 Bq) {
            const float Bv[4] = {Bq.x, Bq.y, Bq.z, Bq.w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < TC; ++c)
                {
                    const float Av[4] = {A[c].x, A[c].y, A[c].z, A[c].w};
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(Av[j], Bv[j], acc[c], 0, 0, 0);
                }
        };
        // Software pipeline over the input-channel blocks: while the MFMAs of block cib run, the wave reads the filter
        // of block cib + 1 and does that block's depthwise arithmetic.  A wave issues in order, so the overlap only
        // happens if those instructions sit BETWEEN the MFMAs: the scheduling groups below ask for one MFMA, then a
        // couple of LDS reads and a handful of vector instructions, sixteen times (an MFMA occupies the matrix pipe for
        // 32 cycles = 8 issue slots).
        float4 Ac[TC], An[TC];
        filter(0, Ac);
        float4 Bc = depthwise();
        for (int cib = 0; cib + 1 < CiB; ++cib)
        {
            filter(cib + 1, An);
            multiply(Ac, Bc);
            Bc = depthwise();
#pragma unroll
            for (int c = 0; c < TC; ++c) Ac[c] = An[c];
#pragma unroll
            for (int g = 0; g < 4 * TC; ++g)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);      // LDS reads
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);      // vector ALU
            }
        }
        multiply(Ac, Bc);
        if (!pv) continue;
#pragma unroll
        for (int c = 0; c < TC; ++c)
        {
            const int cob = cg * TC + c;
            const float4 bias = *reinterpret_cast<const float4 *>(wl + L.bias2_off + cob * CB + 4 * kq);
            const float4 v = make_float4(act_bf(acc[c][0] + bias.x, L.nscale2), act_bf(acc[c][1] + bias.y, L.nscale2),
                                         act_bf(acc[c][2] + bias.z, L.nscale2), act_bf(acc[c][3] + bias.w, L.nscale2));
            if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + apos(cob, P, p, kq)) = v;
            else *reinterpret_cast<float4 *>(gout + ((size_t)cob * P + p) * CB + 4 * kq) = v;
        }
    }
}

// depthwise convolution, any window: a lane = one output pixel x 4 channels of one block
__device__ __forceinline__ void dw_layer_any(const FMLayer &L, float *lds, const float *wl, float *gout, int tid)
{
    const int kh = L.kh, kw = L.kw;
    const int Pin = L.H * L.W, P = L.Ho * L.Wo, n = (L.Ci / CB) * P * 4;
    const float *src = lds + L.src_off;
    for (int i = tid; i < n; i += NT)
    {
        const int q = i & 3, r = i >> 2;
        const int cb = (int)(((float)r + 0.5f) * L.r_p), p = r - cb * P;
        const int oh = (int)(((float)p + 0.5f) * L.r_wo), ow = p - oh * L.Wo;
        const int ih0 = oh * L.stride - L.pt, iw0 = ow * L.stride - L.pl;
        const float *w = wl + cb * kh * kw * CB + 4 * q;
        float4 acc = *reinterpret_cast<const float4 *>(wl + L.bias_off + cb * CB + 4 * q);
        for (int a = 0; a < kh; ++a)
            for (int b = 0; b < kw; ++b)
            {
                const int ih = ih0 + a, iw = iw0 + b;
                const bool ok = (unsigned)ih < (unsigned)L.H && (unsigned)iw < (unsigned)L.W;
                float4 x = *reinterpret_cast<const float4 *>(src + apos(cb, Pin, ok ? ih * L.W + iw : 0, q));
                if (!ok) x = make_float4(0.f, 0.f, 0.f, 0.f);
                const float4 k = *reinterpret_cast<const float4 *>(w + (a * kw + b) * CB);
                acc.x = fmaf(x.x, k.x, acc.x); acc.y = fmaf(x.y, k.y, acc.y);
                acc.z = fmaf(x.z, k.z, acc.z); acc.w = fmaf(x.w, k.w, acc.w);
            }
        acc.x = act_bf(acc.x, L.nscale); acc.y = act_bf(acc.y, L.nscale);
        acc.z = act_bf(acc.z, L.nscale); acc.w = act_bf(acc.w, L.nscale);
        if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + apos(cb, P, p, q)) = acc;
        else *reinterpret_cast<float4 *>(gout + ((size_t)cb * P + p) * CB + 4 * q) = acc;
    }
}

__device__ __forceinline__ float4 pool_op(bool is_max, float4 acc, float4 v)
{
    if (is_max)
    {
        acc.x = v.x > acc.x ? v.x : acc.x; acc.y = v.y > acc.y ? v.y : acc.y;
        acc.z = v.z > acc.z ? v.z : acc.z; acc.w = v.w > acc.w ? v.w : acc.w;
    }
    else { acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w; }
    return acc;
}

// window == whole image, no padding (AveragePool2D: sum * float(1 / (H * W)), abstract_layer.hpp:514-569).
// A wave owns a channel quad (wave, wave + 16, ...): its lanes fold the pixels lane, lane + 64, ... in that order, then
// the wave folds its 64 partial sums with xor-shuffles (32, 16, ... 1): a fixed order (deterministic), no barrier and no
// LDS staging inside the layer.  (Three stages through LDS with two barriers took 2.4 us of the DS-CNN's 27.)
__device__ __forceinline__ void pool_layer(const FMLayer &L, float *lds, float *part, float *gout, int tid)
{
    (void)part;
    const int C4 = L.Ci / 4, P = L.H * L.W;
    const bool is_max = L.kind == K_POOL_MAX;
    const float *src = lds + L.src_off;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int c4 = wave; c4 < C4; c4 += NW)
    {
        const int cb = c4 >> 2, q = c4 & 3;
        // a lane without a pixel holds the operation's neutral element: pixel 0 again for the maximum, zero for the sum
        float4 acc = is_max ? *reinterpret_cast<const float4 *>(src + apos(cb, P, 0, q)) : make_float4(0.f, 0.f, 0.f, 0.f);
        for (int p = lane; p < P; p += WAVE)
            acc = pool_op(is_max, acc, *reinterpret_cast<const float4 *>(src + apos(cb, P, p, q)));
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
        {
            const float4 o = make_float4(__shfl_xor(acc.x, d, WAVE), __shfl_xor(acc.y, d, WAVE), __shfl_xor(acc.z, d, WAVE),
                                         __shfl_xor(acc.w, d, WAVE));
            acc = pool_op(is_max, acc, o);
        }
        if (lane == 0)
        {
            if (!is_max) { acc.x *= L.norm; acc.y *= L.norm; acc.z *= L.norm; acc.w *= L.norm; }
            if (L.dst_off >= 0) *reinterpret_cast<float4 *>(lds + L.dst_off + apos(cb, 1, 0, q)) = acc;
            else *reinterpret_cast<float4 *>(gout + (size_t)cb * CB + 4 * q) = acc;
        }
    }
}

// n16 16-byte pieces from global memory to LDS without passing through registers (global_load_lds_dwordx4: a wave's
// 64 lanes write 1 KiB of consecutive LDS from the wave-uniform base; each lane supplies its own global address).
// The caller waits (vmcnt) before the data is read.
__device__ __forceinline__ void weights_to_lds(const float *g, float *l, int n16, int tid, int wave)
{
#pragma unroll
    for (int k = 0; k < NPRE; ++k)
    {
        const int i = tid + k * NT;
        if (i < n16)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(g + i * 4),
                                             (__attribute__((address_space(3))) void *)(l + (k * NT + wave * WAVE) * 4), 16, 0, 0);
    }
}

__global__ __launch_bounds__(NT) void fmodel_f32_kernel(const FMHeader *__restrict__ hdr_dev, const float *__restrict__ blob,
                                                        const float *__restrict__ in, float *__restrict__ out)
{
    HeaderPtr hdr = (HeaderPtr)hdr_dev;
    extern __shared__ __align__(16) float lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t n = blockIdx.x;
    const int n_layers = hdr->n_layers;
    float *wbuf = lds + hdr->w_lds;
    const int w_floats = hdr->w_floats;

    // the first layer's weights and the image
    {
        weights_to_lds(blob + hdr->layer[0].blob_off, wbuf, hdr->layer[0].blob16, tid, wave);
        const float *img = in + n * (size_t)hdr->in_elems;
        float *x = lds + hdr->in_off;
        if (hdr->in_C < CB)
            for (int i = tid; i < hdr->in_elems; i += NT) x[i] = img[i];
        else
        {
            const int P = hdr->in_H * hdr->in_W, n4 = hdr->in_elems >> 2;
            for (int i = tid; i < n4; i += NT)
            {
                const int q = i & 3, r = i >> 2, cb = r / P, p = r - cb * P;
                *reinterpret_cast<float4 *>(x + apos(cb, P, p, q)) = reinterpret_cast<const float4 *>(img)[i];
            }
        }
    }
    float *gout = out + n * (size_t)hdr->out_elems;
    float *part = lds + hdr->pool_off;
    const float *zero = lds + hdr->zero_off;
    if (tid < 4) lds[hdr->zero_off + tid] = 0.f;
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    for (int li = 0; li < n_layers; ++li)
    {
        const FMLayer L = load_layer(hdr, li);
        const float *wl = wbuf + (li & 1) * w_floats;
        // the next layer's weights go from global memory straight into the other LDS buffer (no registers are held
        // across the layer): in flight while this layer is computed, waited for before the barrier that ends it
        if (L.next_blob16 > 0)
            weights_to_lds(blob + L.next_blob_off, wbuf + ((li + 1) & 1) * w_floats, L.next_blob16, tid, wave);
        if (L.kind == K_CONV)
        {
            const int n_tiles = ((L.Ho * L.Wo + 15) >> 4) * (L.Co / CB);
            if (n_tiles >= 2 * NW) conv_layer<2>(L, lds, wl, zero, gout, wave, lane);
            else conv_layer<1>(L, lds, wl, zero, gout, wave, lane);
        }
        else if (L.kind == K_STEM)
        {
            // as many output-channel blocks per gathered operand as still leave every wave a pixel tile
            const int CoB = L.Co / CB, n_pt = (L.Ho * L.Wo + 15) >> 4;
            if (CoB % 4 == 0 && n_pt * (CoB / 4) >= NW) stem_layer<4>(L, lds, wl, zero, gout, wave, lane);
            else if (CoB % 2 == 0 && n_pt * (CoB / 2) >= NW) stem_layer<2>(L, lds, wl, zero, gout, wave, lane);
            else stem_layer<1>(L, lds, wl, zero, gout, wave, lane);
        }
        else if (L.kind == K_DWPW)
        {
            // as many output-channel blocks per depthwise result as still leave every wave a pixel tile
            const int CoB = L.Co2 / CB, n_pt = (L.Ho * L.Wo + 15) >> 4;
            if (CoB % 4 == 0 && (n_pt * (CoB / 4) >= NW || CoB == 4)) dwpw_layer<4>(L, lds, wl, zero, gout, wave, lane);
            else if (CoB % 2 == 0) dwpw_layer<2>(L, lds, wl, zero, gout, wave, lane);
            else dwpw_layer<1>(L, lds, wl, zero, gout, wave, lane);
        }
        else if (L.kind == K_DW)
        {
            if (L.kh == 3 && L.kw == 3) dw_layer_win<3, 3>(L, lds, wl, zero, gout, tid);
            else dw_layer_any(L, lds, wl, gout, tid);
        }
        else
            pool_layer(L, lds, part, gout, tid);
        __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0): the weights have landed in LDS
        __syncthreads();
    }
}

// ---- depthwise-separable chains ---------------------------------------------------------------------------------
// First layer of 1..3 channels, pairs of a 3x3 depthwise and a 1x1 convolution, a whole-image pooling, fully connected layers:
// what a keyword-spotting DS-CNN is.  What bounds such a model is the number of instructions between two barriers (a layer is
// a few hundred cycles of arithmetic per wave; the general kernel's address arithmetic with its bounds took as long again), so
// LDS is laid out for addresses that cost nothing:
//   * pixels PITCH floats apart, 16 channels and 4 of padding: eight neighbouring pixels cover all banks without a swizzle,
//   * what a depthwise layer reads has a ring of zeros round it (written once, before the first layer; a tensor of another shape has
//     its own place), so a window is three row addresses with constant column offsets and no bounds,
//   * the image lies in LDS with its padding, so a tap of the first layer is one addition to a table entry.
// An image is one workgroup, or (few images) several: it is cut into bands of rows, and a band computes the rows of every layer that
// its rows of the last pair need (the halo is computed again by the neighbours).  A band stores its rows of the last pair; the
// workgroup that is counted last pools them and goes on.  Nobody waits for anybody: the others have left.  Sums and their
// order do not depend on the cut.
constexpr int PITCH = CB + 4;

struct SepPair
{
    int src, src_plane, src_row;         // LDS floats: the ring tensor's first window position, its channel block, its row
    int c4, stride, Wo;                  // channel quads, depthwise stride, output columns
    int plane;                           // floats of a channel block between the two layers
    int CiB, CoB;
    int bias_off, w2_off, bias2_off;     // inside the unit's weights
    int dst, dst_plane, dst_row;         // LDS floats: the next ring tensor's pixel (0, 0), its channel block, its row
    int next_off, next16;                // the next unit's weights: blob float offset and 16-byte pieces
    float r_wo, r_cob, nscale, nscale2;
};
struct SepArgs
{
    int n_pairs, n_fc;
    int in_elems, out_elems, Ci, W, H;   // the image in memory
    int img, img_row, img_elems;         // the padded image in LDS: float offset, floats per row, floats
    int pt, pl;
    float r_row, r_ci;                   // 1 / img_row, 1 / Ci
    int ring, ring_floats;               // LDS to be cleared
    int w_lds, w_floats, mid, mid2;      // two weight buffers; the tensor between a pair's layers; the other half of the FC ping-pong
    // first layer
    int CoB, P, Wo, stride, chunks, bias_off, ktab_off, blob_off, blob16, next_off, next16;
    int dst, dst_plane, dst_row;
    float r_wo, r_cob, nscale;
    // whole-image pooling of the last pair's output
    int last_P, last_elems, last_Wo, pool_c4, pool_max, last_dst, last_plane, last_row;
    float last_r_wo, norm;
    int last_word;                       // LDS word of the band count
};
typedef const __attribute__((address_space(4))) SepPair *PairPtr;
typedef const __attribute__((address_space(4))) int2 *RangePtr;

__device__ __forceinline__ SepPair load_pair(PairPtr p)
{
    SepPair r;
    __builtin_memcpy(&r, p, sizeof(SepPair));
    return r;
}

__device__ __forceinline__ int div_by(int i, float r) { return (int)(((float)i + 0.5f) * r); }      // i / d for r = 1 / d, i * d small

// output pixels [p0, p1) of the first layer; TC output-channel blocks share a gathered operand
template <int TC>
__device__ __forceinline__ void sep_stem(const SepArgs &a, float *lds, const float *wl, int wave, int lane, int p0, int p1)
{
    const int col = lane & 15, kq = lane >> 4;
    const int n_pt = (p1 - p0 + 15) >> 4, n_cg = a.CoB / TC, n_work = n_pt * n_cg;
    const float r_ncg = a.r_cob * (float)TC;
    const int4 *ktab = reinterpret_cast<const int4 *>(wl + a.ktab_off);
    for (int work = wave; work < n_work; work += NW)
    {
        const int pt = div_by(work, r_ncg), cg = work - pt * n_cg;
        const int p = p0 + pt * 16 + col;
        const bool pv = p < p1;
        const int pc = pv ? p : p0;
        const int oh = div_by(pc, a.r_wo), ow = pc - oh * a.Wo;
        const float *x = lds + a.img + oh * a.stride * a.img_row + ow * a.stride * a.Ci;
        const float *w = wl + (cg * TC * a.chunks * 64 + kq * 16 + col) * 4;
        floatx4 acc[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        for (int ch = 0; ch < a.chunks; ++ch)
        {
            const int4 e4 = ktab[ch * 4 + kq];
            const int ev[4] = {e4.x, e4.y, e4.z, e4.w};
            float4 A[TC];
            float b[4];
#pragma unroll
            for (int c = 0; c < TC; ++c) A[c] = *reinterpret_cast<const float4 *>(w + (c * a.chunks + ch) * 256);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = x[ev[j] < 0 ? 0 : ev[j]];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ev[j] < 0 ? 0.f : b[j];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < TC; ++c)
                {
                    const float Av[4] = {A[c].x, A[c].y, A[c].z, A[c].w};
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(Av[j], b[j], acc[c], 0, 0, 0);
                }
        }
        if (!pv) continue;
        float *d = lds + a.dst + oh * a.dst_row + ow * PITCH + 4 * kq;
#pragma unroll
        for (int c = 0; c < TC; ++c)
        {
            const int cob = cg * TC + c;
            const float4 bias = *reinterpret_cast<const float4 *>(wl + a.bias_off + cob * CB + 4 * kq);
            *reinterpret_cast<float4 *>(d + cob * a.dst_plane) =
                make_float4(act_bf(acc[c][0] + bias.x, a.nscale), act_bf(acc[c][1] + bias.y, a.nscale),
                            act_bf(acc[c][2] + bias.z, a.nscale), act_bf(acc[c][3] + bias.w, a.nscale));
        }
    }
}

// depthwise 3x3, output pixels [p0, p1): a lane owns four channels of a pixel, consecutive lanes consecutive pixels
__device__ __forceinline__ void sep_dw(const SepPair &L, float *lds, const float *wl, float *mid, int tid, int p0, int p1)
{
    const int np = p1 - p0, n = np * L.c4;
    const float r_np = __builtin_amdgcn_rcpf((float)np);
    for (int i = tid; i < n; i += NT)
    {
        const int c = div_by(i, r_np), p = p0 + i - c * np;
        const int oh = div_by(p, L.r_wo), ow = p - oh * L.Wo;
        const int cb = c >> 2, q = (c & 3) * 4;
        const float *x = lds + L.src + cb * L.src_plane + oh * L.stride * L.src_row + ow * L.stride * PITCH + q;
        const float *w = wl + cb * (9 * CB) + q;
        float4 acc = *reinterpret_cast<const float4 *>(wl + L.bias_off + cb * CB + q);
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
#pragma unroll
            for (int b = 0; b < 3; ++b)
            {
                const float4 v = *reinterpret_cast<const float4 *>(x + b * PITCH);
                const float4 k = *reinterpret_cast<const float4 *>(w + (a * 3 + b) * CB);
                acc.x = fmaf(v.x, k.x, acc.x); acc.y = fmaf(v.y, k.y, acc.y);
                acc.z = fmaf(v.z, k.z, acc.z); acc.w = fmaf(v.w, k.w, acc.w);
            }
            x += L.src_row;
        }
        *reinterpret_cast<float4 *>(mid + cb * L.plane + p * PITCH + q) =
            make_float4(act_bf(acc.x, L.nscale), act_bf(acc.y, L.nscale), act_bf(acc.z, L.nscale), act_bf(acc.w, L.nscale));
    }
}

// The same at stride 1 for rows [r0, r1): a lane slides a window of three rows down R output rows of a column, so that a row of
// the input is read once for R outputs and the taps once for all of them.  For maps of more outputs than the workgroup has lanes, where
// LDS reads bound the layer (DS-CNN on whole images: a pixel a lane 29.5 us, three 26.1).
template <int R>
__device__ __forceinline__ void sep_dw_strip(const SepPair &L, float *lds, const float *wl, float *mid, int tid, int r0, int r1)
{
    const int np = (r1 - r0 + R - 1) / R * L.Wo, n = np * L.c4;
    const float r_np = __builtin_amdgcn_rcpf((float)np);
    for (int i = tid; i < n; i += NT)
    {
        const int c = div_by(i, r_np), s = i - c * np;
        const int st = div_by(s, L.r_wo), ow = s - st * L.Wo, oh = r0 + st * R;
        const int cb = c >> 2, q = (c & 3) * 4;
        const float *x = lds + L.src + cb * L.src_plane + oh * L.src_row + ow * PITCH + q;
        const float *w = wl + cb * (9 * CB) + q;
        const float4 bias = *reinterpret_cast<const float4 *>(wl + L.bias_off + cb * CB + q);
        float4 k[9], acc[R];
#pragma unroll
        for (int t = 0; t < 9; ++t) k[t] = *reinterpret_cast<const float4 *>(w + t * CB);
#pragma unroll
        for (int o = 0; o < R; ++o) acc[o] = bias;
#pragma unroll
        for (int a = 0; a < R + 2; ++a)
        {
            float4 v[3];
#pragma unroll
            for (int b = 0; b < 3; ++b) v[b] = *reinterpret_cast<const float4 *>(x + b * PITCH);
            x += oh + a < r1 + 1 ? L.src_row : 0;                // rows of outputs past r1 repeat the last one that exists
#pragma unroll
            for (int o = 0; o < R; ++o)
            {
                if (a < o || a > o + 2) continue;
#pragma unroll
                for (int b = 0; b < 3; ++b)
                {
                    const float4 kk = k[(a - o) * 3 + b];
                    acc[o].x = fmaf(v[b].x, kk.x, acc[o].x); acc[o].y = fmaf(v[b].y, kk.y, acc[o].y);
                    acc[o].z = fmaf(v[b].z, kk.z, acc[o].z); acc[o].w = fmaf(v[b].w, kk.w, acc[o].w);
                }
            }
        }
        float *d = mid + cb * L.plane + (oh * L.Wo + ow) * PITCH + q;
#pragma unroll
        for (int o = 0; o < R; ++o)
            if (oh + o < r1)
                *reinterpret_cast<float4 *>(d + o * L.Wo * PITCH) = make_float4(act_bf(acc[o].x, L.nscale), act_bf(acc[o].y, L.nscale),
                                                                                act_bf(acc[o].z, L.nscale), act_bf(acc[o].w, L.nscale));
    }
}

// 1x1 convolution, pixels [p0, p1) of src [CiB][plane]; TP pixel tiles share a filter operand.  To a ring tensor (TO_RING), to the
// band's slot (TO_SLOT: g is the tensor [CoB][P][16] in memory) or to a vector of one pixel (TO_VECTOR: g in memory, or LDS).
enum { TO_RING, TO_SLOT, TO_VECTOR };
template <int TP, int TO>
__device__ __forceinline__ void sep_pw(const SepPair &L, float *lds, const float *wl, const float *src, float *g, int P, int wave, int lane,
                                       int p0, int p1)
{
    const int col = lane & 15, kq = lane >> 4;
    const int n_pt = (p1 - p0 + 15) >> 4, n_work = (n_pt + TP - 1) / TP * L.CoB;
    for (int work = wave; work < n_work; work += NW)
    {
        const int pg = div_by(work, L.r_cob), cob = work - pg * L.CoB;
        int p[TP];
        const float *x[TP];
        floatx4 acc[TP];
#pragma unroll
        for (int t = 0; t < TP; ++t)
        {
            p[t] = p0 + (pg * TP + t) * 16 + col;
            x[t] = src + (p[t] < p1 ? p[t] : p0) * PITCH + 4 * kq;
            acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const float *w = wl + L.w2_off + (cob * L.CiB * 64 + kq * 16 + col) * 4;
        const float4 bias = *reinterpret_cast<const float4 *>(wl + L.bias2_off + cob * CB + 4 * kq);
        auto blocks = [&](auto n_) {
            constexpr int N = decltype(n_)::value;
            float4 A[N], B[TP][N];
#pragma unroll
            for (int u = 0; u < N; ++u)
            {
                A[u] = *reinterpret_cast<const float4 *>(w + u * 256);
#pragma unroll
                for (int t = 0; t < TP; ++t) { B[t][u] = *reinterpret_cast<const float4 *>(x[t]); x[t] += L.plane; }
            }
            w += N * 256;
#pragma unroll
            for (int u = 0; u < N; ++u)
            {
                const float Av[4] = {A[u].x, A[u].y, A[u].z, A[u].w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < TP; ++t)
                    {
                        const float Bv[4] = {B[t][u].x, B[t][u].y, B[t][u].z, B[t][u].w};
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Av[j], Bv[j], acc[t], 0, 0, 0);
                    }
            }
        };
        int cib = 0;
        for (; cib + 4 <= L.CiB; cib += 4) blocks(std::integral_constant<int, 4>{});
        for (; cib < L.CiB; ++cib) blocks(std::integral_constant<int, 1>{});
#pragma unroll
        for (int t = 0; t < TP; ++t)
        {
            if (p[t] >= p1) continue;
            const float4 v = make_float4(act_bf(acc[t][0] + bias.x, L.nscale2), act_bf(acc[t][1] + bias.y, L.nscale2),
                                         act_bf(acc[t][2] + bias.z, L.nscale2), act_bf(acc[t][3] + bias.w, L.nscale2));
            if (TO == TO_RING)
            {
                const int oh = div_by(p[t], L.r_wo), ow = p[t] - oh * L.Wo;
                *reinterpret_cast<float4 *>(lds + L.dst + cob * L.dst_plane + oh * L.dst_row + ow * PITCH + 4 * kq) = v;
            }
            else if (TO == TO_SLOT) store_shared(g + ((size_t)cob * P + p[t]) * CB + 4 * kq, v);
            else if (g) *reinterpret_cast<float4 *>(g + cob * CB + 4 * kq) = v;
            else *reinterpret_cast<float4 *>(lds + L.dst + cob * PITCH + 4 * kq) = v;
        }
    }
}

// whole-image pooling as pool_layer does it: a wave per channel quad, pixels lane, lane + 64, ..., then xor-folds 32, 16, ... 1
template <bool SLOT>
__device__ __forceinline__ void sep_pool(const SepArgs &a, float *lds, const float *tensor, float *dst, float *g, int wave, int lane)
{
    for (int c = wave; c < a.pool_c4; c += NW)
    {
        const int cb = c >> 2, q = (c & 3) * 4;
        auto value = [&](int p) -> float4 {
            if (SLOT) return load_shared(tensor + ((size_t)cb * a.last_P + p) * CB + q);
            const int oh = div_by(p, a.last_r_wo), ow = p - oh * a.last_Wo;
            return *reinterpret_cast<const float4 *>(lds + a.last_dst + cb * a.last_plane + oh * a.last_row + ow * PITCH + q);
        };
        float4 acc = a.pool_max ? value(0) : make_float4(0.f, 0.f, 0.f, 0.f);
        for (int p = lane; p < a.last_P; p += WAVE) acc = pool_op(a.pool_max, acc, value(p));
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
        {
            const float4 o = make_float4(__shfl_xor(acc.x, d, WAVE), __shfl_xor(acc.y, d, WAVE), __shfl_xor(acc.z, d, WAVE),
                                         __shfl_xor(acc.w, d, WAVE));
            acc = pool_op(a.pool_max, acc, o);
        }
        if (lane == 0)
        {
            if (!a.pool_max) { acc.x *= a.norm; acc.y *= a.norm; acc.z *= a.norm; acc.w *= a.norm; }
            if (g) *reinterpret_cast<float4 *>(g + c * 4) = acc;
            else *reinterpret_cast<float4 *>(dst + cb * PITCH + q) = acc;
        }
    }
}

__global__ __launch_bounds__(NT) void fmodel_f32_sep_kernel(const SepArgs a, const SepPair *__restrict__ pairs_dev, const float *__restrict__ blob,
                                                            const float *__restrict__ in, float *__restrict__ out,
                                                            const int2 *__restrict__ ranges_dev, int bands, float *tensors, unsigned *counters)
{
    extern __shared__ __align__(16) float lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = blockIdx.x / bands, band = blockIdx.x - n * bands;
    PairPtr pairs = (PairPtr)pairs_dev;
    RangePtr ranges = (RangePtr)(ranges_dev + (size_t)band * (a.n_pairs + 1));
    float *wbuf = lds + a.w_lds, *gout = out + (size_t)n * a.out_elems, *tensor = tensors + (size_t)n * a.last_elems;

    // first layer's weights, the image with its padding, zeros for the rings
    weights_to_lds(blob + a.blob_off, wbuf, a.blob16, tid, wave);
    const float *img = in + (size_t)n * a.in_elems;
    for (int i = tid; i < a.img_elems; i += NT)
    {
        const int r = div_by(i, a.r_row), c = i - r * a.img_row, x = div_by(c, a.r_ci), ih = r - a.pt, iw = x - a.pl;
        const bool ok = (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
        lds[a.img + i] = ok ? img[(ih * a.W + iw) * a.Ci + c - x * a.Ci] : 0.f;
    }
    for (int i = tid * 4; i < a.ring_floats; i += NT * 4) *reinterpret_cast<float4 *>(lds + a.ring + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    SepPair L = load_pair(pairs);
    int2 rg;
    __builtin_memcpy(&rg, ranges, sizeof(rg));
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    if (a.next16 > 0) weights_to_lds(blob + a.next_off, wbuf + a.w_floats, a.next16, tid, wave);
    {
        // as many output-channel blocks per gathered operand as still leave every wave a pixel tile
        const int n_pt = (rg.y - rg.x + 15) >> 4;
        if (a.CoB % 4 == 0 && n_pt * (a.CoB / 4) >= NW) sep_stem<4>(a, lds, wbuf, wave, lane, rg.x, rg.y);
        else if (a.CoB % 2 == 0 && n_pt * (a.CoB / 2) >= NW) sep_stem<2>(a, lds, wbuf, wave, lane, rg.x, rg.y);
        else sep_stem<1>(a, lds, wbuf, wave, lane, rg.x, rg.y);
    }
    __builtin_memcpy(&rg, ranges + 1, sizeof(rg));
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    float *mid = lds + a.mid;
    int unit = 1;
    for (int i = 0; i < a.n_pairs; ++i, ++unit)
    {
        const float *wl = wbuf + (unit & 1) * a.w_floats;
        if (L.next16 > 0) weights_to_lds(blob + L.next_off, wbuf + ((unit + 1) & 1) * a.w_floats, L.next16, tid, wave);
        if (L.stride == 1 && (rg.y - rg.x) * L.c4 > NT) sep_dw_strip<3>(L, lds, wl, mid, tid, div_by(rg.x, L.r_wo), div_by(rg.y, L.r_wo));
        else sep_dw(L, lds, wl, mid, tid, rg.x, rg.y);
        // the next pair's record (the fully connected layers' follow the pairs') while this one multiplies
        const SepPair N = load_pair(pairs + i + 1);
        int2 rn;
        __builtin_memcpy(&rn, ranges + (i + 2 <= a.n_pairs ? i + 2 : i + 1), sizeof(rn));
        __syncthreads();
        const int n_work = ((rg.y - rg.x + 15) >> 4) * L.CoB;
        if (i + 1 == a.n_pairs && bands > 1) sep_pw<1, TO_SLOT>(L, lds, wl, mid, tensor, a.last_P, wave, lane, rg.x, rg.y);
        else if (n_work >= 2 * NW) sep_pw<2, TO_RING>(L, lds, wl, mid, nullptr, 0, wave, lane, rg.x, rg.y);
        else sep_pw<1, TO_RING>(L, lds, wl, mid, nullptr, 0, wave, lane, rg.x, rg.y);
        L = N;
        rg = rn;
        // vmcnt(0): the weights have landed in LDS, and the slot's rows where every XCD reads them; with the barrier this is the release in front of
        // the (relaxed) count of a finished band
        keep_order();
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    }

    float *vec = mid, *gpool = a.n_fc == 0 ? gout : nullptr;
    if (bands > 1)
    {
        // every wave has waited for its stores before the band is counted
        unsigned *last = reinterpret_cast<unsigned *>(lds + a.last_word);
        if (tid == 0) *last = __hip_atomic_fetch_add(counters + n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*last != (unsigned)bands - 1) return;        // the whole workgroup leaves together
        keep_order();                                    // the bands' rows are read after the count
        if (tid == 0) __hip_atomic_store(counters + n, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch on this stream
        sep_pool<true>(a, lds, tensor, vec, gpool, wave, lane);
    }
    else sep_pool<false>(a, lds, nullptr, vec, gpool, wave, lane);
    __syncthreads();
    for (int i = 0; i < a.n_fc; ++i, ++unit)
    {
        const float *wl = wbuf + (unit & 1) * a.w_floats;
        if (L.next16 > 0) weights_to_lds(blob + L.next_off, wbuf + ((unit + 1) & 1) * a.w_floats, L.next16, tid, wave);
        const bool end = i + 1 == a.n_fc;
        sep_pw<1, TO_VECTOR>(L, lds, wl, vec, end ? gout : nullptr, 0, wave, lane, 0, 1);
        if (end) break;
        vec = lds + L.dst;
        L = load_pair(pairs + a.n_pairs + i + 1);
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    }
}

int align_up(int v, int a) { return (v + a - 1) / a * a; }

} // namespace

struct small_hip_fmodel
{
    FMHeader hdr;
    void *dev = nullptr;        // [FMHeader, or the records and pixel ranges of a separable chain][weights of every layer][bands' slots]
    size_t blob_off = 0;
    int device = 0;

    // Separable chain.  What the bands of a launch exchange lies in one of a few slots, each taken for good by the first stream that
    // needs one, so that two launches that may run at the same time never share one.  A stream is its handle; a handle that the runtime
    // gives out again belongs to a stream whose work is done, because hipStreamDestroy waits for it (measured with the runtimes of ROCm 7.0
    // and 7.2: 332 ms behind a kernel of that length, created with and without hipStreamNonBlocking).
    static constexpr int SLOTS = 4;
    static constexpr size_t SLOT_BYTES = size_t(4) << 20;
    bool separable = false;
    SepArgs sep;
    size_t ranges_off = 0, slot_bytes = 0;
    int rows = 0, band_batch = 0;                    // rows of the last pair's output; images a slot has room for (0: no slots)
    std::vector<int> ranges_first;                   // [rows per band] -> first range (int2) of that cut, -1: not planned
    std::vector<float> band_work;                    // [rows per band] -> work of the longest band (bands_pay)
    unsigned char *slots = nullptr;                  // [SLOTS][band_batch] tensors
    unsigned *counters = nullptr;                    // [SLOTS][band_batch]
    mutable std::mutex mu;
    mutable int n_slots = 0;
    mutable hipStream_t slot_stream[SLOTS];

    // the slot of this stream, or -1: others got all of them before it (take = false: the slot it would get)
    int slot(hipStream_t s, bool take) const
    {
        std::lock_guard<std::mutex> lk(mu);
        for (int i = 0; i < n_slots; ++i)
            if (slot_stream[i] == s) return i;
        if (n_slots == SLOTS) return -1;
        if (!take) return n_slots;
        slot_stream[n_slots] = s;
        return n_slots++;
    }
};

namespace
{

// Is the model a separable chain that fits LDS in that kernel's layout?  Fills its arguments, records and pixel ranges.
bool plan_separable(const small_hip_flayer *layers, const std::vector<FMLayer> &tmp, small_hip_fmodel *m, std::vector<SepPair> &pairs,
                    std::vector<int> &ranges)
{
    const int n = (int)tmp.size();
    auto at = [&](int i) -> const FMLayer & { return tmp[(size_t)i]; };
    auto pointwise = [&](int i) {
        const FMLayer &L = at(i);
        return L.kind == K_CONV && L.kh == 1 && L.kw == 1 && L.stride == 1 && L.pt == 0 && L.pl == 0 && L.Ho == L.H && L.Wo == L.W;
    };
    for (int i = 1; i < n; ++i)
        if (layers[i].src != layers[i - 1].dst) return false;
    if (at(0).kind != K_STEM) return false;
    int n_pairs = 0, i = 1;
    for (; i + 1 < n && at(i).kind == K_DW; i += 2, ++n_pairs)
    {
        const FMLayer &D = at(i);
        // the window stays within one pixel of the image
        if (D.kh != 3 || D.kw != 3 || D.pt > 1 || D.pl > 1 || (D.Ho - 1) * D.stride - D.pt + 2 > D.H || (D.Wo - 1) * D.stride - D.pl + 2 > D.W ||
            !pointwise(i + 1) || D.blob16 + at(i + 1).blob16 > NPRE * NT)
            return false;
    }
    if (n_pairs == 0 || i >= n || (at(i).kind != K_POOL_AVG && at(i).kind != K_POOL_MAX)) return false;
    const int pool = i, n_fc = n - 1 - pool;
    for (int k = pool + 1; k < n; ++k)
        if (!pointwise(k) || at(k).H != 1 || at(k).W != 1) return false;

    SepArgs &a = m->sep;
    std::memset(&a, 0, sizeof(a));
    a.n_pairs = n_pairs; a.n_fc = n_fc;
    const FMLayer &S = at(0);
    const small_hip_flayer &l0 = layers[0];
    a.Ci = S.Ci; a.H = S.H; a.W = S.W; a.in_elems = S.Ci * S.H * S.W;
    a.out_elems = at(n - 1).Co * at(n - 1).Ho * at(n - 1).Wo;
    a.pt = l0.t_pad; a.pl = l0.l_pad;
    a.img_row = ((S.Wo - 1) * S.stride + S.kw) * S.Ci;
    a.img_elems = ((S.Ho - 1) * S.stride + S.kh) * a.img_row;
    a.r_row = 1.0f / (float)a.img_row; a.r_ci = 1.0f / (float)S.Ci;

    // LDS (floats): [weights x2][word][image][ring tensors, one place per map size][between a pair's layers][vectors]
    struct Ring { int H, W, blocks, off; };
    std::vector<Ring> rings;
    auto ring = [&](int blocks, int H, int W) -> Ring & {
        for (Ring &r : rings)
            if (r.H == H && r.W == W) { r.blocks = blocks > r.blocks ? blocks : r.blocks; return r; }
        rings.push_back(Ring{H, W, blocks, 0});
        return rings.back();
    };
    int mid = 0, mid2 = 0, unit = S.blob16;
    ring(S.Co / CB, S.Ho, S.Wo);
    for (int p = 0; p < n_pairs; ++p)
    {
        const FMLayer &D = at(1 + 2 * p), &C = at(2 + 2 * p);
        ring(C.Co / CB, C.Ho, C.Wo);
        mid = std::max(mid, D.Co / CB * D.Ho * D.Wo * PITCH);
        unit = std::max(unit, D.blob16 + C.blob16);
    }
    mid = std::max(mid, at(pool).Ci / CB * PITCH);
    for (int k = pool + 1; k < n; ++k)
    {
        unit = std::max(unit, at(k).blob16);
        mid = std::max(mid, at(k).Co / CB * PITCH);
        mid2 = std::max(mid2, at(k).Co / CB * PITCH);
    }
    long off = 0;
    a.w_lds = 0; a.w_floats = unit * 4; off += 2L * a.w_floats;
    a.last_word = (int)off; off += 4;
    a.img = (int)off; off += align_up(a.img_elems, 4);
    a.ring = (int)off;
    for (Ring &r : rings) { r.off = (int)off; off += (long)r.blocks * (r.H + 2) * (r.W + 2) * PITCH; }
    a.ring_floats = (int)(off - a.ring);
    a.mid = (int)off; off += mid;
    a.mid2 = (int)off; off += mid2;
    if (off * 4 > LDS_LIMIT) return false;
    m->hdr.lds_bytes = (int)off * 4;

    auto window = [](const Ring &r, int pt, int pl) { return r.off + ((1 - pt) * (r.W + 2) + 1 - pl) * PITCH; };
    auto row = [](const Ring &r) { return (r.W + 2) * PITCH; };
    auto plane = [](const Ring &r) { return (r.H + 2) * (r.W + 2) * PITCH; };
    auto weights = [&](int k, int *o, int *n16) {                       // of the unit that begins with layer k
        if (k >= n) { *o = *n16 = 0; return; }
        *o = at(k).blob_off;
        *n16 = at(k).blob16 + (k < pool ? at(k + 1).blob16 : 0);
    };
    {
        const Ring &r = ring(S.Co / CB, S.Ho, S.Wo);
        a.CoB = S.Co / CB; a.P = S.Ho * S.Wo; a.Wo = S.Wo; a.stride = S.stride; a.chunks = S.chunks;
        a.bias_off = S.bias_off; a.ktab_off = S.ktab_off; a.blob_off = S.blob_off; a.blob16 = S.blob16;
        weights(1, &a.next_off, &a.next16);
        a.dst = window(r, 0, 0); a.dst_row = row(r); a.dst_plane = plane(r);
        a.r_wo = S.r_wo; a.r_cob = S.r_cob; a.nscale = S.nscale;
    }
    pairs.assign((size_t)(n_pairs + n_fc + 1), SepPair{});
    for (int p = 0; p < n_pairs; ++p)
    {
        const FMLayer &D = at(1 + 2 * p), &C = at(2 + 2 * p);
        SepPair &L = pairs[(size_t)p];
        const Ring &src = ring(D.Ci / CB, D.H, D.W), &dst = ring(C.Co / CB, C.Ho, C.Wo);
        L.src = window(src, D.pt, D.pl); L.src_row = row(src); L.src_plane = plane(src);
        L.c4 = D.Ci / 4; L.stride = D.stride; L.Wo = D.Wo; L.plane = D.Ho * D.Wo * PITCH;
        L.CiB = C.Ci / CB; L.CoB = C.Co / CB;
        L.bias_off = D.bias_off; L.w2_off = C.blob_off - D.blob_off; L.bias2_off = L.w2_off + C.bias_off;
        L.dst = window(dst, 0, 0); L.dst_row = row(dst); L.dst_plane = plane(dst);
        weights(p + 1 < n_pairs ? 3 + 2 * p : pool + 1, &L.next_off, &L.next16);
        L.r_wo = D.r_wo; L.r_cob = C.r_cob; L.nscale = D.nscale; L.nscale2 = C.nscale;
        if (p + 1 == n_pairs)
        {
            a.last_P = C.Ho * C.Wo; a.last_elems = C.Co * a.last_P; a.last_Wo = C.Wo; a.last_r_wo = C.r_wo;
            a.last_dst = L.dst; a.last_row = L.dst_row; a.last_plane = L.dst_plane;
        }
    }
    a.pool_c4 = at(pool).Ci / 4; a.pool_max = at(pool).kind == K_POOL_MAX; a.norm = at(pool).norm;
    for (int k = pool + 1; k < n; ++k)
    {
        const FMLayer &C = at(k);
        SepPair &L = pairs[(size_t)(n_pairs + k - pool - 1)];
        L.plane = PITCH; L.CiB = C.Ci / CB; L.CoB = C.Co / CB; L.bias2_off = C.bias_off;
        L.dst = (k - pool) & 1 ? a.mid2 : a.mid;
        weights(k + 1, &L.next_off, &L.next16);
        L.r_wo = 1.f; L.r_cob = C.r_cob; L.nscale2 = C.nscale;
    }

    // for each number of rows per band: the output pixels of the first layer and of every pair that each band computes
    const int rows = at(pool).H;
    m->rows = rows;
    m->ranges_first.assign((size_t)rows + 1, -1);
    m->band_work.assign((size_t)rows + 1, 0.f);
    for (int rb = 1; rb <= rows; rb = rb < rows && rb + 1 > (rows + 1) / 2 ? rows : rb + 1)
    {
        m->ranges_first[(size_t)rb] = (int)ranges.size() / 2;
        for (int r = 0; r < rows; r += rb)
        {
            std::vector<int> band((size_t)(n_pairs + 1) * 2);
            int lo = r, hi = std::min(r + rb, rows);
            float work = 0.f;
            for (int u = n_pairs; u >= 0; --u)
            {
                if (lo >= hi) return false;          // a band that reads padding only
                const int Wo = u == 0 ? S.Wo : at(2 * u - 1).Wo;
                band[(size_t)u * 2] = lo * Wo;
                band[(size_t)u * 2 + 1] = hi * Wo;
                if (u == 0) break;
                const FMLayer &D = at(2 * u - 1), &C = at(2 * u);
                const int np = (hi - lo) * Wo;
                work += (float)(np * (D.Ci / 4)) / (float)NT + 0.25f * (float)((np + 15) / 16 * (C.Co / CB) * (C.Ci / CB)) / (float)NW;
                const int in_lo = lo * D.stride - D.pt, in_hi = (hi - 1) * D.stride - D.pt + 3;
                lo = std::max(in_lo, 0);
                hi = std::min(in_hi, D.H);
            }
            ranges.insert(ranges.end(), band.begin(), band.end());
            m->band_work[(size_t)rb] = std::max(m->band_work[(size_t)rb], work);
        }
    }
    return true;
}

// Rows per band for this batch (all rows: whole images): as many bands as compute units take at once, where they pay.
// DS-CNN (25 rows; us of a launch), general kernel / whole images here / bands: batch 1 26.9 / 25.6 / 15.6 (1 row), 16 27.4 / 25.9 / 17.9 (2),
// 41 27.4 / 26.1 / 19.6 (5), 85 27.6 / 26.2 / 22.1 (9), 128 27.7 / 26.3 / 23.9 (13), 256 27.8 / 26.4; a second round of bands costs more than it
// gives (batch 100 in three bands: 34.2).
int rows_per_band(const small_hip_fmodel *m, int batch)
{
    static const int force = tune_int("fmodel_band", -1);
    if (batch > m->band_batch || force == 0) return m->rows;
    const int most = NUM_CU / batch;                 // bands, two at least: band_batch
    const int rows = std::min(force > 0 ? force : (m->rows + most - 1) / most, m->rows);
    if (m->ranges_first[(size_t)rows] < 0) return m->rows;
    const float saved = m->band_work[(size_t)m->rows] - m->band_work[(size_t)rows];
    return force > 0 || bands_pay(saved, batch, (m->rows + rows - 1) / rows) ? rows : m->rows;
}

// The stream's slot; none (-1) for a stream that is being captured (a graph may be replayed on any stream, at the same time as other
// launches) and for the per-thread default stream, whose handle stands for several streams.
int band_slot(const small_hip_fmodel *m, hipStream_t s, bool take)
{
    if (s == hipStreamPerThread) return -1;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) { (void)hipGetLastError(); return -1; }
    return st == hipStreamCaptureStatusNone ? m->slot(s, take) : -1;
}

} // namespace

extern "C" {

int small_hip_fmodel_create(int n_layers, const small_hip_flayer *layers, small_hip_fmodel **model,
                            small_hip_stream_t stream)
{
    const char *op = "small_hip_fmodel_create";
    if (!model) return einval("small_hip_fmodel_create: null result pointer");
    *model = nullptr;
    if (n_layers <= 0 || n_layers > MAX_LAYERS || !layers)
    { set_error("%s: 1..%d layers", op, MAX_LAYERS); return SMALL_HIP_EINVAL; }
    small_hip_fmodel *m = new (std::nothrow) small_hip_fmodel();
    if (!m) return SMALL_HIP_ENOMEM;
    std::memset(&m->hdr, 0, sizeof(m->hdr));
    FMHeader &h = m->hdr;
    auto fail = [&](int rc) { delete m; return rc; };
    std::vector<FMLayer> tmp((size_t)n_layers);          // one record per layer as given; fused pairs are formed below
    std::memset(tmp.data(), 0, sizeof(FMLayer) * (size_t)n_layers);

    int written_by[MAX_TENSORS];
    for (int t = 0; t < MAX_TENSORS; ++t) written_by[t] = -1;
    int blob_floats = 0, max_blob = 0;
    bool any_pool = false;
    std::vector<int> w_floats((size_t)n_layers, 0);
    for (int i = 0; i < n_layers; ++i)
    {
        const small_hip_flayer &l = layers[i];
        FMLayer &L = tmp[(size_t)i];
        const bool pool = l.kind == SMALL_HIP_FL_GLOBAL_AVGPOOL || l.kind == SMALL_HIP_FL_GLOBAL_MAXPOOL;
        if (l.kind != SMALL_HIP_FL_CONV && l.kind != SMALL_HIP_FL_DWCONV && !pool)
        { set_error("%s: layer %d: unknown kind", op, i); return fail(SMALL_HIP_EINVAL); }
        const int Ci = l.input_channels, H = l.input_height, W = l.input_width;
        if (H <= 0 || W <= 0 || Ci <= 0 || H > 4096 || W > 4096) { set_error("%s: layer %d: bad size", op, i); return fail(SMALL_HIP_EINVAL); }
        const bool from_input = l.src == SMALL_HIP_QM_INPUT;
        if (from_input != (i == 0)) { set_error("%s: exactly the first layer reads the model input", op); return fail(SMALL_HIP_EINVAL); }
        if (!from_input && (l.src < 0 || l.src >= MAX_TENSORS || written_by[l.src] < 0))
        { set_error("%s: layer %d reads a tensor that no earlier layer wrote", op, i); return fail(SMALL_HIP_EINVAL); }
        if (l.dst != SMALL_HIP_QM_OUTPUT && (l.dst < 0 || l.dst >= MAX_TENSORS || l.dst == l.src))
        { set_error("%s: layer %d: bad destination tensor", op, i); return fail(SMALL_HIP_EINVAL); }
        if ((l.dst == SMALL_HIP_QM_OUTPUT) != (i == n_layers - 1))
        { set_error("%s: exactly the last layer writes the model output", op); return fail(SMALL_HIP_EINVAL); }
        if (!from_input)
        {
            const FMLayer &S = tmp[(size_t)written_by[l.src]];
            if (S.Ho != H || S.Wo != W || S.Co != Ci)
            { set_error("%s: layer %d: input shape differs from what layer %d produces", op, i, written_by[l.src]); return fail(SMALL_HIP_EINVAL); }
        }
        L.Ci = Ci; L.H = H; L.W = W;
        L.nscale = 1.f;
        if (pool)
        {
            if (Ci % CB != 0 || Ci / 4 > NT) { set_error("%s: layer %d: pooling over %d channels", op, i, Ci); return fail(SMALL_HIP_EUNSUPPORTED); }
            if (l.kernel_height != H || l.kernel_width != W || l.t_pad || l.b_pad || l.l_pad || l.r_pad || from_input ||
                l.act != SMALL_HIP_ACT_NONE)
            { set_error("%s: layer %d: only whole-image pooling without padding or activation, after another layer", op, i); return fail(SMALL_HIP_EUNSUPPORTED); }
            L.kind = l.kind == SMALL_HIP_FL_GLOBAL_AVGPOOL ? K_POOL_AVG : K_POOL_MAX;
            L.Co = Ci; L.Ho = 1; L.Wo = 1; L.kh = H; L.kw = W; L.stride = 1;
            L.norm = (float)(1.0 / ((double)H * W));
            any_pool = true;
        }
        else
        {
            const int kh = l.kernel_height, kw = l.kernel_width, s = l.stride;
            const bool dw = l.kind == SMALL_HIP_FL_DWCONV;
            const int Co = dw ? Ci : l.output_channels;
            const bool stem = !dw && Ci < CB;
            if (stem ? !(Ci >= 1 && Ci <= 3) : Ci % CB != 0) { set_error("%s: layer %d: %d input channels", op, i, Ci); return fail(SMALL_HIP_EUNSUPPORTED); }
            if (stem && !from_input) { set_error("%s: layer %d: 1..3 input channels only on the model input", op, i); return fail(SMALL_HIP_EUNSUPPORTED); }
            if (dw && from_input) { set_error("%s: layer %d: the first layer must be a convolution", op, i); return fail(SMALL_HIP_EUNSUPPORTED); }
            if (s != 1 && s != 2) { set_error("%s: layer %d: stride %d", op, i, s); return fail(SMALL_HIP_EUNSUPPORTED); }
            if (kh <= 0 || kw <= 0 || kh > 255 || kw > 255 || Co <= 0 || Co % CB != 0 || !l.filter || !aligned16(l.filter) ||
                (l.bias && !aligned16(l.bias)) || !pads_ok(l.t_pad, l.b_pad, l.l_pad, l.r_pad))
            { set_error("%s: layer %d: bad convolution arguments", op, i); return fail(SMALL_HIP_EINVAL); }
            if (l.act < SMALL_HIP_ACT_NONE || l.act > SMALL_HIP_ACT_LEAKY) { set_error("%s: layer %d: bad activation", op, i); return fail(SMALL_HIP_EINVAL); }
            const int Ho = out_dim(H, l.t_pad, l.b_pad, kh, s), Wo = out_dim(W, l.l_pad, l.r_pad, kw, s);
            if (Ho <= 0 || Wo <= 0) { set_error("%s: layer %d: empty output", op, i); return fail(SMALL_HIP_EINVAL); }
            L.kind = dw ? K_DW : stem ? K_STEM : K_CONV;
            L.Co = Co; L.Ho = Ho; L.Wo = Wo; L.kh = kh; L.kw = kw; L.stride = s; L.pt = l.t_pad; L.pl = l.l_pad;
            L.nscale = l.act == SMALL_HIP_ACT_RELU ? 0.f : l.act == SMALL_HIP_ACT_LEAKY ? l.slope : 1.f;
            const long taps = (long)kh * kw;
            long wf;
            if (dw) wf = (long)Ci * taps;
            else if (stem)
            {
                L.K = (int)(taps * Ci);
                L.chunks = (L.K + 15) / 16;
                wf = (long)Co * L.chunks * 16;
            }
            else wf = (long)Co * Ci * taps;
            long bf = wf + Co + (stem ? L.chunks * 16 : 0);
            bf = (bf + 3) & ~3L;
            if (bf > (long)NPRE * NT * 4) { set_error("%s: layer %d: more than %d KB of weights", op, i, NPRE * NT * 16 / 1024); return fail(SMALL_HIP_EUNSUPPORTED); }
            w_floats[(size_t)i] = (int)wf;
            L.bias_off = (int)wf;
            L.ktab_off = (int)wf + Co;
            L.blob_off = blob_floats;
            L.blob16 = (int)(bf >> 2);
            blob_floats += (int)bf;
        }
        L.r_wo = 1.0f / (float)L.Wo;
        L.r_cob = 1.0f / (float)(L.Co / CB);
        L.r_p = 1.0f / (float)(L.Ho * L.Wo);
        if ((long)L.Co * L.Ho * L.Wo > LDS_LIMIT / 4)
        { set_error("%s: layer %d: output tensor larger than LDS", op, i); return fail(SMALL_HIP_EUNSUPPORTED); }
        if (l.dst >= 0) written_by[l.dst] = i;
    }

    static const bool sep_off = tune_int("fmodel_sep", 1) == 0;
    std::vector<SepPair> pairs;
    std::vector<int> ranges;
    m->separable = !sep_off && plan_separable(layers, tmp, m, pairs, ranges);

    // The launch's layer list.  A 3x3 depthwise convolution whose only reader is the 1x1 stride-1 convolution right
    // after it becomes one layer with it (their weights already lie back to back in the blob); the depthwise tensor
    // then needs no LDS.  SMALL_HIP_TUNE key fmodel_fuse=0 keeps the layers apart (a measurement aid).
    static const bool fuse_off = tune_int("fmodel_fuse", 1) == 0;
    int tensor_floats[MAX_TENSORS] = {};
    int dev_src[MAX_LAYERS], dev_dst[MAX_LAYERS], n_dev = 0;
    // where a caller's tensor id lives: a fused pair must not write the tensor it reads (callers ping-pong between two
    // ids, so the 1x1 convolution's destination usually IS the depthwise input, whose neighbouring pixels other waves
    // still read); its result then goes to the tensor the depthwise result would have had, and the two ids trade places
    int phys[MAX_TENSORS];
    for (int t = 0; t < MAX_TENSORS; ++t) phys[t] = t;
    for (int i = 0; i < n_layers; ++i)
    {
        FMLayer L = tmp[(size_t)i];
        const int lsrc = layers[i].src, ldst = layers[i].dst;
        int src = lsrc >= 0 ? phys[lsrc] : lsrc, dst = ldst >= 0 ? phys[ldst] : ldst;
        if (!fuse_off && L.kind == K_DW && L.kh == 3 && L.kw == 3 && i + 1 < n_layers)
        {
            const FMLayer &N = tmp[(size_t)i + 1];
            bool ok = N.kind == K_CONV && N.kh == 1 && N.kw == 1 && N.stride == 1 && N.Ho == N.H && N.Wo == N.W &&
                      layers[i + 1].src == ldst && L.blob16 + N.blob16 <= NPRE * NT;
            for (int j = i + 2; ok && j < n_layers; ++j)      // nobody else reads the depthwise result
            {
                if (layers[j].src == ldst) ok = false;
                if (layers[j].dst == ldst) break;
            }
            if (ok)
            {
                L.kind = K_DWPW;
                L.Co2 = N.Co;
                L.w2_off = N.blob_off - L.blob_off;
                L.bias2_off = L.w2_off + N.bias_off;
                L.nscale2 = N.nscale;
                L.r_cob2 = 1.0f / (float)(N.Co / CB);
                L.blob16 += N.blob16;
                const int odst = layers[i + 1].dst;
                if (odst >= 0 && phys[odst] == src)
                {
                    const int free_id = phys[ldst];
                    phys[ldst] = phys[odst];
                    phys[odst] = free_id;
                }
                dst = odst >= 0 ? phys[odst] : odst;
                ++i;
            }
        }
        if (dst >= 0 && dst == src) { set_error("%s: layer %d writes the tensor it reads", op, i); return fail(SMALL_HIP_EINVAL); }
        h.layer[n_dev] = L;
        dev_src[n_dev] = src; dev_dst[n_dev] = dst;
        max_blob = L.blob16 * 4 > max_blob ? L.blob16 * 4 : max_blob;
        if (dst >= 0)
        {
            const int Co = L.kind == K_DWPW ? L.Co2 : L.Co;
            const int fl = Co * L.Ho * L.Wo;
            tensor_floats[dst] = fl > tensor_floats[dst] ? fl : tensor_floats[dst];
        }
        ++n_dev;
    }
    h.n_layers = n_dev;
    for (int i = 0; i + 1 < n_dev; ++i)
    {
        h.layer[i].next_blob_off = h.layer[i + 1].blob_off;
        h.layer[i].next_blob16 = h.layer[i + 1].blob16;
    }

    // LDS plan (floats): [weights x2][pooling partials][input][tensors]
    int off = 0;
    h.w_lds = off; h.w_floats = max_blob; off += 2 * max_blob;
    h.pool_off = off; off += any_pool ? NT * 4 + NT / 2 * 4 : 0;
    h.zero_off = off; off += 4;
    const small_hip_flayer &l0 = layers[0];
    h.in_C = l0.input_channels; h.in_H = l0.input_height; h.in_W = l0.input_width;
    h.in_elems = h.in_C * h.in_H * h.in_W;
    h.in_off = off; off += align_up(h.in_elems, 4);
    int tensor_off[MAX_TENSORS];
    for (int t = 0; t < MAX_TENSORS; ++t) { tensor_off[t] = off; off += tensor_floats[t]; }
    if (!m->separable) h.lds_bytes = off * 4;
    if ((long)off * 4 > LDS_LIMIT)
    {
        set_error("%s: the model needs %ld bytes of LDS (activations %ld, weights of two layers %d), the limit is %d: run it "
                  "layer by layer", op, (long)off * 4, (long)(off - h.in_off) * 4, 2 * max_blob * 4, LDS_LIMIT);
        return fail(SMALL_HIP_EUNSUPPORTED);
    }
    for (int i = 0; i < n_dev; ++i)
    {
        FMLayer &L = h.layer[i];
        L.src_off = i == 0 ? h.in_off : tensor_off[dev_src[i]];
        L.dst_off = dev_dst[i] >= 0 ? tensor_off[dev_dst[i]] : -1;
    }
    const FMLayer &last = tmp[(size_t)n_layers - 1];
    h.out_elems = last.Co * last.Ho * last.Wo;

    hipStream_t s = as_stream(stream);
    hipError_t e = hipGetDevice(&m->device);
    if (e != hipSuccess) return fail(fail_hip(e, "hipGetDevice"));
    // what precedes the weights, uploaded in one piece
    auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
    m->ranges_off = up256(pairs.size() * sizeof(SepPair));
    m->blob_off = m->separable ? m->ranges_off + up256(ranges.size() * sizeof(int)) : up256(sizeof(FMHeader));
    std::vector<unsigned char> head(m->blob_off);
    if (m->separable)
    {
        std::memcpy(head.data(), pairs.data(), pairs.size() * sizeof(SepPair));
        std::memcpy(head.data() + m->ranges_off, ranges.data(), ranges.size() * sizeof(int));
    }
    else std::memcpy(head.data(), &m->hdr, sizeof(FMHeader));
    // the weights, and behind them the bands' slots (without memory for those the model runs on whole images)
    const size_t own_bytes = up256(m->blob_off + (size_t)blob_floats * 4 + 256);
    size_t slot_bytes = 0, counter_bytes = 0;
    if (m->separable && m->rows > 1)
    {
        const size_t per_image = (size_t)m->sep.last_elems * 4, fit = small_hip_fmodel::SLOT_BYTES / per_image;
        m->band_batch = (int)std::min<size_t>(fit, NUM_CU / 2);
        while (m->band_batch > 0 && rows_per_band(m, m->band_batch) == m->rows) --m->band_batch;      // the largest batch whose bands pay
        m->slot_bytes = up256(m->band_batch * per_image);
        slot_bytes = m->slot_bytes * small_hip_fmodel::SLOTS;
        counter_bytes = (size_t)m->band_batch * small_hip_fmodel::SLOTS * sizeof(unsigned);
    }
    e = hipMalloc(&m->dev, own_bytes + slot_bytes + counter_bytes);
    if (e == hipErrorOutOfMemory && slot_bytes > 0)
    {
        (void)hipGetLastError();
        m->band_batch = 0;
        e = hipMalloc(&m->dev, own_bytes);
    }
    if (e != hipSuccess)
    {
        (void)hipGetLastError();
        set_error("%s: hipMalloc: %s", op, hipGetErrorString(e));
        return fail(e == hipErrorOutOfMemory ? SMALL_HIP_ENOMEM : SMALL_HIP_EHIP);
    }
    auto fail_dev = [&](int rc) { (void)hipFree(m->dev); return fail(rc); };
    if (m->band_batch > 0)
    {
        m->slots = static_cast<unsigned char *>(m->dev) + own_bytes;
        m->counters = reinterpret_cast<unsigned *>(m->slots + slot_bytes);
        e = hipMemsetAsync(m->counters, 0, counter_bytes, s);
        if (e != hipSuccess) return fail_dev(fail_hip(e, "small_hip_fmodel_create: counters"));
    }
    float *dblob = reinterpret_cast<float *>(static_cast<uint8_t *>(m->dev) + m->blob_off);
    std::vector<std::vector<int>> ktabs((size_t)n_layers);          // alive until the stream has been waited for
    for (int i = 0; i < n_layers; ++i)
    {
        const FMLayer &L = tmp[(size_t)i];
        if (L.kind != K_CONV && L.kind != K_STEM && L.kind != K_DW) continue;
        const int wf = w_floats[(size_t)i];
        const int nthreads = wf > L.Co ? wf : L.Co;
        hipLaunchKernelGGL(fm_prep_kernel, dim3((unsigned)((nthreads + 255) / 256)), dim3(256), 0, s, L.kind, layers[i].filter,
                           layers[i].bias, dblob + L.blob_off, L.Co, L.Ci, L.kh * L.kw, L.K, L.chunks, wf);
        e = hipGetLastError();
        if (e != hipSuccess) return fail_dev(fail_hip(e, "small_hip_fmodel_create: pre-pass"));
        if (L.kind == K_STEM)
        {
            std::vector<int> &kt = ktabs[(size_t)i];
            // entry [chunk][kq][j] describes reduction element k = 16 chunk + 4 j + kq
            kt.assign((size_t)L.chunks * 16, -1);
            for (int k = 0; k < L.K; ++k)
            {
                const int tap = k / L.Ci, ci = k - tap * L.Ci, a = tap / L.kw, b = tap - a * L.kw;
                const int chunk = k / 16, j = (k % 16) / 4, kq = k % 4;
                kt[(size_t)((chunk * 4 + kq) * 4 + j)] = m->separable ? a * m->sep.img_row + b * L.Ci + ci : a | (b << 8) | (ci << 16);
            }
            e = hipMemcpyAsync(dblob + L.blob_off + L.ktab_off, kt.data(), kt.size() * sizeof(int), hipMemcpyHostToDevice, s);
            if (e != hipSuccess) return fail_dev(fail_hip(e, "small_hip_fmodel_create: tables"));
        }
    }
    e = hipMemcpyAsync(m->dev, head.data(), head.size(), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);       // the caller's filters and the host-side tables may go
    if (e != hipSuccess) return fail_dev(fail_hip(e, "small_hip_fmodel_create: upload"));
    e = hipFuncSetAttribute(m->separable ? reinterpret_cast<const void *>(fmodel_f32_sep_kernel) : reinterpret_cast<const void *>(fmodel_f32_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS_LIMIT);
    if (e != hipSuccess) return fail_dev(fail_hip(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)"));
    *model = m;
    return SMALL_HIP_OK;
}

int small_hip_fmodel_forward(const small_hip_fmodel *model, int batch, const float *input, float *output,
                             small_hip_stream_t stream)
{
    if (!model || !model->dev) return einval("small_hip_fmodel_forward: null model");
    if (batch < 0 || !input || !output) return einval("small_hip_fmodel_forward: bad argument");
    if (batch == 0) return SMALL_HIP_OK;
    if (!aligned16(output) || (model->hdr.in_C >= CB && !aligned16(input)))
        return einval("small_hip_fmodel_forward: misaligned pointer");
    const unsigned char *dev = static_cast<const unsigned char *>(model->dev);
    const float *dblob = reinterpret_cast<const float *>(dev + model->blob_off);
    if (model->separable)
    {
        int rows = rows_per_band(model, batch), slot = 0;
        if (rows < model->rows && (slot = band_slot(model, as_stream(stream), true)) < 0) rows = model->rows;
        const int bands = (model->rows + rows - 1) / rows;
        hipLaunchKernelGGL(fmodel_f32_sep_kernel, dim3((unsigned)batch * bands), dim3(NT), (size_t)model->hdr.lds_bytes, as_stream(stream),
                           model->sep, reinterpret_cast<const SepPair *>(dev), dblob, input, output,
                           reinterpret_cast<const int2 *>(dev + model->ranges_off) + model->ranges_first[(size_t)rows], bands,
                           bands > 1 ? reinterpret_cast<float *>(model->slots + slot * model->slot_bytes) : nullptr,
                           bands > 1 ? model->counters + slot * model->band_batch : nullptr);
        SHP_LAUNCH_CHECK("small_hip_fmodel_forward");
        return SMALL_HIP_OK;
    }
    hipLaunchKernelGGL(fmodel_f32_kernel, dim3((unsigned)batch), dim3(NT), (size_t)model->hdr.lds_bytes, as_stream(stream),
                       static_cast<const FMHeader *>(model->dev), dblob, input, output);
    SHP_LAUNCH_CHECK("small_hip_fmodel_forward");
    return SMALL_HIP_OK;
}

size_t small_hip_fmodel_output_elems(const small_hip_fmodel *model) { return model ? (size_t)model->hdr.out_elems : 0; }
int small_hip_fmodel_bands(const small_hip_fmodel *model, int batch, small_hip_stream_t stream)
{
    if (!model || batch <= 0) return 0;
    if (!model->separable) return 1;
    const int rows = rows_per_band(model, batch);
    return rows < model->rows && band_slot(model, as_stream(stream), false) >= 0 ? (model->rows + rows - 1) / rows : 1;
}

size_t small_hip_fmodel_lds_bytes(const small_hip_fmodel *model) { return model ? (size_t)model->hdr.lds_bytes : 0; }

int small_hip_fmodel_destroy(small_hip_fmodel *model)
{
    if (!model) return SMALL_HIP_OK;
    int rc = SMALL_HIP_OK;
    if (model->dev)
    {
        hipError_t e = hipFree(model->dev);
        if (e != hipSuccess) rc = fail_hip(e, "small_hip_fmodel_destroy: hipFree");
    }
    delete model;
    return rc;
}

} // extern "C"
