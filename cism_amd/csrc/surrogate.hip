// surrogate.hip -- learned initial guess for the velocity solve (no reference
// counterpart): a fully convolutional 4-level encoder-decoder (~1.0M
// parameters) mapping 2D ice-sheet fields on the vertex grid to u, v at every
// level plus a per-column preconditioner scale, with hand-written forward and
// backward kernels and Adam.
//
// Precision: FP32 master weights and activations; every convolution runs as an
// implicit GEMM on gfx950's MFMA (v_mfma_f32_16x16x32_bf16) with BF16 operands and FP32
// accumulation.  Activations are NHWC (channels fastest); 3x3 convolutions use
// periodic (circular) padding, matching the periodic grids of the solver.
//
//   enc0  3x3 16->32, 32->32          (H x W; 5 input channels zero-padded to 16)
//   enc1  pool, 3x3 32->64, 64->64    (H/2)
//   enc2  pool, 3x3 64->128, 128->128 (H/4)
//   mid   pool, 3x3 128->128 x2       (H/8)
//   dec2  up, cat enc2, 3x3 256->128
//   dec1  up, cat enc1, 3x3 192->64
//   dec0  up, cat enc0, 3x3 96->32
//   head  1x1 32->32 (24 used: u, v at nz<=11 levels and two log-scales)
// ReLU after every convolution except the head.
#include "internal.h"

#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline short f2bf(float f) {
    // round to nearest even
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}

#define SG_IN_RAW 5
#define SG_IN 16
#define SG_OUT 24
#define SG_OUT_PAD 32

// ---------------------------------------------------------------------------
// implicit-GEMM convolution: out[p][co] = act(bias[co] + sum_k W[co][k] * X(p, k))
// k = tap*Ci + ci, tap = ky*3 + kx (ks = 3) or 0 (ks = 1); X(p, k) = in at pixel p
// shifted by (ky-1, kx-1) with periodic wrap.  Ci is a multiple of 16, Co of 32.
// ---------------------------------------------------------------------------
struct ConvDims {
    int B, H, W, Ci, Co, ks, relu;
};

// A convolution's input: one image a of Ca channels, or (b not null) the decoder's
// concatenation, read in place: channels [0, Ca) from a at half the resolution (nearest
// upsampling), the Cb after them from b.  Ca and Cb are multiples of 8 (of 32 with b).
struct ConvSrc {
    const float *a, *b;
    int Ca, Cb;
};

// Images are worked on in patches of 8 x 8 output pixels.
#define CONV_P 8

// 8 channels from c of pixel (y, x) of image n (y, x inside the image) as BF16
__device__ __forceinline__ const float *conv_src_at(const ConvDims &d, const ConvSrc &s, int n, int y, int x, int c) {
    if (!s.b) return s.a + (((long long)n * d.H + y) * d.W + x) * s.Ca + c;
    if (c < s.Ca) return s.a + (((long long)n * (d.H >> 1) + (y >> 1)) * (d.W >> 1) + (x >> 1)) * s.Ca + c;
    return s.b + (((long long)n * d.H + y) * d.W + x) * s.Cb + (c - s.Ca);
}

__device__ __forceinline__ uint4 pack_bf16(const float4 &f, const float4 &h) {
    auto two = [](float lo, float hi) {
        return (unsigned)(unsigned short)f2bf(lo) | ((unsigned)(unsigned short)f2bf(hi) << 16);
    };
    return make_uint4(two(f.x, f.y), two(f.z, f.w), two(h.x, h.y), two(h.z, h.w));
}

// source of patch pixel (ly, lx) of a patch with a halo of `off` pixels whose first output
// pixel is (y0, x0): the wrapped coordinates, or false for a pixel no output needs
__device__ __forceinline__ bool patch_pixel(const ConvDims &d, int off, int y0, int x0, int ly, int lx, int &y,
                                            int &x) {
    y = y0 + ly - off;
    x = x0 + lx - off;
    if (y >= d.H + off || x >= d.W + off) return false;
    y = y < 0 ? y + d.H : (y >= d.H ? y - d.H : y);
    x = x < 0 ? x + d.W : (x >= d.W ? x - d.W : x);
    return true;
}

// One workgroup: 32 NA output channels of one patch; wave (w >> 1, w & 1) takes 16 NA of the
// channels and 32 of the pixels (4 patch rows), NA x 2 MFMA tiles.  The patch with its halo is
// staged once, as BF16, all Ci channels of a pixel together: each input value is loaded and
// converted once per workgroup instead of once per tap, and every tap's operand is the same
// rows of LDS at another pixel offset.  The row stride Ci + 8 puts the 16-byte reads of eight
// neighbouring pixels on disjoint banks for every Ci here.  The weights come from L2 in the
// order the MFMA reads them (Wf[co / 16][k / 32][lane][8], k_prep_weights): 1 KB contiguous
// per fragment.  k ascends in steps of 32 from one accumulator, zeros past K (3x3 over 16
// channels: 144), so an output does not depend on the tiling.
// Lane l of an MFMA holds row (l & 15) of A and column (l & 15) of B with 8 consecutive
// k from 8 (l >> 4); its 4 results are rows 4 (l >> 4) + i of column (l & 15).
// mask (the data gradient of an input that went through a ReLU): zero where mask is not
// positive.
// Bound: the MFMA operands' L1 and LDS reads (2 + 2 KB per 4 MFMAs of a wave) at the deep
// levels, the FP32 activations' traffic at the full resolution.  The weights of four steps
// are loaded ahead of the four being multiplied: waiting for each step's from L2 cost 6 to
// 20% of a layer.  The twelve layers at 512 x 512: 0.64 ms with every tap loaded and converted
// again and the concatenations written out, 0.29 ms with the patches and each step's weights
// loaded as they were needed, 0.25 ms here.
template <int NA>
__global__ __launch_bounds__(256) void k_conv_patch(ConvDims d, ConvSrc src, const short *__restrict__ Wf,
                                                    const float *__restrict__ bias, const float *__restrict__ mask,
                                                    float *__restrict__ out) {
    extern __shared__ __align__(16) short X[];   // [pixel][Ci + 8]
    const int ld = d.Ci + 8, off = d.ks == 3 ? 1 : 0, R = CONV_P + 2 * off, G = d.Ci >> 3;
    const int tw = (d.W + CONV_P - 1) / CONV_P, th = (d.H + CONV_P - 1) / CONV_P;
    const int n = blockIdx.x / (tw * th), pt = blockIdx.x - n * (tw * th);
    const int y0 = pt / tw * CONV_P, x0 = (pt - pt / tw * tw) * CONV_P;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int items = R * R * G;   // 8 channels of a pixel each
    for (int i0 = t; i0 < items; i0 += 4 * 256) {
        float4 v[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int it = i0 + u * 256, px = it / G, ly = px / R;
            int y, x;
            v[u][0] = v[u][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (it < items && patch_pixel(d, off, y0, x0, ly, px - ly * R, y, x)) {
                const float4 *p = reinterpret_cast<const float4 *>(conv_src_at(d, src, n, y, x, (it - px * G) * 8));
                v[u][0] = p[0];
                v[u][1] = p[1];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int it = i0 + u * 256, px = it / G;
            if (it < items) *reinterpret_cast<uint4 *>(&X[px * ld + (it - px * G) * 8]) = pack_bf16(v[u][0], v[u][1]);
        }
    }
    __syncthreads();
    const int K = d.ks * d.ks * d.Ci, S = (K + 31) >> 5;
    const int co0 = blockIdx.y * 32 * NA + (wave >> 1) * 16 * NA, row0 = (wave & 1) * 4;
    f32x4 acc[NA][2];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const bf16x8 *wf = reinterpret_cast<const bf16x8 *>(Wf) + (long long)(co0 >> 4) * S * 64 + lane;
    // this lane's pixel of the two B tiles, and its k within the step as (tap, channel)
    const int c15 = lane & 15;
    const short *xb0 = X + ((row0 + (c15 >> 3)) * R + (c15 & 7)) * ld;
    const short *xb1 = xb0 + 2 * R * ld;
    int tap = 0, ci = 8 * (lane >> 4);
    if (ci >= d.Ci) {   // Ci = 16: the step's second half is the next tap
        ci -= d.Ci;
        tap = 1;
    }
    // four steps' weights at a time, the next four on their way while these are multiplied
    bf16x8 w0[4][NA], w1[4][NA];
    auto weights = [&](bf16x8(&w)[4][NA], int s0) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s0 + u < S)
#pragma unroll
                for (int a = 0; a < NA; ++a) w[u][a] = wf[((long long)a * S + s0 + u) * 64];
    };
    auto multiply = [&](const bf16x8(&w)[4][NA], int s0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (s0 + u >= S) break;
            bf16x8 b0 = {}, b1 = {};
            if (tap < d.ks * d.ks) {
                const int ky = tap / 3, o = (ky * R + tap - 3 * ky) * ld + ci;
                b0 = *reinterpret_cast<const bf16x8 *>(xb0 + o);
                b1 = *reinterpret_cast<const bf16x8 *>(xb1 + o);
            }
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                acc[a][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][a], b0, acc[a][0], 0, 0, 0);
                acc[a][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][a], b1, acc[a][1], 0, 0, 0);
            }
            ci += 32;
            if (ci >= d.Ci) {   // the next tap, or the one after it (16 channels)
                const int over = d.Ci == 16 ? 2 : 1;
                ci -= over * d.Ci;
                tap += over;
            }
        }
    };
    weights(w0, 0);
    for (int s = 0; s < S; s += 8) {
        weights(w1, s + 4);
        multiply(w0, s);
        weights(w0, s + 8);
        multiply(w1, s + 4);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int y = y0 + row0 + 2 * b + (c15 >> 3), x = x0 + (c15 & 7);
        if (y >= d.H || x >= d.W) continue;
        const long long p = ((long long)n * d.H + y) * d.W + x;
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const int oc = co0 + 16 * a + 4 * (lane >> 4);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[a][b][i] + (bias ? bias[oc + i] : 0.f);
                if (d.relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
            }
            if (mask) {
                const float4 m = *reinterpret_cast<const float4 *>(mask + p * d.Co + oc);
                v[0] = m.x > 0.f ? v[0] : 0.f;
                v[1] = m.y > 0.f ? v[1] : 0.f;
                v[2] = m.z > 0.f ? v[2] : 0.f;
                v[3] = m.w > 0.f ? v[3] : 0.f;
            }
            *reinterpret_cast<float4 *>(out + p * d.Co + oc) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

// Weight and bias gradients: dW[co][k] = sum_p dY[p][co] * X(p, k), db[co] = sum_p dY[p][co].
// One workgroup: 32 output x 32 input channels, every tap, over a run of patches; wave
// (w >> 1, w & 1) has 16 x 16 of them, KS * KS MFMA tiles.  The contraction runs over pixels,
// which neither operand has contiguous: both patches are staged [pixel][channel] as BF16
// and gfx950's transposing LDS reads (ds_read_b64_tr_b16: 16 lanes read 4 pixels x 16
// channels, each lane receives one channel of the 4 pixels) give the MFMA's 8 consecutive
// pixels of a channel in two reads.  A k step of 32 is 4 patch rows.  dY is staged once for
// the nine taps, and the next patch is loaded while this one is multiplied.  The bias
// gradient adds the loader's FP32 values of dY (the workgroups of the first 32 input
// channels).  Partials per run, part[run][Co * K weights, then Co biases], are added by
// k_wgrad_reduce in a fixed order.  A patch's staging (FP32 loads and conversions) bounds it
// at 32 x 32 channels.  The twelve layers at 4 x 256 x 256, with the reductions: 4.9 ms with
// dY and X staged transposed once per tap and a pass per channel for the biases, 0.35 ms here.
#define WG_LD 48   // staged channels of a pixel: 32 and a pad that keeps 4 pixels on disjoint banks
template <int KS>
__global__ __launch_bounds__(256) void k_wgrad_patch(ConvDims d, ConvSrc src, const float *__restrict__ dY,
                                                     float *__restrict__ part, int per) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef short s8 __attribute__((ext_vector_type(8)));
    constexpr int OFF = KS == 3 ? 1 : 0, R = CONV_P + 2 * OFF, NX = (R * R * 4 + 255) / 256;
    alignas(16) __shared__ short Ys[CONV_P * CONV_P * WG_LD];
    alignas(16) __shared__ short Xs[R * R * WG_LD];
    const int tw = (d.W + CONV_P - 1) / CONV_P, th = (d.H + CONV_P - 1) / CONV_P, np = d.B * tw * th;
    const int ci0 = blockIdx.x * 32, co0 = blockIdx.y * 32;
    const int q0 = blockIdx.z * per, q1 = min(np, q0 + per);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    float4 vy[2], vx[NX][2];
    float bsum[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) bsum[c] = 0.f;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load = [&](int q) {
        const int n = q / (tw * th), pt = q - n * (tw * th);
        const int y0 = pt / tw * CONV_P, x0 = (pt - pt / tw * tw) * CONV_P;
        {
            const int y = y0 + (t >> 5), x = x0 + ((t >> 2) & 7);
            vy[0] = vy[1] = zero;
            if (y < d.H && x < d.W) {
                const float4 *p = reinterpret_cast<const float4 *>(
                    dY + (((long long)n * d.H + y) * d.W + x) * d.Co + co0 + 8 * (t & 3));
                vy[0] = p[0];
                vy[1] = p[1];
            }
        }
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            const int it = t + 256 * u, px = it >> 2, ly = px / R, c = ci0 + 8 * (it & 3);
            int y, x;
            vx[u][0] = vx[u][1] = zero;
            if (px < R * R && c < d.Ci && patch_pixel(d, OFF, y0, x0, ly, px - ly * R, y, x)) {
                const float4 *p = reinterpret_cast<const float4 *>(conv_src_at(d, src, n, y, x, c));
                vx[u][0] = p[0];
                vx[u][1] = p[1];
            }
        }
    };
    f32x4 acc[KS * KS];
#pragma unroll
    for (int k = 0; k < KS * KS; ++k) acc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int g = lane >> 4, l4 = (lane & 15) >> 2, ch = 4 * (lane & 3);
    // 8 consecutive pixels of one channel: two transposing reads of 4 pixels
    auto frag = [&](const short *p) {
        using lds4 = __attribute__((address_space(3))) s4;
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(p + 4 * WG_LD));
        const s8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(bf16x8, v);
    };
    if (q0 < q1) load(q0);
    for (int q = q0; q < q1; ++q) {
        __syncthreads();   // the last patch's reads are done
        *reinterpret_cast<uint4 *>(&Ys[(t >> 2) * WG_LD + 8 * (t & 3)]) = pack_bf16(vy[0], vy[1]);
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            const int it = t + 256 * u;
            if ((it >> 2) < R * R)
                *reinterpret_cast<uint4 *>(&Xs[(it >> 2) * WG_LD + 8 * (it & 3)]) = pack_bf16(vx[u][0], vx[u][1]);
        }
        bsum[0] += vy[0].x; bsum[1] += vy[0].y; bsum[2] += vy[0].z; bsum[3] += vy[0].w;
        bsum[4] += vy[1].x; bsum[5] += vy[1].y; bsum[6] += vy[1].z; bsum[7] += vy[1].w;
        __syncthreads();
        if (q + 1 < q1) load(q + 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 4 * h + g;
            const bf16x8 af = frag(&Ys[(row * CONV_P + l4) * WG_LD + (wave >> 1) * 16 + ch]);
#pragma unroll
            for (int k = 0; k < KS * KS; ++k) {
                const bf16x8 bf = frag(&Xs[((row + k / KS) * R + l4 + k % KS) * WG_LD + (wave & 1) * 16 + ch]);
                acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, acc[k], 0, 0, 0);
            }
        }
    }
    const long long K = (long long)KS * KS * d.Ci;
    float *pz = part + (long long)blockIdx.z * (d.Co * K + d.Co);
    const int ci = ci0 + (wave & 1) * 16 + (lane & 15);
    if (ci < d.Ci)
#pragma unroll
        for (int k = 0; k < KS * KS; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                pz[(co0 + (wave >> 1) * 16 + 4 * g + i) * K + k * d.Ci + ci] = acc[k][i];
    if (blockIdx.x == 0) {
        // a channel's 64 pixel sums in LDS, added in pixel order by one lane
        __shared__ float bs[CONV_P * CONV_P][33];
#pragma unroll
        for (int c = 0; c < 8; ++c) bs[t >> 2][8 * (t & 3) + c] = bsum[c];
        __syncthreads();
        if (t < 32) {
            float s = 0.f;
            for (int p = 0; p < CONV_P * CONV_P; ++p) s += bs[p][t];
            pz[d.Co * K + co0 + t] = s;
        }
    }
}

// dW[e] = sum over the runs of part[run][e]: 64 entries a workgroup of NW waves, wave w on runs
// 4 w .. 4 w + 3, then 4 NW further on (4 loads in flight a lane), the waves added in order.
// 16 waves where there are many runs of a small layer (512 runs of 9,248 entries).
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_wgrad_reduce(const float *__restrict__ part, int runs, long long n,
                                                          float *__restrict__ dW) {
    __shared__ float red[NW][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long e = (long long)blockIdx.x * 64 + lane;
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    if (e < n)
        for (int z = 4 * w; z < runs; z += 4 * NW)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (z + u < runs) a[u] += part[(long long)(z + u) * n + e];
    red[w][lane] = (a[0] + a[1]) + (a[2] + a[3]);
    __syncthreads();
    if (w == 0 && e < n) {
        float s = red[0][lane];
#pragma unroll
        for (int v = 1; v < NW; ++v) s += red[v][lane];
        dW[e] = s;
    }
}

// 2x2 average pool and nearest 2x upsample, NHWC, with their adjoints
__global__ void k_pool(int B, int H, int W, int C, const float *__restrict__ in, float *__restrict__ out) {
    const long long n = (long long)B * (H / 2) * (W / 2) * C;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int c = (int)(t % C);
    long long r = t / C;
    const int x = (int)(r % (W / 2));
    r /= (W / 2);
    const int y = (int)(r % (H / 2));
    const long long b = r / (H / 2);
    auto at = [&](int yy, int xx) { return in[((b * H + yy) * W + xx) * C + c]; };
    out[t] = 0.25f * (at(2 * y, 2 * x) + at(2 * y, 2 * x + 1) + at(2 * y + 1, 2 * x) + at(2 * y + 1, 2 * x + 1));
}

// gradient of an encoder output that feeds a 2x2 pool and, through the decoder's
// concatenation, channels [Ca, Ca + C) of dcat: the sum of both, zero where the output y
// (a ReLU's) is not positive
__global__ void k_skip_bwd(int B, int H, int W, int C, int Ca, const float *__restrict__ dcat,
                           const float *__restrict__ dpool, const float *__restrict__ y, float *__restrict__ dy) {
    const long long n = (long long)B * H * W * (C / 4);
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int c = (int)(t % (C / 4)) * 4;
    const long long p = t / (C / 4);
    const long long r = p / W;
    const int x = (int)(p - r * W), yy = (int)(r % H);
    const long long b = r / H;
    const float4 a = *reinterpret_cast<const float4 *>(dcat + p * (Ca + C) + Ca + c);
    const float4 q = *reinterpret_cast<const float4 *>(dpool + ((b * (H / 2) + yy / 2) * (W / 2) + x / 2) * C + c);
    const float4 m = *reinterpret_cast<const float4 *>(y + p * C + c);
    float4 o;
    o.x = m.x > 0.f ? a.x + 0.25f * q.x : 0.f;
    o.y = m.y > 0.f ? a.y + 0.25f * q.y : 0.f;
    o.z = m.z > 0.f ? a.z + 0.25f * q.z : 0.f;
    o.w = m.w > 0.f ? a.w + 0.25f * q.w : 0.f;
    *reinterpret_cast<float4 *>(dy + p * C + c) = o;
}

// gradient of the low-resolution input of the decoder's up + concat: the sum over its 4
// children of channels [0, Ca) of dcat, zero where the input y (a ReLU's) is not positive
__global__ void k_up_cat_bwd(int B, int H, int W, int Ca, int Cs, const float *__restrict__ dcat,
                             const float *__restrict__ y, float *__restrict__ da) {
    const int Ct = Ca + Cs, h = H / 2, w = W / 2;
    const long long n = (long long)B * h * w * (Ca / 4);
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int c = (int)(t % (Ca / 4)) * 4;
    const long long p = t / (Ca / 4);
    const long long r = p / w;
    const int x = (int)(p - r * w), yy = (int)(r % h);
    const long long b = r / h;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int dy = 0; dy < 2; ++dy)
        for (int dx = 0; dx < 2; ++dx) {
            const float4 v = *reinterpret_cast<const float4 *>(
                dcat + ((b * H + 2 * yy + dy) * W + 2 * x + dx) * Ct + c);
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
    const float4 m = *reinterpret_cast<const float4 *>(y + p * Ca + c);
    *reinterpret_cast<float4 *>(da + p * Ca + c) = make_float4(m.x > 0.f ? s.x : 0.f, m.y > 0.f ? s.y : 0.f,
                                                               m.z > 0.f ? s.z : 0.f, m.w > 0.f ? s.w : 0.f);
}

// masked mean squared error over the SG_OUT used channels; out has SG_OUT_PAD channels
__global__ __launch_bounds__(256) void k_loss(long long P, int nch, const float *__restrict__ out,
                                              const float *__restrict__ tgt,
                                              const float *__restrict__ mask,
                                              const float *__restrict__ chw,
                                              double *__restrict__ partials) {
    double s = 0.0, m = 0.0;
    // a lane per (pixel, channel) of the targets, so that a wave reads both images in runs
    const long long n = P * SG_OUT, step = (long long)gridDim.x * 256;
    for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < n; t += step) {
        const long long p = t / SG_OUT;
        const int c = (int)(t - p * SG_OUT);
        const float mk = mask[p];
        if (mk == 0.f) continue;
        if (c == 0) m += mk;
        if (c < nch) {
            const double e = (double)out[p * SG_OUT_PAD + c] - tgt[t];
            s += mk * chw[c] * e * e;
        }
    }
    double v[2] = {s, m};
    block_reduce_store<2>(v, partials);
}

__global__ __launch_bounds__(256) void k_loss_final(const double *__restrict__ partials, int nb,
                                                    double *__restrict__ res) {
    double v[2] = {0.0, 0.0};
    for (int b = threadIdx.x; b < nb; b += 256) {
        v[0] += partials[2 * b];
        v[1] += partials[2 * b + 1];
    }
    __shared__ double tot[2];
    block_reduce_store<2>(v, tot, 0);
    __syncthreads();
    if (threadIdx.x == 0) {
        res[0] = tot[1] > 0 ? tot[0] / tot[1] : 0.0;
        res[1] = tot[1];
    }
}

__global__ void k_loss_grad(long long P, int nch, const float *__restrict__ out,
                            const float *__restrict__ tgt, const float *__restrict__ mask,
                            const float *__restrict__ chw, const double *__restrict__ res,
                            float *__restrict__ dout) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P * SG_OUT_PAD) return;
    const long long p = t / SG_OUT_PAD;
    const int c = (int)(t % SG_OUT_PAD);
    const double m = res[1];
    float g = 0.f;
    if (c < nch && m > 0) g = (float)(2.0 * mask[p] * chw[c] * ((double)out[t] - tgt[p * SG_OUT + c]) / m);
    dout[t] = g;
}

// Adam on FP32 masters
__global__ void k_adam(long long n, float *__restrict__ w, const float *__restrict__ g,
                       float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float gg = g[t];
    const float mm = b1 * m[t] + (1.f - b1) * gg;
    const float vv = b2 * v[t] + (1.f - b2) * gg * gg;
    m[t] = mm;
    v[t] = vv;
    w[t] = w[t] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}

// BF16 copies of the weights in the order k_conv_patch reads them, [row / 16][k / 32][lane][8]
// (lane l: row l & 15, k from 8 (l >> 4)), zeros past K: the forward weights W[co][k], and the
// data gradient's W'[ci][k'] (k' = tap'*Co + co, tap' = 8 - tap): dX = conv(dY, W') with the
// flipped kernel, periodic padding making it exact.  One lane per BF16 value of either copy.
__host__ __device__ inline long long frag_size(int rows, int K) { return (long long)rows * ((K + 31) / 32 * 32); }

__global__ void k_prep_weights(int Co, int Ci, int ks, const float *__restrict__ W,
                               short *__restrict__ Wf, short *__restrict__ Wt) {
    const int kk = ks * ks;
    const long long nf = frag_size(Co, kk * Ci), nt = frag_size(Ci, kk * Co);
    long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nf + nt) return;
    const bool fwd = t < nf;
    if (!fwd) t -= nf;
    const int K = fwd ? kk * Ci : kk * Co, S = (K + 31) / 32;
    const int j = (int)(t & 7), lane = (int)(t >> 3) & 63;
    const long long f = t >> 9;
    const int row = (int)(f / S) * 16 + (lane & 15), k = (int)(f % S) * 32 + 8 * (lane >> 4) + j;
    short v = 0;
    if (k < K) {
        if (fwd) {
            v = f2bf(W[(long long)row * K + k]);
        } else {
            const int tap = k / Co, co = k - tap * Co;
            v = f2bf(W[((long long)co * kk + (ks == 3 ? 8 - tap : 0)) * Ci + row]);
        }
    }
    (fwd ? Wf : Wt)[t] = v;
}

// ---------------------------------------------------------------------------
// network container
// ---------------------------------------------------------------------------
struct ConvLayer {
    int ks, Ci, Co, relu;
    long long woff, boff;   // offsets into the parameter vector: the biases follow the weights
    long long nparams() const { return (long long)Co * ks * ks * Ci + Co; }
    short *Wf, *Wt;         // BF16 forward / data-gradient weights, as the MFMA reads them
};

struct Act {
    int H, W, C;
    float *y, *dy;
    long long n(int B) const { return (long long)B * H * W * C; }
};

struct cism_surrogate {
    int B, H, W;
    std::vector<ConvLayer> L;
    long long nparams;
    float *w, *g, *m, *v;   // params, grads, Adam moments
    long long step;
    // activations: 0 in; conv outputs and pool/cat buffers
    std::vector<Act> A;
    float *raw, *tgt, *mask, *chw, *wpart;
    long long wpart_n;
    double *lpart, *lres;
    hipStream_t stream;
    hipEvent_t ev0, ev1;
    float last_forward_ms;   // device time of the last forward pass (kernels only)
    int wprep_ok;            // the BF16 copies Wf, Wt match w (cleared whenever w changes)
};

// activation indices
enum {
    A_IN, A_E0a, A_E0b, A_P0, A_E1a, A_E1b, A_P1, A_E2a, A_E2b, A_P2, A_M0, A_M1, A_C2, A_D2,
    A_C1, A_D1, A_C0, A_D0, A_OUT, A_N
};
// layer indices
enum { L_E0a, L_E0b, L_E1a, L_E1b, L_E2a, L_E2b, L_M0, L_M1, L_D2, L_D1, L_D0, L_HEAD, L_N };

static const int LAYER_IN[L_N] = {A_IN, A_E0a, A_P0, A_E1a, A_P1, A_E2a, A_P2, A_M0, A_C2, A_C1, A_C0, A_D0};
static const int LAYER_OUT[L_N] = {A_E0a, A_E0b, A_E1a, A_E1b, A_E2a, A_E2b, A_M0, A_M1, A_D2, A_D1, A_D0, A_OUT};

// the weight gradient's split of a layer's patches into runs of `per`: about 512 workgroups,
// with at least 4 patches each so that the partials (Co * K floats a run) stay a small part
// of the traffic
static void wgrad_runs(const ConvLayer &c, int B, int H, int W, int &runs, int &per) {
    const int np = B * ((H + CONV_P - 1) / CONV_P) * ((W + CONV_P - 1) / CONV_P);
    const int tiles = ((c.Ci + 31) / 32) * (c.Co / 32);
    int want = (512 + tiles - 1) / tiles;
    if (want > (np + 3) / 4) want = (np + 3) / 4;
    per = (np + want - 1) / want;
    runs = (np + per - 1) / per;
}

static int sg_alloc(float **p, long long n) {
    hipError_t e = hipMalloc(p, sizeof(float) * (n > 0 ? n : 1));
    if (e != hipSuccess) {
        cism_set_error("surrogate allocation failed: %s", hipGetErrorString(e));
        return CISM_ERR_NOMEM;
    }
    // null-stream memset: complete it before anything runs on the non-blocking stream
    HIP_TRY(hipMemset(*p, 0, sizeof(float) * (n > 0 ? n : 1)));
    HIP_TRY(hipDeviceSynchronize());
    return CISM_OK;
}

extern "C" int cism_surrogate_destroy(cism_surrogate *s);

extern "C" int cism_surrogate_create(int H, int W, int batch, int device, cism_surrogate **out) {
    if (!out || H % 8 || W % 8 || H < 8 || W < 8 || batch < 1) {
        cism_set_error("surrogate: H and W must be positive multiples of 8 (got %d x %d)", H, W);
        return CISM_ERR_ARG;
    }
    HIP_TRY(hipSetDevice(device));
    cism_surrogate *s = new cism_surrogate();
    s->B = batch; s->H = H; s->W = W;
    const int spec[L_N][4] = {{3, SG_IN, 32, 1}, {3, 32, 32, 1}, {3, 32, 64, 1}, {3, 64, 64, 1},
                              {3, 64, 128, 1}, {3, 128, 128, 1}, {3, 128, 128, 1}, {3, 128, 128, 1},
                              {3, 256, 128, 1}, {3, 192, 64, 1}, {3, 96, 32, 1}, {1, 32, SG_OUT_PAD, 0}};
    long long off = 0;
    for (int l = 0; l < L_N; ++l) {
        ConvLayer c;
        c.ks = spec[l][0]; c.Ci = spec[l][1]; c.Co = spec[l][2]; c.relu = spec[l][3];
        c.woff = off;
        off += (long long)c.Co * c.ks * c.ks * c.Ci;
        c.boff = off;
        off += c.Co;
        c.Wf = c.Wt = nullptr;
        s->L.push_back(c);
    }
    s->nparams = off;
    const int dims[A_N][3] = {{H, W, SG_IN}, {H, W, 32}, {H, W, 32}, {H / 2, W / 2, 32},
                              {H / 2, W / 2, 64}, {H / 2, W / 2, 64}, {H / 4, W / 4, 64},
                              {H / 4, W / 4, 128}, {H / 4, W / 4, 128}, {H / 8, W / 8, 128},
                              {H / 8, W / 8, 128}, {H / 8, W / 8, 128}, {H / 4, W / 4, 256},
                              {H / 4, W / 4, 128}, {H / 2, W / 2, 192}, {H / 2, W / 2, 64},
                              {H, W, 96}, {H, W, 32}, {H, W, SG_OUT_PAD}};
    int st = CISM_OK;
    for (int a = 0; a < A_N; ++a) {
        Act x;
        x.H = dims[a][0]; x.W = dims[a][1]; x.C = dims[a][2];
        x.y = x.dy = nullptr;
        s->A.push_back(x);
    }
    for (int a = 0; a < A_N && !st; ++a) {
        // the concatenations exist as gradients only: the convolutions read their parts
        const bool cat = a == A_C0 || a == A_C1 || a == A_C2;
        if (!cat) st = sg_alloc(&s->A[a].y, s->A[a].n(batch));
        if (!st) st = sg_alloc(&s->A[a].dy, s->A[a].n(batch));
    }
    for (int l = 0; l < L_N && !st; ++l) {
        const ConvLayer &c = s->L[l];
        if (hipMalloc(&s->L[l].Wf, sizeof(short) * frag_size(c.Co, c.ks * c.ks * c.Ci)) != hipSuccess ||
            hipMalloc(&s->L[l].Wt, sizeof(short) * frag_size(c.Ci, c.ks * c.ks * c.Co)) != hipSuccess)
            st = CISM_ERR_NOMEM;
    }
    if (!st) st = sg_alloc(&s->w, s->nparams);
    if (!st) st = sg_alloc(&s->g, s->nparams);
    if (!st) st = sg_alloc(&s->m, s->nparams);
    if (!st) st = sg_alloc(&s->v, s->nparams);
    const long long P = (long long)batch * H * W;
    if (!st) st = sg_alloc(&s->raw, P * SG_IN_RAW);
    if (!st) st = sg_alloc(&s->tgt, P * SG_OUT);
    if (!st) st = sg_alloc(&s->mask, P);
    if (!st) st = sg_alloc(&s->chw, SG_OUT);
    // weight-gradient partials: the largest layer's runs
    s->wpart_n = 0;
    for (int l = 0; l < L_N; ++l) {
        int runs, per;
        wgrad_runs(s->L[l], batch, s->A[LAYER_OUT[l]].H, s->A[LAYER_OUT[l]].W, runs, per);
        const long long n = (long long)runs * s->L[l].nparams();
        if (n > s->wpart_n) s->wpart_n = n;
    }
    if (!st) st = sg_alloc(&s->wpart, s->wpart_n);
    if (!st && hipMalloc(&s->lpart, sizeof(double) * 2 * 1024) != hipSuccess) st = CISM_ERR_NOMEM;
    if (!st && hipMalloc(&s->lres, sizeof(double) * 2) != hipSuccess) st = CISM_ERR_NOMEM;
    if (!st && hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess) st = CISM_ERR_HIP;
    if (!st && (hipEventCreate(&s->ev0) != hipSuccess || hipEventCreate(&s->ev1) != hipSuccess))
        st = CISM_ERR_HIP;
    if (st) {
        cism_surrogate_destroy(s);
        return st;
    }
    // default initialisation: He-normal from a fixed LCG, zero biases, zero head
    std::vector<float> h(s->nparams, 0.f);
    unsigned long long rs = 0x9E3779B97F4A7C15ull;
    auto unif = [&]() {
        rs = rs * 6364136223846793005ull + 1442695040888963407ull;
        return ((rs >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    for (int l = 0; l < L_N; ++l) {
        const ConvLayer &c = s->L[l];
        const long long nw = (long long)c.Co * c.ks * c.ks * c.Ci;
        const double sd = l == L_HEAD ? 1e-3 : sqrt(2.0 / (c.ks * c.ks * c.Ci));
        for (long long i = 0; i < nw; ++i) {
            const double u1 = unif(), u2 = unif();
            h[c.woff + i] = (float)(sd * sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
        }
    }
    float ones[SG_OUT];
    for (int c = 0; c < SG_OUT; ++c) ones[c] = 1.f;
    HIP_TRY(hipMemcpyAsync(s->chw, ones, sizeof ones, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemcpyAsync(s->w, h.data(), sizeof(float) * s->nparams, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    s->step = 0;
    s->wprep_ok = 0;
    *out = s;
    return CISM_OK;
}

extern "C" int cism_surrogate_destroy(cism_surrogate *s) {
    if (!s) return CISM_OK;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    for (auto &a : s->A) {
        if (a.y) (void)hipFree(a.y);
        if (a.dy) (void)hipFree(a.dy);
    }
    for (auto &l : s->L) {
        if (l.Wf) (void)hipFree(l.Wf);
        if (l.Wt) (void)hipFree(l.Wt);
    }
    void *ptrs[] = {s->w, s->g, s->m, s->v, s->raw, s->tgt, s->mask, s->chw, s->wpart, s->lpart, s->lres};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (s->ev0) (void)hipEventDestroy(s->ev0);
    if (s->ev1) (void)hipEventDestroy(s->ev1);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
    return CISM_OK;
}

extern "C" long long cism_surrogate_num_params(const cism_surrogate *s) { return s ? s->nparams : 0; }

extern "C" double cism_surrogate_last_forward_ms(const cism_surrogate *s) {
    return s ? (double)s->last_forward_ms : -1.0;
}

// Host transfers of the weights go through the network's own (non-blocking) stream and
// wait for it, so they are ordered after every kernel launched before them.
extern "C" int cism_surrogate_get_params(cism_surrogate *s, float *host) {
    HIP_TRY(hipMemcpyAsync(host, s->w, sizeof(float) * s->nparams, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return CISM_OK;
}

extern "C" int cism_surrogate_set_params(cism_surrogate *s, const float *host) {
    s->wprep_ok = 0;
    HIP_TRY(hipMemcpyAsync(s->w, host, sizeof(float) * s->nparams, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipMemsetAsync(s->m, 0, sizeof(float) * s->nparams, s->stream));
    HIP_TRY(hipMemsetAsync(s->v, 0, sizeof(float) * s->nparams, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    s->step = 0;
    return CISM_OK;
}

// BF16 copies of the weights, rebuilt only after the weights changed (creation,
// cism_surrogate_set_params, a training step)
static int prep_weights(cism_surrogate *s) {
    if (s->wprep_ok) return CISM_OK;
    for (auto &c : s->L) {
        const long long n = frag_size(c.Co, c.ks * c.ks * c.Ci) + frag_size(c.Ci, c.ks * c.ks * c.Co);
        hipLaunchKernelGGL(k_prep_weights, dim3(nblocks_for(n)), dim3(256), 0, s->stream, c.Co, c.Ci, c.ks,
                           s->w + c.woff, c.Wf, c.Wt);
    }
    HIP_TRY(hipGetLastError());
    s->wprep_ok = 1;
    return CISM_OK;
}

static int conv_launch(cism_surrogate *s, const ConvDims &d, const ConvSrc &src, const short *Wf,
                       const float *bias, const float *mask, float *out) {
    if (d.Ci % 16 != 0 || d.Co % 32 != 0 || (d.ks != 1 && d.ks != 3)) {
        cism_set_error("surrogate convolution: Ci %% 16 and Co %% 32 must be 0 and the kernel 1x1 or 3x3");
        return CISM_ERR_ARG;
    }
    const int R = CONV_P + (d.ks == 3 ? 2 : 0);
    const size_t lds = sizeof(short) * R * R * (d.Ci + 8);   // at most 52.8 KB (256 channels)
    const unsigned np = (unsigned)(d.B * ((d.H + CONV_P - 1) / CONV_P) * ((d.W + CONV_P - 1) / CONV_P));
    // 64 output channels a workgroup read each staged patch half as often; 32 where that
    // leaves fewer than two workgroups a CU
    if (d.Co % 64 == 0 && np * (d.Co / 64) >= 512)
        hipLaunchKernelGGL(k_conv_patch<2>, dim3(np, d.Co / 64), dim3(256), lds, s->stream, d, src, Wf, bias, mask,
                           out);
    else
        hipLaunchKernelGGL(k_conv_patch<1>, dim3(np, d.Co / 32), dim3(256), lds, s->stream, d, src, Wf, bias, mask,
                           out);
    HIP_TRY(hipGetLastError());
    return CISM_OK;
}

// what layer l reads
static ConvSrc layer_src(const cism_surrogate *s, int l) {
    auto cat = [&](int low, int skip) {
        return ConvSrc{s->A[low].y, s->A[skip].y, s->A[low].C, s->A[skip].C};
    };
    if (l == L_D2) return cat(A_M1, A_E2b);
    if (l == L_D1) return cat(A_D2, A_E1b);
    if (l == L_D0) return cat(A_D1, A_E0b);
    const Act &in = s->A[LAYER_IN[l]];
    return ConvSrc{in.y, nullptr, in.C, 0};
}

static int forward(cism_surrogate *s) {
    const int B = s->B;
    CISM_TRY(prep_weights(s));
    auto conv = [&](int l) -> int {
        const ConvLayer &c = s->L[l];
        const Act &out = s->A[LAYER_OUT[l]];
        ConvDims d = {B, out.H, out.W, c.Ci, c.Co, c.ks, c.relu};
        return conv_launch(s, d, layer_src(s, l), c.Wf, s->w + c.boff, nullptr, out.y);
    };
    auto pool = [&](int a_in, int a_out) {
        const Act &x = s->A[a_in];
        hipLaunchKernelGGL(k_pool, dim3(nblocks_for(s->A[a_out].n(B))), dim3(256), 0, s->stream, B, x.H, x.W,
                           x.C, x.y, s->A[a_out].y);
    };
    CISM_TRY(conv(L_E0a)); CISM_TRY(conv(L_E0b)); pool(A_E0b, A_P0);
    CISM_TRY(conv(L_E1a)); CISM_TRY(conv(L_E1b)); pool(A_E1b, A_P1);
    CISM_TRY(conv(L_E2a)); CISM_TRY(conv(L_E2b)); pool(A_E2b, A_P2);
    CISM_TRY(conv(L_M0)); CISM_TRY(conv(L_M1));
    CISM_TRY(conv(L_D2)); CISM_TRY(conv(L_D1)); CISM_TRY(conv(L_D0));
    CISM_TRY(conv(L_HEAD));
    HIP_TRY(hipGetLastError());
    return CISM_OK;
}

// backward of layer l given dY of its output (already ReLU-masked): its parameter gradients
// and, when want_dx, the gradient of its input, zeroed where mask (the input itself, when
// it is a ReLU's output used by this layer alone) is not positive
static int conv_backward(cism_surrogate *s, int l, bool want_dx, bool mask) {
    const int B = s->B;
    const ConvLayer &c = s->L[l];
    const Act &in = s->A[LAYER_IN[l]], &out = s->A[LAYER_OUT[l]];
    int runs, per;
    wgrad_runs(c, B, out.H, out.W, runs, per);
    ConvDims d = {B, out.H, out.W, c.Ci, c.Co, c.ks, 0};
    const dim3 grid((unsigned)((c.Ci + 31) / 32), (unsigned)(c.Co / 32), (unsigned)runs);
    hipLaunchKernelGGL(c.ks == 3 ? k_wgrad_patch<3> : k_wgrad_patch<1>, grid, dim3(256), 0, s->stream, d,
                       layer_src(s, l), out.dy, s->wpart, per);
    const dim3 gred((unsigned)((c.nparams() + 63) / 64));
    if (runs > 64)
        hipLaunchKernelGGL(k_wgrad_reduce<16>, gred, dim3(1024), 0, s->stream, s->wpart, runs, c.nparams(),
                           s->g + c.woff);
    else
        hipLaunchKernelGGL(k_wgrad_reduce<4>, gred, dim3(256), 0, s->stream, s->wpart, runs, c.nparams(),
                           s->g + c.woff);
    HIP_TRY(hipGetLastError());
    if (want_dx) {
        // dX = conv(dY, W') : channels Co -> Ci
        ConvDims dd = {B, out.H, out.W, c.Co, c.Ci, c.ks, 0};
        CISM_TRY(conv_launch(s, dd, ConvSrc{out.dy, nullptr, c.Co, 0}, c.Wt, nullptr, mask ? in.y : nullptr, in.dy));
    }
    return CISM_OK;
}

static int backward(cism_surrogate *s) {
    const int B = s->B;
    // the low-resolution input of a concatenation
    auto upcat_bwd = [&](int a_low, int a_skip, int a_cat) {
        const Act &o = s->A[a_cat], &low = s->A[a_low];
        hipLaunchKernelGGL(k_up_cat_bwd, dim3(nblocks_for(low.n(B) / 4)), dim3(256), 0, s->stream, B, o.H, o.W, low.C,
                           s->A[a_skip].C, o.dy, low.y, low.dy);
    };
    // an encoder output, from the concatenation and from the pool after it
    auto skip_bwd = [&](int a_low, int a, int a_cat, int a_pool) {
        const Act &x = s->A[a];
        hipLaunchKernelGGL(k_skip_bwd, dim3(nblocks_for(x.n(B) / 4)), dim3(256), 0, s->stream, B, x.H, x.W, x.C,
                           s->A[a_low].C, s->A[a_cat].dy, s->A[a_pool].dy, x.y, x.dy);
    };
    CISM_TRY(conv_backward(s, L_HEAD, true, true));     // dOUT set by the loss -> dD0
    CISM_TRY(conv_backward(s, L_D0, true, false));      // -> dC0
    upcat_bwd(A_D1, A_E0b, A_C0);
    CISM_TRY(conv_backward(s, L_D1, true, false));      // -> dC1
    upcat_bwd(A_D2, A_E1b, A_C1);
    CISM_TRY(conv_backward(s, L_D2, true, false));      // -> dC2
    upcat_bwd(A_M1, A_E2b, A_C2);
    CISM_TRY(conv_backward(s, L_M1, true, true));       // -> dM0
    CISM_TRY(conv_backward(s, L_M0, true, false));      // -> dP2
    skip_bwd(A_M1, A_E2b, A_C2, A_P2);
    CISM_TRY(conv_backward(s, L_E2b, true, true));      // -> dE2a
    CISM_TRY(conv_backward(s, L_E2a, true, false));     // -> dP1
    skip_bwd(A_D2, A_E1b, A_C1, A_P1);
    CISM_TRY(conv_backward(s, L_E1b, true, true));
    CISM_TRY(conv_backward(s, L_E1a, true, false));     // -> dP0
    skip_bwd(A_D1, A_E0b, A_C0, A_P0);
    CISM_TRY(conv_backward(s, L_E0b, true, true));
    CISM_TRY(conv_backward(s, L_E0a, false, false));
    HIP_TRY(hipGetLastError());
    return CISM_OK;
}

// inputs arrive with SG_IN_RAW channels; the first layer reads SG_IN (zero padded)
__global__ void k_widen(long long P, const float *__restrict__ raw, float *__restrict__ in) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P * SG_IN) return;
    const long long p = t / SG_IN;
    const int c = (int)(t % SG_IN);
    in[t] = c < SG_IN_RAW ? raw[p * SG_IN_RAW + c] : 0.f;
}

static int upload_batch(cism_surrogate *s, const float *in, const float *tgt, const float *mask) {
    const long long P = (long long)s->B * s->H * s->W;
    HIP_TRY(hipMemcpyAsync(s->raw, in, sizeof(float) * P * SG_IN_RAW, hipMemcpyHostToDevice, s->stream));
    hipLaunchKernelGGL(k_widen, dim3(nblocks_for(P * SG_IN)), dim3(256), 0, s->stream, P, s->raw,
                       s->A[A_IN].y);
    if (tgt) HIP_TRY(hipMemcpyAsync(s->tgt, tgt, sizeof(float) * P * SG_OUT, hipMemcpyHostToDevice, s->stream));
    if (mask) HIP_TRY(hipMemcpyAsync(s->mask, mask, sizeof(float) * P, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return CISM_OK;
}

static int loss_and_grad(cism_surrogate *s, int nch, double *loss) {
    const long long P = (long long)s->B * s->H * s->W;
    const int nb = (int)(P * SG_OUT < 1024 * 256 ? (P * SG_OUT + 255) / 256 : 1024);
    hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, s->stream, P, nch, s->A[A_OUT].y, s->tgt, s->mask,
                       s->chw, s->lpart);
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(256), 0, s->stream, s->lpart, nb, s->lres);
    hipLaunchKernelGGL(k_loss_grad, dim3(nblocks_for(P * SG_OUT_PAD)), dim3(256), 0, s->stream, P, nch,
                       s->A[A_OUT].y, s->tgt, s->mask, s->chw, s->lres, s->A[A_OUT].dy);
    HIP_TRY(hipGetLastError());
    double res[2];
    HIP_TRY(hipMemcpyAsync(res, s->lres, sizeof res, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    if (loss) *loss = res[0];
    return CISM_OK;
}

__global__ void k_narrow(long long P, const float *__restrict__ o, float *__restrict__ out) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P * SG_OUT) return;
    out[t] = o[(t / SG_OUT) * SG_OUT_PAD + t % SG_OUT];
}

// forward on host inputs (B x H x W x 5, NHWC) -> host outputs (B x H x W x 24)
extern "C" int cism_surrogate_forward(cism_surrogate *s, const float *in, float *out) {
    if (!s) return CISM_ERR_ARG;
    CISM_TRY(upload_batch(s, in, nullptr, nullptr));
    HIP_TRY(hipEventRecord(s->ev0, s->stream));
    CISM_TRY(forward(s));
    HIP_TRY(hipEventRecord(s->ev1, s->stream));
    const long long P = (long long)s->B * s->H * s->W;
    // narrow SG_OUT_PAD -> SG_OUT channels into the target buffer (free during inference)
    hipLaunchKernelGGL(k_narrow, dim3(nblocks_for(P * SG_OUT)), dim3(256), 0, s->stream, P, s->A[A_OUT].y,
                       s->tgt);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, s->tgt, sizeof(float) * P * SG_OUT, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    HIP_TRY(hipEventElapsedTime(&s->last_forward_ms, s->ev0, s->ev1));
    return CISM_OK;
}

// loss and gradient w.r.t. all parameters (grad may be NULL) without an update
extern "C" int cism_surrogate_loss_grad(cism_surrogate *s, const float *in, const float *tgt,
                                        const float *mask, int nch, double *loss, float *grad) {
    if (!s || nch < 1 || nch > SG_OUT) return CISM_ERR_ARG;
    CISM_TRY(upload_batch(s, in, tgt, mask));
    CISM_TRY(forward(s));
    CISM_TRY(loss_and_grad(s, nch, loss));
    CISM_TRY(backward(s));
    if (grad) {
        HIP_TRY(hipMemcpyAsync(grad, s->g, sizeof(float) * s->nparams, hipMemcpyDeviceToHost, s->stream));
        HIP_TRY(hipStreamSynchronize(s->stream));
    }
    return CISM_OK;
}

extern "C" int cism_surrogate_train_step(cism_surrogate *s, const float *in, const float *tgt,
                                         const float *mask, int nch, float lr, double *loss) {
    CISM_TRY(cism_surrogate_loss_grad(s, in, tgt, mask, nch, loss, nullptr));
    s->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)s->step), c2 = 1.f - powf(b2, (float)s->step);
    hipLaunchKernelGGL(k_adam, dim3(nblocks_for(s->nparams)), dim3(256), 0, s->stream, s->nparams, s->w, s->g,
                       s->m, s->v, lr, b1, b2, 1e-8f, c1, c2);
    s->wprep_ok = 0;
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s->stream));
    return CISM_OK;
}

extern "C" int cism_surrogate_set_channel_weights(cism_surrogate *s, const float *w24) {
    HIP_TRY(hipMemcpyAsync(s->chw, w24, sizeof(float) * SG_OUT, hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return CISM_OK;
}

// ---------------------------------------------------------------------------
// The learned initial guess on a solver context (cism_learned_guess*): features
// from the context's resident fields, the network, and the decoded velocity written
// into the context's x, all on the device.
//
// Image layout: pixel (y, x) is owned vertex (i, j) = (x + ilo, y + jlo).  A periodic
// grid's owned vertices are the whole image (their count must be a multiple of 8 in
// each direction, the network's periodic padding then matches the grid's).  An
// outflow grid's owned vertices sit in the corner of a canvas at least 8 pixels wider
// and taller, rounded up to a multiple of 8, whose other pixels carry zero features
// (no ice) and separate the domain's edges across the periodic wrap.
// ---------------------------------------------------------------------------
#define SG_V_CH 11             // output channels: u at levels 0..10, v at 11..21
#define SG_NZ_MAX 11

struct cism_guess {
    cism_surrogate *net;
    int W, H, Wown, Hown, i0, j0;
    int nz, encoding;          // encoding 0: v = uscale o; 1: v = sign(o) uscale expm1(|o|)
    double uscale;
};

// features of one pixel (stagthck / 1000, 100 ds/dx, 100 ds/dy, (ln max(beta, 1e-3) - 7) / 2,
// log10 of the column-mean flow factor + 16; zero at inactive vertices and off the grid),
// the column-mean A of each of the vertex's four cells from flwafact = A^(-1/3) / 2
__global__ __launch_bounds__(256) void k_guess_features(GridDev g, int W, int H, int Wown, int Hown, int i0,
                                                        int j0, const int32_t *__restrict__ av,
                                                        const double *__restrict__ sthck,
                                                        const double *__restrict__ dsdx,
                                                        const double *__restrict__ dsdy,
                                                        const double *__restrict__ beta,
                                                        const double *__restrict__ ff, float *__restrict__ in) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long long)W * H) return;
    const int y = (int)(p / W), x = (int)(p % W);
    float f[SG_IN_RAW] = {0.f, 0.f, 0.f, 0.f, 0.f};
    if (x < Wown && y < Hown) {
        const int i = x + i0, j = y + j0;
        const long long v = i + (long long)g.sx * j;
        if (av[v]) {
            double vA = 0.0;
            for (int dj = 0; dj < 2; ++dj)
                for (int di = 0; di < 2; ++di) {
                    const long long cell = (i + di) + (long long)g.nx * (j + dj);
                    double colA = 0.0;
                    for (int k = 0; k < g.nz - 1; ++k) {
                        const double t = ff[k + (long long)(g.nz - 1) * cell];
                        colA += t > 0.0 ? 1.0 / (8.0 * t * t * t) : 0.0;
                    }
                    vA += colA / (g.nz - 1);
                }
            vA *= 0.25;
            f[0] = (float)(sthck[v] / 1000.0);
            f[1] = (float)(dsdx[v] * 100.0);
            f[2] = (float)(dsdy[v] * 100.0);
            f[3] = (float)((log(fmax(beta[v], 1e-3)) - 7.0) / 2.0);
            f[4] = (float)(log10(fmax(vA, 1e-30)) + 16.0);
        }
    }
#pragma unroll
    for (int c = 0; c < SG_IN; ++c) in[p * SG_IN + c] = c < SG_IN_RAW ? f[c] : 0.f;
}

// largest |output| decoded (network units), as the host decoder clips
__device__ inline double guess_decode(float o, int encoding, double uscale) {
    const double lim = encoding == 1 ? 10.0 : 1000.0;
    const double t = fmin(lim, fmax(-lim, (double)o));
    if (encoding == 1) return (t < 0 ? -uscale : uscale) * expm1(fabs(t));
    return uscale * t;
}

// x = the decoded velocity at owned active vertices, 0 elsewhere (halo images follow)
__global__ __launch_bounds__(256) void k_guess_decode(GridDev g, int W, int Wown, int Hown, int i0, int j0,
                                                      int encoding, double uscale,
                                                      const int32_t *__restrict__ av,
                                                      const float *__restrict__ out, double *__restrict__ x) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.nn) return;
    const int k = node_level(g, q);
    const long long col = node_col(g, q);
    const int i = col_i(g, col), j = col_j(g, col);
    const int px = i - i0, py = j - j0;
    double u = 0.0, v = 0.0;
    if (px >= 0 && px < Wown && py >= 0 && py < Hown && av[col]) {
        const long long p = (long long)py * W + px;
        u = guess_decode(out[p * SG_OUT_PAD + k], encoding, uscale);
        v = guess_decode(out[p * SG_OUT_PAD + SG_V_CH + k], encoding, uscale);
    }
    x[2 * q] = u;
    x[2 * q + 1] = v;
}

void learned_guess_free(cism_ctx *c) {
    if (!c || !c->guess) return;
    cism_surrogate_destroy(c->guess->net);
    delete c->guess;
    c->guess = nullptr;
}

int learned_guess_device(cism_ctx *c) {
    cism_guess *gs = c->guess;
    if (!gs) {
        cism_set_error("learned guess: no network loaded (cism_learned_guess_load)");
        return CISM_ERR_ARG;
    }
    const GridDev &g = c->g;
    cism_surrogate *s = gs->net;
    const long long P = (long long)gs->W * gs->H;
    hipLaunchKernelGGL(k_guess_features, dim3(nblocks_for(P)), dim3(256), 0, c->stream, g, gs->W, gs->H, gs->Wown,
                       gs->Hown, gs->i0, gs->j0, c->av, c->sthck, c->dsdx, c->dsdy, c->beta, c->flwafact,
                       s->A[A_IN].y);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    HIP_TRY(hipEventRecord(s->ev0, s->stream));
    CISM_TRY(forward(s));
    HIP_TRY(hipEventRecord(s->ev1, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    HIP_TRY(hipEventElapsedTime(&s->last_forward_ms, s->ev0, s->ev1));
    hipLaunchKernelGGL(k_guess_decode, dim3(nblocks_for(g.nn)), dim3(256), 0, c->stream, g, gs->W, gs->Wown,
                       gs->Hown, gs->i0, gs->j0, gs->encoding, gs->uscale, c->av, s->A[A_OUT].y, c->x);
    HIP_TRY(hipGetLastError());
    return launch_halo_vec(c, c->x);
}

extern "C" int cism_learned_guess_load(cism_ctx *c, const float *params, long long nparams, int nz, int encoding,
                                       double uscale) {
    if (!c || !params || (encoding != 0 && encoding != 1) || !(uscale > 0)) {
        cism_set_error("learned_guess_load: invalid arguments");
        return CISM_ERR_ARG;
    }
    HIP_TRY(hipSetDevice(c->device));
    const GridDev &g = c->g;
    if (nz != g.nz || nz > SG_NZ_MAX) {
        // the output channels hold nz levels of u then of v from channel 11: another nz
        // would read the wrong channels
        cism_set_error("learned_guess_load: the weights predict %d levels, the grid has nz = %d (at most %d)", nz,
                       g.nz, SG_NZ_MAX);
        return CISM_ERR_ARG;
    }
    const int Wown = g.ihi - g.ilo + 1, Hown = g.jhi - g.jlo + 1;
    int W = Wown, H = Hown;
    if (g.periodic) {
        if (Wown % 8 || Hown % 8) {
            cism_set_error("learned_guess_load: a periodic grid needs ewn and nsn divisible by 8 (got %d x %d)",
                           Wown, Hown);
            return CISM_ERR_UNSUPPORTED;
        }
    } else {
        W = (Wown + 8 + 7) / 8 * 8;
        H = (Hown + 8 + 7) / 8 * 8;
    }
    learned_guess_free(c);
    cism_surrogate *s = nullptr;
    CISM_TRY(cism_surrogate_create(H, W, 1, c->device, &s));
    if (nparams != s->nparams) {
        cism_surrogate_destroy(s);
        cism_set_error("learned_guess_load: %lld parameters given, the network has %lld", nparams, s->nparams);
        return CISM_ERR_ARG;
    }
    const int st = cism_surrogate_set_params(s, params);
    if (st) {
        cism_surrogate_destroy(s);
        return st;
    }
    cism_guess *gs = new cism_guess();
    gs->net = s;
    gs->W = W; gs->H = H; gs->Wown = Wown; gs->Hown = Hown; gs->i0 = g.ilo; gs->j0 = g.jlo;
    gs->nz = nz; gs->encoding = encoding; gs->uscale = uscale;
    c->guess = gs;
    return CISM_OK;
}

// weight file: "CISMSG01", int32 nz, int32 encoding, float64 uscale, int64 nparams, then
// nparams float32 (little endian)
extern "C" int cism_learned_guess_load_file(cism_ctx *c, const char *path) {
    if (!c || !path) {
        cism_set_error("learned_guess_load_file: invalid arguments");
        return CISM_ERR_ARG;
    }
    FILE *f = fopen(path, "rb");
    if (!f) {
        cism_set_error("learned_guess_load_file: cannot open %s", path);
        return CISM_ERR_ARG;
    }
    char magic[8];
    int32_t nz = 0, enc = 0;
    double uscale = 0.0;
    long long n = 0;
    int ok = fread(magic, 1, 8, f) == 8 && memcmp(magic, "CISMSG01", 8) == 0 && fread(&nz, 4, 1, f) == 1 &&
             fread(&enc, 4, 1, f) == 1 && fread(&uscale, 8, 1, f) == 1 && fread(&n, 8, 1, f) == 1 && n > 0 &&
             n < (1LL << 28);
    std::vector<float> w;
    if (ok) {
        w.resize((size_t)n);
        ok = fread(w.data(), sizeof(float), (size_t)n, f) == (size_t)n;
    }
    fclose(f);
    if (!ok) {
        cism_set_error("learned_guess_load_file: %s is not a weight file", path);
        return CISM_ERR_ARG;
    }
    return cism_learned_guess_load(c, w.data(), n, nz, enc, uscale);
}

extern "C" int cism_learned_guess(cism_ctx *c, const double *stagthck, const double *dusrf_dx,
                                  const double *dusrf_dy, const double *beta_internal, const double *flwafact,
                                  const int32_t *active_vertex, double *uvel, double *vvel) {
    if (!c) {
        cism_set_error("learned_guess: null context");
        return CISM_ERR_ARG;
    }
    HIP_TRY(hipSetDevice(c->device));
    const GridDev &g = c->g;
    const size_t ncol = (size_t)g.sx * g.sy;
    struct { double *dst; const double *src; size_t n; } ins[] = {
        {c->sthck, stagthck, ncol}, {c->dsdx, dusrf_dx, ncol}, {c->dsdy, dusrf_dy, ncol},
        {c->beta, beta_internal, ncol}, {c->flwafact, flwafact, (size_t)g.ne}};
    for (auto &t : ins)
        if (t.src) HIP_TRY(hipMemcpyAsync(t.dst, t.src, sizeof(double) * t.n, hipMemcpyHostToDevice, c->stream));
    if (active_vertex)
        HIP_TRY(hipMemcpyAsync(c->av, active_vertex, sizeof(int32_t) * ncol, hipMemcpyHostToDevice, c->stream));
    CISM_TRY(learned_guess_device(c));
    if (uvel && vvel) CISM_TRY(download_vec(c, c->x, uvel, vvel));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return CISM_OK;
}

extern "C" double cism_learned_guess_last_ms(const cism_ctx *c) {
    return c && c->guess ? (double)c->guess->net->last_forward_ms : 0.0;
}
