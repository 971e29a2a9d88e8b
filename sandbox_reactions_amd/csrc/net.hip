// The learned FLD preconditioner on the device: a 3-level U-Net (16/32/64 channels, 3x3 convolutions, BF16
// activations and weights, FP32 accumulation), its backward pass and Adam.
//
// The reference has no learned part (its preconditioners are Jacobi and the multigrid of
// crates/sr-engine/shaders/heat.wgsl:1160-1526); the network's definition is this library's, stated layer by layer in
// the f64 numpy oracle, oracle/unet.py, whose names the kernels follow.
//
//   * activations are channels-last BF16 (pixel-major, channels contiguous), so a lane's eight consecutive K values
//     of the implicit GEMM are one 16-byte load;
//   * k_conv is the implicit-GEMM 3x3 convolution on the matrix cores: M = output channels, N = pixels (16 x R rows per
//     wave, the tile's input staged in LDS 32 channels at a time), K = taps x input channels in chunks of 32
//     (v_mfma_f32_16x16x32_bf16). The same kernel computes the backward-data pass with mirrored, transposed weights and
//     the ReLU mask applied while staging; upsample + concat of the decoder is folded into the staging, the encoder's
//     2x2 pooling and the output 1x1 layer into the epilogue;
//   * the weight gradient (k_dw) is a matrix product too, K the pixels: channels-last LDS tiles read transposed
//     (ds_read_b64_tr_b16), FP32 accumulation, per-block partials summed in a fixed order by k_dw_reduce (deterministic,
//     no atomics);
//   * the features and the energy-norm loss are elementwise / stencil kernels.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"
#include "net.hpp"

namespace sr {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

#define NTH 256
#define NB_FEAT 1024
#define DW_FLOATS (1 << 22)  // a layer's weight-gradient partials: so many, and 256 to 1024 blocks
#define DW_TW 32         // its tile
#define DW_TH 4
#define LOG_CLAMP 20.0f
// Blocks that a convolution's launch keeps the chip busy with: below it a wave takes half the rows. An application with 128,
// 256, 512, 1024 and 2048: 91 / 91 / 87 / 90 / 90 us at 516 x 260, 112 / 102 / 99 / 99 / 108 at 512^2, 196 / 201 / 208 / 205
// / 229 at 1024^2, 444 / 445 / 445 / 460 / 462 at 1540^2, 673 / 673 / 673 / 672 / 703 at 2048^2.
#define CONV_FILL 512

__device__ __forceinline__ bf16x8 ld8(const bf16 *p) { return *(const bf16x8 *)p; }
__device__ __forceinline__ void st8(bf16 *p, bf16x8 v) { *(bf16x8 *)p = v; }

// the sum of a cell's four face couplings (rim faces included, as the features read them)
__device__ __forceinline__ float coupling_sum(int w, const float *kx, const float *ky, int i, int y, int x) {
    return kx[(size_t)y * (w + 1) + x] + kx[(size_t)y * (w + 1) + x + 1] + ky[i] + ky[i + w];
}

// ------------------------------------------------------------------------------------------------------- features
// partials of sum (r d^-1/2)^2 and sum log(mean coupling)
__global__ void __launch_bounds__(NTH) k_feat_sums(int w, int h, const float *__restrict__ own,
                                                   const float *__restrict__ kx, const float *__restrict__ ky,
                                                   const float *__restrict__ r, double *part) {
    double v[2] = {0.0, 0.0};
    const int n = w * h;
    for (int i = blockIdx.x * NTH + threadIdx.x; i < n; i += gridDim.x * NTH) {
        const int y = i / w, x = i - y * w;
        const float ks = coupling_sum(w, kx, ky, i, y, x);
        const float rt = r[i] * rsqrtf(own[i] + ks);
        v[0] += (double)rt * rt;
        v[1] += (double)logf(fmaxf(0.25f * ks, 1e-30f));
    }
    block_partials<2>(v, part, gridDim.x);
}

// the three input channels (padded to 8): r d^-1/2 / s, log mean coupling - its mean (clamped), log(own / d);
// d^-1/2 kept for the output's scaling; scal = {s, mean}
__global__ void __launch_bounds__(NTH) k_feat(int w, int h, const float *__restrict__ own, const float *__restrict__ kx,
                                              const float *__restrict__ ky, const float *__restrict__ r,
                                              const double *part, int nb, bf16 *__restrict__ x,
                                              float *__restrict__ dis, float *scal) {
    const double s2 = sum_partials(part, nb), sl = sum_partials(part + nb, nb);
    const int n = w * h;
    const float s = s2 > 0.0 ? (float)sqrt(s2 / n) : 1.0f, mean = (float)(sl / n);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal[0] = s;
        scal[1] = mean;
    }
    const float is = 1.0f / s;
    for (int i = blockIdx.x * NTH + threadIdx.x; i < n; i += gridDim.x * NTH) {
        const int y = i / w, xx = i - y * w;
        const float ks = coupling_sum(w, kx, ky, i, y, xx);
        const float d = own[i] + ks;
        const float di = rsqrtf(d);
        dis[i] = di;
        bf16x8 f = {};
        f[0] = (bf16)(r[i] * di * is);
        f[1] = (bf16)fminf(fmaxf(logf(fmaxf(0.25f * ks, 1e-30f)) - mean, -LOG_CLAMP), LOG_CLAMP);
        f[2] = (bf16)logf(own[i] / d);
        st8(x + (size_t)8 * i, f);
    }
}

// ------------------------------------------------------------------------------------------- implicit-GEMM conv 3x3
// K's order. Input channels go by slabs of 32 (the last what is left: 8 or 16); within a slab by row tap ty, then the
// (column tap tx, channel octet) pairs, tx-major, four pairs of eight channels to a chunk of 32, the last chunk's missing
// pairs zero. A chunk holds one row tap alone, so the pixels' operand of an input row serves all three output rows
// around it.
__host__ __device__ constexpr int conv_chunks(int sc) { return (3 * (sc / 8) + 3) / 4; }
__host__ __device__ constexpr int conv_kp(int cin) {
    return cin / 32 * 3 * 32 * conv_chunks(32) + (cin % 32 ? 3 * 32 * conv_chunks(cin % 32) : 0);
}
// the tap (3 ty + tx) and channel of K index k, false for the padding
__device__ inline bool conv_k(int cin, int k, int &tap, int &ci) {
    const int per = 3 * 32 * conv_chunks(32);
    int slab = k / per, sc = 32;
    if (slab >= cin / 32) {
        slab = cin / 32;
        sc = cin % 32;
    }
    k -= slab * per;
    const int oct = sc / 8, c32 = 32 * conv_chunks(sc), ty = k / c32, pair = (k - ty * c32) / 8;
    if (pair >= 3 * oct) return false;
    tap = 3 * ty + pair / oct;
    ci = 32 * slab + 8 * (pair % oct) + k % 8;
    return true;
}

struct ConvArgs {
    const bf16 *in;    // (H, W, CIN - cup): channels [cup, CIN)
    const bf16 *up;    // (H/2, W/2, cup): channels [0, cup), nearest-upsampled; null when cup == 0 (a multiple of 32)
    const bf16 *mask;  // (H, W, CIN): entries whose mask is not > 0 read as zero; or null (only with cup == 0)
    const bf16 *wt;    // (COUT, conv_kp(CIN))
    const float *bias; // (COUT) or null
    bf16 *out;         // (H, W, COUT)
    int H, W, cup, relu;
    bf16 *half = nullptr;  // CONV_POOL, CONV_SPLIT: the half-resolution output
    // CONV_OUT: zn = (b + w . out) s d^-1/2, z = zadd + zn and/or err = zn - e (each null when not wanted)
    const float *wout = nullptr, *scal = nullptr, *dis = nullptr, *zadd = nullptr, *e = nullptr;
    float *z = nullptr, *err = nullptr;
};

// What a convolution does with its result (rounded to BF16) besides storing it; the fused forms take an even H and W
enum {
    CONV_PLAIN,
    CONV_POOL,   // also its 2x2 mean into half (H/2, W/2, COUT)
    CONV_OUT,    // COUT = 16: also the output 1x1 layer and the scaling back to the system's units
    CONV_SPLIT,  // a concat's gradient: channels [0, 32) (COUT = 48) or [0, 64) (96), summed over 2x2 pixels, into
                 // half, the rest into out (H, W, COUT - those)
    CONV_UNPOOL  // a pooled gradient: a quarter of it added to each of the four pixels of out (2 H, 2 W, COUT)
};

#define TW 64
// One slab of a tile's input: SC channels from channel cb. The loads of a thread's items are issued together and the next
// slab's go out before this one's products, whose time covers them; in LDS the pixel stride is an odd number of 16-byte
// slots, so eight lanes' reads take eight slots. The tile is zero outside the image.
template <int CIN, int R, int S> struct ConvSlab {
    static constexpr int SC = 32 * S < CIN / 32 * 32 ? 32 : CIN % 32, OCT = SC / 8, CP = SC == 8 ? 8 : SC + 8;
    static constexpr int RW = TW + 2, RH = R + 2, N = RH * RW * OCT, IT = (N + NTH - 1) / NTH, CB = 32 * S;
    static constexpr int C = conv_chunks(SC), KB = S * 3 * 32 * conv_chunks(32);
    bf16x8 v[IT];
    __device__ inline void load(const ConvArgs &a, int x0, int y0) {
        const int H = a.H, W = a.W, cup = a.cup, cs = CIN - cup;
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int t = threadIdx.x + k * NTH;
            const int o = t % OCT, px = t / OCT, lx = px % RW, ly = px / RW;
            const int xx = x0 + lx - 1, yy = y0 + ly - 1, ci = CB + 8 * o;
            v[k] = bf16x8{};
            if (t < N && xx >= 0 && xx < W && yy >= 0 && yy < H) {
                if (ci < cup)
                    v[k] = ld8(a.up + ((size_t)(yy >> 1) * (W >> 1) + (xx >> 1)) * cup + ci);
                else
                    v[k] = ld8(a.in + ((size_t)yy * W + xx) * cs + (ci - cup));
                if (a.mask) {
                    const bf16x8 mv = ld8(a.mask + ((size_t)yy * W + xx) * CIN + ci);
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        if (!((float)mv[j] > 0.0f)) v[k][j] = (bf16)0.0f;
                }
            }
        }
    }
    __device__ inline void store(bf16 *tile) const {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int t = threadIdx.x + k * NTH;
            if (t < N) st8(tile + (t / OCT) * CP + 8 * (t % OCT), v[k]);
        }
    }
    // chunk c's weights for the three row taps
    template <int NT> static __device__ inline void weights(const bf16 *wt, int c, bf16x8 (&w)[3][NT]) {
        const int g = (threadIdx.x & 63) >> 4, c16 = threadIdx.x & 15;
#pragma unroll
        for (int ty = 0; ty < 3; ty++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                w[ty][t] = ld8(wt + (size_t)(t * 16 + c16) * conv_kp(CIN) + KB + (ty * C + c) * 32 + 8 * g);
    }
    // every chunk's products, the wave walking its R + 2 input rows, each row's pixels read once and used by up to three
    // output rows, the next chunk's weights loading meanwhile. Lane l of an MFMA holds A[m = l % 16][k = 8 (l / 16) + j],
    // B[k = 8 (l / 16) + j][n = l % 16] and D[m = 4 (l / 16) + j][n = l % 16]: m the output channel, n the pixel, so a
    // lane ends with four consecutive channels of one pixel. A padded pair's zero weights meet the zeros at `zeros` (not a
    // pixel, which may be infinite).
    template <int NT>
    static __device__ inline void products(const bf16 *wt, const bf16 *tile, const bf16 *zeros, bf16x8 (&w)[3][NT],
                                           f32x4 (&acc)[R][NT]) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c16 = lane & 15;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int pair = 4 * c + g, tx = pair / OCT, o = pair % OCT;
            const bf16 *px = tile + (16 * wave + c16 + tx) * CP + 8 * o;
            int row = RW * CP;
            if (4 * c + 3 >= 3 * OCT && pair >= 3 * OCT) {
                px = zeros;
                row = 0;
            }
            bf16x8 wn[3][NT];
            if (c + 1 < C) weights<NT>(wt, c + 1, wn);
#pragma unroll
            for (int i = 0; i < RH; i++) {
                const bf16x8 p = ld8(px + i * row);
#pragma unroll
                for (int ty = 0; ty < 3; ty++) {
                    const int r = i - ty;
                    if (r < 0 || r >= R) continue;
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ty][t], p, acc[r][t], 0, 0, 0);
                }
            }
            if (c + 1 < C)
#pragma unroll
                for (int ty = 0; ty < 3; ty++)
#pragma unroll
                    for (int t = 0; t < NT; t++) w[ty][t] = wn[ty][t];
        }
    }
};

template <int CIN, int R, int NT, int S>
__device__ inline void conv_slabs(const ConvArgs &a, bf16 *tile, const bf16 *zeros, int x0, int y0,
                                  const ConvSlab<CIN, R, S> &slab, f32x4 (&acc)[R][NT]) {
    using SL = ConvSlab<CIN, R, S>;
    bf16x8 w[3][NT];
    SL::template weights<NT>(a.wt, 0, w);
    slab.store(tile);
    __syncthreads();
    if constexpr (SL::CB + SL::SC < CIN) {
        ConvSlab<CIN, R, S + 1> next;
        next.load(a, x0, y0);
        SL::template products<NT>(a.wt, tile, zeros, w, acc);
        __syncthreads();  // the slab is read
        conv_slabs<CIN, R, NT, S + 1>(a, tile, zeros, x0, y0, next, acc);
    } else {
        SL::template products<NT>(a.wt, tile, zeros, w, acc);
    }
}

// the value of the lane beside (lane ^ 1), without the LDS unit
__device__ __forceinline__ float beside(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

// a and b summed over pairs of 16-lane rows, and over the two halves: rows (a0 + a1, b0 + b1, a2 + a3, b2 + b3), and
// halves (a.low + a.high, b.low + b.high)
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float swap16_add(float a, float b) {
    const u32x2 r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                     false, false);
    const unsigned lo = r[0], hi = r[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float swap32_add(float a, float b) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                     false, false);
    const unsigned lo = r[0], hi = r[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}

// A block computes TW x R pixels (a wave 16 columns of every row) x all COUT channels. Measured at 2048^2 (nine tap reads
// of LDS per product row and COUT-scattered 2-byte stores before): 48 -> 16 channels 296 -> 136 us, 96 -> 32 at 1024^2
// 168 -> 92, 64 -> 64 at 512^2 81 -> 56; the wide-image 16-channel layers are bound by HBM (8 -> 16: 38 us, 5.3 TB/s).
template <int CIN, int COUT, int R, int EPI>
__global__ void __launch_bounds__(NTH) k_conv(ConvArgs a) {
    constexpr int NT = COUT / 16, FULL = CIN / 32, REST = CIN % 32;
    constexpr int CPM = FULL ? 40 : REST == 8 ? 8 : REST + 8;
    constexpr int SUMMED = EPI == CONV_SPLIT ? COUT / 3 * 2 : 0;  // the concat's upsampled channels
    static_assert(CIN % 8 == 0 && COUT % 16 == 0 && R % 2 == 0, "channel counts, rows");
    static_assert(EPI != CONV_OUT || COUT == 16, "the output layer reads 16 channels");
    constexpr int PIXELS = (R + 2) * (TW + 2) * CPM;
    __shared__ __attribute__((aligned(16))) bf16 tile[PIXELS + 8];  // and eight zeros
    if (threadIdx.x == 0) st8(tile + PIXELS, bf16x8{});
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c16 = lane & 15;
    const int blk = xcd_tile(), x0 = (blk % gridDim.x) * TW, y0 = (blk / gridDim.x) * R;
    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    {
        ConvSlab<CIN, R, 0> first;
        first.load(a, x0, y0);
        conv_slabs<CIN, R, NT, 0>(a, tile, tile + PIXELS, x0, y0, first, acc);
    }
    const int x = x0 + 16 * wave + c16, H = a.H, W = a.W;
    if (x0 + 16 * wave >= W) return;  // the whole wave is past the image
    float o[R];
#pragma unroll
    for (int r = 0; r < R; r++) o[r] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int co = t * 16 + 4 * g;
        const bool summed = t * 16 < SUMMED;
        float b[4] = {0.0f, 0.0f, 0.0f, 0.0f}, wv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (a.bias) b[j] = a.bias[co + j];
            if (EPI == CONV_OUT) wv[j] = a.wout[co + j];
        }
        bf16x4 s[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const bool in = x < W && y0 + r < H;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v = acc[r][t][j] + b[j];
                if (a.relu) v = fmaxf(v, 0.0f);
                s[r][j] = (bf16)v;
                if (EPI == CONV_OUT) o[r] += wv[j] * (float)s[r][j];
            }
            if (EPI == CONV_UNPOOL) {
                if (in)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        bf16x4 *p = (bf16x4 *)(a.out + ((size_t)(2 * (y0 + r) + (q >> 1)) * (2 * W) + 2 * x + (q & 1)) * COUT + co);
                        bf16x4 f = *p;
#pragma unroll
                        for (int j = 0; j < 4; j++) f[j] = (bf16)((float)f[j] + 0.25f * (float)s[r][j]);
                        *p = f;
                    }
            } else if (!summed && in) {
                *(bf16x4 *)(a.out + ((size_t)(y0 + r) * W + x) * (COUT - SUMMED) + co - SUMMED) = s[r];
            }
        }
        if (EPI == CONV_POOL || summed) {
            constexpr int HC = EPI == CONV_POOL ? COUT : SUMMED;
            const float f = EPI == CONV_POOL ? 0.25f : 1.0f;
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                bf16x4 h;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float v0 = (float)s[r][j], v1 = (float)s[r + 1][j];
                    h[j] = (bf16)(f * (((v0 + beside(v0)) + v1) + beside(v1)));
                }
                if (!(c16 & 1) && x < W && y0 + r < H)
                    *(bf16x4 *)(a.half + ((size_t)((y0 + r) >> 1) * (W >> 1) + (x >> 1)) * HC + co) = h;
            }
        }
    }
    if (EPI == CONV_OUT) {
        const float s = a.scal[0], bo = a.wout[16];
        // the four groups' sums of two or four rows joined by lane swaps, group g ending with row g (of two: g % 2)
        constexpr int Q = R < 4 ? 2 : 4;
#pragma unroll
        for (int r0 = 0; r0 < R; r0 += Q) {
            float v = swap16_add(o[r0], o[r0 + 1]);
            v = swap32_add(v, Q == 4 ? swap16_add(o[r0 + Q - 2], o[r0 + Q - 1]) : v);
            const int y = y0 + r0 + g;
            if (g < Q && x < W && y < H) {
                const size_t i = (size_t)y * W + x;
                const float zn = (v + bo) * s * a.dis[i];
                if (a.err) a.err[i] = zn - a.e[i];
                if (a.z) a.z[i] = (a.zadd ? a.zadd[i] : 0.0f) + zn;
            }
        }
    }
}

// Rows per wave: the more rows, the fewer reads of LDS and of the halo per product (R + 2 for 3 R NT products), as long
// as the launch still fills the chip; wide outputs keep four (eight take the registers of two waves a SIMD, and an
// application at 2048^2 674 us as with four, a training step at 1024^2 972 against 965).
template <int CIN, int COUT, int EPI = CONV_PLAIN> static void conv(hipStream_t s, const ConvArgs &a) {
    auto blocks = [&](int r) { return ((a.W + TW - 1) / TW) * ((a.H + r - 1) / r); };
    auto go = [&](auto kernel, int r) {
        hipLaunchKernelGGL(kernel, dim3((a.W + TW - 1) / TW, (a.H + r - 1) / r), dim3(NTH), 0, s, a);
    };
    if constexpr (COUT <= 48)
        if (blocks(8) >= CONV_FILL) return go(k_conv<CIN, COUT, 8, EPI>, 8);
    if (blocks(4) >= CONV_FILL) return go(k_conv<CIN, COUT, 4, EPI>, 4);
    go(k_conv<CIN, COUT, 2, EPI>, 2);
}

// ------------------------------------------------------------------------------------------------------- training
// A v in face form (own v + sum over interior faces k (v_i - v_j)), as the solver's level 0 applies it
__device__ __forceinline__ float apply_a(int w, int h, const float *own, const float *kx, const float *ky,
                                         const float *v, int i, int y, int x) {
    const float vi = v[i];
    float s = own[i] * vi;
    if (x > 0) s += kx[(size_t)y * (w + 1) + x] * (vi - v[i - 1]);
    if (x < w - 1) s += kx[(size_t)y * (w + 1) + x + 1] * (vi - v[i + 1]);
    if (y > 0) s += ky[i] * (vi - v[i - w]);
    if (y < h - 1) s += ky[i + w] * (vi - v[i + w]);
    return s;
}

// aerr = A err; partials of err . A err and e . A e
__global__ void __launch_bounds__(NTH) k_loss(int w, int h, const float *__restrict__ own, const float *__restrict__ kx,
                                              const float *__restrict__ ky, const float *__restrict__ err,
                                              const float *__restrict__ e, float *__restrict__ aerr, double *part) {
    double v[2] = {0.0, 0.0};
    const int n = w * h;
    for (int i = blockIdx.x * NTH + threadIdx.x; i < n; i += gridDim.x * NTH) {
        const int y = i / w, x = i - y * w;
        const float ae = apply_a(w, h, own, kx, ky, err, i, y, x);
        aerr[i] = ae;
        v[0] += (double)err[i] * ae;
        v[1] += (double)e[i] * apply_a(w, h, own, kx, ky, e, i, y, x);
    }
    block_partials<2>(v, part, gridDim.x);
}

// dL/d(out) = 2 A err / (e . A e) * s d^-1/2; then dL/d(d1) = gout w_out and partials of dL/dw_out, dL/db_out
__global__ void __launch_bounds__(NTH) k_out_back(int n, const float *__restrict__ aerr, const double *lpart, int nbl,
                                                  const float *scal, const float *__restrict__ dis,
                                                  const bf16 *__restrict__ d1, const float *__restrict__ wout,
                                                  float *__restrict__ gout, bf16 *__restrict__ g_d1, double *part) {
    const double norm = sum_partials(lpart + nbl, nbl);
    const float f = norm > 0.0 ? (float)(2.0 / norm) * scal[0] : 0.0f;
    double v[17];
#pragma unroll
    for (int c = 0; c < 17; c++) v[c] = 0.0;
    float wv[16];
#pragma unroll
    for (int c = 0; c < 16; c++) wv[c] = wout[c];
    for (int i = blockIdx.x * NTH + threadIdx.x; i < n; i += gridDim.x * NTH) {
        const float go = f * aerr[i] * dis[i];
        gout[i] = go;
        const bf16x8 a = ld8(d1 + (size_t)16 * i), b = ld8(d1 + (size_t)16 * i + 8);
        bf16x8 ga, gb;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            v[j] += (double)((float)a[j] * go);
            v[8 + j] += (double)((float)b[j] * go);
            ga[j] = (bf16)(go * wv[j]);
            gb[j] = (bf16)(go * wv[8 + j]);
        }
        v[16] += go;
        st8(g_d1 + (size_t)16 * i, ga);
        st8(g_d1 + (size_t)16 * i + 8, gb);
    }
    block_partials<17>(v, part, gridDim.x);
}

// out[k] = sum of part[k nb .. k nb + nb), one block per k (a fixed order)
__global__ void __launch_bounds__(NTH) k_reduce_rows(const double *part, int nb, float *out) {
    const double s = sum_partials(part + (size_t)blockIdx.x * nb, nb);
    if (threadIdx.x == 0) out[blockIdx.x] = (float)s;
}

// Weight and bias gradients of one layer: dW[tap][ci][co] = sum_p x[p + tap][ci] ga[p][co], ga = gy (y > 0): per tap a
// (CIN x pixels) (pixels x COUT) product on the matrix cores, FP32 accumulation of BF16 products (each exact in FP32).
// A block walks 32 x 4 pixel tiles; the x tile (with its one-pixel rim) and ga lie channels-last in LDS and both operands
// are read transposed (ds_read_b64_tr_b16: of four pixels x 16 channels over 16 lanes, lane i gets channel i of the four
// pixels), so a lane's eight K values are eight consecutive pixels of one channel. The (tap, 16 input channels) pairs are
// dealt to the four waves, each holding its pairs' accumulators for every output channel over all tiles; the last wave
// also sums the biases' gradients (a row of ones). The pixel stride is an odd number of 32-byte slots: the eight pixels
// that half a wave reads take eight slots. At 512^2 the ten layers' launches take 0.19 ms (vector FMAs from FP32 tiles:
// 1.87 ms).
template <int CIN, int COUT>
__global__ void __launch_bounds__(NTH) k_dw(const bf16 *__restrict__ in, const bf16 *__restrict__ up, int cup,
                                            const bf16 *__restrict__ gy, const bf16 *__restrict__ y, int H, int W,
                                            float *__restrict__ part) {
    constexpr int CI = CIN < 16 ? 16 : CIN, MB = CI / 16, NBK = COUT / 16, PAIRS = 9 * MB, PPW = (PAIRS + 3) / 4;
    constexpr int XP = MB % 2 ? CI : CI + 16, GP = NBK % 2 ? COUT : COUT + 16;  // pixel strides
    constexpr int RW = DW_TW + 2, OX = CI / 8, OG = COUT / 8;
    __shared__ __attribute__((aligned(16))) bf16 xs[(DW_TH + 2) * RW * XP];
    __shared__ __attribute__((aligned(16))) bf16 gs[DW_TH * DW_TW * GP];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    f32x4 acc[PPW][NBK], bacc[NBK];
#pragma unroll
    for (int t = 0; t < NBK; t++) {
        bacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < PPW; q++) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; j++) ones[j] = (bf16)1.0f;
    // eight pixels from p on of 16 channels: pixels 8 g .. 8 g + 7 of the lane's group
    auto tr8 = [&](const bf16 *p, int stride) {
        const bf16 *q = p + (8 * g + (i16 >> 2)) * stride + 4 * (i16 & 3);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)q);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(q + 4 * stride));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const int cs = CIN - cup, spr = (W + DW_TW - 1) / DW_TW, ntile = spr * ((H + DW_TH - 1) / DW_TH);
    for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int y0 = tile / spr * DW_TH, x0 = tile % spr * DW_TW;
        __syncthreads();
        for (int t = threadIdx.x; t < (DW_TH + 2) * RW * OX; t += NTH) {
            const int o = t % OX, px = t / OX, lx = px % RW, ly = px / RW, ci = 8 * o;
            const int xx = x0 + lx - 1, yy = y0 + ly - 1;
            bf16x8 v = {};
            if (ci < CIN && xx >= 0 && xx < W && yy >= 0 && yy < H)
                v = ci < cup ? ld8(up + ((size_t)(yy >> 1) * (W >> 1) + (xx >> 1)) * cup + ci)
                             : ld8(in + ((size_t)yy * W + xx) * cs + (ci - cup));
            st8(xs + px * XP + ci, v);
        }
        for (int t = threadIdx.x; t < DW_TH * DW_TW * OG; t += NTH) {
            const int o = t % OG, px = t / OG, xx = x0 + px % DW_TW, yy = y0 + px / DW_TW;
            bf16x8 v = {};
            if (xx < W && yy < H) {
                const size_t i = ((size_t)yy * W + xx) * COUT + 8 * o;
                v = ld8(gy + i);
                const bf16x8 yv = ld8(y + i);
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (!((float)yv[j] > 0.0f)) v[j] = (bf16)0.0f;
            }
            st8(gs + px * GP + 8 * o, v);
        }
        __syncthreads();
        const int rows = min(DW_TH, H - y0);  // a row below the image takes no part (its zeros may meet infinite pixels)
#pragma unroll 1
        for (int r = 0; r < rows; r++) {
            bf16x8 gv[NBK];
#pragma unroll
            for (int t = 0; t < NBK; t++) gv[t] = tr8(gs + r * DW_TW * GP + 16 * t, GP);
#pragma unroll
            for (int q = 0; q < PPW; q++) {
                const int pr = wave + 4 * q, tap = pr / MB, mb = pr - tap * MB;
                if (pr >= PAIRS) continue;
                const bf16x8 xv = tr8(xs + ((r + tap / 3) * RW + tap % 3) * XP + 16 * mb, XP);
#pragma unroll
                for (int t = 0; t < NBK; t++)
                    acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv, gv[t], acc[q][t], 0, 0, 0);
            }
            if (wave == 3)
#pragma unroll
                for (int t = 0; t < NBK; t++)
                    bacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, gv[t], bacc[t], 0, 0, 0);
        }
    }
    float *pb = part + (size_t)blockIdx.x * (9 * CIN * COUT + COUT);
#pragma unroll
    for (int q = 0; q < PPW; q++) {
        const int pr = wave + 4 * q, tap = pr / MB, mb = pr - tap * MB;
        if (pr >= PAIRS) continue;
#pragma unroll
        for (int t = 0; t < NBK; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int ci = 16 * mb + 4 * g + j;
                if (ci < CIN) pb[((size_t)tap * CIN + ci) * COUT + 16 * t + i16] = acc[q][t][j];
            }
    }
    if (wave == 3 && g == 0)
#pragma unroll
        for (int t = 0; t < NBK; t++) pb[9 * CIN * COUT + 16 * t + i16] = bacc[t][0];
}

// Every layer's k_dw partials summed into the gradients in one launch: a block takes 32 consecutive values of one
// layer's (3, 3, cin, cout) + (cout), eight threads a value, each a strided run of the layer's blocks (in FP64), the runs
// joined in order. (One thread a value walking all blocks took 63 us a layer: a chain of 256 loads.)
struct DwTable {
    int n;
    int start[10], nb[10], cinp[10], cin[10], cout[10];  // first block, k_dw blocks, the layer's shape
    size_t part[10], w[10], b[10];                       // offsets of the partials and of the gradients
};

__global__ void __launch_bounds__(NTH) k_dw_reduce(DwTable T, const float *__restrict__ part, float *__restrict__ grads) {
    int l = 0;
    while (l + 1 < T.n && (int)blockIdx.x >= T.start[l + 1]) l++;
    const int cin = T.cin[l], cout = T.cout[l], cinp = T.cinp[l], nw = 9 * cin * cout, nb = T.nb[l];
    const int v = threadIdx.x & 31, run = threadIdx.x >> 5, o = ((int)blockIdx.x - T.start[l]) * 32 + v;
    const size_t stride = (size_t)9 * cinp * cout + cout;
    __shared__ double sh[NTH / 32][32];
    double s = 0.0;
    if (o < nw + cout) {
        size_t src = (size_t)9 * cinp * cout + (o - nw);
        if (o < nw) {
            const int co = o % cout, rest = o / cout, ci = rest % cin, tap = rest / cin;
            src = ((size_t)tap * cinp + ci) * cout + co;
        }
        const float *p = part + T.part[l] + src;
#pragma unroll 8
        for (int b = run; b < nb; b += NTH / 32) s += p[(size_t)b * stride];
    }
    sh[run][v] = s;
    __syncthreads();
    if (run == 0 && o < nw + cout) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < NTH / 32; k++) t += sh[k][v];
        grads[o < nw ? T.w[l] + o : T.b[l] + (o - nw)] = (float)t;
    }
}

// Adam (Kingma and Ba 2015, Algorithm 1) on the FP32 master parameters
__global__ void k_adam(int n, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float bc1, float bc2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi, vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

// The BF16 weight layouts of every layer from the FP32 (3, 3, cin, cout) masters, K in k_conv's order: forward (cout, kp)
// over the taps and input channels, backward-data (cin, kpb) over the mirrored taps and output channels (wb null: none).
// One launch for all layers (a launch each, ten of them, cost a training step 45 us).
struct PackTable {
    int start[11];  // first value of each layer's two layouts, the total last
    int cin[10], cinp[10], cout[10], kp[10], kpb[10];
    size_t w[10];
    bf16 *wt[10], *wb[10];
};

__global__ void k_pack(PackTable T, const float *__restrict__ params) {
    int i = blockIdx.x * blockDim.x + threadIdx.x, l = 0;
    if (i >= T.start[10]) return;
    while (i >= T.start[l + 1]) l++;
    i -= T.start[l];
    const int cin = T.cin[l], cout = T.cout[l], kp = T.kp[l], kpb = T.kpb[l], nf = cout * kp;
    const float *w = params + T.w[l];
    int tap, c;
    if (i < nf) {
        const int co = i / kp;
        const bool in = conv_k(T.cinp[l], i - co * kp, tap, c) && c < cin;
        T.wt[l][i] = (bf16)(in ? w[((size_t)tap * cin + c) * cout + co] : 0.0f);
    } else {
        const int j = i - nf, ci = j / kpb;
        const bool in = conv_k(cout, j - ci * kpb, tap, c);
        T.wb[l][j] = (bf16)(in ? w[((size_t)(8 - tap) * cin + ci) * cout + c] : 0.0f);
    }
}

// ------------------------------------------------------------------------------------------------------ host side
static const int LAYER_SHAPE[10][2] = {{3, 16}, {16, 16}, {16, 32}, {32, 32}, {32, 64},
                                       {64, 64}, {96, 32}, {32, 32}, {48, 16}, {16, 16}};
enum { E1A, E1, E2A, E2, E3A, E3, D2A, D2, D1A, D1 };

Net::~Net() {
    for (auto &l : L) {
        if (l.wt) (void)hipFree(l.wt);
        if (l.wb) (void)hipFree(l.wb);
    }
    void *ps[] = {params, grads, m, v, x, e1a, e1, p1, e2a, e2, p2, e3a, e3, d2a, d2, d1a, d1, g_d1, g_d1a,
                  g_d2, g_d2a, g_e3, g_e3a, g_e2, g_e2a, g_e1, g_e1a, dis, err, aerr, gout, wpart,
                  part, lpart, opart, scal};
    for (void *q : ps)
        if (q) (void)hipFree(q);
    if (host) (void)hipHostFree(host);
}

template <typename T> static int dalloc(T **p, size_t count) {
    SR_HIP(hipMalloc((void **)p, sizeof(T) * std::max<size_t>(count, 1)));
    SR_HIP(hipMemset(*p, 0, sizeof(T) * std::max<size_t>(count, 1)));
    return SR_OK;
}

int Net::init(int mw, int mh) {
    if (mw <= 0 || mh <= 0 || mw % 4 || mh % 4)
        return fail(SR_ERR_ARGUMENT, "the network's grid sides must be positive multiples of 4");
    max_w = mw;
    max_h = mh;
    size_t off = 0;
    for (int i = 0; i < 10; i++) {
        NetLayer l;
        l.cin = LAYER_SHAPE[i][0];
        l.cout = LAYER_SHAPE[i][1];
        l.cinp = i == E1A ? 8 : l.cin;
        l.kp = conv_kp(l.cinp);
        l.kpb = conv_kp(l.cout);
        l.w_off = off;
        off += (size_t)9 * l.cin * l.cout;
        l.b_off = off;
        off += l.cout;
        SR_TRY(dalloc(&l.wt, (size_t)l.cout * l.kp));
        if (i != E1A) SR_TRY(dalloc(&l.wb, (size_t)l.cin * l.kpb));
        L.push_back(l);
    }
    out_off = off;
    nparams = off + 17;
    SR_TRY(dalloc(&params, nparams));
    SR_TRY(dalloc(&grads, nparams));
    SR_TRY(dalloc(&m, nparams));
    SR_TRY(dalloc(&v, nparams));
    const size_t n = (size_t)mw * mh, n2 = n / 4, n4 = n / 16;
    SR_TRY(dalloc(&x, 8 * n));
    SR_TRY(dalloc(&e1a, 16 * n));
    SR_TRY(dalloc(&e1, 16 * n));
    SR_TRY(dalloc(&p1, 16 * n2));
    SR_TRY(dalloc(&e2a, 32 * n2));
    SR_TRY(dalloc(&e2, 32 * n2));
    SR_TRY(dalloc(&p2, 32 * n4));
    SR_TRY(dalloc(&e3a, 64 * n4));
    SR_TRY(dalloc(&e3, 64 * n4));
    SR_TRY(dalloc(&d2a, 32 * n2));
    SR_TRY(dalloc(&d2, 32 * n2));
    SR_TRY(dalloc(&d1a, 16 * n));
    SR_TRY(dalloc(&d1, 16 * n));
    SR_TRY(dalloc(&dis, n));
    SR_TRY(dalloc(&part, 2 * NB_FEAT));
    SR_TRY(dalloc(&scal, 4));
    SR_HIP(hipHostMalloc((void **)&host, sizeof(double) * 4 * NB_FEAT));
    return SR_OK;
}

int Net::set_params(const float *h, size_t n) {
    if (n != nparams) return fail(SR_ERR_LENGTH, "network parameters: expected " + std::to_string(nparams));
    SR_HIP(hipMemcpy(params, h, sizeof(float) * n, hipMemcpyHostToDevice));
    SR_HIP(hipMemset(m, 0, sizeof(float) * n));
    SR_HIP(hipMemset(v, 0, sizeof(float) * n));
    adam_t = 0;
    packed = false;
    return SR_OK;
}

int Net::get_params(float *h, size_t n) {
    if (n != nparams) return fail(SR_ERR_LENGTH, "network parameters: expected " + std::to_string(nparams));
    SR_HIP(hipMemcpy(h, params, sizeof(float) * n, hipMemcpyDeviceToHost));
    return SR_OK;
}

int Net::get_grads(float *h, size_t n) {
    if (n != nparams) return fail(SR_ERR_LENGTH, "network gradients: expected " + std::to_string(nparams));
    SR_HIP(hipMemcpy(h, grads, sizeof(float) * n, hipMemcpyDeviceToHost));
    return SR_OK;
}

int Net::pack(hipStream_t s) {
    PackTable T;
    T.start[0] = 0;
    for (int i = 0; i < 10; i++) {
        const NetLayer &l = L[i];
        T.cin[i] = l.cin;
        T.cinp[i] = l.cinp;
        T.cout[i] = l.cout;
        T.kp[i] = l.kp;
        T.kpb[i] = l.kpb;
        T.w[i] = l.w_off;
        T.wt[i] = l.wt;
        T.wb[i] = l.wb;
        T.start[i + 1] = T.start[i] + l.cout * l.kp + (l.wb ? l.cin * l.kpb : 0);
    }
    hipLaunchKernelGGL(k_pack, dim3((T.start[10] + 255) / 256), dim3(256), 0, s, T, (const float *)params);
    SR_HIP(hipGetLastError());
    packed = true;
    return SR_OK;
}

static ConvArgs cargs(const bf16 *in, const bf16 *up, int cup, const bf16 *mask, const bf16 *wt, const float *bias,
                      bf16 *out, int H, int W, int relu) {
    ConvArgs a;
    a.in = in;
    a.up = up;
    a.mask = mask;
    a.wt = wt;
    a.bias = bias;
    a.out = out;
    a.H = H;
    a.W = W;
    a.cup = cup;
    a.relu = relu;
    return a;
}

static int grid_of(size_t n) { return (int)std::min<size_t>(NB_FEAT, (n + NTH - 1) / NTH); }

int Net::forward(int w, int h, const float *own, const float *kx, const float *ky, const float *r, const float *zadd,
                 float *z, const float *e, float *err, hipStream_t s) {
    if (w <= 0 || h <= 0 || w % 4 || h % 4 || w > max_w || h > max_h || (size_t)w * h > (size_t)max_w * max_h)
        return fail(SR_ERR_ARGUMENT, "network input size outside the multiples of 4 it was created for");
    if (!own || !kx || !ky || !r) return fail(SR_ERR_ARGUMENT, "network: null system array");
    if (!packed) SR_TRY(pack(s));
    const size_t n = (size_t)w * h;
    const int nb = grid_of(n);
    nb_feat = nb;
    last_w = w;
    last_h = h;
    hipLaunchKernelGGL(k_feat_sums, dim3(nb), dim3(NTH), 0, s, w, h, own, kx, ky, r, part);
    hipLaunchKernelGGL(k_feat, dim3(nb), dim3(NTH), 0, s, w, h, own, kx, ky, r, (const double *)part, nb, x, dis, scal);
    const int w2 = w / 2, h2 = h / 2, w4 = w / 4, h4 = h / 4;
    auto B = [&](int i) { return (const float *)(params + L[i].b_off); };
    auto with_half = [](ConvArgs a, bf16 *half) {
        a.half = half;
        return a;
    };
    conv<8, 16>(s, cargs(x, nullptr, 0, nullptr, L[E1A].wt, B(E1A), e1a, h, w, 1));
    conv<16, 16, CONV_POOL>(s, with_half(cargs(e1a, nullptr, 0, nullptr, L[E1].wt, B(E1), e1, h, w, 1), p1));
    conv<16, 32>(s, cargs(p1, nullptr, 0, nullptr, L[E2A].wt, B(E2A), e2a, h2, w2, 1));
    conv<32, 32, CONV_POOL>(s, with_half(cargs(e2a, nullptr, 0, nullptr, L[E2].wt, B(E2), e2, h2, w2, 1), p2));
    conv<32, 64>(s, cargs(p2, nullptr, 0, nullptr, L[E3A].wt, B(E3A), e3a, h4, w4, 1));
    conv<64, 64>(s, cargs(e3a, nullptr, 0, nullptr, L[E3].wt, B(E3), e3, h4, w4, 1));
    conv<96, 32>(s, cargs(e2, e3, 64, nullptr, L[D2A].wt, B(D2A), d2a, h2, w2, 1));
    conv<32, 32>(s, cargs(d2a, nullptr, 0, nullptr, L[D2].wt, B(D2), d2, h2, w2, 1));
    conv<48, 16>(s, cargs(e1, d2, 32, nullptr, L[D1A].wt, B(D1A), d1a, h, w, 1));
    ConvArgs last = cargs(d1a, nullptr, 0, nullptr, L[D1].wt, B(D1), d1, h, w, 1);
    last.wout = params + out_off;
    last.scal = scal;
    last.dis = dis;
    last.zadd = zadd;
    last.z = z;
    last.e = e;
    last.err = err;
    conv<16, 16, CONV_OUT>(s, last);
    SR_HIP(hipGetLastError());
    return SR_OK;
}

int Net::apply(int w, int h, const float *own, const float *kx, const float *ky, const float *r, const float *zadd,
               float *z, hipStream_t s) {
    if (!z) return fail(SR_ERR_ARGUMENT, "network: null output");
    return forward(w, h, own, kx, ky, r, zadd, z, nullptr, nullptr, s);
}

// The weight gradient's blocks for an image: a tile each up to as many as the partials' size allows (four to a CU where
// the layer is small: a block waits on its tile's loads before it computes; one where every block's partials are 100 KB),
// then as few as take the same number of turns.
static int dw_blocks_most(int size) { return std::max(256, std::min(1024, DW_FLOATS / size)); }
static int dw_tiles(int H, int W) { return ((W + DW_TW - 1) / DW_TW) * ((H + DW_TH - 1) / DW_TH); }
static int dw_blocks(int H, int W, int size) {
    const int nt = dw_tiles(H, W), most = dw_blocks_most(size), turns = (nt + most - 1) / most;
    return (nt + turns - 1) / turns;
}

template <int CIN, int COUT>
static void dw(hipStream_t s, const bf16 *in, const bf16 *up, int cup, const bf16 *gy, const bf16 *y, int H, int W,
               float *wpart, const NetLayer &l, DwTable &T) {
    const int nb = dw_blocks(H, W, 9 * CIN * COUT + COUT), k = T.n++, nout = 9 * l.cin * l.cout + l.cout;
    T.nb[k] = nb;
    T.cinp[k] = l.cinp;
    T.cin[k] = l.cin;
    T.cout[k] = l.cout;
    T.w[k] = l.w_off;
    T.b[k] = l.b_off;
    if (k == 0) {
        T.start[0] = 0;
        T.part[0] = 0;
    }
    hipLaunchKernelGGL((k_dw<CIN, COUT>), dim3(nb), dim3(NTH), 0, s, in, up, cup, gy, y, H, W, wpart + T.part[k]);
    if (k + 1 < 10) {
        T.start[k + 1] = T.start[k] + (nout + 31) / 32;
        T.part[k + 1] = T.part[k] + (size_t)nb * (9 * l.cinp * l.cout + l.cout);
    }
}

int Net::loss_grad(int w, int h, const float *own, const float *kx, const float *ky, const float *r, const float *e,
                   double *loss, hipStream_t s) {
    if (!e) return fail(SR_ERR_ARGUMENT, "network: null target");
    if (!g_d1) {  // training buffers, allocated at the first training call
        const size_t n = (size_t)max_w * max_h, n2 = n / 4, n4 = n / 16;
        SR_TRY(dalloc(&g_d1, 16 * n));
        SR_TRY(dalloc(&g_d1a, 16 * n));
        SR_TRY(dalloc(&g_d2, 32 * n2));
        SR_TRY(dalloc(&g_d2a, 32 * n2));
        SR_TRY(dalloc(&g_e3, 64 * n4));
        SR_TRY(dalloc(&g_e3a, 64 * n4));
        SR_TRY(dalloc(&g_e2, 32 * n2));
        SR_TRY(dalloc(&g_e2a, 32 * n2));
        SR_TRY(dalloc(&g_e1, 16 * n));
        SR_TRY(dalloc(&g_e1a, 16 * n));
        SR_TRY(dalloc(&err, n));
        SR_TRY(dalloc(&aerr, n));
        SR_TRY(dalloc(&gout, n));
        SR_TRY(dalloc(&lpart, 2 * NB_FEAT));
        SR_TRY(dalloc(&opart, 17 * NB_FEAT));
        // every layer's weight-gradient partials, each layer's at its own resolution
        const int shift[10] = {0, 0, 1, 1, 2, 2, 1, 1, 0, 0};
        size_t parts = 0;
        for (int i = 0; i < 10; i++) {
            const int size = 9 * L[i].cinp * L[i].cout + L[i].cout;
            parts += (size_t)std::min(dw_blocks_most(size), dw_tiles(max_h >> shift[i], max_w >> shift[i])) * size;
        }
        SR_TRY(dalloc(&wpart, parts));
    }
    SR_TRY(forward(w, h, own, kx, ky, r, nullptr, nullptr, e, err, s));
    const size_t n = (size_t)w * h;
    const int nb = grid_of(n);
    const int w2 = w / 2, h2 = h / 2, w4 = w / 4, h4 = h / 4;
    DwTable T;
    T.n = 0;
    hipLaunchKernelGGL(k_loss, dim3(nb), dim3(NTH), 0, s, w, h, own, kx, ky, (const float *)err, e, aerr, lpart);
    hipLaunchKernelGGL(k_out_back, dim3(nb), dim3(NTH), 0, s, (int)n, (const float *)aerr, (const double *)lpart, nb,
                       (const float *)scal, (const float *)dis, (const bf16 *)d1, (const float *)(params + out_off),
                       gout, g_d1, opart);
    hipLaunchKernelGGL(k_reduce_rows, dim3(17), dim3(NTH), 0, s, (const double *)opart, nb, grads + out_off);
    // decoder, level 1
    dw<16, 16>(s, d1a, nullptr, 0, g_d1, d1, h, w, wpart, L[D1], T);
    conv<16, 16>(s, cargs(g_d1, nullptr, 0, d1, L[D1].wb, nullptr, g_d1a, h, w, 0));
    dw<48, 16>(s, e1, d2, 32, g_d1a, d1a, h, w, wpart, L[D1A], T);
    ConvArgs cat = cargs(g_d1a, nullptr, 0, d1a, L[D1A].wb, nullptr, g_e1, h, w, 0);
    cat.half = g_d2;
    conv<16, 48, CONV_SPLIT>(s, cat);
    // decoder, level 2
    dw<32, 32>(s, d2a, nullptr, 0, g_d2, d2, h2, w2, wpart, L[D2], T);
    conv<32, 32>(s, cargs(g_d2, nullptr, 0, d2, L[D2].wb, nullptr, g_d2a, h2, w2, 0));
    dw<96, 32>(s, e2, e3, 64, g_d2a, d2a, h2, w2, wpart, L[D2A], T);
    cat = cargs(g_d2a, nullptr, 0, d2a, L[D2A].wb, nullptr, g_e2, h2, w2, 0);
    cat.half = g_e3;
    conv<32, 96, CONV_SPLIT>(s, cat);
    // encoder, level 3
    dw<64, 64>(s, e3a, nullptr, 0, g_e3, e3, h4, w4, wpart, L[E3], T);
    conv<64, 64>(s, cargs(g_e3, nullptr, 0, e3, L[E3].wb, nullptr, g_e3a, h4, w4, 0));
    dw<32, 64>(s, p2, nullptr, 0, g_e3a, e3a, h4, w4, wpart, L[E3A], T);
    conv<64, 32, CONV_UNPOOL>(s, cargs(g_e3a, nullptr, 0, e3a, L[E3A].wb, nullptr, g_e2, h4, w4, 0));
    // encoder, level 2
    dw<32, 32>(s, e2a, nullptr, 0, g_e2, e2, h2, w2, wpart, L[E2], T);
    conv<32, 32>(s, cargs(g_e2, nullptr, 0, e2, L[E2].wb, nullptr, g_e2a, h2, w2, 0));
    dw<16, 32>(s, p1, nullptr, 0, g_e2a, e2a, h2, w2, wpart, L[E2A], T);
    conv<32, 16, CONV_UNPOOL>(s, cargs(g_e2a, nullptr, 0, e2a, L[E2A].wb, nullptr, g_e1, h2, w2, 0));
    // encoder, level 1
    dw<16, 16>(s, e1a, nullptr, 0, g_e1, e1, h, w, wpart, L[E1], T);
    conv<16, 16>(s, cargs(g_e1, nullptr, 0, e1, L[E1].wb, nullptr, g_e1a, h, w, 0));
    dw<8, 16>(s, x, nullptr, 0, g_e1a, e1a, h, w, wpart, L[E1A], T);
    const NetLayer &l0 = L[E1A];  // the last in the table
    const int rblocks = T.start[9] + (9 * l0.cin * l0.cout + l0.cout + 31) / 32;
    hipLaunchKernelGGL(k_dw_reduce, dim3(rblocks), dim3(NTH), 0, s, T, (const float *)wpart, grads);
    SR_HIP(hipGetLastError());
    if (loss) {
        SR_HIP(hipMemcpyAsync(host, lpart, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, s));
        SR_HIP(hipStreamSynchronize(s));
        double a = 0.0, b = 0.0;
        for (int i = 0; i < nb; i++) {
            a += host[i];
            b += host[nb + i];
        }
        *loss = b > 0.0 ? a / b : 0.0;
    }
    return SR_OK;
}

int Net::adam(double lr, hipStream_t s) {
    adam_t++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float bc1 = 1.0f - powf(b1, (float)adam_t), bc2 = 1.0f - powf(b2, (float)adam_t);
    hipLaunchKernelGGL(k_adam, dim3((nparams + 255) / 256), dim3(256), 0, s, (int)nparams, params,
                       (const float *)grads, m, v, (float)lr, b1, b2, 1e-8f, bc1, bc2);
    SR_HIP(hipGetLastError());
    packed = false;
    return SR_OK;
}

int Net::activation(const char *name, float *out, size_t count) {
    const size_t n = (size_t)last_w * last_h, n2 = n / 4, n4 = n / 16;
    struct A {
        const char *nm;
        const bf16 *p;
        size_t c;
    } t[] = {{"x", x, 8 * n},        {"e1a", e1a, 16 * n}, {"e1", e1, 16 * n},   {"p1", p1, 16 * n2},
             {"e2a", e2a, 32 * n2},  {"e2", e2, 32 * n2},  {"p2", p2, 32 * n4},  {"e3a", e3a, 64 * n4},
             {"e3", e3, 64 * n4},    {"d2a", d2a, 32 * n2}, {"d2", d2, 32 * n2}, {"d1a", d1a, 16 * n},
             {"d1", d1, 16 * n}};
    for (const A &a : t) {
        if (std::strcmp(a.nm, name) != 0) continue;
        if (count != a.c) return fail(SR_ERR_LENGTH, std::string("activation ") + name + ": expected " + std::to_string(a.c));
        std::vector<uint16_t> tmp(a.c);
        SR_HIP(hipMemcpy(tmp.data(), a.p, sizeof(uint16_t) * a.c, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < a.c; i++) {
            const uint32_t bits = (uint32_t)tmp[i] << 16;
            std::memcpy(out + i, &bits, 4);
        }
        return SR_OK;
    }
    return fail(SR_ERR_ARGUMENT, std::string("no activation named ") + name);
}

// HBM bytes of one application by its algorithm: every activation written once and read by its consumers (3x3
// reads counted once), the features' inputs, the output
double Net::bytes_per_apply(int w, int h) const {
    const double n = (double)w * h;
    const double act = 2.0 * (8 + 16 + 16 + 16 + 16) * n                        // x, e1a, e1, d1a, d1
                       + 2.0 * (16 + 32 + 32 + 32 + 32) * n / 4                 // p1, e2a, e2, d2a, d2
                       + 2.0 * (32 + 64 + 64) * n / 16;                         // p2, e3a, e3
    return 2.0 * act + (16.0 + 4.0 + 8.0) * n;
}

double Net::flops_per_apply(int w, int h) const {
    double f = 0.0;
    const double n = (double)w * h;
    const double scale[10] = {1, 1, 0.25, 0.25, 1.0 / 16, 1.0 / 16, 0.25, 0.25, 1, 1};
    for (int i = 0; i < 10; i++) f += 2.0 * 9 * L[i].cin * L[i].cout * n * scale[i];
    return f + 2.0 * 16 * n;
}

} // namespace sr

// ------------------------------------------------------------------------------------------------------------ C ABI
using namespace sr;

struct sr_net {
    Net n;
};

extern "C" int sr_net_create(int max_w, int max_h, sr_net **out) {
    if (!out) return fail(SR_ERR_ARGUMENT, "sr_net_create: null out");
    auto *p = new sr_net();
    const int c = p->n.init(max_w, max_h);
    if (c != SR_OK) {
        delete p;
        return c;
    }
    *out = p;
    return SR_OK;
}

extern "C" int sr_net_param_count(sr_net *p, size_t *n) {
    if (!p || !n) return fail(SR_ERR_ARGUMENT, "sr_net_param_count: null pointer");
    *n = p->n.param_count();
    return SR_OK;
}

extern "C" int sr_net_set_params(sr_net *p, const float *params, size_t n) {
    if (!p || !params) return fail(SR_ERR_ARGUMENT, "sr_net_set_params: null pointer");
    return p->n.set_params(params, n);
}

extern "C" int sr_net_get_params(sr_net *p, float *params, size_t n) {
    if (!p || !params) return fail(SR_ERR_ARGUMENT, "sr_net_get_params: null pointer");
    return p->n.get_params(params, n);
}

extern "C" int sr_net_get_grads(sr_net *p, float *grads, size_t n) {
    if (!p || !grads) return fail(SR_ERR_ARGUMENT, "sr_net_get_grads: null pointer");
    return p->n.get_grads(grads, n);
}

extern "C" int sr_net_apply(sr_net *p, int w, int h, const float *own, const float *kx, const float *ky,
                            const float *r, float *z, void *stream) {
    if (!p) return fail(SR_ERR_ARGUMENT, "sr_net_apply: null network");
    return p->n.apply(w, h, own, kx, ky, r, nullptr, z, (hipStream_t)stream);
}

extern "C" int sr_net_loss_grad(sr_net *p, int w, int h, const float *own, const float *kx, const float *ky,
                                const float *r, const float *e, double *loss, void *stream) {
    if (!p) return fail(SR_ERR_ARGUMENT, "sr_net_loss_grad: null network");
    return p->n.loss_grad(w, h, own, kx, ky, r, e, loss, (hipStream_t)stream);
}

extern "C" int sr_net_adam(sr_net *p, double lr, void *stream) {
    if (!p) return fail(SR_ERR_ARGUMENT, "sr_net_adam: null network");
    if (!(lr > 0.0)) return fail(SR_ERR_ARGUMENT, "sr_net_adam: the learning rate must be positive");
    return p->n.adam(lr, (hipStream_t)stream);
}

extern "C" int sr_net_activation(sr_net *p, const char *name, float *out, size_t count) {
    if (!p || !name || !out) return fail(SR_ERR_ARGUMENT, "sr_net_activation: null pointer");
    return p->n.activation(name, out, count);
}

extern "C" void sr_net_destroy(sr_net *p) { delete p; }

namespace sr {
Net *net_of(sr_net *p) { return p ? &p->n : nullptr; }
}
