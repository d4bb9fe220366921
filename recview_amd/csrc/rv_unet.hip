// rv_unet.hip -- CDNA4 kernels of the learned restoration stage.
//
// 3x3 convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16:
//   forward / data gradient: M = 16 pixels of an image row, N = 16 output
//   channels, K = 32 input channels of one tap.  A block owns a 16 x 16 pixel
//   patch and 16*NF output channels; per 32-channel chunk it stages the 18 x 18
//   halo (96-byte pixel pitch, conflict-free 16-byte reads) and the chunk's
//   weights (already in fragment order) in LDS, then each wave runs
//   9 taps x 4 rows x NF fragments of MFMA.
//   weight gradient: M = 16 output channels, N = 16 input channels, K = 32
//   pixels.  Pixels are the contraction; the LDS transpose reads turn the
//   channel-contiguous dY and X into pixel-contiguous fragments.
// Operand layouts (checked on gfx950): A[i][k] in lane i + 16*(k/8), element
// k%8; B[k][j] in lane j + 16*(k/8), element k%8; D[i][j] in lane j + 16*(i/4),
// element i%4.
#include "rv_unet.h"

#include <algorithm>
#include <cmath>

namespace rv {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ uint16_t f2bf(float f) {
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}
static __device__ __forceinline__ float bf2f(uint16_t u) {
    return __uint_as_float((uint32_t)u << 16);
}
static __device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *(const uint4*)p; }
static __device__ __forceinline__ void st16(uint16_t* p, uint4 v) { *(uint4*)p = v; }

// ------------------------------------------------------------ conv forward
// Row pitches of LDS tiles read as 16-byte fragments (16 rows x 4 groups per
// wave): measured conflict-free on gfx950 when the pitch is 32 mod 64 bytes
// (80, 112, 144, 272, 336 bytes conflict 2x, 128 bytes 4x).
constexpr int HALO_PITCH = 48;          // bf16 per staged pixel: 32 channels + 16 pad
constexpr int CONV_ROWS = 16;           // patch rows (4 per wave)
constexpr int HALO_ROWS = CONV_ROWS + 2;
constexpr int HALO_PIX = HALO_ROWS * 18;
constexpr int HALO_ITEMS = HALO_PIX * 4;          // 16-byte loads per chunk
constexpr int HALO_PER = (HALO_ITEMS + 255) / 256;

// One block: a 16-wide, 4*MR-row pixel patch of one image and 16*NF output
// channels.  Wave w owns patch rows MR*w .. MR*w+MR-1 (MR M fragments) and all
// NF N fragments, so per tap it reads MR A and NF B fragments for MR*NF MFMAs.
// The next 32-channel chunk is fetched into registers while the current one is
// multiplied; the epilogue goes through LDS so every store is 16 bytes.
template <int NF, int MR>
__global__ __launch_bounds__(256, 2) void conv3x3_kernel(ConvArgs a) {
    constexpr int ROWS = 4 * MR;
    constexpr int HALO_PIX_K = (ROWS + 2) * 18;
    constexpr int HALO_ITEMS_K = HALO_PIX_K * 4;
    constexpr int HALO_PER_K = (HALO_ITEMS_K + 255) / 256;
    constexpr int NPIX = 16 * ROWS;
    constexpr int HSZ = HALO_PIX_K * HALO_PITCH;
    constexpr int WSZ = NF * 576 * 8;
    constexpr int TC = 16 * NF;
    constexpr int OPITCH = TC + 8;
    constexpr int OSZ = NPIX * OPITCH;
    constexpr int SMEM = HSZ + WSZ > OSZ ? HSZ + WSZ : OSZ;
    constexpr int W_ITEMS = NF * 576;
    constexpr int W_PER = (W_ITEMS + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t smem[SMEM];
    uint16_t* in_s = smem;
    uint16_t* w_s = smem + HSZ;
    const int tiles_x = (a.W + 15) >> 4;
    const int x0 = (blockIdx.x % tiles_x) * 16, y0 = (blockIdx.x / tiles_x) * ROWS;
    const int bb = blockIdx.z, f0 = blockIdx.y * NF;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int nch = a.Cin >> 5;
    const uint16_t* in = a.in + (long long)bb * a.H * a.W * a.in_stride + a.in_off;
    const uint16_t* up = a.up ? a.up + (long long)bb * (a.H >> 1) * (a.W >> 1) * a.Cup : nullptr;
    floatx4 acc[MR][NF];
#pragma unroll
    for (int m = 0; m < MR; m++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};

    uint4 hreg[HALO_PER_K], wreg[W_PER];
    auto fetch = [&](int cc) {
#pragma unroll
        for (int k = 0; k < HALO_PER_K; k++) {
            const int i = t + 256 * k;
            const int hp = i >> 2, g = i & 3;
            const int hy = hp / 18, hx = hp - hy * 18;
            const int y = y0 - 1 + hy, x = x0 - 1 + hx;
            hreg[k] = make_uint4(0, 0, 0, 0);
            if (i < HALO_ITEMS_K && y >= 0 && y < a.H && x >= 0 && x < a.W) {
                if (cc * 32 < a.Cup)
                    hreg[k] = ld16(up + ((long long)(y >> 1) * (a.W >> 1) + (x >> 1)) * a.Cup + cc * 32 +
                                   g * 8);
                else
                    hreg[k] = ld16(in + ((long long)y * a.W + x) * a.in_stride + cc * 32 + g * 8);
            }
        }
#pragma unroll
        for (int k = 0; k < W_PER; k++) {
            const int i = t + 256 * k;
            if (i < W_ITEMS) {
                const int f = i / 576, r = i - f * 576;
                wreg[k] = ld16(a.wfrag + ((long long)((f0 + f) * nch + cc) * 576 + r) * 8);
            }
        }
    };
    fetch(0);
    for (int cc = 0; cc < nch; cc++) {
#pragma unroll
        for (int k = 0; k < HALO_PER_K; k++) {
            const int i = t + 256 * k;
            if (i < HALO_ITEMS_K) st16(in_s + (i >> 2) * HALO_PITCH + (i & 3) * 8, hreg[k]);
        }
#pragma unroll
        for (int k = 0; k < W_PER; k++) {
            const int i = t + 256 * k;
            if (i < W_ITEMS) st16(w_s + i * 8, wreg[k]);
        }
        __syncthreads();
        if (cc + 1 < nch) fetch(cc + 1);
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int ky = tap / 3, kx = tap % 3;
            bf16x8 av[MR], bv[NF];
#pragma unroll
            for (int m = 0; m < MR; m++)
                av[m] = *(const bf16x8*)(in_s + ((MR * w + m + ky) * 18 + (l & 15) + kx) * HALO_PITCH +
                                         8 * (l >> 4));
#pragma unroll
            for (int f = 0; f < NF; f++) bv[f] = *(const bf16x8*)(w_s + ((f * 9 + tap) * 64 + l) * 8);
            // all fragment reads of the tap are in flight before its first MFMA
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < NF; f++)
#pragma unroll
                for (int m = 0; m < MR; m++)
                    acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv[f], acc[m][f], 0, 0, 0);
        }
        __syncthreads();
    }
    // epilogue: bias, ReLU, bf16 into an LDS tile [NPIX pixels][TC], then 16-byte stores
    uint16_t* o_s = smem;
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int co = f * 16 + (l & 15);
        const float bias = a.bias ? a.bias[(f0 * 16) + co] : 0.f;
#pragma unroll
        for (int m = 0; m < MR; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = acc[m][f][i] + bias;
                if (a.relu) v = fmaxf(v, 0.f);
                o_s[((MR * w + m) * 16 + 4 * (l >> 4) + i) * OPITCH + co] = f2bf(v);
            }
    }
    __syncthreads();
    if (a.pool_out) {
        // 8 x ROWS/2 pooled pixels of this patch, from the rounded outputs
        const int Ho = a.H >> 1, Wo = a.W >> 1;
        for (int it = t; it < 4 * ROWS * (TC / 8); it += 256) {
            const int q = it / (TC / 8), g = it - q * (TC / 8);
            const int py = q >> 3, pxx = q & 7;
            const int yo = (y0 >> 1) + py, xo = (x0 >> 1) + pxx;
            if (yo >= Ho || xo >= Wo) continue;
            float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int px = (2 * py + (k >> 1)) * 16 + 2 * pxx + (k & 1);
                const uint4 v = ld16(o_s + px * OPITCH + 8 * g);
                const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
                for (int e = 0; e < 8; e++) sum[e] += bf2f(v8[e]);
            }
            uint4 r;
            uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
            for (int e = 0; e < 8; e++) r8[e] = f2bf(0.25f * sum[e]);
            st16(a.pool_out + (((long long)bb * Ho + yo) * Wo + xo) * a.Cout + f0 * 16 + 8 * g, r);
        }
    }
    for (int it = t; it < NPIX * (TC / 8); it += 256) {
        const int px = it / (TC / 8), g = it - px * (TC / 8);
        const int y = y0 + (px >> 4), x = x0 + (px & 15);
        if (y >= a.H || x >= a.W) continue;
        const long long pix = ((long long)bb * a.H + y) * a.W + x;
        const int c = f0 * 16 + 8 * g;
        uint4 v = ld16(o_s + px * OPITCH + 8 * g);
        if (a.mask) {
            const uint4 mv = ld16(a.mask + pix * a.mask_stride + a.mask_off + c);
            uint16_t* v8 = (uint16_t*)&v;
            const uint16_t* m8 = (const uint16_t*)&mv;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (!(bf2f(m8[e]) > 0.f)) v8[e] = 0;
        }
        st16(a.out + pix * a.out_stride + a.out_off + c, v);
    }
}

// 32-channel inputs (one chunk): a block walks PPB consecutive 16 x 16
// patches with the weights staged once.  The next patch's halo is fetched into
// registers while the current one is multiplied; the output tile has its own
// LDS so the weights survive the epilogue.
template <int NF, int PPB>
__global__ __launch_bounds__(256, 2) void conv3x3_c32_kernel(ConvArgs a) {
    constexpr int HSZ = HALO_PIX * HALO_PITCH;
    constexpr int WSZ = NF * 576 * 8;
    constexpr int TC = 16 * NF;
    constexpr int OPITCH = TC + 8;
    constexpr int W_ITEMS = NF * 576;
    constexpr int W_PER = (W_ITEMS + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t smem[HSZ + WSZ + 256 * OPITCH];
    uint16_t* in_s = smem;
    uint16_t* w_s = smem + HSZ;
    uint16_t* o_s = w_s + WSZ;
    const int tiles_x = (a.W + 15) >> 4;
    const int ntiles = tiles_x * ((a.H + CONV_ROWS - 1) / CONV_ROWS);
    const int tile0 = blockIdx.x * PPB;
    const int npatch = ntiles - tile0 < PPB ? ntiles - tile0 : PPB;
    const int bb = blockIdx.z, f0 = blockIdx.y * NF;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const uint16_t* in = a.in + (long long)bb * a.H * a.W * a.in_stride + a.in_off;
    const uint16_t* up = a.up ? a.up + (long long)bb * (a.H >> 1) * (a.W >> 1) * a.Cup : nullptr;

#pragma unroll
    for (int k = 0; k < W_PER; k++) {
        const int i = t + 256 * k;
        if (i < W_ITEMS) {
            const int f = i / 576, r = i - f * 576;
            st16(w_s + i * 8, ld16(a.wfrag + ((long long)(f0 + f) * 576 + r) * 8));
        }
    }
    uint4 hreg[HALO_PER];
    auto fetch = [&](int p) {
        const int tile = tile0 + p;
        const int x0 = (tile % tiles_x) * 16, y0 = (tile / tiles_x) * CONV_ROWS;
#pragma unroll
        for (int k = 0; k < HALO_PER; k++) {
            const int i = t + 256 * k;
            const int hp = i >> 2, g = i & 3;
            const int hy = hp / 18, hx = hp - hy * 18;
            const int y = y0 - 1 + hy, x = x0 - 1 + hx;
            hreg[k] = make_uint4(0, 0, 0, 0);
            if (i < HALO_ITEMS && y >= 0 && y < a.H && x >= 0 && x < a.W) {
                if (a.Cup > 0)
                    hreg[k] = ld16(up + ((long long)(y >> 1) * (a.W >> 1) + (x >> 1)) * a.Cup + g * 8);
                else
                    hreg[k] = ld16(in + ((long long)y * a.W + x) * a.in_stride + g * 8);
            }
        }
    };
    fetch(0);
    for (int p = 0; p < npatch; p++) {
        const int tile = tile0 + p;
        const int x0 = (tile % tiles_x) * 16, y0 = (tile / tiles_x) * CONV_ROWS;
#pragma unroll
        for (int k = 0; k < HALO_PER; k++) {
            const int i = t + 256 * k;
            if (i < HALO_ITEMS) st16(in_s + (i >> 2) * HALO_PITCH + (i & 3) * 8, hreg[k]);
        }
        __syncthreads();
        if (p + 1 < npatch) fetch(p + 1);
        floatx4 acc[4][NF];
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int f = 0; f < NF; f++) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int ky = tap / 3, kx = tap % 3;
            bf16x8 av[4], bv[NF];
#pragma unroll
            for (int m = 0; m < 4; m++)
                av[m] = *(const bf16x8*)(in_s + ((4 * w + m + ky) * 18 + (l & 15) + kx) * HALO_PITCH +
                                         8 * (l >> 4));
#pragma unroll
            for (int f = 0; f < NF; f++) bv[f] = *(const bf16x8*)(w_s + ((f * 9 + tap) * 64 + l) * 8);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < NF; f++)
#pragma unroll
                for (int m = 0; m < 4; m++)
                    acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv[f], acc[m][f], 0, 0, 0);
        }
        // bias, ReLU, bf16 into the output tile [256 pixels][TC]
#pragma unroll
        for (int f = 0; f < NF; f++) {
            const int co = f * 16 + (l & 15);
            const float bias = a.bias ? a.bias[(f0 * 16) + co] : 0.f;
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float v = acc[m][f][i] + bias;
                    if (a.relu) v = fmaxf(v, 0.f);
                    o_s[((4 * w + m) * 16 + 4 * (l >> 4) + i) * OPITCH + co] = f2bf(v);
                }
        }
        __syncthreads();
        if (a.pool_out) {
            const int Ho = a.H >> 1, Wo = a.W >> 1;
            for (int it = t; it < 64 * (TC / 8); it += 256) {
                const int q = it / (TC / 8), g = it - q * (TC / 8);
                const int py = q >> 3, pxx = q & 7;
                const int yo = (y0 >> 1) + py, xo = (x0 >> 1) + pxx;
                if (yo >= Ho || xo >= Wo) continue;
                float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int px = (2 * py + (k >> 1)) * 16 + 2 * pxx + (k & 1);
                    const uint4 v = ld16(o_s + px * OPITCH + 8 * g);
                    const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
                    for (int e = 0; e < 8; e++) sum[e] += bf2f(v8[e]);
                }
                uint4 r;
                uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
                for (int e = 0; e < 8; e++) r8[e] = f2bf(0.25f * sum[e]);
                st16(a.pool_out + (((long long)bb * Ho + yo) * Wo + xo) * a.Cout + f0 * 16 + 8 * g, r);
            }
        }
        for (int it = t; it < 256 * (TC / 8); it += 256) {
            const int px = it / (TC / 8), g = it - px * (TC / 8);
            const int y = y0 + (px >> 4), x = x0 + (px & 15);
            if (y >= a.H || x >= a.W) continue;
            const long long pix = ((long long)bb * a.H + y) * a.W + x;
            const int c = f0 * 16 + 8 * g;
            uint4 v = ld16(o_s + px * OPITCH + 8 * g);
            if (a.mask) {
                const uint4 mv = ld16(a.mask + pix * a.mask_stride + a.mask_off + c);
                uint16_t* v8 = (uint16_t*)&v;
                const uint16_t* m8 = (const uint16_t*)&mv;
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (!(bf2f(m8[e]) > 0.f)) v8[e] = 0;
            }
            st16(a.out + pix * a.out_stride + a.out_off + c, v);
        }
        // the next iteration's halo store and output-tile writes are each
        // separated from this iteration's reads by one barrier
    }
}

// Encoder level 0 in one pass for 32 base channels: the edge convolution
// (1 -> 32, ReLU) of each patch's 18 x 18 halo is computed from a 20 x 20 tile
// of the input image in LDS, in edge_in_kernel's operation order (bias, the
// nine taps by fmaf, ReLU, bf16), straight into the halo tile of the 32 -> 32
// convolution; the MFMA loop and the epilogue (bias, ReLU, 2x2 pool, stores)
// are conv3x3_c32_kernel's.  The 32-channel edge output never goes to HBM.
// Halo item i = t + 256 k covers pixel i / 4 and channel group i % 4 = t % 4,
// so a thread keeps one channel group's 72 edge weights in registers.
template <int PPB>
__global__ __launch_bounds__(256, 2) void edge_c32_kernel(ConvArgs a, const float* x, const float* ew,
                                                          const float* eb) {
    constexpr int NF = 2;
    constexpr int HSZ = HALO_PIX * HALO_PITCH;
    constexpr int WSZ = NF * 576 * 8;
    constexpr int TC = 16 * NF;
    constexpr int OPITCH = TC + 8;
    constexpr int W_ITEMS = NF * 576;
    constexpr int W_PER = (W_ITEMS + 255) / 256;
    constexpr int XW = 20, XPIX = (CONV_ROWS + 4) * XW;     // input tile: halo 2 around the patch
    constexpr int X_PER = (XPIX + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t smem[HSZ + WSZ + 256 * OPITCH];
    __shared__ float xs[XPIX];
    uint16_t* in_s = smem;
    uint16_t* w_s = smem + HSZ;
    uint16_t* o_s = w_s + WSZ;
    const int tiles_x = (a.W + 15) >> 4;
    const int ntiles = tiles_x * ((a.H + CONV_ROWS - 1) / CONV_ROWS);
    const int tile0 = blockIdx.x * PPB;
    const int npatch = ntiles - tile0 < PPB ? ntiles - tile0 : PPB;
    const int bb = blockIdx.z;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const float* xb = x + (long long)bb * a.H * a.W;

#pragma unroll
    for (int k = 0; k < W_PER; k++) {
        const int i = t + 256 * k;
        if (i < W_ITEMS) st16(w_s + i * 8, ld16(a.wfrag + (long long)i * 8));
    }
    const int g = t & 3;
    float ewr[8][9], ebr[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        ebr[e] = eb[8 * g + e];
#pragma unroll
        for (int tap = 0; tap < 9; tap++) ewr[e][tap] = ew[(8 * g + e) * 9 + tap];
    }
    float xreg[X_PER];
    auto fetch = [&](int p) {
        const int tile = tile0 + p;
        const int x0 = (tile % tiles_x) * 16, y0 = (tile / tiles_x) * CONV_ROWS;
#pragma unroll
        for (int k = 0; k < X_PER; k++) {
            const int i = t + 256 * k;
            const int ty = i / XW, tx = i - ty * XW;
            const int y = y0 - 2 + ty, xx = x0 - 2 + tx;
            xreg[k] = (i < XPIX && y >= 0 && y < a.H && xx >= 0 && xx < a.W) ? xb[(long long)y * a.W + xx] : 0.f;
        }
    };
    fetch(0);
    for (int p = 0; p < npatch; p++) {
        const int tile = tile0 + p;
        const int x0 = (tile % tiles_x) * 16, y0 = (tile / tiles_x) * CONV_ROWS;
#pragma unroll
        for (int k = 0; k < X_PER; k++) {
            const int i = t + 256 * k;
            if (i < XPIX) xs[i] = xreg[k];
        }
        __syncthreads();
        if (p + 1 < npatch) fetch(p + 1);
        // edge convolution of the halo: zero outside the image (the 32 -> 32
        // convolution's padding), the tile's zeros are the edge layer's padding
#pragma unroll
        for (int k = 0; k < HALO_PER; k++) {
            const int i = t + 256 * k;
            if (i < HALO_ITEMS) {
                const int hp = i >> 2;
                const int hy = hp / 18, hx = hp - hy * 18;
                const int y = y0 - 1 + hy, xx = x0 - 1 + hx;
                uint4 r = make_uint4(0, 0, 0, 0);
                if (y >= 0 && y < a.H && xx >= 0 && xx < a.W) {
                    float v[9];
#pragma unroll
                    for (int tap = 0; tap < 9; tap++) v[tap] = xs[(hy + tap / 3) * XW + hx + tap % 3];
                    uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        float s = ebr[e];
#pragma unroll
                        for (int tap = 0; tap < 9; tap++) s = fmaf(ewr[e][tap], v[tap], s);
                        r8[e] = f2bf(fmaxf(s, 0.f));
                    }
                }
                st16(in_s + hp * HALO_PITCH + g * 8, r);
            }
        }
        __syncthreads();
        floatx4 acc[4][NF];
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int f = 0; f < NF; f++) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int ky = tap / 3, kx = tap % 3;
            bf16x8 av[4], bv[NF];
#pragma unroll
            for (int m = 0; m < 4; m++)
                av[m] = *(const bf16x8*)(in_s + ((4 * w + m + ky) * 18 + (l & 15) + kx) * HALO_PITCH +
                                         8 * (l >> 4));
#pragma unroll
            for (int f = 0; f < NF; f++) bv[f] = *(const bf16x8*)(w_s + ((f * 9 + tap) * 64 + l) * 8);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < NF; f++)
#pragma unroll
                for (int m = 0; m < 4; m++)
                    acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv[f], acc[m][f], 0, 0, 0);
        }
#pragma unroll
        for (int f = 0; f < NF; f++) {
            const int co = f * 16 + (l & 15);
            const float bias = a.bias ? a.bias[co] : 0.f;
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float v = acc[m][f][i] + bias;
                    if (a.relu) v = fmaxf(v, 0.f);
                    o_s[((4 * w + m) * 16 + 4 * (l >> 4) + i) * OPITCH + co] = f2bf(v);
                }
        }
        __syncthreads();
        if (a.pool_out) {
            const int Ho = a.H >> 1, Wo = a.W >> 1;
            for (int it = t; it < 64 * (TC / 8); it += 256) {
                const int q = it / (TC / 8), gg = it - q * (TC / 8);
                const int py = q >> 3, pxx = q & 7;
                const int yo = (y0 >> 1) + py, xo = (x0 >> 1) + pxx;
                if (yo >= Ho || xo >= Wo) continue;
                float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int px = (2 * py + (k >> 1)) * 16 + 2 * pxx + (k & 1);
                    const uint4 v = ld16(o_s + px * OPITCH + 8 * gg);
                    const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
                    for (int e = 0; e < 8; e++) sum[e] += bf2f(v8[e]);
                }
                uint4 r;
                uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
                for (int e = 0; e < 8; e++) r8[e] = f2bf(0.25f * sum[e]);
                st16(a.pool_out + (((long long)bb * Ho + yo) * Wo + xo) * a.Cout + 8 * gg, r);
            }
        }
        for (int it = t; it < 256 * (TC / 8); it += 256) {
            const int px = it / (TC / 8), gg = it - px * (TC / 8);
            const int y = y0 + (px >> 4), xx = x0 + (px & 15);
            if (y >= a.H || xx >= a.W) continue;
            const long long pix = ((long long)bb * a.H + y) * a.W + xx;
            st16(a.out + pix * a.out_stride + a.out_off + 8 * gg, ld16(o_s + px * OPITCH + 8 * gg));
        }
        // the next patch's tile and halo stores and output-tile writes are each
        // separated from this patch's reads by one barrier
    }
}

hipError_t launch_edge_conv3x3_c32(const ConvArgs& a, const float* x, const float* ew, const float* eb,
                                   hipStream_t s) {
    if (a.Cin != 32 || a.Cout != 32 || a.out_stride % 8 || a.out_off % 8 || a.B <= 0 || a.H <= 0 ||
        a.W <= 0 || a.out_off + a.Cout > a.out_stride || a.up || a.Cup || a.mask ||
        (a.pool_out && (a.H % 2 || a.W % 2)))
        return hipErrorInvalidValue;
    const int tiles = ((a.W + 15) / 16) * ((a.H + CONV_ROWS - 1) / CONV_ROWS);
    hipLaunchKernelGGL((edge_c32_kernel<4>), dim3((tiles + 3) / 4, 1, a.B), dim3(256), 0, s, a, x, ew, eb);
    return hipGetLastError();
}

hipError_t launch_conv3x3(const ConvArgs& a, hipStream_t s) {
    if (a.Cin % 32 || a.Cout % 32 || a.in_stride % 8 || a.in_off % 8 || a.out_stride % 8 ||
        a.out_off % 8 || a.B <= 0 || a.H <= 0 || a.W <= 0 || a.in_off + a.Cin > a.in_stride ||
        a.out_off + a.Cout > a.out_stride ||
        (a.mask && (a.mask_stride % 8 || a.mask_off % 8 || a.mask_off + a.Cout > a.mask_stride)) ||
        (a.up && (a.Cup % 32 || a.Cup > a.Cin || a.H % 2 || a.W % 2)) || (!a.up && a.Cup) ||
        (a.pool_out && (a.H % 2 || a.W % 2)))
        return hipErrorInvalidValue;
    const int tiles = ((a.W + 15) / 16) * ((a.H + CONV_ROWS - 1) / CONV_ROWS);
    const int tiles24 = ((a.W + 15) / 16) * ((a.H + 23) / 24);
    // 32 -> 32 layers (one chunk, 64 output channels of work per 16 KB of halo)
    // walk four patches per block with the weights staged once; other 32-output
    // layers use 24-row patches (6 M fragments per wave against 2 N fragments).
    if (a.Cout % 64 == 0)
        hipLaunchKernelGGL((conv3x3_kernel<4, 4>), dim3(tiles, a.Cout / 64, a.B), dim3(256), 0, s, a);
    else if (a.Cin == 32)
        hipLaunchKernelGGL((conv3x3_c32_kernel<2, 4>), dim3((tiles + 3) / 4, a.Cout / 32, a.B), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((conv3x3_kernel<2, 6>), dim3(tiles24, a.Cout / 32, a.B), dim3(256), 0, s, a);
    return hipGetLastError();
}

// ------------------------------------------------------------ weight gradient
// One block: 16 * NFW output x 32 input channels, all nine taps, over the 8 x 16 pixel
// patches split, split + nsplit, ...  dY and the halo of X are staged as they lie, one
// LDS plane per 16 channels (32 bytes a pixel), and the LDS transpose read hands each
// 16-lane group four pixels of 16 channels: a wave's read is one row of 16 pixels, 512
// contiguous bytes, and a tap is only another address.  A contraction pairs the rows r
// and r + 4, so the six row pairs of the halo serve all nine taps of all four pairs
// from registers.  Bound by the LDS and by the latency of a patch's fetch, which the
// second buffer hides.  Staged transposed instead, X in three shifted copies, 2-byte LDS
// writes were most of the time: a layer of a 16 x 512^2 gradient took 266 us on average
// with 64 and 539 us with 32 outputs per block, now 118 and 230 us.
constexpr int WG_ROWS = 8;
constexpr int DY_PLANE = 128 * 16 + 32;   // bf16 per plane: 128 pixels x 16 channels; the pads spread a
constexpr int XT_PLANE = 180 * 16;        // thread group's writes over all banks (5760 bytes does)

typedef short shortx4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ shortx4 lds_tr(const uint16_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)p);
}
static __device__ __forceinline__ bf16x8 lds_tr2(const uint16_t* p, const uint16_t* q) {
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lds_tr(p), lds_tr(q), 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int NFW>
__global__ __launch_bounds__(256, 2) void conv3x3_wgrad_kernel(WgradArgs a) {
    constexpr int TCO = 16 * NFW, G = TCO / 8;
    constexpr int CO = NFW / 2;                      // output fragments of a wave; one input fragment
    constexpr int DYN = 128 * G / 256, XN = 3;       // 16-byte units of a thread
    constexpr int BUF = NFW * DY_PLANE + 2 * XT_PLANE;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int co0 = blockIdx.x * TCO, cc = blockIdx.y, split = blockIdx.z;
    const int cof = (w & 1) * CO, cif = w >> 1;
    const int tiles_x = (a.W + 15) >> 4, tiles_y = (a.H + WG_ROWS - 1) / WG_ROWS;
    const int per_img = tiles_x * tiles_y, npatch = a.B * per_img;
    floatx4 acc[9][CO];
#pragma unroll
    for (int k = 0; k < 9; k++)
#pragma unroll
        for (int c = 0; c < CO; c++) acc[k][c] = floatx4{0.f, 0.f, 0.f, 0.f};
    float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    const int dg = t % G, dp = t / G;                // dY: channel group, first pixel
    const int xg = t & 3, xp = t >> 2;               // X: channel group, first halo pixel
    uint4 dv[DYN], xv[XN];
    auto fetch = [&](int patch) {
        const int bb = patch / per_img, r = patch - bb * per_img;
        const int y0 = (r / tiles_x) * WG_ROWS, x0 = (r % tiles_x) * 16;
        const long long img = (long long)bb * a.H;
#pragma unroll
        for (int k = 0; k < DYN; k++) {
            const int px = dp + k * (256 / G);
            const int y = y0 + (px >> 4), x = x0 + (px & 15);
            dv[k] = make_uint4(0, 0, 0, 0);
            if (y < a.H && x < a.W) dv[k] = ld16(a.dy + ((img + y) * a.W + x) * a.dy_stride + a.dy_off + co0 + 8 * dg);
        }
#pragma unroll
        for (int k = 0; k < XN; k++) {
            const int hp = xp + 64 * k;
            const int hy = hp / 18, hx = hp - hy * 18;
            const int y = y0 - 1 + hy, x = x0 - 1 + hx;
            xv[k] = make_uint4(0, 0, 0, 0);
            if (hp < 180 && y >= 0 && y < a.H && x >= 0 && x < a.W)
                xv[k] = ld16(a.x + ((img + y) * a.W + x) * a.x_stride + a.x_off + cc * 32 + 8 * xg);
        }
    };
    int buf = 0;
    if (split < npatch) fetch(split);
    for (int patch = split; patch < npatch; patch += a.nsplit) {
        uint16_t* dy_s = lds + buf;
        uint16_t* x_s = dy_s + NFW * DY_PLANE;
#pragma unroll
        for (int k = 0; k < DYN; k++)
            st16(dy_s + (dg >> 1) * DY_PLANE + (dp + k * (256 / G)) * 16 + 8 * (dg & 1), dv[k]);
#pragma unroll
        for (int k = 0; k < XN; k++)
            if (xp + 64 * k < 180) st16(x_s + (xg >> 1) * XT_PLANE + (xp + 64 * k) * 16 + 8 * (xg & 1), xv[k]);
        if (cc == 0) {
#pragma unroll
            for (int k = 0; k < DYN; k++) {
                const uint16_t* e8 = (const uint16_t*)&dv[k];
#pragma unroll
                for (int e = 0; e < 8; e++) bsum[e] += bf2f(e8[e]);
            }
        }
        __syncthreads();
        if (patch + a.nsplit < npatch) fetch(patch + a.nsplit);
        const uint16_t* xr = x_s + cif * XT_PLANE + 4 * l;
        const uint16_t* dr = dy_s + cof * DY_PLANE + 4 * l;
        bf16x8 bv[6][3];                             // halo rows r and r + 4, shift kx
        auto rows = [&](int r) {
#pragma unroll
            for (int kx = 0; kx < 3; kx++) bv[r][kx] = lds_tr2(xr + (r * 18 + kx) * 16, xr + ((r + 4) * 18 + kx) * 16);
        };
        rows(0);
        rows(1);
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
            rows(kb + 2);
            bf16x8 av[CO];
#pragma unroll
            for (int c = 0; c < CO; c++)
                av[c] = lds_tr2(dr + c * DY_PLANE + kb * 256, dr + c * DY_PLANE + (kb + 4) * 256);
#pragma unroll
            for (int tap = 0; tap < 9; tap++)
#pragma unroll
                for (int c = 0; c < CO; c++)
                    acc[tap][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[c], bv[kb + tap / 3][tap % 3],
                                                                          acc[tap][c], 0, 0, 0);
        }
        buf = BUF - buf;
    }
    float* P = a.part + (long long)split * a.Cout * 9 * a.Cin;
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int c = 0; c < CO; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int co = co0 + (cof + c) * 16 + 4 * (l >> 4) + e;
                const int ci = cc * 32 + cif * 16 + (l & 15);
                P[((long long)co * 9 + tap) * a.Cin + ci] = acc[tap][c][e];
            }
    if (cc == 0) {
        float* red = (float*)lds;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; e++) red[t * 8 + e] = bsum[e];
        __syncthreads();
        if (t < TCO) {
            float s = 0.f;
            for (int k = t / 8; k < 256; k += G) s += red[k * 8 + t % 8];
            a.partb[(long long)split * a.Cout + co0 + t] = s;
        }
    }
}

int wgrad_splits(int Cin, int Cout, int B, int H, int W) {
    const int nfw = Cout % 64 == 0 ? 4 : 2;
    const int tiles = (Cout / (16 * nfw)) * (Cin / 32);
    const long long npatch = (long long)B * ((H + 7) / 8) * ((W + 15) / 16);
    long long ns = (1024 + tiles - 1) / tiles;
    return (int)std::max(1LL, std::min(ns, npatch));
}

hipError_t launch_conv3x3_wgrad(const WgradArgs& a, hipStream_t s) {
    if (a.Cin % 32 || a.Cout % 32 || a.dy_stride % 8 || a.dy_off % 8 || a.x_stride % 8 ||
        a.x_off % 8 || a.nsplit <= 0 || a.dy_off + a.Cout > a.dy_stride || a.x_off + a.Cin > a.x_stride ||
        a.B <= 0 || a.H <= 0 || a.W <= 0)
        return hipErrorInvalidValue;
    if (a.Cout % 64 == 0)
        hipLaunchKernelGGL(conv3x3_wgrad_kernel<4>, dim3(a.Cout / 64, a.Cin / 32, a.nsplit), dim3(256),
                           0, s, a);
    else
        hipLaunchKernelGGL(conv3x3_wgrad_kernel<2>, dim3(a.Cout / 32, a.Cin / 32, a.nsplit), dim3(256),
                           0, s, a);
    return hipGetLastError();
}

// Column sums of part[nsplit][n] into out and, in the last blocks, of part2[nsplit][n2]
// into out2.  WAVES waves share 64 columns (256-byte rows), wave w taking the splits w, w +
// WAVES, ..., eight loads in flight, and their sums meet in LDS; a workgroup holds GROUPS
// such columns.  Bound by reading the parts: one thread per column had too few waves
// (n = 9216, 1024 splits: 36 blocks) and a serial chain of loads, 3.2 ms of the 14.0 ms of
// a 16 x 512^2 gradient; that now takes 10.9 ms.
template <int WAVES, int GROUPS>
__global__ __launch_bounds__(64 * WAVES * GROUPS) void sum_splits_kernel(const float* part, int nsplit, int n,
                                                                         float* out, const float* part2, int n2,
                                                                         float* out2) {
    constexpr int COLS = 64 * GROUPS;
    __shared__ float red[WAVES][COLS];
    const int wave = threadIdx.x >> 6, w = wave % WAVES, c = (wave / WAVES) * 64 + (threadIdx.x & 63);
    const int nb = (n + COLS - 1) / COLS;
    int i = blockIdx.x * COLS + c;
    if (blockIdx.x >= nb) {
        i -= nb * COLS;
        part = part2;
        n = n2;
        out = out2;
    }
    float s = 0.f;
    if (i < n) {
        const float* p = part + i;
        int k = w;
        for (; k + 7 * WAVES < nsplit; k += 8 * WAVES) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = p[(long long)(k + e * WAVES) * n];
            s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
        for (; k < nsplit; k += WAVES) s += p[(long long)k * n];
    }
    if constexpr (WAVES > 1) {
        red[w][c] = s;
        __syncthreads();
        if (w == 0 && i < n) {
#pragma unroll
            for (int k = 1; k < WAVES; k++) s += red[k][c];
            out[i] = s;
        }
    } else if (i < n) {
        out[i] = s;
    }
}

template <int WAVES, int GROUPS>
static void sum_splits(const float* part, int nsplit, int n, float* out, hipStream_t s, const float* part2, int n2,
                       float* out2) {
    constexpr int COLS = 64 * GROUPS;
    hipLaunchKernelGGL((sum_splits_kernel<WAVES, GROUPS>), dim3((n + COLS - 1) / COLS + (n2 + COLS - 1) / COLS),
                       dim3(64 * WAVES * GROUPS), 0, s, part, nsplit, n, out, part2, n2, out2);
}

hipError_t launch_sum_splits(const float* part, int nsplit, int n, float* out, hipStream_t s, const float* part2,
                             int n2, float* out2) {
    // as many waves as the chip needs: with sixteen for 64 columns of a wide layer, which has
    // few parts, most found nothing to add (whole weight gradient, 16 / 4 / 1 waves, us: 1179648
    // columns of 4 parts 96 / 75 / 73, 589824 of 16 87 / 79 / 73, 147456 of 16 65 / 64 / 62;
    // 9216 of 1024 75 / 82 / 115)
    if (n >= 1 << 18) sum_splits<1, 4>(part, nsplit, n, out, s, part2, n2, out2);
    else if (n >= 1 << 16) sum_splits<4, 1>(part, nsplit, n, out, s, part2, n2, out2);
    else sum_splits<16, 1>(part, nsplit, n, out, s, part2, n2, out2);
    return hipGetLastError();
}

// ------------------------------------------------------------ weight packing
__global__ void pack_kernel(const float* w, int Cin, int Cout, int transpose, uint16_t* out,
                            long long total) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int CinP = transpose ? Cout : Cin;   // contraction channels of the launch
    const int nch = CinP / 32;
    const int e = idx & 7, l = (idx >> 3) & 63;
    const long long r = idx >> 9;              // (f*nch + cc)*9 + tap
    const int tap = (int)(r % 9);
    const long long fc = r / 9;
    const int cc = (int)(fc % nch), f = (int)(fc / nch);
    const int o = f * 16 + (l & 15);           // output channel of the launch
    const int c = cc * 32 + 8 * (l >> 4) + e;  // contraction channel of the launch
    const float v = transpose ? w[((long long)c * 9 + (8 - tap)) * Cin + o]
                              : w[((long long)o * 9 + tap) * Cin + c];
    out[idx] = f2bf(v);
}

hipError_t launch_pack_conv_weights(const float* w, int Cin, int Cout, int transpose,
                                    uint16_t* wfrag, hipStream_t s) {
    if (Cin % 32 || Cout % 32) return hipErrorInvalidValue;
    const long long total = (long long)Cin * Cout * 9;
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, w, Cin,
                       Cout, transpose, wfrag, total);
    return hipGetLastError();
}

// ------------------------------------------------------------ edge layers
static __device__ __forceinline__ void pix_coords(long long p, int H, int W, int& b, int& y, int& x) {
    x = (int)(p % W);
    const long long r = p / W;
    y = (int)(r % H);
    b = (int)(r / H);
}

// One block = 256 consecutive pixels; outputs are staged in LDS so the stores
// are contiguous 16-byte chunks.
template <int C>
__global__ __launch_bounds__(256) void edge_in_kernel(const float* x, const float* w, const float* b,
                                                      uint16_t* out, int os, int oo, int B, int H, int W) {
    constexpr int PITCH = C + 8;
    __shared__ __attribute__((aligned(16))) uint16_t o_s[256 * PITCH];
    const long long n = (long long)B * H * W;
    const long long p0 = (long long)blockIdx.x * 256;
    const long long p = p0 + threadIdx.x;
    if (p < n) {
        int bb, y, xx;
        pix_coords(p, H, W, bb, y, xx);
        float v[9];
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int yy = y + tap / 3 - 1, x2 = xx + tap % 3 - 1;
            v[tap] = (yy >= 0 && yy < H && x2 >= 0 && x2 < W) ? x[((long long)bb * H + yy) * W + x2] : 0.f;
        }
#pragma unroll
        for (int g = 0; g < C / 8; g++) {
            uint4 r;
            uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int c = 8 * g + e;
                float s = b[c];
#pragma unroll
                for (int tap = 0; tap < 9; tap++) s = fmaf(w[c * 9 + tap], v[tap], s);
                r8[e] = f2bf(fmaxf(s, 0.f));
            }
            st16(o_s + threadIdx.x * PITCH + 8 * g, r);
        }
    }
    __syncthreads();
    for (int it = threadIdx.x; it < 256 * (C / 8); it += 256) {
        const int px = it / (C / 8), g = it - px * (C / 8);
        if (p0 + px < n) st16(out + (p0 + px) * os + oo + 8 * g, ld16(o_s + px * PITCH + 8 * g));
    }
}

hipError_t launch_edge_in(const float* x, const float* w, const float* b, int C, uint16_t* out,
                          int out_stride, int out_off, int B, int H, int W, hipStream_t s) {
    const long long n = (long long)B * H * W;
    const dim3 g((unsigned)((n + 255) / 256));
    if (out_stride % 8 || out_off % 8) return hipErrorInvalidValue;
    if (C == 32)
        hipLaunchKernelGGL(edge_in_kernel<32>, g, dim3(256), 0, s, x, w, b, out, out_stride, out_off, B, H, W);
    else if (C == 64)
        hipLaunchKernelGGL(edge_in_kernel<64>, g, dim3(256), 0, s, x, w, b, out, out_stride, out_off, B, H, W);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// Gradients of the two edge layers, whose one side is an image v (the input, or dy of the
// output layer) and whose other side is activations c of C channels: every pixel's C
// channels against the 3 x 3 neighbours in v,
//   first layer: dW[c][tap] = sum_p dy[p][c] x[p + d(tap)], dB[c] = sum_p dy[p][c];
//   last layer (OUT): dW[tap][c] = sum_p X[p][c] dy[p - d(tap)], dB = sum_p dy[p], and on
//   the way dX[p][c] = (X[p][c] > 0) sum_tap W[tap][c] dy[p - d(tap)].
// Bound by the activations: each is read once, the neighbours move down a strip of
// 256 / (C / 8) columns x kEdgeRows rows in registers (three loads a row), and the
// activations of the next row load meanwhile.  Thread t handles channel group t % (C / 8).
// part[blk]: the layout of the parameters, sums of the strips blk, blk + gridDim.x, ...
// 16 x 512^2 x 32: last layer 350 us (each activation read for nine taps) and 240 us for
// dX apart -> 227 us in one; first layer 196 -> 92 us.
constexpr int kEdgeRows = 8;

// A workgroup per strip, up to 1024, which fill the chip and bound the parts (one per
// 4096 pixels, 8 for 2 x 128^2, left most of it idle: that whole gradient took 1290 us, with
// 64 workgroups 1200; 4 x 256^2 1700 and 1600).
int edge_blocks(int C, int B, int H, int W) {
    const int lanes = 256 / (C / 8);
    const long long strips = (long long)B * ((H + kEdgeRows - 1) / kEdgeRows) * ((W + lanes - 1) / lanes);
    return (int)std::max(1LL, std::min(1024LL, strips));
}

template <int C, bool OUT>
__global__ __launch_bounds__(256) void edge_grad_kernel(const float* v, const uint16_t* c, const float* w,
                                                        uint16_t* dx, float* part, int B, int H, int W) {
    constexpr int G = C / 8, LANES = 256 / G, NB = OUT ? 9 * C + 1 : 10 * C;
    __shared__ float red[4][10 * C];
    const int t = threadIdx.x, g = t % G;
    float acc[9][8], bs[8], wr[OUT ? 9 : 1][8];
#pragma unroll
    for (int k = 0; k < 9; k++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            acc[k][e] = 0.f;
            if constexpr (OUT) wr[k][e] = w[k * C + 8 * g + e];
        }
#pragma unroll
    for (int e = 0; e < 8; e++) bs[e] = 0.f;
    const int ncol = (W + LANES - 1) / LANES, nrow = (H + kEdgeRows - 1) / kEdgeRows;
    for (int s = blockIdx.x; s < B * nrow * ncol; s += gridDim.x) {
        const int x = s % ncol * LANES + t / G, y0 = s / ncol % nrow * kEdgeRows;
        const int y1 = min(H, y0 + kEdgeRows);
        const long long img = (long long)(s / ncol / nrow) * H * W;
        float win[3][3];
        auto load_row = [&](int y, float (&r)[3]) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const int xx = x + k - 1;
                // nothing past the image, whose zero activations would make NaN of an infinity
                const bool in = y >= 0 && y < H && xx >= 0 && xx < W && x < W;
                r[k] = in ? v[img + (long long)y * W + xx] : 0.f;
            }
        };
        auto load_c = [&](int y) {
            uint4 q = {0, 0, 0, 0};
            if (x < W && y < y1) q = ld16(c + (img + (long long)y * W + x) * C + 8 * g);
            return q;
        };
        load_row(y0 - 1, win[0]);
        load_row(y0, win[1]);
        uint4 next = load_c(y0);
        for (int y = y0; y < y1; y++) {
            load_row(y + 1, win[2]);
            const uint4 cur = next;
            next = load_c(y + 1);
            const uint16_t* c8 = (const uint16_t*)&cur;
            // the neighbour of a tap: p + d(tap), for the last layer p - d(tap)
            auto nb = [&](int tap) { return OUT ? win[2 - tap / 3][2 - tap % 3] : win[tap / 3][tap % 3]; };
            uint4 r;
            uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float a = bf2f(c8[e]);
#pragma unroll
                for (int tap = 0; tap < 9; tap++) acc[tap][e] = fmaf(a, nb(tap), acc[tap][e]);
                if constexpr (OUT) {
                    float d = 0.f;
#pragma unroll
                    for (int tap = 0; tap < 9; tap++) d = fmaf(wr[tap][e], nb(tap), d);
                    r8[e] = f2bf(a > 0.f ? d : 0.f);
                } else {
                    bs[e] += a;
                }
            }
            if constexpr (OUT) {
                if (x < W) {
                    bs[0] += win[1][1];
                    st16(dx + (img + (long long)y * W + x) * C + 8 * g, r);
                }
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                win[0][k] = win[1][k];
                win[1][k] = win[2][k];
            }
        }
    }
    auto sum = [&](float a) {
        for (int off = 32; off >= G; off >>= 1) a += __shfl_xor(a, off);
        return a;
    };
    float* mine = red[t >> 6];
    const bool first = (t & 63) < G;
#pragma unroll
    for (int e = 0; e < 8; e++) {
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const float a = sum(acc[k][e]);
            if (first) mine[OUT ? k * C + 8 * g + e : (8 * g + e) * 9 + k] = a;
        }
        if (!OUT || e == 0) {
            const float a = sum(bs[e]);
            if (first && (!OUT || g == 0)) mine[9 * C + (OUT ? 0 : 8 * g + e)] = a;
        }
    }
    __syncthreads();
    for (int i = t; i < NB; i += 256)
        part[(long long)blockIdx.x * NB + i] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
}

hipError_t launch_edge_in_wgrad(const uint16_t* dy, int C, const float* x, float* part, int nblk,
                                int B, int H, int W, hipStream_t s) {
    if (C == 32)
        hipLaunchKernelGGL((edge_grad_kernel<32, false>), dim3(nblk), dim3(256), 0, s, x, dy, nullptr, nullptr, part,
                           B, H, W);
    else if (C == 64)
        hipLaunchKernelGGL((edge_grad_kernel<64, false>), dim3(nblk), dim3(256), 0, s, x, dy, nullptr, nullptr, part,
                           B, H, W);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// One block = a 16 x 16 pixel patch; the 18 x 18 halo of X is staged in LDS
// with coalesced 16-byte loads, then each thread reduces 9 taps x C channels.
template <int C>
__global__ __launch_bounds__(256) void edge_out_kernel(const uint16_t* x, const float* w, const float* b,
                                                       const float* xres, float* y, int B, int H, int W) {
    constexpr int PITCH = C + 8;
    constexpr int G = C / 8;
    __shared__ __attribute__((aligned(16))) uint16_t h_s[324 * PITCH];
    const int tiles_x = (W + 15) >> 4;
    const int x0 = (blockIdx.x % tiles_x) * 16, y0 = (blockIdx.x / tiles_x) * 16;
    const int bb = blockIdx.y;
    for (int i = threadIdx.x; i < 324 * G; i += 256) {
        const int hp = i / G, g = i - hp * G;
        const int hy = hp / 18, hx = hp - hy * 18;
        const int yy = y0 - 1 + hy, xx = x0 - 1 + hx;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (yy >= 0 && yy < H && xx >= 0 && xx < W) v = ld16(x + (((long long)bb * H + yy) * W + xx) * C + 8 * g);
        st16(h_s + hp * PITCH + 8 * g, v);
    }
    __syncthreads();
    const int py = threadIdx.x >> 4, pxl = threadIdx.x & 15;
    const int yy = y0 + py, xx = x0 + pxl;
    if (yy >= H || xx >= W) return;
    float s = b[0];
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
        const uint16_t* q = h_s + ((py + tap / 3) * 18 + pxl + tap % 3) * PITCH;
#pragma unroll
        for (int g = 0; g < G; g++) {
            const uint4 v = ld16(q + 8 * g);
            const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
            for (int e = 0; e < 8; e++) s = fmaf(w[tap * C + 8 * g + e], bf2f(v8[e]), s);
        }
    }
    const long long p = ((long long)bb * H + yy) * W + xx;
    y[p] = xres[p] + s;
}

hipError_t launch_edge_out(const uint16_t* x, int C, const float* w, const float* b,
                           const float* xres, float* y, int B, int H, int W, hipStream_t s) {
    const dim3 g((unsigned)(((W + 15) / 16) * ((H + 15) / 16)), (unsigned)B);
    if (C == 32)
        hipLaunchKernelGGL(edge_out_kernel<32>, g, dim3(256), 0, s, x, w, b, xres, y, B, H, W);
    else if (C == 64)
        hipLaunchKernelGGL(edge_out_kernel<64>, g, dim3(256), 0, s, x, w, b, xres, y, B, H, W);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_edge_out_grad(const float* dy, const uint16_t* x, int C, const float* w, uint16_t* dx,
                                float* part, int nblk, int B, int H, int W, hipStream_t s) {
    if (C == 32)
        hipLaunchKernelGGL((edge_grad_kernel<32, true>), dim3(nblk), dim3(256), 0, s, dy, x, w, dx, part, B, H, W);
    else if (C == 64)
        hipLaunchKernelGGL((edge_grad_kernel<64, true>), dim3(nblk), dim3(256), 0, s, dy, x, w, dx, part, B, H, W);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// ------------------------------------------------------------ pooling / upsampling
__global__ void avgpool2_kernel(const uint16_t* in, int is, int io, int C, uint16_t* out, int B,
                                int H, int W) {
    const int G = C / 8, Ho = H / 2, Wo = W / 2;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)B * Ho * Wo * G) return;
    const int g = (int)(i % G);
    const long long q = i / G;
    int bb, y, x;
    pix_coords(q, Ho, Wo, bb, y, x);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const long long p = ((long long)bb * H + 2 * y + (k >> 1)) * W + 2 * x + (k & 1);
        const uint4 v = ld16(in + p * is + io + 8 * g);
        const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] += bf2f(v8[e]);
    }
    uint4 r;
    uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
    for (int e = 0; e < 8; e++) r8[e] = f2bf(0.25f * s[e]);
    st16(out + q * C + 8 * g, r);
}

hipError_t launch_avgpool2(const uint16_t* in, int in_stride, int in_off, int C, uint16_t* out,
                           int B, int H, int W, hipStream_t s) {
    if (C % 8 || in_stride % 8 || in_off % 8 || H % 2 || W % 2) return hipErrorInvalidValue;
    const long long n = (long long)B * (H / 2) * (W / 2) * (C / 8);
    hipLaunchKernelGGL(avgpool2_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in,
                       in_stride, in_off, C, out, B, H, W);
    return hipGetLastError();
}

__global__ void upsample2_kernel(const uint16_t* in, int C, uint16_t* out, int os, int oo, int B,
                                 int H, int W) {
    const int G = C / 8;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)B * H * W * G) return;
    const int g = (int)(i % G);
    const long long p = i / G;
    int bb, y, x;
    pix_coords(p, H, W, bb, y, x);
    const long long q = ((long long)bb * (H / 2) + y / 2) * (W / 2) + x / 2;
    st16(out + p * os + oo + 8 * g, ld16(in + q * C + 8 * g));
}

hipError_t launch_upsample2(const uint16_t* in, int C, uint16_t* out, int out_stride, int out_off,
                            int B, int H, int W, hipStream_t s) {
    if (C % 8 || out_stride % 8 || out_off % 8 || H % 2 || W % 2) return hipErrorInvalidValue;
    const long long n = (long long)B * H * W * (C / 8);
    hipLaunchKernelGGL(upsample2_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, in, C,
                       out, out_stride, out_off, B, H, W);
    return hipGetLastError();
}

// H, W: full-resolution size of g; out is H/2 x W/2 with C channels.
__global__ void upsample2_bwd_kernel(const uint16_t* g, int gs, int go, int C, uint16_t* out, int B,
                                     int H, int W) {
    const int G = C / 8, Ho = H / 2, Wo = W / 2;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)B * Ho * Wo * G) return;
    const int gg = (int)(i % G);
    const long long q = i / G;
    int bb, y, x;
    pix_coords(q, Ho, Wo, bb, y, x);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const long long p = ((long long)bb * H + 2 * y + (k >> 1)) * W + 2 * x + (k & 1);
        const uint4 v = ld16(g + p * gs + go + 8 * gg);
        const uint16_t* v8 = (const uint16_t*)&v;
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] += bf2f(v8[e]);
    }
    uint4 r;
    uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
    for (int e = 0; e < 8; e++) r8[e] = f2bf(s[e]);
    st16(out + q * C + 8 * gg, r);
}

hipError_t launch_upsample2_bwd(const uint16_t* g, int g_stride, int g_off, int C, uint16_t* out,
                                int B, int H, int W, hipStream_t s) {
    if (C % 8 || g_stride % 8 || g_off % 8 || H % 2 || W % 2) return hipErrorInvalidValue;
    const long long n = (long long)B * (H / 2) * (W / 2) * (C / 8);
    hipLaunchKernelGGL(upsample2_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g,
                       g_stride, g_off, C, out, B, H, W);
    return hipGetLastError();
}

__global__ void pool_bwd_add_kernel(const uint16_t* skip, int ss, int so, const uint16_t* dp,
                                    const uint16_t* e, int es, int eo, int C, uint16_t* out, int B,
                                    int H, int W) {
    const int G = C / 8;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)B * H * W * G) return;
    const int g = (int)(i % G);
    const long long p = i / G;
    int bb, y, x;
    pix_coords(p, H, W, bb, y, x);
    const long long q = ((long long)bb * (H / 2) + y / 2) * (W / 2) + x / 2;
    const uint4 sv = ld16(skip + p * ss + so + 8 * g), dv = ld16(dp + q * C + 8 * g),
                ev = ld16(e + p * es + eo + 8 * g);
    const uint16_t *s8 = (const uint16_t*)&sv, *d8 = (const uint16_t*)&dv, *e8 = (const uint16_t*)&ev;
    uint4 r;
    uint16_t* r8 = (uint16_t*)&r;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float v = fmaf(0.25f, bf2f(d8[k]), bf2f(s8[k]));
        r8[k] = f2bf(bf2f(e8[k]) > 0.f ? v : 0.f);
    }
    st16(out + p * C + 8 * g, r);
}

hipError_t launch_pool_bwd_add(const uint16_t* skip, int skip_stride, int skip_off,
                               const uint16_t* dp, const uint16_t* e, int e_stride, int e_off,
                               int C, uint16_t* out, int B, int H, int W, hipStream_t s) {
    if (C % 8 || skip_stride % 8 || skip_off % 8 || e_stride % 8 || e_off % 8 || H % 2 || W % 2)
        return hipErrorInvalidValue;
    const long long n = (long long)B * H * W * (C / 8);
    hipLaunchKernelGGL(pool_bwd_add_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, skip,
                       skip_stride, skip_off, dp, e, e_stride, e_off, C, out, B, H, W);
    return hipGetLastError();
}

// ------------------------------------------------------------ loss / optimiser
__global__ void scale_kernel(const float* x, float scale, float* y, long long n) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = x[i] * scale;
}

hipError_t launch_scale(const float* x, float scale, float* y, long long n, hipStream_t s) {
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, scale, y, n);
    return hipGetLastError();
}

int loss_blocks(long long n) { return (int)std::max(1LL, std::min(1024LL, (n + 2047) / 2048)); }

__global__ void mse_kernel(const float* y, const float* t, float* dy, float* part, long long n) {
    __shared__ float red[4];
    float s = 0.f;
    const float k = 2.f / (float)n;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float d = y[i] - t[i];
        dy[i] = k * d;
        s = fmaf(d, d, s);
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

hipError_t launch_mse(const float* y, const float* t, float* dy, float* part, long long n,
                      hipStream_t s) {
    hipLaunchKernelGGL(mse_kernel, dim3(loss_blocks(n)), dim3(256), 0, s, y, t, dy, part, n);
    return hipGetLastError();
}

__global__ void adam_kernel(float* p, const float* g, float* m, float* v, long long n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = fmaf(b1, m[i], (1.f - b1) * gi);
    const float vi = fmaf(b2, v[i], (1.f - b2) * gi * gi);
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

hipError_t launch_adam(float* p, const float* g, float* m, float* v, long long n, float lr,
                       float b1, float b2, float eps, int step, hipStream_t s) {
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)b1, step)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)b2, step)));
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, g, m, v, n,
                       lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

}  // namespace rv
