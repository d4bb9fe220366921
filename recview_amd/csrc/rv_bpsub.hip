// rv_bpsub.hip -- back-projection of launches with few tiles (gfx950).
//
// BP_LINEAR / BP_LINEAR2 / BP_LINEAR4 on parts of a tile, for launches whose tiles are
// too few to fill the chip (bp_sub_parts).  A workgroup owns 16 PX x 16 PY pixels of a
// tile and forms coordinates and samples as bp_tiled_kernel does on the whole tile (same
// origin, same operations, same order of the sums), so the images are the same bit for
// bit.  It stages only the samples its part sees; the rows of the next chunk of angles
// and the angle entries of the one after load while a chunk is summed.  Bound by the
// waves in flight (512^2 x 450: 8 workgroups a tile, 2 waves per SIMD) and by one LDS
// read and five vector instructions per update.
//
// A file of its own: in one file with it the compiler allocates bp_tiled_kernel's
// registers differently (one slice of 2048^2 x 1800 or 4096^2 x 3600 0.3 to 0.9% slower).
// Compiled with -ffp-contract=off; FMAs are written explicitly.
#include "rv_bp.h"
#include <type_traits>

namespace rv {

template <int NS, int PX, int PY>
struct SubCfg {
    using C = TileCfg<PX, PY>;
    static constexpr int NQ = NS == 1 ? 1 : NS / 2;               // LDS planes per angle
    static constexpr int CH = NS == 1 ? 32 : 16;                  // angles per chunk
    static constexpr int TPA = 256 / CH;                          // staging threads per angle
    static constexpr int PER = (C::SEG + TPA - 1) / TPA;          // samples per staging thread
    using T = typename std::conditional<NS == 1, float2, float4>::type;
};

// The tile: w x h pixels, and the bits of a pixel's offset in it that bp_tiled_kernel
// covers in steps of 8 i and 8 j (8 (PX - 1), 8 (PY - 1) of its instantiation).
struct SubTile {
    int w, h, mx, my;
};

template <int NS, int PX, int PY>
__global__ void __launch_bounds__(256) bp_sub_kernel(BpLaunch L, SubTile E)
{
    using F = SubCfg<NS, PX, PY>;
    using C = typename F::C;
    using T = typename F::T;
    constexpr int SEG = C::SEG, CH = F::CH, NQ = F::NQ;
    const int nsx = E.w / C::TW, nsub = nsx * (E.h / C::TH);
    __shared__ float4 tab[CH];
    __shared__ T data[CH * NQ * SEG];

    int item = blockIdx.x / nsub;
    const int sub = blockIdx.x % nsub;
    if (L.item_order) item = L.item_order[item];
    int lo = 0, hi = L.nslices - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (L.slices[mid].tile_base <= item) lo = mid; else hi = mid - 1;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    const BpSlice& S = L.slices[lo];
    const int t = item - S.tile_base;
    const int X0 = (t % S.tiles_x) * E.w, Y0 = (t / S.tiles_x) * E.h;
    const int sx = (sub % nsx) * C::TW, sy = (sub / nsx) * C::TH;       // the part's place in the tile
    const int out_n = S.out_n, nang = S.nang, N = S.row_len;
    if (X0 + sx >= out_n || Y0 + sy >= out_n) return;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wx = sx + (wave & 1) * C::WX, wy = sy + (wave >> 1) * C::WY;     // the wave's pixels in the tile
    // bp_tiled_kernel's lane offset and pixel steps 8 i, 8 j of the lane's first pixel
    const float dxl = (float)((wx & ~E.mx) + (lane & 7)), dyl = (float)((wy & ~E.my) + (lane >> 3));
    const float xi = (float)(wx & E.mx), yj = (float)(wy & E.my);

    // staging: one angle of the chunk per thread, samples j0, j0 + TPA, ... of its part
    const int sa = tid / F::TPA, j0 = tid % F::TPA;
    AngleEntry e{};
    auto fetch_entry = [&](int a0) {
        if (a0 + sa < nang) e = S.ang[a0 + sa];
    };
    T raw[F::PER][NQ];                                 // NS 1: (p_k, p_k+1); else the packed (p, d, p', d')
    float4 geo;
    int jlo, k0;                                       // first staged sample: from the tile's s0, in the row
    auto fetch_rows = [&](int a0) {
        const bool ok = a0 + sa < nang;
        const double ut = e.u0 + (double)X0 * e.dux + (double)Y0 * e.duy;
        const double utile = ut + fmin(0.0, (E.w - 1) * e.dux) + fmin(0.0, (E.h - 1) * e.duy);
        const int s0 = (int)floor(utile) - 1;                                    // the tile's
        const double us = ut + sx * e.dux + sy * e.duy + fmin(0.0, (C::TW - 1) * e.dux) +
                          fmin(0.0, (C::TH - 1) * e.duy);
        jlo = max((int)floor(us) - 1 - s0, 0);                                  // the part's, from the tile's
        geo = ok ? make_float4((float)e.dux, (float)e.duy, (float)(ut - (double)s0),
                               __int_as_float(sa * NQ * SEG - jlo))
                 : make_float4(0.f, 0.f, 1.f, __int_as_float(sa * NQ * SEG - 1));
        if (!ok) jlo = 1;
        k0 = s0 + jlo;
#pragma unroll
        for (int m = 0; m < F::PER; m++) {
            const int j = j0 + m * F::TPA;
            const int k = k0 + j;
            const bool in = ok && j < SEG && k >= 0 && k < N;
            if constexpr (NS == 1) {
                raw[m][0] = make_float2(0.f, 0.f);
                if (in) {
                    raw[m][0].x = load_row_val(S, e.row, k);
                    if (k < N - 1) raw[m][0].y = load_row_val(S, e.row, k + 1);
                }
            } else {
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    raw[m][q] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (in) raw[m][q] = ((const float4*)S.rows)[((long long)e.row * S.row_stride + k) * NQ + q];
                }
            }
        }
    };
    auto stage = [&]() {
        if (j0 == 0) tab[sa] = geo;
#pragma unroll
        for (int m = 0; m < F::PER; m++) {
            const int j = j0 + m * F::TPA;
            if (j >= SEG) continue;
            const float fj = -(float)(jlo + j);
            if constexpr (NS == 1) {
                const float2 v = raw[m][0];
                const float d = k0 + j < N - 1 ? v.y - v.x : 0.f;      // the last sample is held
                data[sa * SEG + j] = make_float2(fmaf(fj, d, v.x), d);
            } else {
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    const float4 v = raw[m][q];
                    data[(sa * NQ + q) * SEG + j] =
                        make_float4(fmaf(fj, v.y, v.x), v.y, fmaf(fj, v.w, v.z), v.w);
                }
            }
        }
    };

    float acc[NS][PY][PX];
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int j = 0; j < PY; j++)
#pragma unroll
            for (int i = 0; i < PX; i++) acc[s][j][i] = 0.f;

    fetch_entry(0);
    fetch_rows(0);
    fetch_entry(CH);
    for (int a0 = 0; a0 < nang; a0 += CH) {
        stage();
        __syncthreads();
        if (a0 + CH < nang) {
            fetch_rows(a0 + CH);
            fetch_entry(a0 + 2 * CH);
        }
#pragma unroll 4
        for (int a = 0; a < CH; a++) {                 // angles past the last add zeros
            const float4 tb = tab[a];
            const T* seg = data + __float_as_int(tb.w);
            const float base = fmaf(dyl, tb.y, fmaf(dxl, tb.x, tb.z));
#pragma unroll
            for (int j = 0; j < PY; j++) {
                const float bj = fmaf(yj + 8 * j, tb.y, base);
#pragma unroll
                for (int i = 0; i < PX; i++) {
                    const float u = fmaf(xi + 8 * i, tb.x, bj);
                    const T* p = seg + (int)u;
                    if constexpr (NS == 1) {
                        const float2 v = p[0];
                        acc[0][j][i] += fmaf(u, v.y, v.x);
                    } else {
#pragma unroll
                        for (int q = 0; q < NQ; q++) {
                            const float4 v = p[q * SEG];
                            acc[2 * q][j][i] += fmaf(u, v.y, v.x);
                            acc[2 * q + 1][j][i] += fmaf(u, v.w, v.z);
                        }
                    }
                }
            }
        }
        __syncthreads();
    }

#pragma unroll
    for (int j = 0; j < PY; j++) {
        const int iy = Y0 + wy + (lane >> 3) + 8 * j;
        if (iy >= out_n) continue;
#pragma unroll
        for (int i = 0; i < PX; i++) {
            const int ix = X0 + wx + (lane & 7) + 8 * i;
            if (ix >= out_n) continue;
            const long long o = (long long)iy * out_n + ix;
#pragma unroll
            for (int s = 0; s < NS; s++) {
                float* out = (float*)(s == 0 ? S.out : S.out_x[s - 1]);
                const float v = acc[s][j][i] * S.out_scale;
                out[o] = S.accumulate ? out[o] + v : v;
            }
        }
    }
}

// Whole tiles need about three workgroups per CU; below that a launch waits on each
// wave's own chain of staging, barriers and LDS reads.  The smaller the part, the more
// of its time is staging and coordinates, so the parts only get as small as the launch
// needs.  One slice, whole execution, whole tiles / 4 / 8 / 16 parts (us):
//   333^2 x 240 (36 tiles)     125 / 43 / 37 / 33     512^2 x 450 (64)    221 / 72 / 60 / 63
//   700^2 x 500 (121)          238 / 82 / 82 / 107   1024^2 x 900 (256)  418 / 192 / 224 / 289
//   1536^2 x 1200 (576)        620 / 507 / 552 / 767 2048^2 x 1800 (1024) 1085 / 1244 / 1423 / 1997
//   1700^2 x 900 (729)         499 / 505
// Four slices per item: 384^2 x 225 (36 tiles) 236 / 124 / 71 / 62, 384^2 x 225 x 16
// (144) 249 / 137 / 130 / 132, 800^2 x 600 (169) 621 / 287 / 301 / 313, 1024^2 x 900 x 8
// (512) 905 / 882 / 1097 / 1213, 2048^2 x 1800 (1024) 2311 / 3393 / 4171 / 4608.  Pairs, whole
// tiles (64 x 128 and 128 x 64 below 700^2) / parts: 384^2 x 225 270 / 52, 512^2 x 450 505 / 91,
// 600^2 x 450 506 / 109, 1024^2 x 900 562 / 268, 1400^2 x 1200 (484) 767 / 642.
// (Tiles counted as 64 x 64 pixels, whatever the tile configuration.)
// Where whole tiles take over depends on what each side costs.  Parts of 32 x 32 pixels fill
// the chip once with 256 tiles and twice with 512, and sum whole chunks of 16 angles in
// pairs and fours (1400^2 x 20, fours: 50 whole, 60 in parts).  32 x 32 and 32 x 64 tiles are
// two to four times as many, so that whole they fill it sooner (four slices of 1200^2 x 900
// on 32 x 32: 500 / 764, pairs of 1400^2 x 900 on 32 x 64 408 / 479); lone ones sit six to a CU,
// a second set beginning with 1536 of them (1280^2 x 1500 641 / 495).  16-bit rows cost
// parts more to stage (1600^2 x 900 493 / 525); chunks below the default cost whole pairs more
// (1100^2 x 700 on 32 x 64 in chunks of 12: 353 / 287).  A queue costs whole tiles an atomic each and a
// launch that clears its counter, which is most of their time when angles are few (pairs of
// 1376^2 x 24 on 32 x 32: 63 / 34, without a queue 33 / 34).  The lines below were read off
// 6960 measured launches; they make none more than 5% slower than whole tiles.
static int bp_sub_most(int mode, int tile, int chunk, long long n, int nang, bool rows16, bool queue)
{
    const int filled = n > 384 ? 512 : 256;                 // small tiles: gains up to here, and again from 384 on
    if (mode == BP_LINEAR) {
        if (tile == 2) {
            if (queue) return nang < 200 || !rows16 ? 640 : filled;
            return nang >= 32 ? filled : rows16 ? 512 : 640;
        }
        if (tile == 4) {
            if (queue) return nang < 200 ? 640 : rows16 ? 430 : 512;
            return rows16 || nang < 32 ? 256 : 430;
        }
        if (tile == 0 && rows16) return queue && nang < 100 ? 640 : nang < 64 ? 440 : 512;
        return queue || nang >= 32 ? 640 : 570;
    }
    if (mode == BP_LINEAR2) {
        if (tile == 2 || tile == 4) {
            if (queue) return nang < 200 || chunk < bp_default_chunk(mode, tile) ? 512 : 256;
            return tile == 4 ? (nang < 32 ? 128 : 256) : nang < 100 ? 80 : 128;
        }
        if (tile == 0 && !queue)                            // 380: over a fifth more angles summed than there are
            return nang < 8 ? 150 : nang < 20 ? 256 : 5 * (-nang & 15) > nang ? 380 : 512;
        return 512;
    }
    if (mode == BP_LINEAR4) {
        if (tile == 2) {
            if (queue) return nang < 32 ? 512 : nang < 100 ? filled : 128;
            return nang < 40 ? 80 : 128;
        }
        if (tile == 4) return queue ? (nang < 16 ? 512 : 256) : nang < 40 ? 80 : 256;
        if (tile == 0) {
            if (queue) return nang < 36 ? 256 : 512;
            return nang < 8 ? 100 : nang < 100 ? 256 : nang < 200 ? 400 : 512;
        }
        return !queue && nang < 8 ? 256 : 512;
    }
    return 0;
}

int bp_sub_parts(int mode, int tile, int chunk, int total_items, int nang, bool rows16, bool queue)
{
    const long long n = (long long)total_items * bp_tile_side(tile) * bp_tile_h(tile) / 4096;
    if (n > bp_sub_most(mode, tile, chunk, n, nang, rows16, queue)) return 0;
    if (mode == BP_LINEAR) return n <= 48 ? 16 : n <= 96 ? 8 : 4;
    return n <= 80 ? 16 : n <= (tile == 2 ? 128 : 150) ? 8 : 4;
}

template <int NS, int PX, int PY>
static void launch_sub(const BpLaunch& L, hipStream_t stream)
{
    using C = TileCfg<PX, PY>;
    SubTile E{bp_tile_side(L.tile), bp_tile_h(L.tile), 24, 24};      // <4, 4>
    if (L.tile == 1) E.my = 56;                                     // <4, 8>
    if (L.tile == 2) E.mx = E.my = 8;                               // <2, 2>
    if (L.tile == 3) E.mx = 56;                                     // <8, 4>
    if (L.tile == 4) E.mx = 8;                                      // <2, 4>
    const int nsub = (E.w / C::TW) * (E.h / C::TH);
    hipLaunchKernelGGL((bp_sub_kernel<NS, PX, PY>), dim3(L.total_items * nsub), dim3(256), 0, stream, L, E);
}

template <int NS>
static void launch_sub_parts(const BpLaunch& L, int parts, hipStream_t stream)
{
    if (parts == 16) launch_sub<NS, 1, 1>(L, stream);
    else if (parts == 8) launch_sub<NS, 2, 1>(L, stream);
    else launch_sub<NS, 2, 2>(L, stream);
}

void launch_bp_sub(const BpLaunch& L, int parts, hipStream_t stream)
{
    if (L.mode == BP_LINEAR) launch_sub_parts<1>(L, parts, stream);
    else if (L.mode == BP_LINEAR2) launch_sub_parts<2>(L, parts, stream);
    else launch_sub_parts<4>(L, parts, stream);
}

}  // namespace rv
