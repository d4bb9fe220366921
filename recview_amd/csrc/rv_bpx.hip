// rv_bpx.hip -- back-projection of FP32 stacks on the matrix cores (gfx950).
//
// Slices of one geometry share every interpolation weight, so for one angle and
// one 4 x 4-pixel block the linear interpolation of 16 slices is a matrix product
// over a window of eight detector samples j0 .. j0 + 7 (pixels are at most a sample apart,
// pix_zoom >= 1 in every plan, so a block spans at most 3 (|cos| + |sin|) <= 4.25 samples;
// j0 is even):
//
//   D[slice][pixel] += sum_k P[slice][k] * W[k][pixel],
//   W[k][pixel] = max(0, 1 - |u_pixel - j0 - k|).
//
// FP32 operands are kept as sums of two FP16 values, p = ph + pl and w = wh + wl
// (each rounded to nearest: 22 significant bits and the sign of the low part; samples are
// scaled by one power of two per slice, so those below 2^-17 of the slice's largest are
// kept to 2^-40 of that instead).  The
// 32-long contraction of v_mfma_f32_16x16x32_f16 is two angles x eight samples x
// {ph, pl}; against it stand wh twice and wl twice, so two products do the whole
// (ph + pl) (wh + wl) of 2 x 256 updates with FP32 sums and drop nothing.
// Operand layouts (checked on gfx950): A[i][k] in lane i + 16 (k / 8), element
// k % 8; B[k][j] in lane j + 16 (k / 8), element k % 8; D[i][j] in lane
// j + 16 (i / 4), element i % 4.  Lane group g = lane / 16 holds samples 2g and
// 2g + 1 of the window, as [ph ph pl pl] of the first angle, then of the second.
//
// Slices that this does not suit -- samples that are not finite, which would reach every
// pixel of a window (0 * NaN), or a few rows far above all others -- are back-projected
// again by the vector kernel (bpx_apart_kernel).
#include "rv_internal.h"

#include <cfloat>
#include <type_traits>

namespace rv {

typedef _Float16 xhalf2 __attribute__((ext_vector_type(2)));
typedef _Float16 xhalf8 __attribute__((ext_vector_type(8)));
typedef float xfloat2 __attribute__((ext_vector_type(2)));
typedef float xfloat4 __attribute__((ext_vector_type(4)));
typedef unsigned int xuint2 __attribute__((ext_vector_type(2)));
typedef unsigned int xuint4 __attribute__((ext_vector_type(4)));

// global (not flat) pointers: flat loads would count with the LDS reads
typedef const __attribute__((address_space(1))) unsigned char* gbytes;
typedef const __attribute__((address_space(1))) xfloat4* gfloat4;
typedef const __attribute__((address_space(1))) float* gfloat;

namespace bpx {
constexpr int kTile = 32;                  // pixels per tile side: 8 x 8 blocks
constexpr int kSeg = 48;                   // staged samples per angle: a tile spans at most 31 sqrt 2 = 43.9
constexpr int kPairs = kSeg / 2;
constexpr int kMaxJ0 = kSeg - 8;           // last window start
constexpr int kAng = 4;                    // angles per chunk (one contraction)
constexpr int kWaves = 8;                  // waves of a workgroup
constexpr int kGroups = bp_slices_per_item(BP_LINEAR_X64) / 16;     // groups of 16 slices
constexpr int kPlane = kPairs * 128 + 16;  // LDS bytes of one plane (16 slices); the 16 keeps reads of
                                           // different planes from pairing into ds_read2 (whose results
                                           // would need moves into place)
// three chunks of rows, eight waves' tables of row ends, the work item
constexpr int kLdsBytes = 3 * kAng * kGroups * kPlane + kWaves * 8 * 16 + 16;
}  // namespace bpx

// Tile geometry entry of (tile, angle): cos, sin, the tile origin's coordinate
// relative to s0, and s0 (even) with bit 0 set when the tile meets the ends of the
// detector row.  A tile that sees no sample reads the zero padding.
__global__ void __launch_bounds__(256) bpx_geometry_kernel(const AngleEntry* ang, int nang, int nang_pad, int tiles_x,
                                                           int ntiles, int N, float4* out)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)nang_pad * ntiles) return;
    const int t = (int)(i / nang_pad);
    const int a = (int)(i - (long long)t * nang_pad);
    float4 r = make_float4(0.f, 0.f, 0.f, __int_as_float(-kBpxPad));
    if (a < nang) {
        const AngleEntry e = ang[a];
        const int X0 = (t % tiles_x) * bpx::kTile, Y0 = (t / tiles_x) * bpx::kTile;
        const double ut = e.u0 + (double)X0 * e.dux + (double)Y0 * e.duy;
        const double m = bpx::kTile - 1;
        const double umin = ut + fmin(0.0, m * e.dux) + fmin(0.0, m * e.duy);
        const double umax = ut + fmax(0.0, m * e.dux) + fmax(0.0, m * e.duy);
        if (umax > -0.5 && umin < N + 0.5) {
            const int s0 = (int)floor(umin) & ~1;
            const int edge = (umin < 0.5 || umax > N - 1.5) ? 1 : 0;
            r = make_float4((float)e.dux, (float)e.duy, (float)(ut - (double)s0), __int_as_float(s0 | edge));
        }
    }
    out[i] = r;
}

void launch_bpx_geometry(const AngleEntry* ang, int nang, int tiles_x, int ntiles, int N, float4* out,
                         hipStream_t stream)
{
    const int np = bpx_angles(nang);
    const long long n = (long long)np * ntiles;
    if (n <= 0) return;
    hipLaunchKernelGGL(bpx_geometry_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, ang, nang, np,
                       tiles_x, ntiles, N, out);
}

// lane n of every 16-lane row, broadcast within the row
template <int N>
__device__ __forceinline__ float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ int row_bcast(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + N, 0xf, 0xf, true);
}

template <int I>
using Int = std::integral_constant<int, I>;

template <int I, int E, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < E) {
        f(Int<I>{});
        static_for<I + 1, E>(f);
    }
}

// One work item: kGroups groups of 16 slices of one 32 x 32 tile, by kWaves waves of a row
// of eight blocks each.
__device__ __forceinline__ void bpx_item(const BpSlice& S, int t, float minus_one, xfloat4* part)
{
    using namespace bpx;
    extern __shared__ xuint4 lds16[];
    unsigned char* lds = (unsigned char*)lds16;
    constexpr int NG = kGroups, NW = kWaves;
    constexpr int NB = 64 / NW, NSET = NB / 4;         // blocks per wave, in sets of four
    static_assert(NB == 8, "a wave's blocks are a row of the tile");
    constexpr int ABYTES = NG * kPlane;                // one staged angle
    constexpr int CBYTES = kAng * ABYTES;              // one chunk
    const int N = S.row_len;
    const int nch = bpx_angles(S.nang) / kAng;
    const gfloat4 tg = (gfloat4)S.tgeom + (size_t)t * (nch * kAng);
    const unsigned int plane_stride = (unsigned int)bpx_pairs(N) * 128u;     // bytes of one plane of a packed row
    const unsigned int row_stride = plane_stride * NG;
    const gbytes packed = (gbytes)S.rows;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, n = lane & 15;
    const float xl = (float)(n & 3), yl = (float)(n >> 2), gneg = -2.f * (float)g;
    // table lane: angle (lane % 16) / 4 of the chunk, block lane % 4 of the wave
    const int ta = (lane >> 2) & 3;
    const int wy0 = 4 * wave;
    const float bx = (float)(4 * (lane & 3)), by = (float)wy0;

    const int X0 = (t % S.tiles_x) * kTile, Y0 = (t / S.tiles_x) * kTile;
    const int ox = X0 & 32, oy = Y0 & 32;              // offset inside the 64 x 64 tile

    // staging: a unit is 1 KB (a third) of one plane of one angle, copied by one wave
    constexpr int UNITS = kAng * NG * 3, PER = (UNITS + NW - 1) / NW;
    xuint4 sreg[PER];
    const unsigned int lane16 = 16u * lane;
    // rows: the chunk's first row; w: its table entries, angle a's in lanes 4a .. 4a + 3
    auto fetch = [&](auto ki, gbytes rows, float w) {
        constexpr int k = decltype(ki)::value;
        const int u = NW * k + wave;
        if (UNITS % NW == 0 || u < UNITS) {
            const int a = u / (3 * NG), pl = u / 3 % NG;
            const int s0 = __builtin_amdgcn_readlane(__float_as_int(w), 4 * a) & ~1;
            const unsigned int off = (unsigned int)a * row_stride + (unsigned int)pl * plane_stride +
                                     (unsigned int)(s0 + kBpxPad) * 64u + (unsigned int)(u % 3) * 1024u;
            sreg[k] = *(const __attribute__((address_space(1))) xuint4*)(rows + off + lane16);
        }
    };
    auto stage = [&](auto ki, int buf) {                   // buf: byte offset
        constexpr int k = decltype(ki)::value;
        const int u = NW * k + wave;
        if (UNITS % NW == 0 || u < UNITS)
            *(xuint4*)(lds + (buf + (u / 3) * kPlane + (u % 3) * 1024 + lane16)) = sreg[k];
    };

    xfloat4 acc[NB][NG];

    // A chunk's window of this lane's (angle, block): the block origin's coordinate
    // relative to the even window start j0, and the LDS offset of the window's first
    // pair; the coordinate of the lane's pixel and sample relative to the origin's
    struct Window {
        float bp[NSET], lp[kAng];
        int adr[NSET], buf, c, sw;
        bool edge;
    };
    struct Origin {
        float ub[NSET], m;
        int j0[NSET];
    };
    // the wave's own table of the chunk's angles on the 64 x 64 tile, two chunks deep
    xfloat4* ends = (xfloat4*)(lds + 3 * CBYTES) + 8 * wave;
    // in kWin pieces of a few vector instructions
    auto window = [&](auto piece_, Window& k, Origin& f, const xfloat4 geo, int c, int buf) {
        constexpr int piece = decltype(piece_)::value;
#pragma unroll
        for (int z = 0; z < NSET; z++) {
            if constexpr (piece == 0) f.ub[z] = fmaf(bx + 16.f * z, geo.x, geo.z);
            if constexpr (piece == 1) f.ub[z] = fmaf(by, geo.y, f.ub[z]);
            if constexpr (piece == 3) f.j0[z] = (int)(f.ub[z] + f.m) & ~1;
            if constexpr (piece == 4) f.j0[z] = min(max(f.j0[z], 0), kMaxJ0);
            if constexpr (piece == 5) k.bp[z] = f.ub[z] - (float)f.j0[z];
            if constexpr (piece == 6) k.adr[z] = buf + ta * ABYTES + f.j0[z] * 64;
        }
        if constexpr (piece == 2) f.m = fminf(0.f, 3.f * geo.x) + fminf(0.f, 3.f * geo.y);
        if constexpr (piece >= 7) {
            constexpr int a = piece - 7;
            k.lp[a] = fmaf(yl, row_bcast<4 * a>(geo.y), fmaf(xl, row_bcast<4 * a>(geo.x), gneg));
        }
        if constexpr (piece == 0) {
            k.buf = buf;
            k.c = c;
            k.sw = __float_as_int(geo.w);
            k.edge = __builtin_amdgcn_ballot_w64((k.sw & 1) != 0) != 0;
            if (__builtin_expect(k.edge, false)) {
                    // the 64 x 64 tile's origin of the lane's angle, as bp_tiled_kernel forms it
                    const AngleEntry& e = S.ang[min(c * kAng + ta, S.nang - 1)];
                    const double ut = e.u0 + (double)(X0 - ox) * e.dux + (double)(Y0 - oy) * e.duy;
                    const int s0 = (int)floor(ut + fmin(0.0, 63.0 * e.dux) + fmin(0.0, 63.0 * e.duy)) - 1;
                    ends[4 * (c & 1) + ta] = xfloat4{(float)e.dux, (float)e.duy, (float)(ut - (double)s0),
                                                     __int_as_float(s0)};
                }
        }
    };
    constexpr int kWin = 7 + kAng;
    const int lane8 = 8 * lane;

    // Weights of block b for angles 2p and 2p + 1: W(k) of the lane's samples 2g and
    // 2g + 1, in kWeights pieces of two to four vector instructions: they end a slot before the
    // products that read them.
    constexpr int kWeights = 7;
    struct Weights {
        float r[2], t[2], w[2][2];
        xhalf2 h[2], l[2];
    };
    auto weights = [&](auto piece_, auto bi, auto pi, const Window& k, Weights& f, xhalf8& Wh, xhalf8& Wl) {
        constexpr int piece = decltype(piece_)::value, b = decltype(bi)::value, p = decltype(pi)::value, z = b / 4;
        if constexpr (piece == 0) {
            static_for<0, 2>([&](auto ai) {
                constexpr int a = decltype(ai)::value, e = 4 * (2 * p + a) + b % 4;
                f.r[a] = row_bcast<e>(k.bp[z]) + k.lp[2 * p + a];
            });
            if (__builtin_expect(k.edge, false)) {
                    // some angle of the chunk meets an end of the row: nothing before the first
                    // sample and after the last, which is held for one step, decided by the
                    // vector kernels' coordinate on their 64 x 64 tile (bp_tiled_kernel)
                    const int j0 = (k.adr[z] - k.buf - ta * ABYTES) / 64;
                    const float last = (float)(N - 1 - (k.sw & ~1) - j0);  // last sample, from the window's start
                    const float dxl = (float)(ox + 4 * (b & 1) + (n & 3)), xi = (float)((4 * b) & 24);
                    const float dyl = (float)(oy + wy0 % 8 + (n >> 2)), yj = (float)(wy0 & 24);
                    static_for<0, 2>([&](auto ai) {
                        constexpr int a = decltype(ai)::value, A = 2 * p + a, e = 4 * A + b % 4;
                        const xfloat4 g64 = ends[4 * (k.c & 1) + A];
                        const float u = fmaf(xi, g64.x, fmaf(yj, g64.y, fmaf(dyl, g64.y, fmaf(dxl, g64.x, g64.z))));
                        const int q = __float_as_int(g64.w) + (int)u;
                        const float rl = row_bcast<e>(last) + gneg;
                        f.r[a] = (q < 0 || q >= N) ? -64.f : q == N - 1 ? rl : f.r[a];
                    });
                }
        }
        if constexpr (piece == 1)
            for (int a = 0; a < 2; a++) {
                f.t[a] = f.r[a] - 1.f;
                f.w[a][0] = __builtin_amdgcn_fmed3f(1.f - fabsf(f.r[a]), 0.f, 1.f);
            }
        if constexpr (piece == 2)
            for (int a = 0; a < 2; a++) f.w[a][1] = __builtin_amdgcn_fmed3f(1.f - fabsf(f.t[a]), 0.f, 1.f);
        if constexpr (piece == 3)
            for (int a = 0; a < 2; a++) f.h[a] = __builtin_convertvector((xfloat2{f.w[a][0], f.w[a][1]}), xhalf2);
        if constexpr (piece == 4)
            for (int a = 0; a < 2; a++) f.l[a].x = (_Float16)fmaf((float)f.h[a].x, minus_one, f.w[a][0]);
        if constexpr (piece == 5)
            for (int a = 0; a < 2; a++) f.l[a].y = (_Float16)fmaf((float)f.h[a].y, minus_one, f.w[a][1]);
        if constexpr (piece == 6) {
            Wh = __builtin_shufflevector(f.h[0], f.h[1], 0, 1, 0, 1, 2, 3, 2, 3);
            Wl = __builtin_shufflevector(f.l[0], f.l[1], 0, 1, 0, 1, 2, 3, 2, 3);
        }
    };
    // LDS address of angle 2p + a's window of block b
    auto address = [&](auto bi, auto pi, auto ai, const Window& k) {
        constexpr int b = decltype(bi)::value, A = 2 * decltype(pi)::value + decltype(ai)::value;
        return row_bcast<4 * A + b % 4>(k.adr[b / 4]) + lane8;
    };
    auto sample = [&](int va, int q, int a, xuint4& pv) {
        const xuint2 d = *(const xuint2*)(lds + va + q * kPlane);
        pv[2 * a] = d.x;
        pv[2 * a + 1] = d.y;
    };

    // A step is one angle pair of one block: 2 NG products, in as many slots.  Each slot
    // also issues one LDS read for the next step and a piece of the next step's weights,
    // so that the three pipes run side by side with two waves per SIMD.
    // Three LDS buffers: in the first half of chunk c the rows of chunk c + 1 (fetched
    // a chunk earlier) go into the buffer chunk c - 2 used; in its middle one barrier makes
    // them visible and keeps every wave within a chunk of the others, and then the rows of
    // chunk c + 2 are fetched; the products of a wave run on from chunk to chunk.
    constexpr int SLOTS = 2 * NG, NSLOT = 2 * NB * SLOTS;      // slots of a step and of a chunk
    constexpr int ST0 = NSLOT / 2 - 2 * SLOTS - PER, BAR = NSLOT / 2, FE0 = BAR + 1, WI0 = BAR + PER + 2;
    constexpr int WID = (NSLOT - SLOTS - WI0) / kWin;          // slots between the window's pieces
    static_assert(ST0 >= 0 && WID >= 1 && kWeights < SLOTS, "the parts fit their slots");
    int c0 = 0, c1 = nch;                                  // chunks of the segment
    auto at = [&](int c) { return min(c, c1 - 1); };       // chunks past the last repeat it, unused
    auto rows_at = [&](int c) { return packed + (size_t)at(c) * kAng * row_stride; };
    const gfloat tw = (gfloat)tg + 4 * ta + 3;             // s0 of the lane's angle
    auto w_at = [&](int c) { return tw[at(c) * 4 * kAng]; };
    // The products round the sums oftener than one addition per angle does, so the
    // angles are summed in segments whose totals are added apart (through the
    // workgroup's own 256 KB of workspace): with two segments the error against FP64 is
    // below the vector kernels'.
    const int nseg = max(2, (nch * kAng + 1023) / 1024);
    for (int seg = 0; seg < nseg; seg++) {
        c0 = (int)((long long)nch * seg / nseg);
        c1 = (int)((long long)nch * (seg + 1) / nseg);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int q = 0; q < NG; q++) acc[b][q] = xfloat4{0.f, 0.f, 0.f, 0.f};
        if (c0 == c1) continue;
        __syncthreads();                                   // the last segment's reads are done
        static_for<0, PER>([&](auto k) { fetch(k, rows_at(c0), w_at(c0)); });
        static_for<0, PER>([&](auto k) { stage(k, 0); });
        static_for<0, PER>([&](auto k) { fetch(k, rows_at(c0 + 1), w_at(c0 + 1)); });
        xfloat4 gn = tg[at(c0 + 1) * kAng + ta];
        float w2 = w_at(c0 + 2);
        __syncthreads();
        Window win;
        Origin org;
        static_for<0, kWin>([&](auto i) { window(i, win, org, tg[c0 * kAng + ta], c0, 0); });
        xuint4 pv[2][NG];
        xhalf8 Wh[2], Wl[2];
        {
            Weights f;
            static_for<0, kWeights>([&](auto i) { weights(i, Int<0>{}, Int<0>{}, win, f, Wh[0], Wl[0]); });
            const int v0 = address(Int<0>{}, Int<0>{}, Int<0>{}, win), v1 = address(Int<0>{}, Int<0>{}, Int<1>{}, win);
    #pragma unroll
            for (int q = 0; q < NG; q++) {
                sample(v0, q, 0, pv[0][q]);
                sample(v1, q, 1, pv[0][q]);
            }
        }
        for (int c = c0; c < c1; c++) {
            Window next;
            const int nbuf = win.buf == 2 * CBYTES ? 0 : win.buf + CBYTES;
            const gbytes rows2 = rows_at(c + 2);
            static_for<0, 2 * NB>([&](auto hi_) {
                constexpr int h = decltype(hi_)::value, b = h / 2, p = h & 1;
                constexpr bool wrap = h + 1 == 2 * NB;
                constexpr int nb = wrap ? 0 : (h + 1) / 2;             // the next step's block; its pair is 1 - p
                const Window& k = wrap ? next : win;
                Weights f;
                int va[2];
                static_for<0, SLOTS>([&](auto si) {
                    constexpr int i = decltype(si)::value, q = i / 2, slot = h * SLOTS + i;
                    xfloat4& A = acc[b][q];
                    const xhalf8 P = __builtin_bit_cast(xhalf8, pv[p][q]);
                    A = __builtin_amdgcn_mfma_f32_16x16x32_f16(P, (i & 1) ? Wl[p] : Wh[p], A, 0, 0, 0);
                    if constexpr (i < 2) va[i] = address(Int<nb>{}, Int<1 - p>{}, Int<i>{}, k);
                    sample(va[i & 1], q, i & 1, pv[1 - p][q]);
                    if constexpr (i < kWeights) weights(si, Int<nb>{}, Int<1 - p>{}, k, f, Wh[1 - p], Wl[1 - p]);
                    if constexpr (slot >= ST0 && slot < ST0 + PER) stage(Int<slot - ST0>{}, nbuf);
                    if constexpr (slot == BAR) {
                        // the rows were written 2 SLOTS reads ago and more: all but the last
                        // SLOTS LDS operations done means they are in place
                        asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"i"(SLOTS) : "memory");
                    }
                    if constexpr (slot >= FE0 && slot < FE0 + PER) fetch(Int<slot - FE0>{}, rows2, w2);
                    if constexpr (slot >= WI0 && slot < WI0 + kWin * WID && (slot - WI0) % WID == 0)
                        window(Int<(slot - WI0) / WID>{}, next, org, gn, c + 1, nbuf);
                    if constexpr (slot == WI0 + kWin * WID) {
                        gn = tg[at(c + 2) * kAng + ta];
                        w2 = w_at(c + 3);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            win = next;
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int q = 0; q < NG; q++) {
                xfloat4* p = part + (b * NG + q) * (64 * NW) + tid;
                if (seg > 0) acc[b][q] += *p;
                if (seg + 1 < nseg) *p = acc[b][q];
            }
    }

    // lane l, element e of group q: slice 16 q + 4 (l / 16) + e of pixel l % 16
    const int X = X0 + (n & 3);
    const int Y = Y0 + wy0 + (n >> 2);
    const int out_n = S.out_n;
    const int* ex = (const int*)S.gscale;
#pragma unroll
    for (int q = 0; q < NG; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int sl = 16 * q + 4 * g + e;
            float* out = (float*)(sl == 0 ? S.out : S.out_x[sl - 1]);
            const int sh = ex[sl];
#pragma unroll
            for (int b = 0; b < NB; b++)
                if (X + 4 * b < out_n && Y < out_n)
                    out[(long long)Y * out_n + X + 4 * b] = ldexpf(acc[b][q][e], sh) * S.out_scale;
        }
}

// Two waves per SIMD (512 registers a lane between them): 128 sums, 64 registers of
// operands in flight and 24 of rows on their way to LDS.
// 64 slices of 2048^2 x 1800: 29.5 ms, 1.64e13 updates/s (four slices per item on the
// vector ALU: 36.5 ms).  Bound by instruction issue: a slot of one product (16 clocks of
// its pipe), one 8-byte LDS read and three vector instructions takes 24.9 clocks per
// SIMD alone and 26 here.  Slower than this form when tried: items of 32 or 16 slices (weights
// shared by fewer updates; not compared with four per item), four angles per contraction with three products (half the LDS reads, but
// 16-byte reads of four rows each), a second body without the row-end test.
__global__ void __launch_bounds__(64 * bpx::kWaves, 2) bpx_kernel(BpLaunch L, float minus_one)
{
    extern __shared__ xuint4 lds16[];
    xfloat4* part = (xfloat4*)L.part + (size_t)blockIdx.x * (kBpxPart / 4);
    int* item_sh = (int*)((unsigned char*)lds16 + bpx::kLdsBytes - 16);
    // the list in eight contiguous parts, one per XCD; a workgroup whose own part is
    // taken goes on with the next
    const int per_xcd = (L.total_items + kXcds - 1) / kXcds;
    int probe = 0;
    while (true) {
        __syncthreads();
        if (threadIdx.x == 0) {
            int pos = L.total_items;
            for (; probe < kXcds; probe++) {
                const int q = (int)((blockIdx.x + probe) % kXcds);
                const int k = (int)atomicAdd(L.counter + q * kCounterStride, 1u);
                if (k < per_xcd && q * per_xcd + k < L.total_items) {
                    pos = q * per_xcd + k;
                    break;
                }
            }
            *item_sh = pos;
        }
        __syncthreads();
        const int pos = __builtin_amdgcn_readfirstlane(*item_sh);
        if (pos >= L.total_items) break;
        const int item = L.item_order[pos];
        int lo = 0, hi = L.nslices - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (L.slices[mid].tile_base <= item) lo = mid; else hi = mid - 1;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        const BpSlice& S = L.slices[lo];
        bpx_item(S, item - S.tile_base, minus_one, part);
    }
}

// ------------------------------------------------------------ packed rows
// Largest magnitude of every filtered row, infinity where a sample is not finite: one
// wave per row, rows of slice y of job z.
__global__ void __launch_bounds__(256) bpx_row_max_kernel(const PackJob* jobs)
{
    const PackJob& J = jobs[blockIdx.z];
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= J.nrows) return;
    const float* src = (const float*)J.rows[blockIdx.y] + (long long)row * J.N;
    float m = 0.f;
    auto take = [&](float x) {
        const float v = fabsf(x);
        m = v <= FLT_MAX ? fmaxf(m, v) : INFINITY;
    };
    const int head = min(J.N, (int)(((16 - ((uintptr_t)src & 15)) & 15) / 4)), quads = (J.N - head) / 4;
    const float4* body = (const float4*)(src + head);
    for (int i = lane; i < quads; i += 64) {
        const float4 v = body[i];
        take(v.x); take(v.y); take(v.z); take(v.w);
    }
    // the values before and after the 16-byte quads (at most six)
    const int rest = lane < head ? lane : lane + 4 * quads;
    if (rest < J.N) take(src[rest]);
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) J.row_max[(size_t)blockIdx.y * J.nrows + row] = m;
}

// Exponent of each slice: its samples times 2^-e lie within 2^15.  A slice runs apart
// (bpx_apart_kernel) where the matrix products would lose what it holds: when a sample
// is not finite, and when one of a few rows is so large that most others lie below 2^-14
// of it, from where on the split would leave them fewer bits than FP32 does (rows at
// 2^-16 of the largest still keep 23, at 2^-20 they keep 20, at 2^-24 16).  Rows of
// zeros are exact and do not count.
__global__ void __launch_bounds__(256) bpx_exponent_kernel(const PackJob* jobs)
{
    const PackJob& J = jobs[blockIdx.y];
    const float* row_max = J.row_max + (size_t)blockIdx.x * J.nrows;
    __shared__ float red[4];
    float m = 0.f;
    for (int k = threadIdx.x; k < J.nrows; k += 256) m = fmaxf(m, row_max[k]);
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float low = m * 0x1p-14f;
    int weak = 0, strong = 0;
    for (int k0 = 0; k0 < J.nrows; k0 += 256) {
        const float v = k0 + threadIdx.x < J.nrows ? row_max[k0 + threadIdx.x] : 0.f;
        weak += __syncthreads_count(v > 0.f && v < low);
        strong += __syncthreads_count(v >= low && v > 0.f);
    }
    if (threadIdx.x == 0) {
        int e = 15;
        const bool finite = m <= FLT_MAX;
        if (finite && m > 0.f) frexpf(m, &e);
        ((int*)J.gscale)[blockIdx.x] = e - 15;
        ((int*)J.gscale)[J.ns + blockIdx.x] = !finite || weak > strong;
    }
}

// Packed row: [plane 2 q + part][pair][16 slices] of FP16 pairs (samples 2j, 2j + 1),
// part 0 the high and part 1 the low halves of group q, kBpxPad zero samples on
// either side.  A slice's samples only reach its own sums, so those of slices that run
// apart may be anything.  Thread: one slice, eight consecutive samples.
__global__ void __launch_bounds__(256) bpx_pack_kernel(const PackJob* jobs)
{
    const PackJob& J = jobs[blockIdx.z];
    const int N = J.N, pairs = bpx_pairs(N);
    const int row = blockIdx.x;
    if (row >= bpx_angles(J.nrows)) return;
    const bool used = row < J.nrows;               // rows up to a whole chunk are zero
    const int i = threadIdx.x & 15, q = blockIdx.y;
    const int sh = -((const int*)J.gscale)[16 * q + i];
    const float* src = (const float*)J.rows[16 * q + i] + (long long)row * N;
    xuint2* o = (xuint2*)J.out + ((size_t)row * bpx::kGroups + q) * pairs * 16 + i;
    const bool aligned = ((uintptr_t)src & 15) == 0;       // then src + j is, j being a multiple of four
    for (int p0 = 4 * (threadIdx.x >> 4); p0 < pairs; p0 += 64) {
        const int j0 = 2 * p0 - kBpxPad;
        float v[8];
        if (used && aligned && j0 >= 0 && j0 + 8 <= N) {
            const float4 a = *(const float4*)(src + j0), b = *(const float4*)(src + j0 + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = (used && j0 + k >= 0 && j0 + k < N) ? src[j0 + k] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = ldexpf(v[k], sh);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (p0 + k >= pairs) break;
            const xhalf2 h = __builtin_convertvector((xfloat2{v[2 * k], v[2 * k + 1]}), xhalf2);
            const xhalf2 l = __builtin_convertvector(
                (xfloat2{v[2 * k] - (float)h.x, v[2 * k + 1] - (float)h.y}), xhalf2);
            o[(size_t)(p0 + k) * 16] = xuint2{__builtin_bit_cast(unsigned int, h), __builtin_bit_cast(unsigned int, l)};
        }
    }
}

// Work list of the slices that run apart, one slice per item on the vector ALU
// (bp_tiled_kernel, whose images they keep bit for bit): rest holds an entry for every
// slice of the items, in order; the tiles of those marked fill the end of the list and
// the persistent launch's counter starts there, so that nothing marked is nothing to do.
__global__ void __launch_bounds__(1024) bpx_apart_kernel(const BpSlice* items, int nitems, BpSlice* rest, int* order,
                                                         int total, unsigned int* counter)
{
    constexpr int NS = bp_slices_per_item(BP_LINEAR_X64);
    __shared__ int marked[NS];
    const int tid = threadIdx.x;
    int end = total;
    for (int q = 0; q < nitems; q++) {
        const int mark = tid < NS ? ((const int*)items[q].gscale)[NS + tid] : 0;
        if (tid < NS) marked[tid] = mark;
        if (!__syncthreads_or(mark)) continue;
        for (int e = 0; e < NS; e++) {
            if (!marked[e]) continue;
            BpSlice& R = rest[NS * q + e];
            const int n = R.tiles_x * R.tiles_y;
            end -= n;
            for (int t = tid; t < n; t += 1024) order[end + t] = R.tile_base + t;
            if (tid == 0) R.out = e == 0 ? items[q].out : items[q].out_x[e - 1];
        }
        __syncthreads();
    }
    if (tid == 0) *counter = end;
}

void launch_bpx_pack(const PackJob* d_jobs, int njobs, int max_rows, hipStream_t stream)
{
    constexpr int ns = bp_slices_per_item(BP_LINEAR_X64);
    if (njobs <= 0 || max_rows <= 0) return;
    hipLaunchKernelGGL(bpx_row_max_kernel, dim3((max_rows + 3) / 4, ns, njobs), dim3(256), 0, stream, d_jobs);
    hipLaunchKernelGGL(bpx_exponent_kernel, dim3(ns, njobs), dim3(256), 0, stream, d_jobs);
    hipLaunchKernelGGL(bpx_pack_kernel, dim3(bpx_angles(max_rows), bpx::kGroups, njobs), dim3(256), 0, stream, d_jobs);
}

void launch_bpx_apart(const BpSlice* items, int nitems, BpSlice* rest, int* order, int total, unsigned int* counter,
                      hipStream_t stream)
{
    hipLaunchKernelGGL(bpx_apart_kernel, dim3(1), dim3(1024), 0, stream, items, nitems, rest, order, total, counter);
}

void bpx_prepare()
{
    (void)hipFuncSetAttribute((const void*)&bpx_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bpx::kLdsBytes);
}

void launch_bpx(const BpLaunch& L, int grid, hipStream_t stream)
{
    hipLaunchKernelGGL(bpx_kernel, dim3(grid), dim3(64 * bpx::kWaves), bpx::kLdsBytes, stream, L, -1.f);
}

}  // namespace rv
