// rv_sinogram.hip -- sinogram generation on the GPU: dark / incident (flat)
// correction with the incident interpolated in exposure time, -ln(I/I0) x
// LOG_SCALE (or the Zernike ratio), the pixel-count floor and the drift shift,
// with the production semantics of GenerateSinogramThread (general.cpp:2377-2532).
// A grid row per frame (a job), its multiplex lines side by side in the grid's columns; the
// host resolves the incident frames, weights and shifts (the sequential part) into the
// job table.
#include "rv_internal.h"

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace rv {

// log(a / b) to 2^-39 for a finite a > 0 and an integer b in [1, 65535], as
// k ln 2 + 2 atanh((a - b 2^k) / (a + b 2^k)) with b 2^k within a factor sqrt 2 of a
// (the area hyperbolic tangent's power series, |argument| <= 0.1716): one reciprocal
// and 16 operations of 64 bits instead of a division and a logarithm.  What it is
// rounded to is FP32: of 14 million ratios, near 1 and near the factor sqrt 2 among them,
// 40 round differently than the library's log of the quotient, the largest error being
// 0.50001 of a unit in the last place against 0.512 (near 1, where the quotient's own
// rounding shows).
__device__ __forceinline__ float log_ratio(float a, int b)
{
    const float fb = (float)b;
    const float ma = __builtin_amdgcn_frexp_mantf(a), mb = __builtin_amdgcn_frexp_mantf(fb);
    int k = __builtin_amdgcn_frexp_expf(a) - __builtin_amdgcn_frexp_expf(fb);
    if (ma > 1.4142135f * mb) k++;
    else if (1.4142135f * ma < mb) k--;
    const double x = (double)a, y = ldexp((double)b, k);
    const double den = x + y;
    double r = __builtin_amdgcn_rcp(den);                  // 2^-22 and better
    r = fma(fma(-den, r, 1.0), r, r);
    const double s = (x - y) * r, z = s * s;
    double q = fma(z, 1.0 / 13, 1.0 / 11);
    q = fma(q, z, 1.0 / 9);
    q = fma(q, z, 1.0 / 7);
    q = fma(q, z, 1.0 / 5);
    q = fma(q, z, 1.0 / 3);
    const double s2 = s + s;
    return (float)fma((double)k, 0.69314718055994530942, fma(s2 * z, q, s2));
}

// One sample: dark-corrected, against the interpolated incident frames.
// kOut 0: int16 as the reference; 1: float, without the x3000 scale and rounding.
template <int kOut>
__device__ __forceinline__ auto convert(int row, int dark, int a0, int a1, float t0, int pixmin, int zernike)
{
    int16_t v = 0;
    float fv = 0.f;
    // unsigned short + float arithmetic in float, kept as double (general.cpp:2483)
    const float fa = (float)(a1 - a0) * t0;
    const float inc = ((float)a0 + fa) - (float)dark;
    const int is = row - dark;
    if (inc > 0 && is >= pixmin) {
        if constexpr (kOut == 1) {
            if (zernike) fv = (float)((double)inc / is);
            else if (inc <= FLT_MAX) fv = log_ratio(inc, is);
            else fv = (float)log((double)inc / is);
        } else {
            v = zernike ? (int16_t)(int)((double)inc * 1000 / is + 0.5)
                        : (int16_t)(int)(log((double)inc / is) * 3000 + 0.5);
        }
    }
    if constexpr (kOut == 1) return fv;
    else return v;
}

typedef unsigned int su4 __attribute__((ext_vector_type(4)));

// out_full = 1 writes row frame * mult + k (the frames' layout), 0 writes row
// j * mult + k of job j.  Block: 2048 samples of one row, eight consecutive ones per
// thread with 16-byte loads where rows are 16-byte aligned and not shifted (vec), else
// eight 256 apart.
// 2048 x 8 lines x 1803 frames to float (0.18 GB moved): 52 us, bound by the 64-bit
// operations of log_ratio; 139 us with one sample per thread, 64-bit division and log.
template <int kOut>
__global__ void __launch_bounds__(256) sinogram_kernel(const uint16_t* frames, int nframes, int mult, int W,
                                                       const SinoJob* jobs, void* out, int pixmin, int zernike,
                                                       int out_full, int vec)
{
    using T = typename std::conditional<kOut == 1, float, int16_t>::type;
    const SinoJob J = jobs[blockIdx.y];
    const int nx = (W + 2047) / 2048, kk = blockIdx.x / nx;
    T* orow = (T*)out + ((size_t)(out_full ? J.frame : (int)blockIdx.y) * mult + kk) * W;
    const uint16_t* dark = frames + ((size_t)(nframes - 1) * mult + kk) * W;
    const uint16_t* a0 = frames + ((size_t)J.i0 * mult + kk) * W;
    const uint16_t* a1 = frames + ((size_t)J.i1 * mult + kk) * W;
    const uint16_t* row = frames + ((size_t)J.frame * mult + kk) * W;
    const int x0 = blockIdx.x % nx * 2048;
    if (vec && J.shift == 0) {
        const int j = x0 + 8 * threadIdx.x;
        if (j >= W) return;                                // W is a multiple of eight
        T v[8] = {};
        if (J.action == 1) {
            const su4 r = *(const su4*)(row + j), d = *(const su4*)(dark + j), p = *(const su4*)(a0 + j),
                      q = *(const su4*)(a1 + j);
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const int sh = 16 * (m & 1);
                v[m] = convert<kOut>((r[m / 2] >> sh) & 0xffff, (d[m / 2] >> sh) & 0xffff, (p[m / 2] >> sh) & 0xffff,
                                     (q[m / 2] >> sh) & 0xffff, J.t0, pixmin, zernike);
            }
        }
        su4* o = (su4*)(orow + j);
        const su4* w = (const su4*)v;
#pragma unroll
        for (int m = 0; m < (int)sizeof(T) / 2; m++) o[m] = w[m];
        return;
    }
    for (int m = 0; m < 8; m++) {
        const int j = x0 + 256 * m + threadIdx.x;
        if (j >= W) return;
        const int src = j - J.shift;                       // general.cpp:2501-2513: out[j] = row[j - shift], zero fill
        T v = 0;
        if (J.action == 1 && src >= 0 && src < W)
            v = convert<kOut>(row[src], dark[src], a0[src], a1[src], J.t0, pixmin, zernike);
        orow[j] = v;
    }
}

void launch_sinogram(const uint16_t* frames, int nframes, int mult, int W, const SinoJob* jobs,
                     int njobs, void* out, int pixmin, int zernike, int out_float, int out_full,
                     hipStream_t stream)
{
    if (njobs <= 0) return;
    const int vec = W % 8 == 0 && (((uintptr_t)frames | (uintptr_t)out) & 15) == 0;
    for (int k0 = 0; k0 < njobs; k0 += 65535) {
        const dim3 grid((W + 2047) / 2048 * mult, std::min(njobs - k0, 65535));     // grid y ends there
        void* o = out_full ? out : (char*)out + (size_t)k0 * mult * W * (out_float ? 4 : 2);
        if (out_float)
            hipLaunchKernelGGL(sinogram_kernel<1>, grid, dim3(256), 0, stream, frames, nframes, mult, W, jobs + k0, o,
                               pixmin, zernike, out_full, vec);
        else
            hipLaunchKernelGGL(sinogram_kernel<0>, grid, dim3(256), 0, stream, frames, nframes, mult, W, jobs + k0, o,
                               pixmin, zernike, out_full, vec);
    }
}

}  // namespace rv
