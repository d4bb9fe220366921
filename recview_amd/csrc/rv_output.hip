// rv_output.hip -- caller-side output stage on the GPU (gazoDoc.cpp:3993-4021):
// min / max over the whole square (imax starts at 0, imin at INT_MAX), then
// every pixel inside the circle of radius min(z*c/bin, N - z*c/bin) becomes
// (int)((float)(v - imin) * 65534 / (imax - imin)) and everything outside 0.
// Two launches: per-block min/max, normalise.
#include "recview_hip.h"
#include "rv_common.h"

#include <climits>
#include <cfloat>
#include <map>
#include <mutex>

namespace rv {

template <typename T>
struct Lim;
template <>
struct Lim<int> {
    static __device__ int lo() { return INT_MAX; }
};
template <>
struct Lim<float> {
    static __device__ float lo() { return FLT_MAX; }
};

template <typename T>
struct Quad {
    typedef T type __attribute__((ext_vector_type(4)));
};

// Minimum and maximum over a workgroup of 256, in every thread; NaN is passed over.
template <typename T>
__device__ __forceinline__ void block_minmax(T& mn, T& mx)
{
    __shared__ T smin[4], smax[4];
    auto take = [&](T a, T b) {
        mn = a < mn ? a : mn;
        mx = b > mx ? b : mx;
    };
    for (int off = 32; off > 0; off >>= 1) take(__shfl_xor(mn, off), __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) {
        smin[threadIdx.x >> 6] = mn;
        smax[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    for (int w = 0; w < 4; w++) take(smin[w], smax[w]);
}

template <typename T>
__global__ void __launch_bounds__(256) minmax_kernel(const T* img, long long n, T* part_min, T* part_max)
{
    using Q = typename Quad<T>::type;
    T mn = Lim<T>::lo(), mx = (T)0;
    auto take = [&](T v) {
        mn = v < mn ? v : mn;
        mx = v > mx ? v : mx;
    };
    const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
    // 16-byte loads from the first aligned value on; the values around them one by one
    const long long head = min(n, (long long)((16 - ((uintptr_t)img & 15)) & 15) / 4), quads = (n - head) / 4;
    const Q* body = (const Q*)(img + head);
    for (long long i = id; i < quads; i += (long long)gridDim.x * 256) {
        const Q v = body[i];
        take(v.x); take(v.y); take(v.z); take(v.w);
    }
    if (blockIdx.x == 0) {
        const long long rest = threadIdx.x < head ? threadIdx.x : threadIdx.x + 4 * quads;
        if (rest < n) take(img[rest]);
    }
    block_minmax(mn, mx);
    if (threadIdx.x == 0) {
        part_min[blockIdx.x] = mn;
        part_max[blockIdx.x] = mx;
    }
}

// Every workgroup reduces the nparts partial minima / maxima itself (4 KB at most, from
// L2) instead of waiting for a launch that does; the first one writes them to range
// (max bumped by one unit when equal to the min, gazoDoc.cpp:3999).  Threads take four
// pixels of a row at a time; vec: rows are 16-byte (image) and 8-byte (out) aligned.
template <typename T>
__global__ void __launch_bounds__(256) normalise_kernel(const T* img, int N, int irad2, const T* part_min,
                                                        const T* part_max, int nparts, T* range, uint16_t* out,
                                                        int vec)
{
    using Q = typename Quad<T>::type;
    T mn = Lim<T>::lo(), mx = (T)0;
    for (int i = threadIdx.x; i < nparts; i += 256) {
        mn = part_min[i] < mn ? part_min[i] : mn;
        mx = part_max[i] > mx ? part_max[i] : mx;
    }
    block_minmax(mn, mx);
    if (mx == mn) mx = mx + (T)1;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        range[0] = mn;
        range[1] = mx;
    }
    const float span = (float)(mx - mn);
    const unsigned int per_row = (N + 3) / 4;
    const int h = N / 2;
    const long long total = (long long)N * per_row;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
        const int r = total <= 0xffffffffll ? (int)((unsigned int)i / per_row) : (int)(i / per_row);
        const int c = (int)(i - (long long)r * per_row) * 4;
        const long long o = (long long)r * N + c;
        const int i2 = (r - h) * (r - h);
        uint16_t v[4] = {};
        T x[4];
        if (vec) *(Q*)x = *(const Q*)(img + o);
        else
            for (int k = 0; k < 4; k++) x[k] = c + k < N ? img[o + k] : (T)0;
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (i2 + (c + k - h) * (c + k - h) <= irad2) {
                const float d = (float)(x[k] - mn);
                v[k] = (uint16_t)(int)(d * (float)(65535 - 1) / span);
            }
        if (vec) *(uint2*)(out + o) = make_uint2(v[0] | (unsigned int)v[1] << 16, v[2] | (unsigned int)v[3] << 16);
        else
            for (int k = 0; k < 4 && c + k < N; k++) out[o + k] = v[k];
    }
}

// 2048^2 floats (25 MB): 13.9 us; three launches of one pixel per thread took 18.5.  The
// rest of a call is two launches and the wait for the range.
template <typename T>
static void run(const T* img, int N, int irad2, uint16_t* out, T* part, T* range, hipStream_t s)
{
    const long long n = (long long)N * N;
    // eight 16-byte loads per thread, two workgroups per CU at most
    const int nparts = (int)std::min<long long>(kOutputParts, (n + 8191) / 8192);
    T* pmin = part;
    T* pmax = part + kOutputParts;
    const int vec = N % 4 == 0 && ((uintptr_t)img & 15) == 0 && ((uintptr_t)out & 7) == 0;
    const long long groups = ((long long)N * ((N + 3) / 4) + 255) / 256;
    hipLaunchKernelGGL(minmax_kernel<T>, dim3(nparts), dim3(256), 0, s, img, n, pmin, pmax);
    hipLaunchKernelGGL(normalise_kernel<T>, dim3((unsigned)std::min<long long>(groups, 2048)), dim3(256), 0, s, img,
                       N, irad2, (const T*)pmin, (const T*)pmax, nparts, range, out, vec);
}

void launch_output_stage_parts(const void* img, int is_float, int N, int irad2, uint16_t* out, void* part,
                               void* range, hipStream_t s)
{
    if (is_float)
        run<float>((const float*)img, N, irad2, out, (float*)part, (float*)range, s);
    else
        run<int>((const int*)img, N, irad2, out, (int*)part, (int*)range, s);
}

}  // namespace rv

// ------------------------------------------------ allocation-free output stage
// The partial minima and maxima of RecviewOutputStageNoAlloc live in this
// array: 512 + 512 four-byte values (4 KiB) on every GPU the library runs on,
// held until the process ends.  The partials are capped at 512 whatever the
// image side, so the array serves every image the entry point accepts.  Host
// code never passes the array's name to a kernel: it passes the device address
// hipGetSymbolAddress returns for the current device, kept per device.
static __device__ __align__(256) unsigned int scratch[2 * rv::kOutputParts];

namespace {

std::mutex g_scratch_mu;
std::map<int, void*> g_scratch_ptr;

// The device address of `scratch` on the current device (looked up on the first
// call on that device), or nullptr with the message set.
void* scratch_on_current_device()
{
    int dev = 0;
    if (!rv::hip_ok(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch_ptr.find(dev);
    if (it != g_scratch_ptr.end()) return it->second;
    void* ptr = nullptr;
    if (!rv::hip_ok(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)"))
        return nullptr;
    g_scratch_ptr[dev] = ptr;
    return ptr;
}

}  // namespace

extern "C" int RecviewOutputStageNoAlloc(const void* d_img, int is_float, int N, double center,
                                         int iInterpolation, unsigned short* d_out, void* d_range,
                                         rv_stream_t stream)
{
    if (!d_img || !d_out || !d_range || N <= 0 || iInterpolation < 0 || iInterpolation > 5) {
        rv::set_message("RecviewOutputStageNoAlloc: bad arguments");
        return -1;
    }
    if (N > RV_OUTPUT_NOALLOC_MAX_SIDE) {
        rv::set_message("RecviewOutputStageNoAlloc: image side N exceeds 65536");
        return -1;
    }
    void* part = scratch_on_current_device();
    if (!part) return -1;
    // every partial the second launch reads is written by the first, so nothing needs
    // clearing
    rv::launch_output_stage_parts(d_img, is_float, N, rv::output_irad2(N, center, iInterpolation), d_out,
                                  part, d_range, (hipStream_t)stream);
    return rv::hip_ok(hipGetLastError(), "output stage") ? 0 : -1;
}
