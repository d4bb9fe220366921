// Back-projection kernels on the vector ALU: tile shapes and row access shared by
// rv_bp.hip (whole tiles) and rv_bpsub.hip (parts of tiles).
#ifndef RV_BP_H
#define RV_BP_H

#include "rv_internal.h"
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>

namespace rv {

// smallest integer >= sqrt(v)
constexpr int isqrt_ceil(int v)
{
    int r = 0;
    while (r * r < v) r++;
    return r;
}

template <int PX, int PY, int NW = 4>
struct TileCfg {
    static constexpr int WX = 8 * PX, WY = 8 * PY;   // wave block
    static constexpr int TW = 2 * WX, TH = (NW / 2) * WY;   // 2 x NW/2 waves
    static constexpr int T = 64 * NW;
    // detector footprint of a tile: (TW-1)|cos| + (TH-1)|sin| <= the tile diagonal D;
    // with s0 = floor(umin) - 1 every index used is <= D + 2, so SEG >= D + 3
    static constexpr int SEG = (isqrt_ceil((TW - 1) * (TW - 1) + (TH - 1) * (TH - 1)) + 7) / 4 * 4;
};

__device__ __forceinline__ float load_row_val(const void* rows, const float* scales, const BpSlice& S, int row,
                                              int k)
{
    const long long off = (long long)row * S.row_stride + k;
    if (S.store == 0) return ((const float*)rows)[off];
    const float sc = scales[row];
    if (S.store == 1) return __half2float(((const __half*)rows)[off]) * sc;
    return __bfloat162float(((const __hip_bfloat16*)rows)[off]) * sc;
}

__device__ __forceinline__ float load_row_val(const BpSlice& S, int row, int k)
{
    return load_row_val(S.rows, S.scales, S, row, k);
}

}  // namespace rv

#endif
