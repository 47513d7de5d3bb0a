// The sum of a row's partial sums (sigmoid attention's splits), for the kernels that take it.
#pragma once
#include "common.h"

// Partial sums part[row, split, dv] of `dv` numbers a row, added in ascending order: number d of row r.
__device__ __forceinline__ float merged_shares(const float* __restrict__ part, int64_t r, int d, int S, int dv) {
    const float* p = part + r * S * dv + d;
    float acc = 0.f;
    int s = 0;
    for (; s + 8 <= S; s += 8) {               // eight loads in flight, added in ascending order
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = p[(int64_t)(s + i) * dv];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc += v[i];
    }
    for (; s < S; ++s) acc += p[(int64_t)s * dv];
    return acc;
}
