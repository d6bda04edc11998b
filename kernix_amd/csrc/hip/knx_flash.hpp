// knx_flash.hpp — attention over any number of keys (knx_flash.hip), internal to this library.
#pragma once

#include "knx_xgemm.hpp"

struct knx_flash_args {
    const float* Q;
    int ldq;
    const float* K;
    int ldk;
    const float* V;
    int ldv;
    float* ctx;
    int B, H, Rq, S, d;  // d: head size of Q, K and V
    float scale;
    int causal;
    float qmul;  // set by knx_flash
};

// the sum of both half-waves' values
static __device__ __forceinline__ float knx_lane_group_sum_halves(float v)
{
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

// Returns 1 without launching where the shape does not fit (d > 128 or no multiple of 4).
int knx_flash(const knx_flash_args& p, hipStream_t s, const char* name);
