// knx_xgemm.hpp — the fp32 GEMM on the bf16 matrix cores (knx_xgemm.hip), internal to this library.
#pragma once

#include "knx_pipe.hpp"

// ---- an fp32 value as three bf16 values ----
typedef float knx_v2f __attribute__((ext_vector_type(2)));
typedef float knx_v4fu __attribute__((ext_vector_type(4), aligned(4)));  // 16-byte global access at any float address
typedef __bf16 knx_v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 knx_v8bf __attribute__((ext_vector_type(8)));

// two fp32 values → two bf16 (round to nearest even) in one register
static __device__ __forceinline__ unsigned knx_pk(float a, float b)
{
    const knx_v2f v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, knx_v2bf));
}
// what is left of a and b after their bf16 parts h (exact)
static __device__ __forceinline__ void knx_rest(float& a, float& b, unsigned h)
{
    a = a - __builtin_bit_cast(float, h << 16);
    b = b - __builtin_bit_cast(float, h & 0xffff0000u);
}
// four values into their three bf16 parts
static __device__ __forceinline__ void knx_split4(float4 v, uint2& h, uint2& m, uint2& l)
{
    h = make_uint2(knx_pk(v.x, v.y), knx_pk(v.z, v.w));
    knx_rest(v.x, v.y, h.x);
    knx_rest(v.z, v.w, h.y);
    m = make_uint2(knx_pk(v.x, v.y), knx_pk(v.z, v.w));
    knx_rest(v.x, v.y, m.x);
    knx_rest(v.z, v.w, m.y);
    l = make_uint2(knx_pk(v.x, v.y), knx_pk(v.z, v.w));
}

static __device__ __forceinline__ float4 knx_load4(const float* p)
{
    const knx_v4fu v = *reinterpret_cast<const knx_v4fu*>(p);
    return make_float4(v.x, v.y, v.z, v.w);
}

struct knx_xargs {
    int M, N, K;
    const float* A;  // M rows, stride lda
    int lda;
    const float* B;  // N rows, stride ldb
    int ldb;
    float* C;
    int ldc;
    const float* bias;
    int act;
    float act_alpha;
    float alpha;  // C = alpha·(A·Bᵀ) before bias
    int causal;   // C[i][j] = −inf for j > i (attention scores)
    int tiles_m, tiles_n;
    int zh;  // batch index z = zb·zh + zi
    long long sAb, sAh, sBb, sBh, sCb, sCh;
    const float* R;  // residual added after the activation (stride ldr), or null; batch 1 only
    int ldr;
    knx_conv_geom cv;  // convolutions: A rows are output pixels gathered from x
    int cgc;           // input channels per group
};

// the output tile of a workgroup; 0: picked by the shape
enum { KNX_X64x64 = 1, KNX_X64x64K2, KNX_X128x64, KNX_X256x64, KNX_X128x128, KNX_X256x128, KNX_X256x256 };

// Both return 1 without launching where the shape does not fit (the caller has a general kernel).
int knx_xgemm(const knx_xargs& p, int batch, int tile, hipStream_t s, const char* name);
// the estimated time of knx_xgemm in µs, on the tile it would pick
float knx_xgemm_us(const knx_xargs& p, int batch);
// y = act(conv(x, Wt) + bias) (+ R), Wt Co × (kh·kw·C/groups)
int knx_xconv(const knx_conv_geom* g, const float* x, const float* wt, const float* bias, int act, float alpha,
              const float* R, float* y, int tile, hipStream_t s, const char* name);
