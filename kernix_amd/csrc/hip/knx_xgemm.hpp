// knx_xgemm.hpp — the fp32 GEMM on the bf16 matrix cores (knx_xgemm.hip), internal to this library.
#pragma once

#include "knx_pipe.hpp"

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
enum { KNX_X64x64 = 1, KNX_X128x64, KNX_X256x64, KNX_X128x128, KNX_X256x128, KNX_X256x256 };

// Both return 1 without launching where the shape does not fit (the caller has a general kernel).
int knx_xgemm(const knx_xargs& p, int batch, int tile, hipStream_t s, const char* name);
// the estimated time of knx_xgemm in µs, on the tile it would pick
float knx_xgemm_us(const knx_xargs& p, int batch);
// y = act(conv(x, Wt) + bias) (+ R), Wt Co × (kh·kw·C/groups)
int knx_xconv(const knx_conv_geom* g, const float* x, const float* wt, const float* bias, int act, float alpha,
              const float* R, float* y, int tile, hipStream_t s, const char* name);
