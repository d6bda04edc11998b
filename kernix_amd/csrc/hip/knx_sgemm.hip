// knx_sgemm.hip — fp32 GEMM with fused epilogue on v_mfma_f32_32x32x2_f32 (gfx950), one whole-GPU tiling.
//
// Replaces the reference's row split of one GEMM between MPS (GPU) and cblas_sgemm (AMX) with its separate bias/act
// pass (reference src/kernix_metal.m:161-265, include/kernix.h:951-977, include/kernix_model.h:528-550):
// every output tile is computed by one workgroup and leaves the chip already biased and activated.
//
// GEMMs with both operands K-contiguous (A M×K, Bt N×K: the device layout of Linear and attention weights) run on the
// bf16 matrix cores at fp32 accuracy (knx_xgemm.hip); here are their dispatch and three kernels:
//   sgemm_skinny  few output tiles (a small batch through a Linear): 16×16 tiles, K split over the waves;
//   sgemm_k32   at most one 64×64 tile per CU, K % 32 == 0: 128-byte k-tiles moved HBM → LDS by global_load_lds;
//   sgemm_tile  the general kernel (any shape, B K×N or N×K): BM×BN per workgroup of WM×WN waves, K streamed in
//               16-float k-tiles through double-buffered LDS, both tiles stored k-major (As[k][m], Bs[k][n]) so each
//               MFMA operand read is 32 consecutive floats per half-wave.  An optional batch index (grid.y) with
//               two-level strides serves the per-(batch, head) attention GEMMs.
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "knx_xgemm.hpp"

typedef float v16f __attribute__((ext_vector_type(16)));

namespace {

using SgArgs = knx_xargs;

constexpr int BK = 16;

template <int BM, int BN, int WM, int WN, bool TB>
__global__ void __launch_bounds__(WM * WN * 64) sgemm_tile(SgArgs p)
{
    constexpr int NT = WM * WN * 64;
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int FM = TM / 32, FN = TN / 32;
    constexpr int SA = BM + 4, SB = BN + 4;  // LDS row strides (floats)
    constexpr int LA = BM * BK / 4 / NT;     // float4 loads per thread (A)
    constexpr int LB = BN * BK / 4 / NT;     // float4 loads per thread (B)
    static_assert(BM * BK / 4 % NT == 0 && BN * BK / 4 % NT == 0, "load split");
    __shared__ __attribute__((aligned(16))) float As[2][BK * SA];
    __shared__ __attribute__((aligned(16))) float Bs[2][BK * SB];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int tm = blockIdx.x / p.tiles_n, tn = blockIdx.x % p.tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    const int z = blockIdx.y, zb = z / p.zh, zi = z % p.zh;
    const float* A = p.A + zb * p.sAb + zi * p.sAh;
    const float* B = p.B + zb * p.sBb + zi * p.sBh;
    float* C = p.C + zb * p.sCb + zi * p.sCh;
    const int M = p.M, N = p.N, K = p.K;
    const bool a_vec = (p.lda & 3) == 0 && ((uintptr_t)A & 15) == 0;
    const bool b_vec = (p.ldb & 3) == 0 && ((uintptr_t)B & 15) == 0;

    float4 ra[LA], rb[LB];

    // A (and NT B): row r, k-chunk kc of 4 floats; zero outside the matrix.
    auto load_rows = [&](const float* X, int ld, bool vec, int r0, int rows, int k0, int i) -> float4 {
        const int idx = i * NT + t, r = idx >> 2, kc = (idx & 3) * 4;
        const int gr = r0 + r, gk = k0 + kc;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (gr < rows) {
            const float* src = X + (size_t)gr * ld + gk;
            if (vec && gk + 3 < K) v = *reinterpret_cast<const float4*>(src);
            else {
                if (gk + 0 < K) v.x = src[0];
                if (gk + 1 < K) v.y = src[1];
                if (gk + 2 < K) v.z = src[2];
                if (gk + 3 < K) v.w = src[3];
            }
        }
        return v;
    };
    // NN B: k row, n-chunk of 4 floats.
    auto load_b_nn = [&](int k0, int i) -> float4 {
        const int idx = i * NT + t, k = idx / (BN / 4), nc = (idx % (BN / 4)) * 4;
        const int gk = k0 + k, gn = n0 + nc;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (gk < K) {
            const float* src = B + (size_t)gk * p.ldb + gn;
            if (b_vec && gn + 3 < N) v = *reinterpret_cast<const float4*>(src);
            else {
                if (gn + 0 < N) v.x = src[0];
                if (gn + 1 < N) v.y = src[1];
                if (gn + 2 < N) v.z = src[2];
                if (gn + 3 < N) v.w = src[3];
            }
        }
        return v;
    };
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < LA; ++i) ra[i] = load_rows(A, p.lda, a_vec, m0, M, k0, i);
#pragma unroll
        for (int i = 0; i < LB; ++i) rb[i] = TB ? load_rows(B, p.ldb, b_vec, n0, N, k0, i) : load_b_nn(k0, i);
    };
    auto swrite = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int idx = i * NT + t, r = idx >> 2, kc = (idx & 3) * 4;
            float* d = &As[buf][kc * SA + r];
            d[0] = ra[i].x; d[SA] = ra[i].y; d[2 * SA] = ra[i].z; d[3 * SA] = ra[i].w;
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            if (TB) {
                const int idx = i * NT + t, r = idx >> 2, kc = (idx & 3) * 4;
                float* d = &Bs[buf][kc * SB + r];
                d[0] = rb[i].x; d[SB] = rb[i].y; d[2 * SB] = rb[i].z; d[3 * SB] = rb[i].w;
            } else {
                const int idx = i * NT + t, k = idx / (BN / 4), nc = (idx % (BN / 4)) * 4;
                *reinterpret_cast<float4*>(&Bs[buf][k * SB + nc]) = rb[i];
            }
        }
    };

    v16f acc[FM][FN];
#pragma unroll
    for (int fi = 0; fi < FM; ++fi)
#pragma unroll
        for (int fj = 0; fj < FN; ++fj)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[fi][fj][e] = 0.0f;

    const int rl = lane & 31, g = lane >> 5;
    const int nk = (K + BK - 1) / BK;
    if (nk > 0) {
        gload(0);
        swrite(0);
        __syncthreads();
    }
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        const bool more = kt + 1 < nk;
        if (more) gload((kt + 1) * BK);
#pragma unroll
        for (int s = 0; s < BK / 2; ++s) {
            float af[FM], bf[FN];
            const int kk = 2 * s + g;
#pragma unroll
            for (int fi = 0; fi < FM; ++fi) af[fi] = As[cur][kk * SA + wm * TM + fi * 32 + rl];
#pragma unroll
            for (int fj = 0; fj < FN; ++fj) bf[fj] = Bs[cur][kk * SB + wn * TN + fj * 32 + rl];
#pragma unroll
            for (int fi = 0; fi < FM; ++fi)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj)
                    acc[fi][fj] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[fi], bf[fj], acc[fi][fj], 0, 0, 0);
        }
        if (more) swrite(cur ^ 1);
        __syncthreads();
    }

    // epilogue: lane holds column (lane & 31), rows 8·(e/4) + 4·(lane/32) + e%4 of each 32×32 block
#pragma unroll
    for (int fj = 0; fj < FN; ++fj) {
        const int n = n0 + wn * TN + fj * 32 + rl;
        if (n >= N) continue;
        const float bn = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm * TM + fi * 32 + 8 * (e >> 2) + 4 * g + (e & 3);
                if (m >= M) continue;
                float v = acc[fi][fj][e];
                if (p.alpha != 1.0f) v = p.alpha * v;
                if (p.bias) v = v + bn;
                if (p.causal && n > m) v = -INFINITY;
                float o = knx_act(v, p.act, p.act_alpha);
                if (p.R) o = o + p.R[(size_t)m * p.ldr + n];
                C[(size_t)m * p.ldc + n] = o;
            }
    }
}

template <int BM, int BN, int WM, int WN, bool TB>
int launch(SgArgs p, int batch, hipStream_t s, const char* name)
{
    p.tiles_n = (p.N + BN - 1) / BN;
    const unsigned tiles = (unsigned)((p.M + BM - 1) / BM) * (unsigned)p.tiles_n;
    hipLaunchKernelGGL((sgemm_tile<BM, BN, WM, WN, TB>), dim3(tiles, batch), dim3(WM * WN * 64), 0, s, p);
    return knx::check_launch(name);
}

template <bool TB>
int dispatch(SgArgs p, int batch, hipStream_t s, const char* name)
{
    const long big = (long)((p.M + 127) / 128) * ((p.N + 127) / 128) * batch;
    if (big >= knx::num_cus()) {
        if (p.N <= 64) return launch<128, 64, 2, 2, TB>(p, batch, s, name);
        return launch<128, 128, 2, 2, TB>(p, batch, s, name);
    }
    return launch<64, 64, 2, 2, TB>(p, batch, s, name);
}

// ---------------------------------------------------------------- pipelined fp32 GEMM, K-contiguous operands
// C = act(alpha·A·Btᵀ + bias) with A M×K and Bt N×K row-major, K % 32 == 0: the int8 128-byte k-tile pipeline applied
// to fp32.  Each 128-byte k-tile (32 floats) of every operand row moves HBM → LDS with global_load_lds_dwordx4 into
// one of two stages, 16-byte chunks swizzled per row (chunk c of row r at c ^ swz8(r)).  K order inside a k-tile:
// lanes 0-31 take floats 0-15 and lanes 32-63 floats 16-31, one per v_mfma_f32_32x32x2_f32 k-step, so a lane reads
// its 16 operand values of a k-tile as four 16-byte chunks ("quads" of four k-steps).  Tiles that would cross M or N
// are moved back inside and store only what they own.
template <int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64) sgemm_k32(SgArgs p)
{
    constexpr int NW = WM * WN;
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int FM = TM / 32, FN = TN / 32;
    constexpr int ROWS = BM + BN;
    constexpr int STAGE = ROWS * 128;
    constexpr int SLOTS = ROWS / 8 / NW;
    constexpr int SA = BM / 8 / NW;
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "load split");
    static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tile");
    static_assert(NW * 16 * (TN + 4) * 4 <= 2 * STAGE, "staging fits in the stages");
    __shared__ __attribute__((aligned(16))) int8_t lds[2 * STAGE];

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    const int mlo = tm * BM, nlo = tn * BN;
    const int m0 = min(mlo, p.M - BM), n0 = min(nlo, p.N - BN);
    const float* bias = p.bias;
    const float* R = p.R;  // batch 1 only (no batch offset)
    const int z = blockIdx.y, zb = z / p.zh, zi = z % p.zh;
    const float* A = p.A + zb * p.sAb + zi * p.sAh;
    const float* B = p.B + zb * p.sBb + zi * p.sBh;
    float* C = p.C + zb * p.sCb + zi * p.sCh;

    const int8_t* tile_a = reinterpret_cast<const int8_t*>(A + (size_t)m0 * p.lda);
    const int8_t* tile_b = reinterpret_cast<const int8_t*>(B + (size_t)n0 * p.ldb);
    const int lda4 = p.lda * 4, ldb4 = p.ldb * 4;  // row strides in bytes
    const int cl = (lane & 7) ^ (lane >> 3), rs = lane >> 3;
    const int nk = p.K / 32;
    auto issue1 = [&](int kt, int i) {
        const int slot = i * NW + wave;
        const bool a = i < SA;
        const int chunk = cl ^ (slot & 7);
        int8_t* dst = lds + (kt & 1) * STAGE + slot * 1024;
        const int ld = a ? lda4 : ldb4;
        const int8_t* base = (a ? tile_a + (size_t)(slot * 8) * ld : tile_b + (size_t)(slot * 8 - BM) * ld) + kt * 128;
        dma16(base, (unsigned)(rs * ld + chunk * 16), dst);
    };

    // fragment offsets: row r + 32·f has swizzle swz8(r) ^ 4·(f & 1), i.e. the chunk of half-wave g ^ (f & 1)
    const int rl = lane & 31, g = lane >> 5;
    int aoff[2][4], boff[2][4];
    {
        const int ra = wm * TM + rl, rb = BM + wn * TN + rl;
        const int sa_ = swz8(ra), sb_ = swz8(rb);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                aoff[h][c] = ra * 128 + (((4 * (g ^ h) + c) ^ sa_) << 4);
                boff[h][c] = rb * 128 + (((4 * (g ^ h) + c) ^ sb_) << 4);
            }
    }
    float4 fa[2][FM], fb[2][FN];
    auto read1 = [&](int kt, int q, int j) {  // fragment j (A if j < FM) of quad q
        const int8_t* cur = lds + (kt & 1) * STAGE;
        if (j < FM) fa[q & 1][j] = *(const float4*)(cur + aoff[j & 1][q] + j * 4096);
        else fb[q & 1][j - FM] = *(const float4*)(cur + boff[(j - FM) & 1][q] + (j - FM) * 4096);
    };
    v16f acc[FM][FN];
#pragma unroll
    for (int fi = 0; fi < FM; ++fi)
#pragma unroll
        for (int fj = 0; fj < FN; ++fj)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[fi][fj][e] = 0.0f;
    auto mfma1 = [&](int q, int j) {  // multiply j of quad q: k-step j / (FM·FN), block j % (FM·FN)
        const int s = j / (FM * FN), b = j % (FM * FN), fi = b / FN, fj = b % FN;
        acc[fi][fj] = __builtin_amdgcn_mfma_f32_32x32x2f32((&fa[q & 1][fi].x)[s], (&fb[q & 1][fj].x)[s], acc[fi][fj], 0, 0, 0);
    };

    // One k-tile, as in the int8 kernel with quads in place of k-steps: quads 0..2 multiply set q & 1 while the
    // fragments of quad q+1 are read; before quad 3's remaining multiplies the wave waits for its loads of tile kt+1
    // and its own LDS reads, then the barrier hands stage kt % 2 over to the loads of tile kt+2.
    constexpr int NM = 4 * FM * FN, NR = FM + FN, PRE = NM / 4;
    constexpr int GAPS = NM - PRE;
    auto ktile = [&](int kt, auto ARRIVE, auto ISSUE) {
        constexpr bool arrive = decltype(ARRIVE)::value, iss = decltype(ISSUE)::value;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
            for (int j = 0; j < NR; ++j) read1(kt, q + 1, j);
#pragma unroll
            for (int j = 0; j < NM; ++j) mfma1(q, j);
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, NM - NR, 0);
        }
        if (!arrive) {
#pragma unroll
            for (int j = 0; j < NM; ++j) mfma1(3, j);
            return;
        }
#pragma unroll
        for (int j = 0; j < PRE; ++j) mfma1(3, j);
        __builtin_amdgcn_sched_barrier(0);
        KNX_WAIT_VM_LDS(0);
        knx_barrier_nofence();
        int r = 0, l = 0;
#pragma unroll
        for (int j = PRE; j < NM; ++j) {
            mfma1(3, j);
            const int rupto = (NR * (j - PRE + 1) + GAPS - 1) / GAPS;
            while (r < rupto) read1(kt + 1, 0, r++);
            if (iss) {
                const int upto = (SLOTS * (j - PRE + 1) + GAPS - 1) / GAPS;
                while (l < upto) issue1(kt + 2, l++);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) issue1(0, i);
    int kt = 0;
    KNX_WAIT_VM_LDS(0);
    knx_barrier_nofence();
    if (nk > 1) {
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) issue1(1, i);
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) read1(0, 0, j);
    for (; kt < nk - 2; ++kt) ktile(kt, yes{}, yes{});
    if (nk >= 2) ktile(kt++, yes{}, no{});
    ktile(kt, no{}, no{});

    // Epilogue: each wave stages 16 rows × TN of its accumulators at a time in its own LDS region (row stride TN+4),
    // then every lane writes 4 consecutive columns of a row with one 16-byte store.
    constexpr int SROW = TN + 4, LPR = TN / 4, RPI = 64 / LPR;
    float* stg = reinterpret_cast<float*>(lds) + wave * 16 * SROW;
    // lanes from LPR·RPI on (when LPR does not divide 64) would repeat rows of other lanes: they store nothing, so with
    // R aliasing C no lane reads a residual element that another lane has already overwritten
    const int cq = (lane % LPR) * 4, rq = lane < LPR * RPI ? lane / LPR : 16;
    const int nb = n0 + wn * TN + cq;
    float bv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bv[q] = bias ? bias[nb + q] : 0.0f;
    const bool vec = nb >= nlo && (p.ldc & 3) == 0 && ((uintptr_t)C & 15) == 0;
    const bool rvec = nb >= nlo && (nb & 3) == 0 && (p.ldr & 3) == 0 && ((uintptr_t)R & 15) == 0;
    const bool relu = p.act == 0;
    const bool fast_res = R && p.alpha == 1.0f && !p.causal && (p.act == -1 || relu);
    static_assert(16 % RPI == 0, "rows per store instruction");
    KNX_WAIT_LDS();
    knx_barrier_nofence();  // nobody reads the operand stages any more
#pragma unroll
    for (int fi = 0; fi < FM; ++fi) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                for (int e = 8 * h; e < 8 * h + 8; ++e)
                    stg[(8 * ((e >> 2) - 2 * h) + 4 * g + (e & 3)) * SROW + fj * 32 + rl] = acc[fi][fj][e];
            KNX_WAIT_LDS();
            asm volatile("" ::: "memory");
            const int mt0 = m0 + wm * TM + fi * 32 + 16 * h;
            if (fast_res) {
                // Residual with no activation or ReLU: the round's residual rows are loaded before any store (R and C
                // may alias, and a load after a store waits for it: one memory round trip per row).  Loading first is
                // right when R is C, since each element is read before its own store and no other store touches it.
                // Unrolled, so the loads sit in registers; the per-row code is a few instructions.
                constexpr int NJ = (16 + RPI - 1) / RPI;
                float4 rres[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int rr = rq + j * RPI, m = mt0 + rr;
                    rres[j] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (rr >= 16 || m < mlo) continue;
                    const float* rp = R + (size_t)m * p.ldr + nb;
                    if (rvec) {
                        rres[j] = *reinterpret_cast<const float4*>(rp);
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (nb + q >= nlo) (&rres[j].x)[q] = rp[q];
                    }
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int rr = rq + j * RPI;  // idle lanes have rq = 16
                    if (rr >= 16) break;
                    const int m = mt0 + rr;
                    if (m < mlo) continue;
                    const float4 a = *reinterpret_cast<const float4*>(&stg[rr * SROW + cq]);
                    float r[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float v = (&a.x)[q];
                        if (bias) v = v + bv[q];
                        if (relu) v = v >= 0.0f ? v : 0.0f;  // the ReLU of knx_act (NaN → 0)
                        r[q] = v + (&rres[j].x)[q];
                    }
                    float* y = C + (size_t)m * p.ldc + nb;
                    if (vec) {
                        *reinterpret_cast<float4*>(y) = make_float4(r[0], r[1], r[2], r[3]);
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (nb + q >= nlo) y[q] = r[q];
                    }
                }
            } else {
                // General epilogue: one row per iteration, a rolled loop; GELU, ReLU and no activation are
                // compile-time cases (an activation switch per element costs as much as GELU itself), any other
                // activation goes through the switch
                auto rows = [&](auto actc) {
                    constexpr int ACT = decltype(actc)::value;
                    for (int rr = rq; rr < 16; rr += RPI) {
                        const int m = mt0 + rr;
                        if (m < mlo) continue;
                        const float4 a = *reinterpret_cast<const float4*>(&stg[rr * SROW + cq]);
                        float r[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            float v = (&a.x)[q];
                            if (p.alpha != 1.0f) v = p.alpha * v;
                            if (bias) v = v + bv[q];
                            if (p.causal && nb + q > m) v = -INFINITY;
                            r[q] = ACT == 1 ? knx_gelu(v) : ACT == 0 ? (v >= 0.0f ? v : 0.0f) : ACT == -1 ? v
                                                                        : knx_act(v, p.act, p.act_alpha);
                        }
                        float* y = C + (size_t)m * p.ldc + nb;
                        if (R) {  // residual after the activation; each element is read before its own store
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                if (nb + q >= nlo) r[q] = r[q] + R[(size_t)m * p.ldr + nb + q];
                        }
                        if (vec) {
                            *reinterpret_cast<float4*>(y) = make_float4(r[0], r[1], r[2], r[3]);
                        } else {
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                if (nb + q >= nlo) y[q] = r[q];
                        }
                    }
                };
                if (p.act == 1) rows(std::integral_constant<int, 1>{});
                else if (p.act == 0) rows(std::integral_constant<int, 0>{});
                else if (p.act == -1) rows(std::integral_constant<int, -1>{});
                else rows(std::integral_constant<int, -2>{});
            }
            asm volatile("" ::: "memory");
        }
    }
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float4 load4(const float* p)
{
    const v4fu v = *reinterpret_cast<const v4fu*>(p);
    return make_float4(v.x, v.y, v.z, v.w);
}

// Small NT GEMMs (a few dozen 64×64 tiles at most, e.g. a batch of 64 rows through a Linear layer): a 16×16 output
// tile per block so that the grid still spreads over the chip, K split over the 4 waves (wave w takes the 16-wide
// k-chunks w, w + 4, …), the partial sums added in wave order through LDS.  Both operands are K-contiguous and read
// straight from global memory as 16-byte vectors (at any float address; the tail K % 16 element by element); 16×16×4 fp32
// MFMA.
__global__ void __launch_bounds__(256) sgemm_skinny(SgArgs p)
{
    __shared__ float part[4][64 * 4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
    const float* a = p.A + (size_t)min(m0 + r, p.M - 1) * p.lda + 4 * kq;
    const float* b = p.B + (size_t)min(n0 + r, p.N - 1) * p.ldb + 4 * kq;
    // step c of a chunk: half-row kq of the lanes contracts over k = 16·chunk + 4·kq + c, for A and B alike
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int nk = p.K / 16;
    int kc = wave;
    for (; kc + 12 < nk; kc += 16) {  // four chunks in flight
        float4 x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = load4(a + 16 * (kc + 4 * u));
            y[u] = load4(b + 16 * (kc + 4 * u));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x4f32((&x[u].x)[c], (&y[u].x)[c], acc, 0, 0, 0);
    }
    for (; kc < nk; kc += 4) {
        const float4 x = load4(a + 16 * kc);
        const float4 y = load4(b + 16 * kc);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x4f32((&x.x)[c], (&y.x)[c], acc, 0, 0, 0);
    }
    if (p.K % 16 != 0 && wave == nk % 4) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = 16 * nk + 4 * kq + c;  // relative to the row starts below
            const bool in = k < p.K;
            const float xa = in ? a[16 * nk + c] : 0.0f, yb = in ? b[16 * nk + c] : 0.0f;
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, yb, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][lane * 4 + e] = acc[e];
    __syncthreads();
    if (wave != 0) return;
    // element e of a lane is row 4·kq + e, column r of the tile
    const int n = n0 + r;
    if (n >= p.N) return;
    const float bv = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int m = m0 + 4 * kq + e;
        if (m >= p.M) break;
        float v = ((part[0][lane * 4 + e] + part[1][lane * 4 + e]) + part[2][lane * 4 + e]) + part[3][lane * 4 + e];
        if (p.alpha != 1.0f) v = p.alpha * v;
        if (p.bias) v = v + bv;
        if (p.causal && n > m) v = -INFINITY;
        float o = knx_act(v, p.act, p.act_alpha);
        if (p.R) o = o + p.R[(size_t)m * p.ldr + n];
        p.C[(size_t)m * p.ldc + n] = o;
    }
}

bool skinny_ok(const SgArgs& p, int batch)
{
    return batch == 1 && p.K >= 16 && (p.N + 15) / 16 <= 0x7fffffff && (p.M + 15) / 16 <= 65535;
}

int launch_skinny(SgArgs p, hipStream_t s, const char* name)
{
    hipLaunchKernelGGL(sgemm_skinny, dim3((p.N + 15) / 16, (p.M + 15) / 16), dim3(256), 0, s, p);
    return knx::check_launch(name);
}

// the pipelined fp32 kernel's 64×64 tiles: K % 32 == 0, 16-byte aligned rows and whole tiles inside M and N
bool k32_ok(const SgArgs& p)
{
    // batch offsets keep every operand base 16-byte aligned
    const bool strides = ((p.sAb | p.sAh | p.sBb | p.sBh) & 3) == 0;
    return p.K > 0 && p.K % 32 == 0 && p.M >= 64 && p.N >= 64 && (p.lda & 3) == 0 && (p.ldb & 3) == 0 && strides &&
           ((uintptr_t)p.A & 15) == 0 && ((uintptr_t)p.B & 15) == 0 && (long)8 * p.lda * 4 < 0x7fffffffL &&
           (long)8 * p.ldb * 4 < 0x7fffffffL;
}

int launch_k32(SgArgs p, int batch, hipStream_t s, const char* name)
{
    p.tiles_m = (p.M + 63) / 64;
    p.tiles_n = (p.N + 63) / 64;
    hipLaunchKernelGGL((sgemm_k32<64, 64, 2, 2>), dim3((unsigned)p.tiles_m * (unsigned)p.tiles_n, batch), dim3(256), 0, s, p);
    return knx::check_launch(name);
}

// NT dispatch: few tiles → the small-GEMM kernel, else the bf16 matrix cores (knx_xgemm.hip), else (K < 16, rows of
// 32 MB) the general kernel
int dispatch_nt(SgArgs p, int batch, hipStream_t s, const char* name)
{
    // KNX_SGEMM_KERNEL forces the general kernel ("general"), the small-GEMM kernel ("skinny") or one tile of the bf16
    // kernel ("t256", "t128", "t128w8", "t64", "t64x64") or the pipelined fp32 kernel ("k32") where the shape allows it, else the general kernel (tests, tuning)
    const char* force = getenv("KNX_SGEMM_KERNEL");
    if (force != nullptr && *force) {
        static const struct { const char* name; int tile; } TILES[] = {
            {"t256", KNX_X256x256}, {"t128", KNX_X256x128}, {"t128w8", KNX_X128x128}, {"t64", KNX_X128x64}, {"t64x64", KNX_X64x64}, {"t64x64k2", KNX_X64x64K2}};
        for (const auto& t : TILES)
            if (strcmp(force, t.name) == 0) {
                const int rc = knx_xgemm(p, batch, t.tile, s, name);
                if (rc != 1) return rc;
            }
        if (strcmp(force, "k32") == 0 && k32_ok(p)) return launch_k32(p, batch, s, name);
        if (strcmp(force, "skinny") == 0 && skinny_ok(p, batch)) return launch_skinny(p, s, name);
        return dispatch<true>(p, batch, s, name);
    }
    // 16×16 tiles with split K where they are estimated to be the faster: bound by a wave's loads up to about a tile per
    // CU (K 0.0022 µs), by the operands each tile reads again beyond (17×1633×2269: 11 µs, against 45 on the bf16
    // kernel's 64×64 tiles and 98 on the general kernel; 2101×93×781 13 against 20; 500×1000×2000 49 against 41)
    // (up to 4.6 tiles per CU it is the faster at every K, without asking)
    const float rounds = (float)((p.M + 15) / 16) * (float)((p.N + 15) / 16) / (float)knx::num_cus();
    if (rounds < 64.0f && skinny_ok(p, batch) &&
        (rounds < 4.6f || 6.0f + (float)p.K * 0.0028f * rounds < knx_xgemm_us(p, batch)))
        return launch_skinny(p, s, name);
    // at most one 64×64 tile per CU: the split and the LDS traffic of the bf16 kernel are not hidden by other workgroups
    // (280×1536×512: 12.7 µs here, 14.6 there; 2048×512×512 13.6 / 15.2; 2048×256×1024 21.4 / 23.9; with two tiles per
    // CU, 4096×512×512, 23.7 / 21.1)
    if ((long)((p.M + 63) / 64) * ((p.N + 63) / 64) * batch <= knx::num_cus() && k32_ok(p)) return launch_k32(p, batch, s, name);
    const int rc = knx_xgemm(p, batch, 0, s, name);
    return rc != 1 ? rc : dispatch<true>(p, batch, s, name);
}

}  // namespace

extern "C" int knx_hip_sgemm_ep(int M, int N, int K, const float* A, int lda, const float* W, int ldw, const float* bias,
                                int act, float alpha, float* C, int ldc, void* stream)
{
    const char* name = "knx_hip_sgemm_ep";
    KNX_ENTRY(name);
    KNX_REQUIRE(M >= 0 && N >= 0 && K >= 0 && act >= -1 && act <= 15, name);
    if (M == 0 || N == 0) return KNX_OK;
    KNX_REQUIRE(C != nullptr && ldc >= N, name);
    KNX_REQUIRE(K == 0 || (A != nullptr && W != nullptr && lda >= K && ldw >= N), name);
    SgArgs p{};
    p.M = M; p.N = N; p.K = K; p.A = A; p.lda = lda; p.B = W; p.ldb = ldw; p.C = C; p.ldc = ldc;
    p.bias = bias; p.act = act; p.act_alpha = alpha; p.alpha = 1.0f; p.causal = 0; p.zh = 1;
    return dispatch<false>(p, 1, knx::as_stream(stream), name);
}

extern "C" int knx_hip_sgemm_nt_ep(int M, int N, int K, const float* A, int lda, const float* Wt, int ldwt,
                                   const float* bias, int act, float alpha, float* C, int ldc, void* stream)
{
    const char* name = "knx_hip_sgemm_nt_ep";
    KNX_ENTRY(name);
    KNX_REQUIRE(M >= 0 && N >= 0 && K >= 0 && act >= -1 && act <= 15, name);
    if (M == 0 || N == 0) return KNX_OK;
    KNX_REQUIRE(C != nullptr && ldc >= N, name);
    KNX_REQUIRE(K == 0 || (A != nullptr && Wt != nullptr && lda >= K && ldwt >= K), name);
    SgArgs p{};
    p.M = M; p.N = N; p.K = K; p.A = A; p.lda = lda; p.B = Wt; p.ldb = ldwt; p.C = C; p.ldc = ldc;
    p.bias = bias; p.act = act; p.act_alpha = alpha; p.alpha = 1.0f; p.causal = 0; p.zh = 1;
    return dispatch_nt(p, 1, knx::as_stream(stream), name);
}

extern "C" int knx_hip_sgemm_nt_ep_res(int M, int N, int K, const float* A, int lda, const float* Wt, int ldwt,
                                       const float* bias, int act, float alpha, const float* R, int ldr, float* C, int ldc,
                                       void* stream)
{
    const char* name = "knx_hip_sgemm_nt_ep_res";
    KNX_ENTRY(name);
    KNX_REQUIRE(M >= 0 && N >= 0 && K >= 0 && act >= -1 && act <= 15, name);
    if (M == 0 || N == 0) return KNX_OK;
    KNX_REQUIRE(C != nullptr && ldc >= N && R != nullptr && ldr >= N, name);
    KNX_REQUIRE(K == 0 || (A != nullptr && Wt != nullptr && lda >= K && ldwt >= K), name);
    SgArgs p{};
    p.M = M; p.N = N; p.K = K; p.A = A; p.lda = lda; p.B = Wt; p.ldb = ldwt; p.C = C; p.ldc = ldc;
    p.bias = bias; p.act = act; p.act_alpha = alpha; p.alpha = 1.0f; p.causal = 0; p.zh = 1;
    p.R = R; p.ldr = ldr;
    return dispatch_nt(p, 1, knx::as_stream(stream), name);
}

// Batched GEMM used by the attention core (internal to this library, declared in knx_attn.hip).
int knx_sgemm_batched(int M, int N, int K, const float* A, int lda, long long sAb, long long sAh, const float* B, int ldb,
                      long long sBb, long long sBh, bool transB, float* C, int ldc, long long sCb, long long sCh, int nb,
                      int nh, float alpha, int causal, hipStream_t s)
{
    const char* name = "knx_sgemm_batched";
    SgArgs p{};
    p.M = M; p.N = N; p.K = K; p.A = A; p.lda = lda; p.B = B; p.ldb = ldb; p.C = C; p.ldc = ldc;
    p.bias = nullptr; p.act = -1; p.act_alpha = 0.0f; p.alpha = alpha; p.causal = causal; p.zh = nh;
    p.sAb = sAb; p.sAh = sAh; p.sBb = sBb; p.sBh = sBh; p.sCb = sCb; p.sCh = sCh;
    return transB ? dispatch_nt(p, nb * nh, s, name) : dispatch<false>(p, nb * nh, s, name);
}
