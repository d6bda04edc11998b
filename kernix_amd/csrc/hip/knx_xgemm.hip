// knx_xgemm.hip — fp32 GEMM and convolution on the bf16 matrix cores (gfx950), at fp32 accuracy.
//
// v_mfma_f32_32x32x2_f32 tops out at 157 TFLOP/s on this chip, v_mfma_f32_32x32x16_bf16 at 16 times that.  Every fp32
// value is the exact sum of three bf16 values (x = h + m + l, each the rounding of what the ones before left: 8 + 8 + 8
// significand bits), so a product of two fp32 values is nine bf16 products, each exact in fp32.  Six of them are
// multiplied here, smallest first: l·h, h·l, m·m, m·h, h·m, h·h; the three left out (m·l, l·m, l·l) are below 2^-25 of
// the product and have either sign.  All six go into one fp32 accumulator: six roundings per 16 values of k, where the
// fp32 instruction rounds every value, so the sum is no further from the exact one.
//
// Where it differs from fp32 products, the fp32 instruction is used instead: an infinity, a NaN or an operand that
// rounds to a bf16 infinity leaves a non-finite accumulator, and a wave that finds one computes its outputs again with
// v_mfma_f32_32x32x2_f32.  (Operands below 2^-110 lose low bits of l to bf16's exponent range; the absolute error is
// then at most 2^-134 of the other operand.)
#include "knx_xgemm.hpp"

typedef float v16f __attribute__((ext_vector_type(16)));

namespace {

// up to four values at p, `left` of them inside the row
__device__ __forceinline__ float4 load4_tail(const float* p, int left)
{
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (left > 0) v.x = p[0];
    if (left > 1) v.y = p[1];
    if (left > 2) v.z = p[2];
    if (left > 3) v.w = p[3];
    return v;
}

// Where a row of A comes from: PLAIN a row of a matrix; CONV4, CONV1 an output pixel of a convolution (implicit GEMM: k
// runs over (ky, kx, channel), the im2col row is gathered and never stored), four adjacent values of k being four
// channels of one tap (CONV4, channels per group a multiple of 4) or anything (CONV1).
enum { PLAIN, CONV4, CONV1 };

__device__ __attribute__((aligned(16))) float x_zeros[4];  // what padding reads: never written

// an output pixel's window: the address of its tap (0, 0), channel 0 (an integer: it may lie outside x) and the taps that
// fall inside the image, bit ky·kw + kx
struct window {
    unsigned long long at, inside;
};
__device__ __forceinline__ window window_of(const knx_xargs& p, int m, int cbase)
{
    const knx_conv_geom& g = p.cv;
    const int ox = m % g.Wo, oy = (m / g.Wo) % g.Ho, b = m / (g.Wo * g.Ho);
    const int iy = oy * g.sh - g.pt, ix = ox * g.sw - g.pl;
    window w;
    w.at = (unsigned long long)(uintptr_t)p.A + (unsigned long long)(((((long long)b * g.H + iy) * g.W + ix) * g.C + cbase) * 4);
    w.inside = 0;
    for (int ky = 0; ky < g.kh; ++ky) {
        const int y = iy + ky * g.dh;
        if (y < 0 || y >= g.H) continue;
        for (int kx = 0; kx < g.kw; ++kx) {
            const int x = ix + kx * g.dw;
            if (x >= 0 && x < g.W) w.inside |= 1ull << (ky * g.kw + kx);
        }
    }
    return w;
}
// a gathered element's place: byte offset from the window's address, and its tap
__device__ __forceinline__ const float* tap_at(const window& w, int2 e)
{
    const unsigned long long a = w.at + (long long)e.x;
    return reinterpret_cast<const float*>((w.inside >> e.y) & 1 ? a : (unsigned long long)(uintptr_t)x_zeros);
}

// C = act(alpha·A·Bᵀ + bias) (+ R): BM×BN outputs per workgroup of WM×WN waves, K streamed 16 values at a time.  Rows of A
// and B (any K, any float alignment) are loaded four values per lane, two k-tiles ahead, split into their bf16 parts by
// the thread that loaded them (5.5 instructions per value, shared by every wave that multiplies it) and written to LDS
// as MFMA fragments: 32 rows × 16 k of one part are 1 KB in lane order (lane = row + 32·(k / 8), 16 bytes each, the
// upper half's rows at row ^ 12 so that the writes of four lanes per row spread over the banks).  Two LDS stages and
// one barrier per k-tile: while the matrix cores work on one, the next is split and written.
// What bounds it: at 4096³ and above the chip's power (1.9 GHz; 237 TFLOP/s of fp32 product are 1420 TFLOP/s of bf16,
// where a plain bf16 GEMM of torch's reaches 1150 on the same card; fp32 instructions: 147 TFLOP/s); the smaller tiles
// the split's instructions and the LDS, which overlap the multiplies only in part (128×128: 54% of the matrix cores'
// cycles).  K-tiles of 32 or 64 values per barrier, four k-tiles of loads in flight and four waves of 64×64 were slower.
// KG = 2: two groups of WM×WN waves, each with stages of its own, take alternate k-tiles of the same outputs, and the second
// hands its sums to the first through LDS at the end: for shapes that give a CU one workgroup, whose waves would wait for
// one another's LDS reads and splits alone.
template <int BM, int BN, int WM, int WN, int OCC, bool PIPE, int MODE, int KG>
__global__ void __launch_bounds__(WM * WN * 64 * KG, OCC) xgemm(knx_xargs p)
{
    constexpr int NW = WM * WN, NT = NW * 64;
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32;
    constexpr int KT = 16, Q = 4, D = 2;  // values of k per k-tile, pieces of four per row, k-tiles of loads in flight
    constexpr int STAGE = (BM + BN) / 32 * 3 * 1024;
    constexpr int P = (BM + BN) * Q / NT, PA = BM * Q / NT;  // pieces per thread and k-tile; of A
    static_assert(BM * Q % NT == 0 && BN * Q % NT == 0 && TM % 32 == 0 && TN % 32 == 0, "load split");
    static_assert(KG == 1 || (KG == 2 && PIPE), "groups of waves");
    __shared__ __attribute__((aligned(16))) int8_t lds0s[KG * STAGE];
    __shared__ __attribute__((aligned(16))) int8_t lds1s[KG * STAGE];

    const int lane = threadIdx.x & 63;
    const int all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int kg = KG == 1 ? 0 : all / NW, wave = KG == 1 ? all : all % NW, t = wave * 64 + lane;  // of this wave's group
    int8_t* const lds0 = lds0s + kg * STAGE;
    int8_t* const lds1 = lds1s + kg * STAGE;
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_of_best(blockIdx.x, p.tiles_m, p.tiles_n, BM, BN, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const float *A = p.A, *B = p.B, *bias = p.bias, *R = p.R;
    float* C = p.C;
    if (MODE == PLAIN) {
        const int z = blockIdx.y, zb = z / p.zh, zi = z % p.zh;
        A += zb * p.sAb + zi * p.sAh;
        B += zb * p.sBb + zi * p.sBh;
        C += zb * p.sCb + zi * p.sCh;
    } else {  // grid.y = group: its channels of x, its rows of Wt, its columns of y, R and the bias
        const size_t first = (size_t)blockIdx.y * p.N;
        B += first * p.ldb;
        C += first;
        if (bias) bias += first;
        if (R) R += first;
    }
    const int K = p.K;
    // convolution: where each k (CONV1) or each four (CONV4) lies in a window
    extern __shared__ __attribute__((aligned(16))) int2 taps[];
    const int cbase = MODE == PLAIN ? 0 : (int)blockIdx.y * p.cgc;
    if (MODE != PLAIN) {
        for (int i = threadIdx.x; i < (MODE == CONV4 ? K / 4 : K); i += NT * KG) {
            const int k = MODE == CONV4 ? 4 * i : i, tap = k / p.cgc, ky = tap / p.cv.kw, kx = tap - ky * p.cv.kw;
            taps[i] = make_int2((int)((((long long)ky * p.cv.dh * p.cv.W + (long long)kx * p.cv.dw) * p.cv.C + (k - tap * p.cgc)) * 4), tap);
        }
        __syncthreads();
    }

    // piece i of this thread: row (i·NT + t) / Q of the tile's A rows then B rows (rows past the matrix repeat its last
    // one: their outputs are not stored), values 4·(t mod Q) … of the k-tile
    const int q = t & (Q - 1);
    unsigned off[P];
    window win[MODE == PLAIN ? 1 : PA];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int r = (i * NT + t) / Q;
        if (MODE != PLAIN && i < PA) {
            win[i] = window_of(p, min(m0 + r, p.M - 1), cbase);
            continue;
        }
        const int row = i < PA ? min(r, p.M - 1 - m0) : min(r - BM, p.N - 1 - n0);
        off[i] = (unsigned)(row * (i < PA ? p.lda : p.ldb) + 4 * q);
    }
    const float* ta = A + (size_t)m0 * p.lda;  // (not used by convolutions)
    const float* tb = B + (size_t)n0 * p.ldb;
    unsigned woff[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int r = (i * NT + t) / Q, h = q >> 1;
        woff[i] = (r >> 5) * 3072 + h * 512 + (((r & 31) ^ (h * 12)) << 4) + (q & 1) * 8;
    }
    // k-tile 0 is the odd one of K % KT values if there is one, the rest follow in order (tiles past the last repeat it:
    // loaded and written, never multiplied)
    auto gather4 = [&](const window& w, int k) __attribute__((always_inline)) {
        if (MODE == CONV4) return knx_load4(tap_at(w, taps[k >> 2]));
        return make_float4(*tap_at(w, taps[k]), *tap_at(w, taps[k + 1]), *tap_at(w, taps[k + 2]), *tap_at(w, taps[k + 3]));
    };
    auto gather4_tail = [&](const window& w, int k, int left) __attribute__((always_inline)) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MODE == CONV4) return left > 0 ? knx_load4(tap_at(w, taps[k >> 2])) : v;
        if (left > 0) v.x = *tap_at(w, taps[k]);
        if (left > 1) v.y = *tap_at(w, taps[k + 1]);
        if (left > 2) v.z = *tap_at(w, taps[k + 2]);
        if (left > 3) v.w = *tap_at(w, taps[k + 3]);
        return v;
    };
    const int part = K % KT, nkt = (K + KT - 1) / KT, shift = part ? KT - part : 0;
    // (KG = 2: this group's k-tile kt is tile 2·kt + kg; past the last one, which the other group may still have, zeros)
    auto gload = [&](int kt, float4 (&v)[P]) __attribute__((always_inline)) {
        const int tile = kt * KG + kg, k = min(tile, nkt - 1) * KT - shift;
        if (KG > 1 && tile >= nkt) {
#pragma unroll
            for (int i = 0; i < P; ++i) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            return;
        }
#pragma unroll
        for (int i = 0; i < P; ++i) {
            if (MODE != PLAIN && i < PA) v[i] = gather4(win[i], k + 4 * q);
            else v[i] = knx_load4((i < PA ? ta : tb) + k + off[i]);
            __builtin_amdgcn_sched_barrier(0x3ff & ~0x30);  // loads stay in order
        }
    };
    auto gload_first = [&](float4 (&v)[P]) __attribute__((always_inline)) {
        if (part == 0 || kg > 0) return gload(0, v);
#pragma unroll
        for (int i = 0; i < P; ++i) {
            if (MODE != PLAIN && i < PA) v[i] = gather4_tail(win[i], 4 * q, part - 4 * q);
            else v[i] = load4_tail((i < PA ? ta : tb) + off[i], part - 4 * q);
        }
    };
    auto put = [&](int8_t* st, const float4& v, int i) __attribute__((always_inline)) {
        uint2 h, m, l;
        knx_split4(v, h, m, l);
        *reinterpret_cast<uint2*>(st + woff[i]) = h;
        *reinterpret_cast<uint2*>(st + woff[i] + 1024) = m;
        *reinterpret_cast<uint2*>(st + woff[i] + 2048) = l;
    };

    const int rl = lane & 31, g = lane >> 5;
    const unsigned roff = g * 512 + ((rl ^ (g * 12)) << 4);
    // a wave with one 32×32 block keeps two accumulators (odd and even products), so that consecutive multiplies do not
    // wait for each other
    constexpr int NA = FM * FN == 1 ? 2 : 1;
    v16f accs[NA][FM][FN];
    auto& acc = accs[0];
#pragma unroll
    for (int c = 0; c < NA; ++c)
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                for (int e = 0; e < 16; ++e) accs[c][fi][fj][e] = 0.0f;

    constexpr int SA[6] = {2, 0, 1, 1, 0, 0}, SB[6] = {0, 2, 1, 0, 1, 0};  // the parts of A and of B, smallest product first
    struct frags { knx_v8bf a[FM][3], b[FN][3]; };
    const int fa = wm * FM * 3072 + roff, fb = (BM / 32 + wn * FN) * 3072 + roff;
    auto fetch = [&](const int8_t* cur, frags& f) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 3; ++s) {
#pragma unroll
            for (int fi = 0; fi < FM; ++fi) f.a[fi][s] = *reinterpret_cast<const knx_v8bf*>(cur + fa + fi * 3072 + s * 1024);
#pragma unroll
            for (int fj = 0; fj < FN; ++fj) f.b[fj][s] = *reinterpret_cast<const knx_v8bf*>(cur + fb + fj * 3072 + s * 1024);
        }
    };
    auto mfma = [&](const knx_v8bf (&a)[3], const knx_v8bf (&b)[3], int s, int fi, int fj) __attribute__((always_inline)) {
        accs[s % NA][fi][fj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[SA[s]], b[SB[s]], accs[s % NA][fi][fj], 0, 0, 0);
    };
    // PIPE: multiply the fragments f, read from LDS a k-tile ahead; meanwhile split and write the pieces in v to `nxt`
    auto mult = [&](const frags& f, int8_t* nxt, const float4 (&v)[P]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 6; ++s) {
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                for (int fi = 0; fi < FM; ++fi) mfma(f.a[fi], f.b[fj], s, fi, fj);
#pragma unroll
            for (int i = s * P / 6; i < (s + 1) * P / 6; ++i) put(nxt, v[i], i);
        }
        constexpr int NMF = 6 * FM * FN, VPM = (22 * P + NMF - 1) / NMF, NR = 3 * (FM + FN);
#pragma unroll
        for (int j = 0; j < NMF; ++j) {  // a multiply, an LDS read, a few of the split's instructions
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (j < NR) __builtin_amdgcn_sched_group_barrier(0x100, (NR + NMF - 1) / NMF, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
        }
    };
    // otherwise (no registers for a second set of fragments): multiply the k-tile in `cur` a column of blocks at a time
    auto ktile = [&](const int8_t* cur, int8_t* nxt, const float4 (&v)[P]) __attribute__((always_inline)) {
        knx_v8bf a[FM][3];
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int s = 0; s < 3; ++s) a[fi][s] = *reinterpret_cast<const knx_v8bf*>(cur + fa + fi * 3072 + s * 1024);
#pragma unroll
        for (int fj = 0; fj < FN; ++fj) {
            knx_v8bf b[3];
#pragma unroll
            for (int s = 0; s < 3; ++s) b[s] = *reinterpret_cast<const knx_v8bf*>(cur + fb + fj * 3072 + s * 1024);
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int fi = 0; fi < FM; ++fi) mfma(a[fi], b, s, fi, fj);
#pragma unroll
            for (int i = fj * P / FN; i < (fj + 1) * P / FN; ++i) put(nxt, v[i], i);
        }
    };
    auto handover = [&]() __attribute__((always_inline)) {
        KNX_WAIT_LDS();
        knx_barrier_nofence();
    };
    auto stage = [&](int j) __attribute__((always_inline)) -> int8_t* { return j & 1 ? lds1 : lds0; };
    float4 v[D][P];
    if constexpr (PIPE) {
        frags f[2];
        float4 w0[P], w1[P];
        gload_first(w0);
        gload(1, w1);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            __builtin_amdgcn_sched_barrier(0);
            gload(2 + d, v[(2 + d) % D]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < P; ++i) put(lds0, w0[i], i);
#pragma unroll
        for (int i = 0; i < P; ++i) put(lds1, w1[i], i);
        handover();
        fetch(lds0, f[0]);
        handover();
        auto step = [&](int kt, int j) __attribute__((always_inline)) {
            fetch(stage(j + 1), f[(j + 1) & 1]);
            mult(f[j & 1], stage(j), v[(j + 2) % D]);
            gload(kt + j + 2 + D, v[(j + 2) % D]);
            handover();
        };
        const int steps = (nkt + KG - 1) / KG;
        int kt = 0;
        for (; kt + D <= steps; kt += D)
#pragma unroll
            for (int j = 0; j < D; ++j) step(kt, j);
#pragma unroll
        for (int j = 0; j < D - 1; ++j)
            if (kt + j < steps) step(kt, j);
    } else {
        float4 w0[P];
        gload_first(w0);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            __builtin_amdgcn_sched_barrier(0);
            gload(1 + d, v[(1 + d) % D]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < P; ++i) put(lds0, w0[i], i);
        handover();
        auto step = [&](int kt, int j) __attribute__((always_inline)) {
            ktile(stage(j), stage(j + 1), v[(j + 1) % D]);
            gload(kt + j + 1 + D, v[(j + 1) % D]);
            handover();
        };
        int kt = 0;
        for (; kt + D <= nkt; kt += D)
#pragma unroll
            for (int j = 0; j < D; ++j) step(kt, j);
#pragma unroll
        for (int j = 0; j < D - 1; ++j)
            if (kt + j < nkt) step(kt, j);
    }
    if (NA == 2)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[0][0][e] = acc[0][0][e] + accs[NA - 1][0][0][e];

    if (KG == 2) {  // the second group's sums to the first (every wave is past its last read of the stages)
        float* part_sums = reinterpret_cast<float*>(lds0s) + wave * FM * FN * 1024 + lane;
        static_assert(KG == 1 || NW * FM * FN * 4096 <= KG * STAGE, "the sums fit the first stages");
        if (kg == 1)
#pragma unroll
            for (int fi = 0; fi < FM; ++fi)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                    for (int e = 0; e < 16; ++e) part_sums[((fi * FN + fj) * 16 + e) * 64] = acc[fi][fj][e];
        handover();
        if (kg == 1) return;
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[fi][fj][e] = acc[fi][fj][e] + part_sums[((fi * FN + fj) * 16 + e) * 64];
    }
    // a non-finite accumulator: this wave's outputs again, in fp32 products
    float nan = 0.0f;
#pragma unroll
    for (int fi = 0; fi < FM; ++fi)
#pragma unroll
        for (int fj = 0; fj < FN; ++fj)
#pragma unroll
            for (int e = 0; e < 16; ++e) nan = __builtin_fmaf(acc[fi][fj][e], 0.0f, nan);
    if (__any(nan != 0.0f)) {
        const float* ra[FM];
        const float* rb[FN];
        window rw[FM];
#pragma unroll
        for (int fi = 0; fi < FM; ++fi) {
            const int m = min(m0 + wm * TM + fi * 32 + rl, p.M - 1);
            if (MODE == PLAIN) ra[fi] = A + (size_t)m * p.lda;
            else rw[fi] = window_of(p, m, cbase);
        }
#pragma unroll
        for (int fj = 0; fj < FN; ++fj) rb[fj] = B + (size_t)min(n0 + wn * TN + fj * 32 + rl, p.N - 1) * p.ldb;
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[fi][fj][e] = 0.0f;
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += 8) {  // step c multiplies k0 + c (lanes 0-31) and k0 + 4 + c (lanes 32-63)
            const int k = k0 + 4 * g;
            float4 xa[FM], xb[FN];
#pragma unroll
            for (int fi = 0; fi < FM; ++fi) xa[fi] = MODE == PLAIN ? load4_tail(ra[fi] + k, K - k) : gather4_tail(rw[fi], k, K - k);
#pragma unroll
            for (int fj = 0; fj < FN; ++fj) xb[fj] = load4_tail(rb[fj] + k, K - k);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int fi = 0; fi < FM; ++fi)
#pragma unroll
                    for (int fj = 0; fj < FN; ++fj)
                        acc[fi][fj] = __builtin_amdgcn_mfma_f32_32x32x2f32((&xa[fi].x)[c], (&xb[fj].x)[c], acc[fi][fj], 0, 0, 0);
        }
    }

    // Epilogue: FN × 4 accumulators of a lane per round (four rows, a column of each block; a store writes two 128-byte
    // row segments).  One copy of the code for all rounds, the round's accumulators picked by uniform branches: unrolled
    // rounds are thousands of instructions run once each, bound by instruction fetch, and rounds through LDS with
    // 16-byte stores wait for their LDS reads (15 µs for 256×256 outputs).
    const int n = n0 + wn * TN + rl;
    float bv[FN];
    bool in[FN];
#pragma unroll
    for (int fj = 0; fj < FN; ++fj) {
        in[fj] = n + 32 * fj < p.N;
        bv[fj] = bias && in[fj] ? bias[n + 32 * fj] : 0.0f;
    }
#pragma unroll 1
    for (int r = 0; r < FM * 4; ++r) {
        float y[4][FN];
#pragma unroll
        for (int rr = 0; rr < FM * 4; ++rr)
            if (r == rr)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int fj = 0; fj < FN; ++fj) y[e][fj] = acc[rr / 4][fj][4 * (rr % 4) + e];
        const int m = m0 + wm * TM + r * 8 + 4 * g;
        float* out = C + (size_t)m * p.ldc + n;
        if (p.alpha != 1.0f || p.causal)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) {
                    if (p.alpha != 1.0f) y[e][fj] = p.alpha * y[e][fj];
                    if (p.causal && n + 32 * fj > m + e) y[e][fj] = -INFINITY;
                }
        if (bias)  // (never with causal)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) y[e][fj] = y[e][fj] + bv[fj];
        float res[4][FN];
        if (R) {  // before the round's stores: R may be C
            const float* rp = R + (size_t)m * p.ldr + n;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj)
                    res[e][fj] = m + e < p.M && in[fj] ? rp[(size_t)e * p.ldr + 32 * fj] : 0.0f;
        }
        if (p.act == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) y[e][fj] = y[e][fj] >= 0.0f ? y[e][fj] : 0.0f;  // the ReLU of knx_act (NaN → 0)
        } else if (p.act == 1) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) y[e][fj] = knx_gelu(y[e][fj]);
        } else if (p.act != -1) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) y[e][fj] = knx_act(y[e][fj], p.act, p.act_alpha);
        }
        if (R)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int fj = 0; fj < FN; ++fj) y[e][fj] = y[e][fj] + res[e][fj];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (m + e >= p.M) break;
#pragma unroll
            for (int fj = 0; fj < FN; ++fj)
                if (in[fj]) out[(size_t)e * p.ldc + 32 * fj] = y[e][fj];
        }
    }
}

template <int MODE, int BM, int BN, int WM, int WN, int OCC, bool PIPE, int KG = 1>
int launch(knx_xargs p, int batch, hipStream_t s, const char* name)
{
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    const unsigned taps = MODE == PLAIN ? 0 : (unsigned)(MODE == CONV4 ? p.K / 4 : p.K) * 8;
    hipLaunchKernelGGL((xgemm<BM, BN, WM, WN, OCC, PIPE, MODE, KG>), dim3((unsigned)p.tiles_m * (unsigned)p.tiles_n, batch),
                       dim3(WM * WN * 64 * KG), taps, s, p);
    return knx::check_launch(name);
}

template <int MODE>
int launch_tile(const knx_xargs& p, int batch, int tile, hipStream_t s, const char* name)
{
    switch (tile) {
    case KNX_X256x256: if (MODE == PLAIN) return launch<PLAIN, 256, 256, 4, 2, 1, false>(p, batch, s, name); [[fallthrough]];
    case KNX_X256x128: return launch<MODE, 256, 128, 4, 2, 1, true>(p, batch, s, name);
    case KNX_X256x64: return launch<MODE, 256, 64, 4, 1, 2, true>(p, batch, s, name);
    case KNX_X128x128: return launch<MODE, 128, 128, 4, 2, 1, true>(p, batch, s, name);
    case KNX_X64x64K2: return launch<MODE, 64, 64, 2, 2, 1, true, 2>(p, batch, s, name);
    case KNX_X128x64: return launch<MODE, 128, 64, 2, 2, 2, true>(p, batch, s, name);
    default: return launch<MODE, 64, 64, 2, 2, 2, true>(p, batch, s, name);
    }
}

// The tile for a shape: the one with the least estimated time, workgroups per CU in whole rounds.  Per tile: µs for 16
// values of k where at most half of the CUs have a workgroup and where all are busy, and µs for the prologue and the
// epilogue, from 500×1000×2000, 8192×512×{512, 2048} and 4096³ on every tile (the tiles picked here: 37, 28, 88 and
// 581 µs; on v_mfma_f32_32x32x2_f32 they took 83, 40, 130 and 930 µs).  Three choices the times make: two groups of waves on
// a 64×64 tile where each CU has at most one (500×1000×2000: 36.5 against 41 µs, 74 images of 14×14×137 → 46: 34 against 49), 256×256 tiles, the
// fewest operand bytes per multiply, wherever they come in full rounds and K is long (4096³: 581 µs, against 602 on
// 256×128 and 652 on 128×128); 64×64 where larger tiles would leave CUs idle.
int pick_tile(const knx_xargs& p, int batch, bool conv, float* us)
{
    static const struct {
        int tile, bm, bn;
        float idle, busy, fixed, windows;  // windows: µs for a convolution's tap windows and table before the first load
    } T[] = {{KNX_X256x256, 256, 256, 1.58f, 2.2f, 18.0f, 0.0f},
             {KNX_X256x128, 256, 128, 0.78f, 1.15f, 10.0f, 3.5f},
             {KNX_X256x64, 256, 64, 0.78f, 0.65f, 9.0f, 4.0f},
             {KNX_X128x128, 128, 128, 0.41f, 0.63f, 8.0f, 2.0f},
             {KNX_X128x64, 128, 64, 0.37f, 0.37f, 7.5f, 5.0f},
             {KNX_X64x64K2, 64, 64, 0.23f, 0.24f, 7.5f, 1.5f},
             {KNX_X64x64, 64, 64, 0.26f, 0.21f, 7.0f, 1.5f}};
    int best = KNX_X64x64;
    *us = 0.0f;
    for (const auto& t : T) {
        if (conv && t.tile == KNX_X256x256) continue;
        const long tiles = (long)((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * batch, cus = knx::num_cus();
        const long rounds = (tiles + cus - 1) / cus;
        const float e = t.fixed + (conv ? t.windows : 0.0f) + (float)p.K / 16.0f * (2 * tiles <= cus ? t.idle : t.busy * (float)rounds);
        if (*us == 0.0f || e < *us) *us = e, best = t.tile;
    }
    return best;
}

bool fits(const knx_xargs& p)  // whole k-tiles, 32-bit offsets within a tile's rows
{
    return p.K >= 16 && (long long)p.lda * 256 <= 0x7fffffffLL && (long long)p.ldb * 256 <= 0x7fffffffLL;
}

}  // namespace

float knx_xgemm_us(const knx_xargs& p, int batch)
{
    float us;
    pick_tile(p, batch, false, &us);
    return fits(p) ? us : 1e30f;
}

int knx_xgemm(const knx_xargs& p, int batch, int tile, hipStream_t s, const char* name)
{
    if (!fits(p)) return 1;
    float us;
    return launch_tile<PLAIN>(p, batch, tile ? tile : pick_tile(p, batch, false, &us), s, name);
}

int knx_xconv(const knx_conv_geom* g, const float* x, const float* wt, const float* bias, int act, float alpha,
              const float* R, float* y, int tile, hipStream_t s, const char* name)
{
    knx_xargs p{};
    p.cgc = g->C / g->groups;
    p.M = g->B * g->Ho * g->Wo;
    p.N = g->Co / g->groups;
    p.K = g->kh * g->kw * p.cgc;
    const bool four = p.cgc % 4 == 0;
    const long long span = (((long long)(g->kh - 1) * g->dh * g->W + (long long)(g->kw - 1) * g->dw) + 1) * g->C * 4;
    // at most 64 taps (the window's mask), 32-bit offsets in a window, a table of taps that leaves room for two workgroups
    p.ldb = p.K;
    if (!fits(p) || g->kh * g->kw > 64 || span > 0x7fffffffLL || (four ? p.K / 4 : p.K) > 5120) return 1;
    p.A = x; p.B = wt; p.C = y; p.ldc = g->Co;
    p.bias = bias; p.act = act; p.act_alpha = alpha; p.alpha = 1.0f; p.zh = 1;
    p.R = R; p.ldr = g->Co;
    p.cv = *g;
    float us;
    if (!tile) tile = pick_tile(p, g->groups, true, &us);
    return four ? launch_tile<CONV4>(p, g->groups, tile, s, name) : launch_tile<CONV1>(p, g->groups, tile, s, name);
}
