// knx_flash.hip — attention of one head at a time over any number of keys, on the bf16 matrix cores at fp32 accuracy
// (gfx950).  ctx = softmax(scale·Q·Kᵀ + causal mask)·V, the loop body of kernix_attention_run (reference
// include/kernix_model.h:1021-1046), with nothing but Q, K, V and the context in HBM.
//
// Both products split their fp32 operands into three bf16 values and sum six of the nine products in fp32, smallest
// first (knx_xgemm.hip says why that is no less exact than fp32 products); the softmax runs in fp32 with a running
// maximum, sums and products rescaled where the maximum grows.
//
// A workgroup takes 128 queries of one (batch, head), each wave 32 of them, Q split once into registers.  Keys come 32 at
// a time: K and V rows are loaded a tile ahead, split by the threads that loaded them and written to LDS as MFMA
// fragments (two stages each, V one tile behind K, one barrier per tile; V transposed in registers, 4 keys × 4 columns per
// thread).  The wave computes Sᵀ = K·Qᵀ, so that a lane holds 16 keys of one query: the row maximum and sum need one
// exchange between the half-waves, and the probabilities, split in place, are the B operand of ctxᵀ = Vᵀ·Pᵀ (the keys of a
// 16-key step in the order the accumulators hold them, V's fragments in the same order).  The scores of tile kt + 1 are
// multiplied while the softmax of tile kt runs on the vector unit.  Causal: tiles past a workgroup's last query are not
// loaded, tiles past a wave's last query not multiplied.
//
// B 4, H 12, S 1000, d 64: 87 µs causal, 92 without the mask (scores, softmax and products as three launches 257 and 262 on
// fp32 matrix instructions, 203 and 207 with the products of knx_xgemm.hip); B 2, H 8, S 2048: 113 (297).  A tile takes a
// lone workgroup 1.6 µs, 0.7 of them the matrix cores': what remains is the waves' own chain from scores to products,
// one or two waves per SIMD.  Not kept: scores and softmax one after the other (118 µs at B 4, H 12, S 1000), a separate
// last tile without the next one's scores (slower by 5-10% at S ≥ 1000).
#include "knx_flash.hpp"

typedef float v16f __attribute__((ext_vector_type(16)));

namespace {

__device__ __attribute__((aligned(16))) float flash_zeros[4];  // rows past the last key, columns past d: never written

constexpr float LOG2E = 1.44269504f;
constexpr float MASKED = -3.0e38f;  // below every score that is finite in fp32, and times anything no NaN

// D: the head size, rounded up to 32 (columns from d on count as zero)
template <int D, int OCC>
__global__ void __launch_bounds__(256, OCC) flash(knx_flash_args p, int qblocks)
{
    constexpr int NS = D / 16, ND = D / 32;  // 16-wide steps of Q·K, 32-wide blocks of the context
    constexpr int KB = NS * 3072, VB = ND * 2 * 3072, STAGE = KB + VB;  // bytes of K and V fragments
    constexpr int UNITS = 4 * D, NU = (UNITS + 255) / 256;              // 16-value load units per tile, per thread
    __shared__ __attribute__((aligned(16))) int8_t lds[2 * STAGE];

    const int t = threadIdx.x, lane = t & 63, col = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // consecutive workgroups go to consecutive XCDs: the query blocks of a head (which read the same K and V) to one of
    // them, the blocks with the most keys first
    int z = blockIdx.x / qblocks, qb = blockIdx.x % qblocks;
    if ((p.B * p.H) % 8 == 0) {
        const int j = blockIdx.x >> 3;
        z = j / qblocks * 8 + (blockIdx.x & 7);
        qb = j % qblocks;
    }
    if (p.causal) qb = qblocks - 1 - qb;
    const int b = z / p.H, h = z % p.H;
    const float* Kh = p.K + (size_t)b * p.S * p.ldk + (size_t)h * p.d;
    const float* Vh = p.V + (size_t)b * p.S * p.ldv + (size_t)h * p.d;
    const int q0 = qb * 128, qw = q0 + wave * 32, qi = qw + col;
    const float* Qr = p.Q + ((size_t)b * p.Rq + min(qi, p.Rq - 1)) * p.ldq + (size_t)h * p.d;
    const int keys = p.causal ? min(p.S, q0 + 128) : p.S, nt = (keys + 31) / 32;

    // Load unit n of this thread, u = 256·n + t: below 2D a block of V (its four rows' quads: keys 4·kq …, columns
    // 4·dq …), from there four quads of K; which of them is the same for a whole wave.  Rows past the last key repeat it
    // (their scores are masked, their probabilities 0) and columns past d the last quad (times Q's zeros, or not stored).
    float4 ld[NU][4];
    auto is_v = [&](int n) __attribute__((always_inline)) { return (n * 4 + wave) * 64 < 2 * D; };
    auto gload = [&](int kt) __attribute__((always_inline)) {  // K of tile kt, V of tile kt − 1
#pragma unroll
        for (int n = 0; n < NU; ++n) {
            const int u = n * 256 + t;
            if (NU * 256 > UNITS && (n * 4 + wave) * 64 >= UNITS) continue;
            const bool v = is_v(n);
            const float* base = v ? Vh : Kh;
            const int rs = v ? p.ldv : p.ldk, first = 32 * (v ? kt - 1 : kt);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int kv = ((u & 3) | (u >> 5 & 1) << 2) * 4 + i, cv = ((u >> 2 & 7) | u >> 6 << 3) * 4;
                const int k = i * 2 * D + (u - 2 * D), kk = k >> 2 & 31, ck = ((k >> 7) * 4 + (k & 3)) * 4;
                const int row = min(max(first + (v ? kv : kk), 0), p.S - 1), c = min(v ? cv : ck, p.d - 4);
                ld[n][i] = knx_load4(base + (size_t)row * rs + c);
            }
        }
    };
    auto put = [&](int kt) __attribute__((always_inline)) {  // what gload(kt) loaded
        int8_t* sk = lds + (kt & 1) * STAGE;
        int8_t* sv = lds + (kt + 1 & 1) * STAGE + KB;
#pragma unroll
        for (int n = 0; n < NU; ++n) {
            const int u = n * 256 + t;
            if (NU * 256 > UNITS && (n * 4 + wave) * 64 >= UNITS) continue;
            uint2 a, m, l;
            if (is_v(n)) {
                // key quad kq: 16-key step kq / 4, half-wave kq & 1, slots 4·(kq / 2 & 1) … of the lane's eight
                const int kq = (u & 3) | (u >> 5 & 1) << 2, dq = (u >> 2 & 7) | u >> 6 << 3;
                const int hv = kq & 1, up = kq >> 1 & 1, step = kq >> 2;
                int8_t* f = sv + ((dq >> 3) * 2 + step) * 3072 + hv * 512 + up * 8;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int c = (dq & 7) * 4 + i;
                    knx_split4(make_float4((&ld[n][0].x)[i], (&ld[n][1].x)[i], (&ld[n][2].x)[i], (&ld[n][3].x)[i]), a, m, l);
                    int8_t* w = f + ((c ^ (c >> 4 << 1) ^ hv) << 4);
                    *reinterpret_cast<uint2*>(w) = a;
                    *reinterpret_cast<uint2*>(w + 1024) = m;
                    *reinterpret_cast<uint2*>(w + 2048) = l;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int k = i * 2 * D + (u - 2 * D), row = k >> 2 & 31, hv = k >> 1 & 1;
                    knx_split4(ld[n][i], a, m, l);
                    int8_t* w = sk + (k >> 7) * 3072 + hv * 512 + ((row ^ (hv * 12)) << 4) + (k & 1) * 8;
                    *reinterpret_cast<uint2*>(w) = a;
                    *reinterpret_cast<uint2*>(w + 1024) = m;
                    *reinterpret_cast<uint2*>(w + 2048) = l;
                }
            }
        }
    };

    // Q fragments: the lane's query, columns 16·s + 8·hf …
    knx_v8bf qf[NS][3];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        uint2 a[2], m[2], l[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = 16 * s + 8 * hf + 4 * i;
            float4 v = knx_load4(c < p.d ? Qr + c : flash_zeros);
            v.x *= p.qmul, v.y *= p.qmul, v.z *= p.qmul, v.w *= p.qmul;
            knx_split4(v, a[i], m[i], l[i]);
        }
        qf[s][0] = __builtin_bit_cast(knx_v8bf, make_uint4(a[0].x, a[0].y, a[1].x, a[1].y));
        qf[s][1] = __builtin_bit_cast(knx_v8bf, make_uint4(m[0].x, m[0].y, m[1].x, m[1].y));
        qf[s][2] = __builtin_bit_cast(knx_v8bf, make_uint4(l[0].x, l[0].y, l[1].x, l[1].y));
    }

    v16f o[ND];
    float top, sum;  // the query's running maximum of q·k, and this half-wave's sum of exp(scale·(q·k − top))
    auto restart = [&]() __attribute__((always_inline)) {
        top = -INFINITY;
        sum = 0.0f;
#pragma unroll
        for (int u = 0; u < ND; ++u)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[u][e] = 0.0f;
    };
    // element e of a tile's scores: key 32·kt + 8·(e / 4) + 4·hf + e % 4
    auto mask = [&](int kt, v16f& sc, float with) __attribute__((always_inline)) {
        if (32 * kt + 32 <= p.S && !(p.causal && 32 * kt + 31 > qw)) return;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int j = 32 * kt + 8 * (e >> 2) + 4 * hf + (e & 3);
            if (j >= p.S || (p.causal && j > qi)) sc[e] = with;
        }
    };
    auto tile_top = [&](const v16f& sc) __attribute__((always_inline)) {
        float m = sc[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) m = __builtin_fmaxf(m, sc[e]);
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        return __builtin_fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
    };
    auto tile_sum = [&](const v16f& sc) __attribute__((always_inline)) {
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = (sc[e] + sc[4 + e]) + (sc[8 + e] + sc[12 + e]);
        return (a[0] + a[1]) + (a[2] + a[3]);
    };
    auto rescale = [&](float c) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < ND; ++u)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[u][e] = o[u][e] * c;
    };

    constexpr int SA[6] = {2, 0, 1, 1, 0, 0}, SB[6] = {0, 2, 1, 0, 1, 0};  // parts of the operands, smallest product first
    const int ka = hf * 512 + ((col ^ (hf * 12)) << 4), va = KB + hf * 512 + ((col ^ (col >> 4 << 1) ^ hf) << 4);
    auto scores = [&](int kt) __attribute__((always_inline)) {
        const int8_t* cur = lds + (kt & 1) * STAGE + ka;
        v16f s0, s1;  // two chains of multiplies
#pragma unroll
        for (int e = 0; e < 16; ++e) s0[e] = s1[e] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            knx_v8bf kf[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) kf[i] = *reinterpret_cast<const knx_v8bf*>(cur + s * 3072 + i * 1024);
#pragma unroll
            for (int i = 0; i < 6; i += 2) {
                s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[SA[i]], qf[s][SB[i]], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[SA[i + 1]], qf[s][SB[i + 1]], s1, 0, 0, 0);
            }
        }
        return s0 + s1;
    };
    // exp(scale·x) = 2^(x·sl), sl = scale·log2(e) in two floats: the hardware exp2 (≤ 1-2 ulp) of x·sl − tl, where tl is
    // top·sl rounded, the same for every key; a tile's older sums move to a new tl by 2^(old tl − new tl), so tl's
    // rounding cancels in the end
    const float sl = p.scale * LOG2E, sl2 = __builtin_fmaf(p.scale, LOG2E, -sl) + p.scale * 1.925963033500e-8f;
    float tl = 0.0f;
    restart();
    gload(0);
    put(0);
    gload(1);
    KNX_WAIT_LDS();
    knx_barrier_nofence();
    v16f sc = scores(0);
    mask(0, sc, MASKED);
    put(1);
    if (nt > 1) gload(2);
    KNX_WAIT_LDS();
    knx_barrier_nofence();
    const int ntw = p.causal ? min(nt, (qw + 31) / 32 + 1) : nt;  // this wave's tiles
    for (int kt = 0; kt < nt; ++kt) {
        if (kt < ntw) {
            v16f next = scores(kt + 1);  // (past the last tile: not used)
            const float m = __builtin_fmaxf(top, tile_top(sc));
            const float tn = m * sl;
            const float c = top == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(tl - tn);
            const bool grown = __any(top != m);
            top = m;
            tl = tn;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                sc[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[e], sl2, __builtin_fmaf(sc[e], sl, -tl)));
            sum = sum * c + tile_sum(sc);
            constexpr int NM = 6 * NS;
#pragma unroll
            for (int j = 0; j < NM; ++j) {  // a multiply, a few of the softmax's instructions
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (j + 3 < NM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x402, (116 + NM - 1) / NM, 0);
            }
            if (grown) rescale(c);
            const int8_t* cur = lds + (kt & 1) * STAGE + va;
#pragma unroll
            for (int step = 0; step < 2; ++step) {
                uint2 a[2], m2[2], l[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int e = 8 * step + 4 * i;
                    knx_split4(make_float4(sc[e], sc[e + 1], sc[e + 2], sc[e + 3]), a[i], m2[i], l[i]);
                }
                const knx_v8bf pf[3] = {__builtin_bit_cast(knx_v8bf, make_uint4(a[0].x, a[0].y, a[1].x, a[1].y)),
                                        __builtin_bit_cast(knx_v8bf, make_uint4(m2[0].x, m2[0].y, m2[1].x, m2[1].y)),
                                        __builtin_bit_cast(knx_v8bf, make_uint4(l[0].x, l[0].y, l[1].x, l[1].y))};
                knx_v8bf vf[ND][3];
#pragma unroll
                for (int u = 0; u < ND; ++u)
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        vf[u][i] = *reinterpret_cast<const knx_v8bf*>(cur + (u * 2 + step) * 3072 + i * 1024);
#pragma unroll
                for (int i = 0; i < 6; ++i)
#pragma unroll
                    for (int u = 0; u < ND; ++u)
                        o[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u][SA[i]], pf[SB[i]], o[u], 0, 0, 0);
            }
            sc = next;
            mask(kt + 1, sc, MASKED);
        }
        // every wave is past its reads of K's stage kt + 2 and V's kt + 1 (tiles kt and kt − 1): the barrier before
        if (kt + 1 < nt) {
            put(kt + 2);
            if (kt + 2 < nt) gload(kt + 3);
        }
        KNX_WAIT_LDS();
        knx_barrier_nofence();
    }

    float inv = 1.0f / knx_lane_group_sum_halves(sum);
    // An infinity or a NaN in Q, K or V (or a value that rounds to a bf16 infinity) leaves a value that is not finite: the
    // wave's queries again, with fp32 products straight from memory.
    float bad = inv * 0.0f;
#pragma unroll
    for (int u = 0; u < ND; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) bad = __builtin_fmaf(o[u][e], 0.0f, bad);
    if (__any(bad != 0.0f)) {
        restart();
#pragma unroll 1
        for (int kt = 0; kt < nt; ++kt) {
            v16f sc;
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = 0.0f;
            const int key = 32 * kt + col;
#pragma unroll 1
            for (int c0 = 0; c0 < D; c0 += 8) {
                const int c = c0 + 4 * hf;
                const float4 kf = knx_load4(key < p.S && c < p.d ? Kh + (size_t)key * p.ldk + c : flash_zeros);
                const float4 qv = knx_load4(c < p.d ? Qr + c : flash_zeros);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    sc = __builtin_amdgcn_mfma_f32_32x32x2f32((&kf.x)[i], (&qv.x)[i] * p.qmul, sc, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = p.scale * sc[e];
            mask(kt, sc, -INFINITY);
            const float m = __builtin_fmaxf(top, tile_top(sc)), from = m == -INFINITY ? 0.0f : m;
            const float c = top == m ? 1.0f : __builtin_amdgcn_exp2f((top - m) * LOG2E);
            top = m;
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = __builtin_amdgcn_exp2f((sc[e] - from) * LOG2E);
            sum = sum * c + tile_sum(sc);
            rescale(c);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = 32 * kt + 8 * (e >> 2) + 4 * hf + (e & 3);
#pragma unroll
                for (int u = 0; u < ND; ++u) {
                    const int c = 32 * u + col;
                    const float vv = *(row < p.S && c < p.d ? Vh + (size_t)row * p.ldv + c : flash_zeros);
                    o[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, sc[e], o[u], 0, 0, 0);
                }
            }
        }
        inv = 1.0f / knx_lane_group_sum_halves(sum);
    }
    if (qi >= p.Rq) return;
    // element e of o[u]: context column 32·u + 8·(e / 4) + 4·hf + e % 4 of the lane's query
    float* y = p.ctx + ((size_t)b * p.Rq + qi) * ((size_t)p.H * p.d) + (size_t)h * p.d;
#pragma unroll
    for (int u = 0; u < ND; ++u)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const int c = 32 * u + 8 * e4 + 4 * hf;
            const knx_v4fu v = {o[u][4 * e4] * inv, o[u][4 * e4 + 1] * inv, o[u][4 * e4 + 2] * inv, o[u][4 * e4 + 3] * inv};
            if (c < p.d) *reinterpret_cast<knx_v4fu*>(y + c) = v;
        }
}

template <int D, int OCC>
int launch(const knx_flash_args& p, hipStream_t s, const char* name)
{
    const int qblocks = (p.Rq + 127) / 128;
    hipLaunchKernelGGL((flash<D, OCC>), dim3((unsigned)qblocks * (unsigned)(p.B * p.H)), dim3(256), 0, s, p, qblocks);
    return knx::check_launch(name);
}

}  // namespace

int knx_flash(const knx_flash_args& args, hipStream_t s, const char* name)
{
    knx_flash_args p = args;
    if (p.d % 4 != 0 || p.d > 128 || (long long)p.B * p.H * ((p.Rq + 127) / 128) > 0x7fffffffLL) return 1;
    // the running maximum is of q·k: a scale that is not positive goes into Q (0 and NaN as they are)
    p.qmul = p.scale > 0.0f ? 1.0f : p.scale < 0.0f ? -1.0f : p.scale;
    p.scale = p.scale > 0.0f ? p.scale : p.scale < 0.0f ? -p.scale : 1.0f;
    if (p.d <= 32) return launch<32, 2>(p, s, name);
    if (p.d <= 64) return launch<64, 2>(p, s, name);
    if (p.d <= 96) return launch<96, 1>(p, s, name);
    return launch<128, 1>(p, s, name);
}
