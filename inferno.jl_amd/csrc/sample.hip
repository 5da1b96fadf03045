// Draft-side sampler on gfx950: softmax_sample (src/ModelCPU.jl:1123-1200)
// with temperature, top-k, top-p and min-p, and the presence / repetition
// penalties the generation loop applies to the logits first
// (apply_presence_penalty!, apply_repetition_penalty!,
// src/ModelCPU.jl:1202-1225).
//
// One workgroup of 1024 threads per row. Every pass over a row reads it in
// rounds of 4096 logits (one float4 per thread, coalesced), so after the
// first pass the row (600 KB at V = 151936) is served from L2.
//
//  * T = 0: Julia's argmax (the first NaN above every number, +0.0 above
//    -0.0, the first of equals) by an integer key.
//  * top-k (1 <= k <= 4096, k < V): exact radix select of the k-th largest
//    z = L / T (buckets, then an order-preserving key's bits), ties at the
//    threshold kept lowest index first (the stable descending sortperm);
//    the k candidates are compacted into LDS in index order, and softmax,
//    top-p (a bitonic sort by probability, then a scan), min-p and the draw
//    run there.
//  * no top-k: softmax statistics by full passes; top-p finds the nucleus by
//    a radix select over the same keys whose buckets carry the probability
//    mass in 2^-40 fixed point (integer LDS atomics: deterministic); min-p
//    is a threshold; the draw sums each round, picks the round, then scans
//    it, the rounds' sums taken from per-wave parts kept by the pass before
//    it (statistics, nucleus mass or min-p mass) where V <= 262144.
//  * the threshold's refinement passes run over the first pass's bucket
//    gathered into LDS when it holds at most 4096 elements.
//  * with a workspace, every setting spreads each row over workgroups of
//    one round (chunk statistics, each chunk's argmax, threshold histograms
//    and candidate lists, kept sums), and one workgroup per row finishes
//    each stage from them (16 or 8 where a few rows' top-p is flat).
// Sums and scans are trees, where the reference accumulates sequentially:
// the drawn token can differ only where u falls within rounding of a CDF
// step.
#include "common.h"

#include <climits>

namespace {

constexpr int SNT = 1024;
constexpr int SNW = SNT / 64;
constexpr int SROUND = 4 * SNT;
constexpr int SK_MAX = 4096;
constexpr int SMAX_ROUNDS = 1024;  // V <= 4194304
constexpr int SPART_ROUNDS = 64;   // plain draws by per-wave parts: V <= 262144

struct SampleArgs {
    float T;       // 0: argmax
    int top_k;     // 0: off (the host maps k >= V to 0)
    float top_p;   // >= 1: off
    float min_p;   // <= 0: off
};

// Order-preserving 32-bit key of a float (larger float, larger key).
__device__ __forceinline__ uint32_t okey(float z) {
    const uint32_t b = __float_as_uint(z);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float okey_inv(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// ---- block primitives (16 waves), fixed reduction trees
// Cross-lane moves of the butterflies on the VALU: the value of lane l ^ O (O
// = 8: a rotation by 8 within a row of 16; 4: row shifts by 4, each into the
// half rows that take it; 2, 1: quad permutes; 32, 16: swap_op). The levels
// and pairs of the reductions are those of shfl_xor.
template <int CTRL, int BANKS = 0xF> __device__ __forceinline__ float dpp(float old, float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v),
                                                                 CTRL, 0xF, BANKS, false));
}
template <int O> __device__ __forceinline__ float lane_xor(float v) {
    if constexpr (O == 8) return dpp<0x128>(v, v);                              // row_ror:8
    if constexpr (O == 4) return dpp<0x114, 0xA>(dpp<0x104, 0x5>(v, v), v);     // row_shl:4, row_shr:4
    if constexpr (O == 2) return dpp<0x4E>(v, v);                               // quad_perm [2,3,0,1]
    return dpp<0xB1>(v, v);                                                     // quad_perm [1,0,3,2]
}
// v of lane l combined with lane l ^ 32 (16): the two halves (rows) of a swap
// of v with itself hold one operand each.
template <int O, class F> __device__ __forceinline__ float swap_op(float v, F &&f) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    if constexpr (O == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
    }
}
template <class F> __device__ __forceinline__ float wave_reduce(float v, F &&f) {
    v = swap_op<32>(v, f);
    v = swap_op<16>(v, f);
    v = f(v, lane_xor<8>(v));
    v = f(v, lane_xor<4>(v));
    v = f(v, lane_xor<2>(v));
    return f(v, lane_xor<1>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
// The same over integers (any order gives the same sum).
template <int O> __device__ __forceinline__ uint32_t lane_xor_u(uint32_t v) {
    return __builtin_bit_cast(uint32_t, lane_xor<O>(__builtin_bit_cast(float, v)));
}
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
    auto join = [](uint32_t lo, uint32_t hi) { return ((unsigned long long)hi << 32) | lo; };
    const auto l32 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
    v = join(l32[0], h32[0]) + join(l32[1], h32[1]);
    const auto l16 = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
    const auto h16 = __builtin_amdgcn_permlane16_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
    v = join(l16[0], h16[0]) + join(l16[1], h16[1]);
    v += join(lane_xor_u<8>((uint32_t)v), lane_xor_u<8>((uint32_t)(v >> 32)));
    v += join(lane_xor_u<4>((uint32_t)v), lane_xor_u<4>((uint32_t)(v >> 32)));
    v += join(lane_xor_u<2>((uint32_t)v), lane_xor_u<2>((uint32_t)(v >> 32)));
    v += join(lane_xor_u<1>((uint32_t)v), lane_xor_u<1>((uint32_t)(v >> 32)));
    return v;
}
// Inclusive scan over the 64 lanes: row shifts inside each row of 16, then
// the rows' totals (row 0 into 1, 2 into 3; 0 and 1 into 2 and 3).
__device__ __forceinline__ uint32_t wave_scan_u(uint32_t v) {
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, true);  // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, true);  // row_bcast:31 into rows 2, 3
    return v;
}
__device__ __forceinline__ uint32_t wave_sum_u(uint32_t v) { return __builtin_amdgcn_readlane(wave_scan_u(v), 63); }
__device__ __forceinline__ int wave_min_i(int v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}
__device__ float block_sum(float v, float *red) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    v = wave_sum(v);
    __syncthreads();  // (red may still be read by the previous call)
    if (l == 0) red[w] = v;
    __syncthreads();
    return wave_sum(l < SNW ? red[l] : 0.f);
}
__device__ float block_max(float v, float *red) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    v = wave_max(v);
    __syncthreads();
    if (l == 0) red[w] = v;
    __syncthreads();
    return wave_max(l < SNW ? red[l] : -__builtin_huge_valf());
}
__device__ __forceinline__ int block_min_i(int v, int *red) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    v = wave_min_i(v);
    __syncthreads();
    if (l == 0) red[w] = v;
    __syncthreads();
    return wave_min_i(l < SNW ? red[l] : INT_MAX);
}
// exclusive scan over the block in thread order; *total = block sum
__device__ __forceinline__ uint32_t block_excl_scan_u(uint32_t v, uint32_t *red, uint32_t &total) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    uint32_t inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(inc, o);
        if (l >= o) inc += y;
    }
    __syncthreads();
    if (l == 63) red[w] = inc;
    __syncthreads();
    uint32_t base = 0, tot = 0;
    for (int i = 0; i < SNW; i++) {
        const uint32_t x = red[i];
        base += i < w ? x : 0u;
        tot += x;
    }
    total = tot;
    return base + inc - v;
}
__device__ __forceinline__ float block_excl_scan_f(float v, float *red, float &total) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    float inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const float y = __shfl_up(inc, o);
        if (l >= o) inc += y;
    }
    __syncthreads();
    if (l == 63) red[w] = inc;
    __syncthreads();
    float base = 0.f, tot = 0.f;
    for (int i = 0; i < SNW; i++) {
        const float x = red[i];
        if (i < w) base += x;
        tot += x;
    }
    total = tot;
    return base + (inc - v);
}

// Round r of a row: this thread's 4 logits z = L * (1 / T) (within an ulp
// of the reference's L / T, the same order and the same ties), in false past
// V. One 16-byte load where the 4 lie inside the row at an aligned address,
// else 4-byte loads; an entry past V reads -Inf, which no draw can select
// (probability 0, below every kept entry, the last in index order among
// ties), so a row of any length or alignment is drawn as the reference
// draws it (the tokens are clamped to V - 1).
__device__ __forceinline__ void load_round(const float *__restrict__ row, int V, int r, float invT, float (&z)[4],
                                           bool &in) {
    const int base = r * SROUND + 4 * (int)threadIdx.x;
    in = base < V;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (in) {
        if (base + 4 <= V && ((uintptr_t)(row + base) & 15) == 0) {
            x = *(const float4 *)(row + base);
        } else {
            const float ninf = -__builtin_huge_valf();
            x.x = row[base];
            x.y = base + 1 < V ? row[base + 1] : ninf;
            x.z = base + 2 < V ? row[base + 2] : ninf;
            x.w = base + 3 < V ? row[base + 3] : ninf;
        }
    }
    z[0] = x.x; z[1] = x.y; z[2] = x.z; z[3] = x.w;
    if (invT != 1.0f) {
#pragma unroll
        for (int e = 0; e < 4; e++) z[e] = z[e] * invT;
    }
}

// A pass over the row: the loads of RB rounds are in flight together, then
// f(z, in, r) runs for each round in order (uniformly, so f may hold
// barriers).
constexpr int RB = 8;
template <class F>
__device__ __forceinline__ void for_rounds(const float *__restrict__ row, int V, int nround, float T, F &&f) {
    for (int r0 = 0; r0 < nround; r0 += RB) {
        float z[RB][4];
        bool in[RB];
#pragma unroll
        for (int b = 0; b < RB; b++) load_round(row, V, r0 + b, T, z[b], in[b]);
#pragma unroll
        for (int b = 0; b < RB; b++)
            if (r0 + b < nround) f(z[b], in[b], r0 + b);
    }
}

// exp for the probabilities (the hardware exp2 after a multiply by log2 e:
// ~1e-6 relative, the same value in every pass)
__device__ __forceinline__ float pexp(float x) { return __expf(x); }

// (m, s) = (max, sum exp(z - max)) merged; symmetric, so both partners of a
// butterfly get the same bits
__device__ __forceinline__ void merge_ms2(float &m, float &s, float m2, float s2) {
    const float mm = fmaxf(m, m2);
    if (mm == -__builtin_huge_valf()) {  // (both sums 0, or NaN from a NaN entry: kept)
        s = s + s2;
        return;
    }
    s = s * pexp(m - mm) + s2 * pexp(m2 - mm);
    m = mm;
}
__device__ void block_ms(float &m, float &s, float *red) {
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(s, o);
        merge_ms2(m, s, m2, s2);
    }
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) {
        red[w] = m;
        red[SNW + w] = s;
    }
    __syncthreads();
    m = l < SNW ? red[l] : -__builtin_huge_valf();
    s = l < SNW ? red[SNW + l] : 0.f;
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(s, o);
        merge_ms2(m, s, m2, s2);
    }
}

// First j in [0, n) of this thread's 4 values (slot 4t + e) with u <= the
// inclusive prefix; the block's scan total goes to *total.
__device__ __forceinline__ int first_cdf_hit(const float (&v)[4], int n_here, float before, float u, float *redf, float &total) {
    float c[4], run = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        run += v[e];
        c[e] = run;
    }
    const float ex = block_excl_scan_f(run, redf, total);
    int hit = INT_MAX;
#pragma unroll
    for (int e = 3; e >= 0; e--)
        if (e < n_here && u <= before + (ex + c[e])) hit = 4 * (int)threadIdx.x + e;
    return hit;
}

// Julia's findmax order as an unsigned key: the order-preserving key of the
// float (+0.0 above -0.0), every NaN the largest (NaNs equal: the first
// wins). A real float's key is at least 1.
__device__ __forceinline__ uint32_t jl_key(float z) { return isnan(z) ? 0xffffffffu : okey(z); }
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}
// The block's first index holding the largest key (INT_MAX when none: all
// keys 0); *best_k gets that key.
__device__ int block_argmax_key(uint32_t k, int i, uint32_t *s_k, int *s_i, uint32_t *best_k = nullptr) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    uint32_t m = wave_max_u(k);
    __syncthreads();
    if (l == 0) s_k[w] = m;
    __syncthreads();
    m = wave_max_u(l < SNW ? s_k[l] : 0u);
    if (best_k) *best_k = m;
    return block_min_i(k == m && m != 0u ? i : INT_MAX, s_i);
}

// Threshold selection counted from the top (the k-th largest z, or the z
// where the probability mass from the top reaches top_p). Pass A buckets
// logits linearly, 8 buckets per unit of log-probability counted down from
// the maximum's (bucket 255: the tail), which spreads real logits over many
// buckets; then passes of 8 key bits each refine inside the chosen bucket,
// over its few elements. The grid is absolute (zq: floor(8 z), saturated far
// past float's fraction), so that a part of a row may count from its own
// maximum: bucket b there is bucket b + zq(row's) - zq(part's) of the row.
// With MASS the buckets also carry each element's probability in 2^-40
// fixed point (integer atomics: the same sums in any order).
__device__ __forceinline__ int zq(float z) {
    return (int)floorf(fminf(fmaxf(z * 8.0f, -0x1p29f), 0x1p29f));  // (-Inf and NaN: the lowest)
}
__device__ __forceinline__ uint32_t zbin(float z, float zmax) { return (uint32_t)min(zq(zmax) - zq(z), 255); }
// The smallest z with zq(z) >= q: bucket b of a row with zq(zmax) = zqm is
// grid_lo(zqm - b) <= z < grid_lo(zqm - b + 1) (b = 255: no lower bound).
__device__ __forceinline__ float grid_lo(int q) {
    return q <= -(1 << 29) ? -__builtin_huge_valf() : q > (1 << 29) ? __builtin_huge_valf() : __int2float_ru(q) * 0.125f;
}
// z's place among the 256 equal parts of its grid cell (never falls as z
// grows; just below 0 the difference rounds up to 1)
__device__ __forceinline__ uint32_t zpart(float z) {
    const float y = fminf(fmaxf(z * 8.0f, -0x1p29f), 0x1p29f);
    return min((uint32_t)((y - floorf(y)) * 256.0f), 255u);
}

struct Select {
    uint32_t zb;             // the bucket of pass A
    uint32_t tau;            // key of the threshold element inside it
    unsigned long long rem;  // units still to reach among the elements equal to tau
    uint32_t cnt;            // elements equal to tau
    bool all;                // (MASS) the total ran short of the target: keep every element
};

// Wave 0 finds, over the 256 buckets (descending or ascending index), the
// one holding the rem-th unit (~0ull in *selm when the total is short).
template <bool MASS>
__device__ __forceinline__ void pick_bucket(const uint32_t *hist, const unsigned long long *mass, unsigned long long rem,
                            uint32_t *sel, unsigned long long *selm, bool descending) {
    const int t = threadIdx.x;
    if (t >= 64) return;
    unsigned long long c[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int b = descending ? 255 - 4 * t - j : 4 * t + j;
        c[j] = MASS ? mass[b] : (unsigned long long)hist[b];
        sum += c[j];
    }
    unsigned long long inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long y = __shfl_up(inc, o);
        if (t >= o) inc += y;
    }
    const unsigned long long before = inc - sum;
    const bool found = before < rem && rem <= inc;
    if (found) {
        unsigned long long cum = before;
        for (int j = 0; j < 4; j++) {
            if (cum + c[j] >= rem) {
                sel[0] = descending ? 255u - 4u * t - j : 4u * t + j;
                selm[0] = cum;
                break;
            }
            cum += c[j];
        }
    }
    if (__ballot(found) == 0ull && t == 0) {
        sel[0] = 0u;
        selm[0] = ~0ull;
    }
}

// Fixed-point probability mass of z: p = exp(z - zmax) / S in units of 2^-40.
__device__ __forceinline__ unsigned long long mass_fx(float z, float zmax, float invS) {
    return (unsigned long long)(pexp(z - zmax) * invS * 1099511627776.0f);
}

// The entries q of a thread's 4 into their buckets b (MASS: their units m);
// uniform over the wave. A wave whose entries all take one bucket adds once:
// on a row of equal logits its adds to one address are what a pass waits for.
template <bool MASS>
__device__ __forceinline__ void hist_add4(uint32_t *hist, unsigned long long *mass, const bool (&q)[4],
                                          const uint32_t (&b)[4], const unsigned long long (&m)[4]) {
    uint32_t b0 = 0, n = 0;
    unsigned long long sum = 0;
    bool same = true;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (q[e]) {
            same &= n == 0 || b[e] == b0;
            b0 = b[e];
            n++;
            if (MASS) sum += m[e];
        }
    const uint64_t any = __ballot(n != 0);
    if (any == 0ull) return;
    const uint32_t bl = __builtin_amdgcn_readlane(b0, __ffsll((unsigned long long)any) - 1);
    if (__ballot(n != 0 && (!same || b0 != bl)) == 0ull) {
        const uint32_t nw = (uint32_t)wave_sum_u64(n);
        if (MASS) sum = wave_sum_u64(sum);
        if ((threadIdx.x & 63) == 0) {
            atomicAdd(&hist[bl], nw);
            if (MASS) atomicAdd(&mass[bl], sum);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (q[e]) {
                atomicAdd(&hist[b[e]], 1u);
                if (MASS) atomicAdd(&mass[b[e]], m[e]);
            }
    }
}

// The threshold inside bucket R.zb, R.rem units still to reach: R.tau, R.rem
// and R.cnt on return, or R.all when (MASS) truncated masses fall just short of
// the target.
// At most SPAIR_MAX gathered elements (keys ck, values cz) are ranked
// directly: tau is the key whose larger keys hold less than R.rem units and
// which with its equals reaches it (integer sums: the key the passes below
// would find; MASS: the elements' units staged in mass[], which holds 256).
constexpr int SPAIR_MAX = 128;
template <bool MASS>
__device__ void refine_pairs(float zmax, float S, int nzb, unsigned long long *mass, uint32_t *sel,
                             unsigned long long *selm, const uint32_t *ck, const float *cz, Select &R) {
    const int t = threadIdx.x;
    const float invS = 1.0f / S;
    if (t == 0) {
        sel[0] = 0u;
        sel[1] = 0u;
        selm[0] = ~0ull;
    }
    if (MASS && t < nzb) mass[t] = mass_fx(cz[t], zmax, invS);  // (each element's units, once)
    __syncthreads();
    // element i = t / P compared with every P-th element from t % P (at
    // most 16 comparisons a lane); the P lanes of an element (adjacent,
    // in one wave) then add their sums
    int lp = 0;
    while (nzb > (16 << lp)) lp++;  // (nzb <= SPAIR_MAX: P = 2^lp <= 8)
    const int P = 1 << lp, i = t >> lp;
    const bool act = i < nzb;
    const uint32_t ki = act ? ck[i] : 0u;
    unsigned long long gt = 0, eq = 0;
    uint32_t ne = 0;
    if (act)
        for (int j = t & (P - 1); j < nzb; j += P) {
            const uint32_t kj = ck[j];
            const unsigned long long mj = MASS ? mass[j] : 1ull;
            if (kj > ki) {
                gt += mj;
            } else if (kj == ki) {
                eq += mj;
                ne++;
            }
        }
    for (int o = 1; o < P; o <<= 1) {
        gt += __shfl_xor(gt, o);
        eq += __shfl_xor(eq, o);
        ne += __shfl_xor(ne, o);
    }
    if (act && (t & (P - 1)) == 0 && gt < R.rem && R.rem <= gt + eq) {  // (every element of key ki writes the same)
        sel[0] = ki;
        sel[1] = ne;
        selm[0] = gt;
    }
    __syncthreads();
    const uint32_t tau = sel[0], cnt = sel[1];
    const unsigned long long above = selm[0];
    __syncthreads();
    if (above == ~0ull) {
        R.all = true;
        return;
    }
    R.rem -= above;
    R.cnt = cnt;
    R.tau = tau;
}

// Passes B: the key 8 bits a pass from the highest that differs in the bucket
// (a cell of the grid: 14 to 20 bits for |z| of 1 to 64, not 32), over the
// nzb gathered elements when gathered, until one is left, else over the row.
// (Four passes of the whole key: 611 elements 9.4 us, 3000 14.7; now 5 and 8.)
template <bool MASS>
__device__ __noinline__ void refine_passes(const float *__restrict__ row, int V, int nround, float T, float zmax, float S,
                                           bool gathered, int nzb, uint32_t *hist, unsigned long long *mass,
                                           uint32_t *sel, unsigned long long *selm, const uint32_t *ck, const float *cz,
                                           Select &R) {
    const int t = threadIdx.x;
    const uint32_t zb = R.zb;
    const float invS = 1.0f / S;
    // the bits below the highest in which two keys of the bucket can differ
    const int zqm = zq(zmax);
    const float lo = zb >= 255u ? -__builtin_huge_valf() : grid_lo(zqm - (int)zb);
    const float hi = grid_lo(zqm - (int)zb + 1);
    const uint32_t khi = okey(hi) - 1u, klo = okey(lo == 0.f ? -0.f : lo);
    const int nbits = max(32 - __clz(klo ^ khi), 1);
    uint32_t pmask = nbits == 32 ? 0u : ~0u << nbits, prefix = khi & pmask;
    for (int top = nbits; top > 0; top -= 8) {
        const int shift = max(top - 8, 0);
        const uint32_t digit = (1u << (top - shift)) - 1u;
        if (t < 256) {
            hist[t] = 0;
            if (MASS) mass[t] = 0;
        }
        __syncthreads();
        if (gathered) {
            for (int i = t; i < nzb; i += SNT) {
                const uint32_t k = ck[i];
                if ((k & pmask) != prefix) continue;
                const uint32_t b = (k >> shift) & digit;
                atomicAdd(&hist[b], 1u);
                if (MASS) atomicAdd(&mass[b], mass_fx(cz[i], zmax, invS));
            }
        } else {
            for_rounds(row, V, nround, T, [&](const float (&z)[4], bool in, int) {
                bool q[4];
                uint32_t b[4];
                unsigned long long m[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t k = okey(z[e]);
                    q[e] = in && (k & pmask) == prefix && z[e] >= lo && z[e] < hi;
                    b[e] = (k >> shift) & digit;
                    m[e] = MASS && q[e] ? mass_fx(z[e], zmax, invS) : 0ull;
                }
                hist_add4<MASS>(hist, mass, q, b, m);
            });
        }
        __syncthreads();
        pick_bucket<MASS>(hist, mass, R.rem, sel, selm, true);
        __syncthreads();
        const uint32_t b = sel[0];
        const unsigned long long above = selm[0];
        const uint32_t cb = hist[b];
        __syncthreads();
        if (above == ~0ull) {  // (MASS: truncated masses just short of the target)
            R.all = true;
            return;
        }
        R.rem -= above;
        prefix |= b << shift;
        pmask |= digit << shift;
        R.cnt = cb;
        if (gathered && cb == 1u && shift > 0) {  // (one element: its key)
            for (int i = t; i < nzb; i += SNT)
                if ((ck[i] & pmask) == prefix) sel[0] = ck[i];
            __syncthreads();
            prefix = sel[0];
            __syncthreads();
            break;
        }
    }
    R.tau = prefix;
}

template <bool MASS>
__device__ __forceinline__ void refine_threshold(const float *__restrict__ row, int V, int nround, float T, float zmax,
                                                 float S, bool gathered, int nzb, uint32_t *hist,
                                                 unsigned long long *mass, uint32_t *sel, unsigned long long *selm,
                                                 const uint32_t *ck, const float *cz, Select &R) {
    if (gathered && nzb <= SPAIR_MAX) refine_pairs<MASS>(zmax, S, nzb, mass, sel, selm, ck, cz, R);
    else refine_passes<MASS>(row, V, nround, T, zmax, S, gathered, nzb, hist, mass, sel, selm, ck, cz, R);
}

// The B passes read only the elements of bucket zb: when it holds at most
// SK_MAX of them, one more pass gathers their keys and values into LDS
// (ck, cz; any order: the passes only count) and the B passes run there
// instead of over the row.
template <bool MASS>
__device__ void select_threshold(const float *__restrict__ row, int V, int nround, float T, float zmax, float S,
                                 unsigned long long target, uint32_t *hist, unsigned long long *mass, uint32_t *sel,
                                 unsigned long long *selm, uint32_t *ck, float *cz, int *ncnt, Select &R) {
    const int t = threadIdx.x;
    R.zb = 255u;
    R.tau = 0u;
    R.rem = target;
    R.cnt = 0;
    R.all = false;
    const float invS = 1.0f / S;
    // pass A: buckets of w = zmax - z, largest z first = bucket 0 first
    if (t < 256) {
        hist[t] = 0;
        if (MASS) mass[t] = 0;
    }
    __syncthreads();
    for_rounds(row, V, nround, T, [&](const float (&z)[4], bool in, int) {
        if (!in) return;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t b = zbin(z[e], zmax);
            atomicAdd(&hist[b], 1u);
            if (MASS) atomicAdd(&mass[b], mass_fx(z[e], zmax, invS));
        }
    });
    __syncthreads();
    pick_bucket<MASS>(hist, mass, R.rem, sel, selm, false);
    __syncthreads();
    const uint32_t zb = sel[0];
    const unsigned long long aboveA = selm[0];
    const uint32_t nzb = hist[zb];
    __syncthreads();
    if (aboveA == ~0ull) {
        R.all = true;
        return;
    }
    R.rem -= aboveA;
    R.zb = zb;
    const bool gathered = nzb <= (uint32_t)SK_MAX;
    if (gathered) {
        if (t == 0) *ncnt = 0;
        __syncthreads();
        const int zqm = zq(zmax);
        const float lo = zb >= 255u ? -__builtin_huge_valf() : grid_lo(zqm - (int)zb), hi = grid_lo(zqm - (int)zb + 1);
        for_rounds(row, V, nround, T, [&](const float (&z)[4], bool in, int) {
            if (!in) return;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (z[e] >= lo && z[e] < hi) {
                    const int p = atomicAdd(ncnt, 1);  // < nzb: the predicate pass A counted
                    ck[p] = okey(z[e]);
                    cz[p] = z[e];
                }
        });
        __syncthreads();
    }
    refine_threshold<MASS>(row, V, nround, T, zmax, S, gathered, (int)nzb, hist, mass, sel, selm, ck, cz, R);
}

// Kept by a threshold: a larger z than the bucket (smaller bucket index), or
// inside it a larger key, or an equal key before index tie_lim.
__device__ __forceinline__ bool above_threshold(float z, int j, float zmax, uint32_t zb, uint32_t tau, int tie_lim) {
    const uint32_t b = zbin(z, zmax);
    if (b != zb) return b < zb;
    const uint32_t k = okey(z);
    return k > tau || (k == tau && j < tie_lim);
}

// draw_candidates for at most 64 of them, one a lane of one wave: the same
// values in the same order (a block sum of one wave's values is that wave's
// sum, a sorted slot the count of the candidates before it), without the
// ~30 barriers of the block form (sort 21, sums and scans 2-3 each), which
// were most of an 18 us draw of 40 candidates.
__device__ __forceinline__ void draw_candidates_wave(int n, SampleArgs a, float ur, int V, const int *s_cidx, float *s_cp,
                                     int *s_sort, int32_t *out_row) {
    const int l = threadIdx.x;
    // first_cdf_hit over slots 4 l + e of the first 16 lanes
    auto cdf_hit = [&](const float (&v)[4], float u) {
        float c[4], run = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            run += v[e];
            c[e] = run;
        }
        float inc = run;
        for (int o = 1; o < 64; o <<= 1) {
            const float y = __shfl_up(inc, o);
            if (l >= o) inc += y;
        }
        const float ex = inc - run;
        int hit = INT_MAX;
#pragma unroll
        for (int e = 3; e >= 0; e--)
            if (4 * l + e < n && u <= ex + c[e]) hit = 4 * l + e;
        return wave_min_i(hit);
    };
    const bool in = l < n;
    const float z = in ? s_cp[l] : -__builtin_huge_valf();
    const float zmax = wave_max(z);  // (all lanes)
    const float w = in ? pexp(z - zmax) : 0.f;
    const float S = wave_sum(w);
    float p = in ? w / S : 0.f;
    float v[4];
    if (a.top_p < 1.0f) {
        int rank = 0;
        for (int j = 0; j < n; j++) {
            const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), j));
            rank += pj > p || (pj == p && j < l);
        }
        if (in) {
            s_cp[l] = p;
            s_sort[rank] = l;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = 4 * l + e < n ? s_cp[s_sort[4 * l + e]] : 0.f;
        const int cut = cdf_hit(v, a.top_p);
        if (cut != INT_MAX && rank > cut) p = 0.f;
        const float total = wave_sum(p);
        if (total > 0.f) p = p / total;
    }
    if (a.min_p > 0.f) {
        const float thr = wave_max(fmaxf(p, 0.f)) * a.min_p;
        if (p < thr) p = 0.f;
        const float total = wave_sum(p);
        if (total > 0.f) p = p / total;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (in) s_cp[l] = p;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = 4 * l + e < n ? s_cp[4 * l + e] : 0.f;
    const int slot = cdf_hit(v, ur);
    if (l == 0) *out_row = slot == INT_MAX ? V - 1 : s_cidx[slot];
}

// The draw over n top-k candidates in LDS in index order (s_cidx: token
// ids, s_cp: z = L / T; s_sort: scratch), shared by draft_sample_kernel and
// the spread top-k draw: softmax over the candidates (the rest are
// exp(-Inf) = 0), top-p by a bitonic sort of their probabilities, min-p,
// then the inverse CDF in index order.
// (n <= 64: by wave 0 alone, draw_candidates_wave.)
__device__ void draw_candidates(int n, SampleArgs a, float ur, int V, int *s_cidx, float *s_cp, int *s_sort,
                                float *s_redf, int *s_redi, int32_t *out_row) {
    const int t = threadIdx.x;
    if (n <= 64) {
        if (t < 64) draw_candidates_wave(n, a, ur, V, s_cidx, s_cp, s_sort, out_row);
        return;
    }
    // softmax over the candidates (the rest are exp(-Inf) = 0)
    float lm = -__builtin_huge_valf();
    for (int i = t; i < n; i += SNT) lm = fmaxf(lm, s_cp[i]);
    const float zmax = block_max(lm, s_redf);
    float ls = 0.f;
    for (int i = t; i < n; i += SNT) {
        const float w = pexp(s_cp[i] - zmax);
        s_cp[i] = w;
        ls += w;
    }
    const float S = block_sum(ls, s_redf);
    for (int i = t; i < n; i += SNT) s_cp[i] = s_cp[i] / S;
    __syncthreads();
    if (a.top_p < 1.0f) {
        // sort the slots by (p descending, slot ascending) = the stable
        // descending sortperm of the probabilities
        int P2 = 1;
        while (P2 < n) P2 <<= 1;
        for (int i = t; i < P2; i += SNT) s_sort[i] = i < n ? i : -1;
        __syncthreads();
        for (int size = 2; size <= P2; size <<= 1)
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int i = t; i < P2 / 2; i += SNT) {
                    const int lo = ((i & ~(stride - 1)) << 1) | (i & (stride - 1));
                    const int hi = lo + stride;
                    const int A = s_sort[lo], B = s_sort[hi];
                    bool a_first;
                    if (A < 0) a_first = false;
                    else if (B < 0) a_first = true;
                    else {
                        const float pa = s_cp[A], pb = s_cp[B];
                        a_first = pa > pb || (pa == pb && A < B);
                    }
                    if (a_first != ((lo & size) == 0)) {
                        s_sort[lo] = B;
                        s_sort[hi] = A;
                    }
                }
                __syncthreads();
            }
        // the shortest sorted prefix whose mass reaches top_p
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int j = 4 * t + e;
            v[e] = j < n ? s_cp[s_sort[j]] : 0.f;
        }
        float tot;
        const int hit = first_cdf_hit(v, n - 4 * t, 0.f, a.top_p, s_redf, tot);
        const int cut = block_min_i(hit, s_redi);
        const int n_keep = cut == INT_MAX ? n : cut + 1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int j = 4 * t + e;
            if (j < n && j >= n_keep) s_cp[s_sort[j]] = 0.f;
        }
        __syncthreads();
        float lt = 0.f;
        for (int i = t; i < n; i += SNT) lt += s_cp[i];
        const float total = block_sum(lt, s_redf);
        if (total > 0.f)
            for (int i = t; i < n; i += SNT) s_cp[i] = s_cp[i] / total;
        __syncthreads();
    }
    if (a.min_p > 0.f) {
        float lm2 = 0.f;
        for (int i = t; i < n; i += SNT) lm2 = fmaxf(lm2, s_cp[i]);
        const float thr = block_max(lm2, s_redf) * a.min_p;
        float lt = 0.f;
        for (int i = t; i < n; i += SNT) {
            float p = s_cp[i];
            if (p < thr) p = 0.f;
            s_cp[i] = p;
            lt += p;
        }
        const float total = block_sum(lt, s_redf);
        if (total > 0.f)
            for (int i = t; i < n; i += SNT) s_cp[i] = s_cp[i] / total;
        __syncthreads();
    }
    // inverse CDF in index order over the candidates
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int j = 4 * t + e;
        v[e] = j < n ? s_cp[j] : 0.f;
    }
    float tot;
    const int hit = first_cdf_hit(v, n - 4 * t, 0.f, ur, s_redf, tot);
    const int slot = block_min_i(hit, s_redi);
    if (t == 0) *out_row = slot == INT_MAX ? V - 1 : s_cidx[slot];
}

__global__ __launch_bounds__(SNT) void draft_sample_kernel(const float *__restrict__ L, int V, SampleArgs a,
                                                           const float *__restrict__ u, int32_t *__restrict__ out) {
    __shared__ float s_redf[2 * SNW];
    __shared__ float s_redv[SNW][RB];
    __shared__ uint32_t s_redu[SNW];
    __shared__ int s_redi[SNW];
    __shared__ uint32_t s_hist[256];
    __shared__ unsigned long long s_mass[256];
    __shared__ uint32_t s_sel[2];
    __shared__ unsigned long long s_selm[2];
    __shared__ float s_round[SMAX_ROUNDS];
    __shared__ float s_before;
    __shared__ int s_cidx[SK_MAX];
    __shared__ float s_cp[SK_MAX];
    __shared__ int s_sort[SK_MAX];
    __shared__ int s_ncnt;
    __shared__ float s_pm[SPART_ROUNDS][SNW], s_ps[SPART_ROUNDS][SNW];
    const int row = blockIdx.x, t = threadIdx.x;
    const float *Lr = L + (size_t)row * V;
    const int nround = (V + SROUND - 1) / SROUND;
    const float ur = u[row];
    const float invT = a.T > 0.f ? 1.0f / a.T : 1.0f;

    if (a.T == 0.0f) {
        // Julia's argmax: findmax order (the first NaN above every number,
        // +0.0 above -0.0), the first index among equals; each thread sees
        // its indices in increasing order
        uint32_t bk = 0u;
        int bi = INT_MAX;
        for_rounds(Lr, V, nround, 1.0f, [&](const float (&z)[4], bool in, int r) {
            if (!in) return;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t k = jl_key(z[e]);
                if (k > bk) {
                    bk = k;
                    bi = r * SROUND + 4 * t + e;
                }
            }
        });
        const int first = block_argmax_key(bk, bi, s_redu, s_redi);
        if (t == 0) out[row] = first == INT_MAX ? 0 : first;
        return;
    }
    const int K = a.top_k;
    if (K > 0 && K <= SK_MAX) {
        // ---- top-k: the k-th largest z, then the k candidates in index order
        float lmax = -__builtin_huge_valf(), nan = 0.f;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int) {
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    lmax = fmaxf(lmax, z[e]);
                    if (z[e] != z[e]) nan = 1.f;
                }
        });
        const float zm = block_max(lmax, s_redf);
        // a degenerate row (the reference's top-k keeps a NaN, its maximum is
        // then NaN; or no finite maximum) has NaN probabilities: last index
        if (block_max(nan, s_redf) > 0.f || !(zm > -__builtin_huge_valf() && zm < __builtin_huge_valf()) ||
            ur != ur) {
            if (t == 0) out[row] = V - 1;
            return;
        }
        // the reference's draw returns index 1 (here 0) when r <= 0: cumsum >= 0
        if (!(ur > 0.f)) {
            if (t == 0) out[row] = 0;
            return;
        }
        Select R;
        select_threshold<false>(Lr, V, nround, invT, zm, 1.f, (unsigned long long)K, s_hist, s_mass, s_sel, s_selm,
                                (uint32_t *)s_cidx, s_cp, &s_ncnt, R);
        const uint32_t tau = R.tau;  // (the keys of a bucket above tau's are larger)
        const int rem = (int)R.rem;  // elements equal to tau that are kept, lowest index first
        int run_kept = 0, run_eq = 0;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            bool g[4], q[4];
            uint32_t ng = 0, nq = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t k = okey(z[e]);
                g[e] = in && k > tau;
                q[e] = in && k == tau;
                ng += g[e];
                nq += q[e];
            }
            uint32_t tot;
            const uint32_t ex = block_excl_scan_u(ng | (nq << 16), s_redu, tot);
            const int eq_before = (int)(ex >> 16);
            int pos = run_kept + (int)(ex & 0xffffu) + min(max(rem - run_eq, 0), eq_before);
            int er = run_eq + eq_before;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (g[e] || (q[e] && er < rem)) {
                    if (pos < SK_MAX) {
                        s_cidx[pos] = r * SROUND + 4 * t + e;
                        s_cp[pos] = z[e];
                    }
                    pos++;
                }
                if (q[e]) er++;
            }
            run_kept += (int)(tot & 0xffffu) + min(max(rem - run_eq, 0), (int)(tot >> 16));
            run_eq += (int)(tot >> 16);
        });
        __syncthreads();
        const int n = min(run_kept, SK_MAX);  // == K
        draw_candidates(n, a, ur, V, s_cidx, s_cp, s_sort, s_redf, s_redi, out + row);
        return;
    }

    // ---- whole-row path: softmax statistics in one pass
    float zmax = -__builtin_huge_valf(), S = 0.f;
    // plain draws (no top-p, no min-p) over at most SPART_ROUNDS rounds:
    // every wave keeps the (max, sum exp(z - max)) of its part of each round,
    // so the rounds' sums for the draw need no second pass over the row
    bool by_parts = K == 0 && a.top_p >= 1.0f && a.min_p <= 0.f && nround <= SPART_ROUNDS;
    if (by_parts) {
        const int w = t >> 6;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            float m = -__builtin_huge_valf();
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++) m = fmaxf(m, z[e]);
            m = wave_max(m);
            float sw = 0.f;
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (z[e] != z[e]) sw = __builtin_nanf("");  // (a NaN entry flags the row)
                    else if (m > -__builtin_huge_valf()) sw += pexp(z[e] - m);
                }
            sw = wave_sum(sw);
            if ((t & 63) == 0) {
                s_pm[r][w] = m;
                s_ps[r][w] = sw;
            }
        });
        __syncthreads();
        const int np = nround * SNW;
        float lm = -__builtin_huge_valf(), nan = 0.f;
        for (int i = t; i < np; i += SNT) {
            lm = fmaxf(lm, s_pm[i / SNW][i % SNW]);
            if (s_ps[i / SNW][i % SNW] != s_ps[i / SNW][i % SNW]) nan = 1.f;
        }
        zmax = block_max(lm, s_redf);
        const bool has_nan = block_max(nan, s_redf) > 0.f;
        float ls = 0.f;
        if (zmax > -__builtin_huge_valf())
            for (int i = t; i < np; i += SNT) {
                const float m = s_pm[i / SNW][i % SNW];
                if (m > -__builtin_huge_valf()) ls += s_ps[i / SNW][i % SNW] * pexp(m - zmax);
            }
        S = block_sum(ls, s_redf);
        if (has_nan) S = __builtin_nanf("");
        // rows without a finite maximum or sum (all -Inf, NaN) take the
        // online pass below, as every other draw does
        by_parts = zmax > -__builtin_huge_valf() && S > 0.f && S < __builtin_huge_valf();
    }
    if (!by_parts) {
        zmax = -__builtin_huge_valf();
        S = 0.f;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int) {
            if (!in) return;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (z[e] != z[e]) {
                    S = __builtin_nanf("");  // (a NaN entry: the row is degenerate)
                } else if (z[e] > zmax) {
                    S = S * pexp(zmax - z[e]) + 1.0f;
                    zmax = z[e];
                } else if (zmax > -__builtin_huge_valf()) {
                    S += pexp(z[e] - zmax);
                }
            }
        });
        block_ms(zmax, S, s_redf);
    }
    // a degenerate row (no finite maximum, or a NaN entry: the reference's
    // maximum is NaN then) has NaN probabilities: the draw returns the last
    // index; otherwise r <= 0 returns the first (cumsum >= 0)
    if (!(zmax > -__builtin_huge_valf() && zmax < __builtin_huge_valf()) || !(S > 0.f && S < __builtin_huge_valf()) ||
        ur != ur) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    if (!(ur > 0.f)) {
        if (t == 0) out[row] = 0;
        return;
    }
    // the index limit of the ties at a threshold: the first n_eq of the
    // elements in bucket zb with key tau are kept (index order)
    auto tie_limit = [&](uint32_t zb, uint32_t tau, unsigned long long n_eq) {
        int run = 0, lim = V;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            bool q[4];
            uint32_t nq = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                q[e] = in && zbin(z[e], zmax) == zb && okey(z[e]) == tau;
                nq += q[e];
            }
            uint32_t tot;
            const uint32_t ex = block_excl_scan_u(nq, s_redu, tot);
            int cand = INT_MAX;
            int c = run + (int)ex;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (q[e]) {
                    c++;
                    if (c == (int)n_eq && cand == INT_MAX) cand = r * SROUND + 4 * t + e + 1;
                }
            const int got = block_min_i(cand, s_redi);
            if (lim == V && got != INT_MAX) lim = got;
            run += (int)tot;
        });
        return lim;
    };
    // top-k above the candidate limit: the k-th largest z by count (the
    // candidate path's threshold), kept by comparison; the softmax is over
    // the kept entries (S their sum), and top-p / min-p act on it below
    uint32_t zbK = 256u, tauK = 0u;
    int tieK = V;
    if (K > 0) {
        Select RK;
        select_threshold<false>(Lr, V, nround, invT, zmax, 1.f, (unsigned long long)K, s_hist, s_mass, s_sel, s_selm,
                                (uint32_t *)s_cidx, s_cp, &s_ncnt, RK);
        if (!RK.all) {
            zbK = RK.zb;
            tauK = RK.tau;
            if (RK.rem < RK.cnt) tieK = tie_limit(zbK, tauK, RK.rem);
        }
        float ls = 0.f;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (zbK == 256u || above_threshold(z[e], r * SROUND + 4 * t + e, zmax, zbK, tauK, tieK))
                        ls += pexp(z[e] - zmax);
        });
        S = block_sum(ls, s_redf);
    }
    auto keptK = [&](float z, int j) { return zbK == 256u || above_threshold(z, j, zmax, zbK, tauK, tieK); };
    // kept: above_threshold(zb, tau, tie_lim); everything without top-p
    uint32_t zb = 256u, tau = 0u;
    int tie_lim = V;
    bool div_total = false;  // top-p renormalizes by the nucleus mass
    float total_p = 1.0f;
    // rounds' sums of the final probabilities from the last pass's per-wave
    // parts (s_ps, times parts_scale) instead of a pass of their own
    bool round_parts = false;
    float parts_scale = 1.0f;
    const float invS = 1.0f / S;  // (probabilities by reciprocals: within an ulp of the divisions)
    if (a.top_p < 1.0f) {
        const float tp = fmaxf(a.top_p, 0.f) * 1099511627776.0f;
        const unsigned long long target = tp < 1.0f ? 1ull : (unsigned long long)ceilf(tp);
        Select R;
        select_threshold<true>(Lr, V, nround, invT, zmax, S, target, s_hist, s_mass, s_sel, s_selm,
                               (uint32_t *)s_cidx, s_cp, &s_ncnt, R);
        if (!R.all) {
            zb = R.zb;
            tau = R.tau;
            // ties at tau share one probability: keep the first n_eq of them
            const float ptau = pexp(okey_inv(tau) - zmax) * invS;
            const unsigned long long mt = (unsigned long long)(ptau * 1099511627776.0f);
            unsigned long long n_eq = mt ? (R.rem + mt - 1) / mt : (unsigned long long)R.cnt;
            if (n_eq < 1) n_eq = 1;
            if (n_eq < R.cnt) tie_lim = tie_limit(zb, tau, n_eq);  // index of the n_eq-th tie
        }
        // mass of the nucleus, then p' = p / total (without min-p, the
        // rounds' sums of the draw come from this pass's per-wave parts)
        const bool parts = a.min_p <= 0.f && nround <= SPART_ROUNDS;
        float lt = 0.f;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            float c = 0.f;
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int j = r * SROUND + 4 * t + e;
                    if (keptK(z[e], j) && (zb == 256u || above_threshold(z[e], j, zmax, zb, tau, tie_lim)))
                        c += pexp(z[e] - zmax) * invS;
                }
            lt += c;
            if (parts) {
                c = wave_sum(c);
                if ((t & 63) == 0) s_ps[r][t >> 6] = c;
            }
        });
        total_p = block_sum(lt, s_redf);
        div_total = total_p > 0.f;
        if (parts) {
            round_parts = true;
            parts_scale = div_total ? 1.0f / total_p : 1.0f;
        }
    }
    const float inv_total = div_total ? 1.0f / total_p : 1.0f;
    auto prob = [&](float z) {
        float p = pexp(z - zmax) * invS;
        if (div_total) p = p * inv_total;
        return p;
    };
    auto kept = [&](float z, int j) {
        return keptK(z, j) && (zb == 256u || above_threshold(z, j, zmax, zb, tau, tie_lim));
    };
    // min-p: the largest probability is the argmax's, exp(0) / S (renormalized)
    float thr = 0.f;
    bool div_total2 = false;
    float total2 = 1.0f;
    if (a.min_p > 0.f) {
        float pmax = invS;
        if (div_total) pmax = pmax * inv_total;
        thr = pmax * a.min_p;
        const bool parts = nround <= SPART_ROUNDS;
        float lt = 0.f;
        for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
            float c = 0.f;
            if (in)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (kept(z[e], r * SROUND + 4 * t + e)) {
                        const float p = prob(z[e]);
                        if (!(p < thr)) c += p;
                    }
            lt += c;
            if (parts) {
                c = wave_sum(c);
                if ((t & 63) == 0) s_ps[r][t >> 6] = c;
            }
        });
        total2 = block_sum(lt, s_redf);
        div_total2 = total2 > 0.f;
        if (parts) {
            round_parts = true;
            parts_scale = div_total2 ? 1.0f / total2 : 1.0f;
        }
    }
    const float inv_total2 = div_total2 ? 1.0f / total2 : 1.0f;
    auto final_p = [&](float z, int j) {
        if (!kept(z, j)) return 0.f;
        float p = prob(z);
        if (a.min_p > 0.f) {
            if (p < thr) return 0.f;
            if (div_total2) p = p * inv_total2;
        }
        return p;
    };
    // the draw: each round's sum (from the waves' parts, or batched: one
    // block reduction per RB rounds), the round, then the index inside it
    if (by_parts) {
        if (t < nround) {
            float sum = 0.f;
            for (int w = 0; w < SNW; w++) {
                const float m = s_pm[t][w];
                if (m > -__builtin_huge_valf()) sum += s_ps[t][w] * pexp(m - zmax);
            }
            s_round[t] = sum * invS;
        }
    } else if (round_parts) {
        if (t < nround) {
            float sum = 0.f;
            for (int w = 0; w < SNW; w++) sum += s_ps[t][w];
            s_round[t] = sum * parts_scale;
        }
    }
    for (int r0 = 0; r0 < (by_parts || round_parts ? 0 : nround); r0 += RB) {
        float part[RB];
#pragma unroll
        for (int b = 0; b < RB; b++) {
            float z[4];
            bool in;
            load_round(Lr, V, r0 + b, invT, z, in);
            float c = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) c += in ? final_p(z[e], (r0 + b) * SROUND + 4 * t + e) : 0.f;
            part[b] = wave_sum(c);
        }
        __syncthreads();
        if ((t & 63) == 0)
#pragma unroll
            for (int b = 0; b < RB; b++) s_redv[t >> 6][b] = part[b];
        __syncthreads();
        if (t < RB && r0 + t < nround) {
            float sum = 0.f;
            for (int w = 0; w < SNW; w++) sum += s_redv[w][t];
            s_round[r0 + t] = sum;
        }
    }
    __syncthreads();
    if (t == 0) {
        float cum = 0.f;
        int rr = -1;
        for (int r = 0; r < nround; r++) {
            const float nc = cum + s_round[r];
            if (ur <= nc) {
                rr = r;
                break;
            }
            cum = nc;
        }
        s_sel[0] = (uint32_t)rr;
        s_before = cum;
    }
    __syncthreads();
    const int rr = (int)s_sel[0];
    const float before = s_before;
    __syncthreads();
    if (rr < 0) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    float z[4], v[4];
    bool in;
    load_round(Lr, V, rr, invT, z, in);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = in ? final_p(z[e], rr * SROUND + 4 * t + e) : 0.f;
    float tot;
    const int hit = first_cdf_hit(v, in ? 4 : 0, before, ur, s_redf, tot);
    const int local = block_min_i(hit, s_redi);
    // (the scan inside the round can end a rounding step below the round's
    // sum that selected it: then the round's last kept entry)
    int last = INT_MAX;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (v[e] > 0.f) last = INT_MAX - (4 * t + e);
    const int lastk = block_min_i(last, s_redi);
    if (t == 0) {
        int tok = local != INT_MAX ? rr * SROUND + local : lastk != INT_MAX ? rr * SROUND + (INT_MAX - lastk) : V - 1;
        out[row] = min(tok, V - 1);
    }
}

// Workspace of the spread draws: float2 part[rows][nround] (each round's
// (max, sum exp(z - max))), then a slot of SLOT_BYTES per round of each row
// (a threshold: uint64 hist[256], at SLOT_LIST the candidate list; min-p: a
// float sum at SLOT_CSUM, once the list is no longer read), then
// ROW_BYTES per row (a threshold: the selection state, then the longer lists
// of a row of few rounds).
constexpr int SLOT_BYTES = 4096;
constexpr int SLOT_LIST = 2048;
constexpr int SLOT_CSUM = 3072;
constexpr size_t ROW_BYTES = 256 + (size_t)SK_MAX * 12;
constexpr int LIST_MAX = 336;  // entries of a list in its slot: (2048 - 16) / 6
struct SpreadWs {
    float2 *part;
    uint8_t *slots, *rows;
    int nround;
    // a round's list: 16 bytes of header, z[lmax], uint16 index in the round
    // [lmax]; above LIST_MAX in the row's ROW_BYTES, else in the round's slot
    int lmax;
    __device__ uint8_t *slot(int row, int c) const { return slots + ((size_t)row * nround + c) * SLOT_BYTES; }
    __device__ uint8_t *rowb(int row) const { return rows + (size_t)row * ROW_BYTES; }
    __device__ uint8_t *list(int row, int c) const {
        return lmax > LIST_MAX ? rowb(row) + 256 + (size_t)c * (16 + 6 * lmax) : slot(row, c) + SLOT_LIST;
    }
};
// The entries of a list: LIST_MAX, or for a top-k of many entries a round
// (twice the mean and 128; a multiple of 8, so that a header stays 8-byte
// aligned) as many as the row's ROW_BYTES hold for each round (top-k 4000 of
// 32000: 31.5 us with lists of LIST_MAX, 24.6 so; 64 rows of 50257 46.7 and
// 31.1). A row of 1 or 2 rounds is read whole instead (gather_far; top-k 4000
// of 8192: 25.4 us, 32.6 with lists of 4088 entries, a wave each).
constexpr int list_max(int nround, int top_k) {
    const int want = (2 * top_k / nround + 128) / 8 * 8, room = ((int)(ROW_BYTES - 256) / nround - 16) / 6 / 8 * 8;
    const int n = want < room ? want : room;
    return nround > 2 && n > LIST_MAX ? n : LIST_MAX;
}

// The row's softmax statistics from its rounds' partials (a fixed order: the
// same bits in every kernel, each wave by itself: the sums of 64 rounds at a
// time, then the sum of those); false for a degenerate row, whose reference
// probabilities are all NaN (the draw returns the last index): no finite
// maximum (all -Inf, or a +Inf) or a NaN entry anywhere (a round's sum is
// NaN then). The reference's top-k keeps a NaN (its descending sortperm
// puts NaN first) and its maximum is then NaN, so this holds with top-k
// too. count (a top-k threshold, whose softmax is over the kept entries
// only): S = 1.
__device__ __forceinline__ bool row_stats(const float2 *pr, int nround, float &zmax, float &S, bool count = false) {
    const int l = threadIdx.x & 63;
    const float ninf = -__builtin_huge_valf();
    const float2 p0 = l < nround ? pr[l] : make_float2(ninf, 0.f);
    float lm = p0.x;
    bool nan = p0.y != p0.y;
    for (int i = l + 64; i < nround; i += 64) {
        const float2 p = pr[i];
        lm = fmaxf(lm, p.x);
        nan |= p.y != p.y;
    }
    zmax = wave_max(lm);
    const bool has_nan = __ballot(nan) != 0ull;
    const bool finite_max = zmax > ninf && zmax < __builtin_huge_valf();
    if (count) {
        S = 1.0f;
        return finite_max && !has_nan;
    }
    float acc = 0.f;
    if (zmax > ninf)
        for (int v = 0; 64 * v < nround; v++) {
            const int i = 64 * v + l;
            const float2 p = v == 0 ? p0 : i < nround ? pr[i] : make_float2(ninf, 0.f);
            const float sv = wave_sum(p.x > ninf ? p.y * pexp(p.x - zmax) : 0.f);
            if (l == v) acc = sv;
        }
    S = wave_sum(acc);
    return finite_max && !has_nan && S > 0.f && S < __builtin_huge_valf();
}

// The chunk kernels (one workgroup per round of a row): CNT threads of 16
// entries. Wave w holds the entries of the one-row kernel's waves 4 w .. 4 w
// + 3 (v = 4 w + r: entries 256 v + 4 lane + e), so a sum over r = one of
// its waves, then over the 16 of them, is block_sum's. (1024 threads of 4
// entries waited on barriers: 64 rows' statistics 16.8 us, 9.3 with 256.)
constexpr int CNT = 256;
constexpr int CNW = CNT / 64;
constexpr int CR = SROUND / (4 * CNT);  // groups of 4 entries per thread
__device__ __forceinline__ int chunk_entry(int r) {  // the first entry of group r
    return (CR * (int)(threadIdx.x >> 6) + r) * 256 + 4 * (int)(threadIdx.x & 63);
}
// Round c of a row: z = L * (1 / T), -Inf past V (load_round's values; 16-byte
// loads at any 4-byte alignment).
__device__ __forceinline__ void load_chunk(const float *__restrict__ row, int V, int c, float invT, float (&z)[CR][4]) {
    const float *src = row + (size_t)c * SROUND;
    const int n = V - c * SROUND;
    if (n >= SROUND) {
#pragma unroll
        for (int r = 0; r < CR; r++) __builtin_memcpy(z[r], src + chunk_entry(r), 16);
    } else {
#pragma unroll
        for (int r = 0; r < CR; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int j = chunk_entry(r) + e;
                z[r][e] = j < n ? src[j] : -__builtin_huge_valf();
            }
    }
    if (invT != 1.0f) {
#pragma unroll
        for (int r = 0; r < CR; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) z[r][e] = z[r][e] * invT;
    }
}
// block_sum of the one-row kernel's 16 waves' values (v[r]: this thread's
// value in wave CR w + r); the sum in thread 0 (wave 0).
__device__ __forceinline__ float chunk_sum(float (&v)[CR], float *red /* [SNW] */) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < CR; r++) {
        v[r] = wave_sum(v[r]);
        if (l == 0) red[CR * w + r] = v[r];
    }
    __syncthreads();
    return wave_sum(l < SNW ? red[l] : 0.f);
}

// (max, sum exp(z - max)) of round blockIdx.x of row blockIdx.y: part[row][round].
__global__ __launch_bounds__(CNT) void chunk_stats_kernel(const float *__restrict__ L, int V, float invT,
                                                          float2 *__restrict__ part) {
    __shared__ float s_m[CNW], s_red[SNW];
    const int c = blockIdx.x, row = blockIdx.y, nround = gridDim.x;
    float z[CR][4];
    load_chunk(L + (size_t)row * V, V, c, invT, z);
    float m = -__builtin_huge_valf();
#pragma unroll
    for (int r = 0; r < CR; r++)
#pragma unroll
        for (int e = 0; e < 4; e++) m = fmaxf(m, z[r][e]);
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
    __syncthreads();
    m = s_m[0];
#pragma unroll
    for (int w = 1; w < CNW; w++) m = fmaxf(m, s_m[w]);
    float sw[CR];
#pragma unroll
    for (int r = 0; r < CR; r++) {
        sw[r] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (z[r][e] != z[r][e]) sw[r] = __builtin_nanf("");  // (flags the row even when m is -Inf)
            else if (m > -__builtin_huge_valf()) sw[r] += pexp(z[r][e] - m);
        }
    }
    const float sum = chunk_sum(sw, s_red);
    if (threadIdx.x == 0) part[(size_t)row * nround + c] = make_float2(m, sum);
}

// The draw of row blockIdx.x from its rounds' statistics: the row's max and
// sum, each round's probability mass, the round holding u (first with u <=
// the running sum), then the index inside it. A row without a finite maximum
// or sum (all -Inf, NaN, +Inf) draws V - 1, as the reference's NaN
// probabilities do; otherwise u <= 0 draws 0.
__global__ __launch_bounds__(SNT) void chunk_draw_kernel(const float *__restrict__ L, int V, float invT,
                                                         const float2 *__restrict__ part, const float *__restrict__ u,
                                                         int32_t *__restrict__ out) {
    __shared__ float s_redf[2 * SNW];
    __shared__ int s_redi[SNW];
    __shared__ float s_round[SMAX_ROUNDS];
    __shared__ float s_before;
    __shared__ int s_rr;
    const int row = blockIdx.x, t = threadIdx.x;
    const int nround = (V + SROUND - 1) / SROUND;
    const float ur = u[row];
    const float2 *pr = part + (size_t)row * nround;
    float zmax, S;
    if (!row_stats(pr, nround, zmax, S) || ur != ur) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    if (!(ur > 0.f)) {  // the reference's draw returns index 1 (here 0) when r <= 0
        if (t == 0) out[row] = 0;
        return;
    }
    const float invS = 1.0f / S;
    for (int i = t; i < nround; i += SNT) {
        const float2 p = pr[i];
        s_round[i] = p.x > -__builtin_huge_valf() ? p.y * pexp(p.x - zmax) * invS : 0.f;
    }
    __syncthreads();
    if (t == 0) {
        float cum = 0.f;
        int rr = -1;
        for (int r = 0; r < nround; r++) {
            const float nc = cum + s_round[r];
            if (ur <= nc) {
                rr = r;
                break;
            }
            cum = nc;
        }
        s_rr = rr;
        s_before = cum;
    }
    __syncthreads();
    const int rr = s_rr;
    const float before = s_before;
    if (rr < 0) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    float z[4], v[4];
    bool in;
    load_round(L + (size_t)row * V, V, rr, invT, z, in);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = in ? pexp(z[e] - zmax) * invS : 0.f;
    float tot;
    const int hit = first_cdf_hit(v, in ? 4 : 0, before, ur, s_redf, tot);
    const int local = block_min_i(hit, s_redi);
    // (the scan inside the round can end a rounding step below the round's
    // sum that selected it: then the round's last nonzero entry)
    int last = INT_MAX;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (v[e] > 0.f) last = INT_MAX - (4 * t + e);
    const int lastk = block_min_i(last, s_redi);
    if (t == 0) {
        const int tok =
            local != INT_MAX ? rr * SROUND + local : lastk != INT_MAX ? rr * SROUND + (INT_MAX - lastk) : V - 1;
        out[row] = min(tok, V - 1);
    }
}

// Spread greedy draws (T = 0): each chunk's first argmax in Julia's order
// (its key and index as float bits) into part[row][chunk], then one
// workgroup per row takes the first of those; an exact order, so the
// tokens are the one-workgroup kernel's.
__global__ __launch_bounds__(CNT) void chunk_argmax_kernel(const float *__restrict__ L, int V,
                                                           float2 *__restrict__ part) {
    __shared__ uint32_t s_k[CNW];
    __shared__ int s_i[CNW];
    const int c = blockIdx.x, row = blockIdx.y, t = threadIdx.x, nround = gridDim.x;
    float z[CR][4];
    load_chunk(L + (size_t)row * V, V, c, 1.0f, z);
    uint32_t bk = 0u;
    int bi = INT_MAX;
#pragma unroll
    for (int r = 0; r < CR; r++)
#pragma unroll
        for (int e = 0; e < 4; e++) {  // (the thread's entries in index order)
            const uint32_t k = jl_key(z[r][e]);
            const int j = c * SROUND + chunk_entry(r) + e;
            if (k > bk && j < V) {
                bk = k;
                bi = j;
            }
        }
    uint32_t best = wave_max_u(bk);
    int first = wave_min_i(bk == best ? bi : INT_MAX);
    if ((t & 63) == 0) {
        s_k[t >> 6] = best;
        s_i[t >> 6] = first;
    }
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < CNW; w++)  // (the waves in index order: the first best stays)
            if (s_k[w] > best) {
                best = s_k[w];
                first = s_i[w];
            }
        part[(size_t)row * nround + c] = make_float2(__uint_as_float(best), __int_as_float(first));
    }
}

__global__ __launch_bounds__(SNT) void argmax_draw_kernel(int V, const float2 *__restrict__ part,
                                                          int32_t *__restrict__ out) {
    __shared__ uint32_t s_k[SNW];
    __shared__ int s_i[SNW];
    const int row = blockIdx.x, t = threadIdx.x;
    const int nround = (V + SROUND - 1) / SROUND;
    uint32_t bk = 0u;
    int bi = INT_MAX;
    for (int c = t; c < nround; c += SNT) {  // (chunks in index order: the first best stays)
        const float2 p = part[(size_t)row * nround + c];
        const uint32_t k = __float_as_uint(p.x);
        if (k > bk) {
            bk = k;
            bi = __float_as_int(p.y);
        }
    }
    const int first = block_argmax_key(bk, bi, s_k, s_i);
    if (t == 0) out[row] = first == INT_MAX ? 0 : first;
}

// Spread thresholds: top-k (the k-th largest z, by count) and top-p (where
// the probability mass from the top reaches top_p), by the one-row kernel's
// rules (buckets below the row maximum, then the key; ties lowest index
// first). One launch over the rounds reads the logits once:
//  * the round's statistics (part, as chunk_stats_kernel's);
//  * hist[256] of the round, its buckets counted down from its own maximum
//    m: per bucket the count and the mass sum exp(z - m), packed as mass << 13
//    | count (one LDS atomic an entry, a copy of the array per wave). Bucket
//    b's mass is in units of 2^-mass_exp(b), ~2^-30 of its largest entry's,
//    so the entries' fp32 exponentials enter exactly (but in bucket 255, the
//    tail); the row kernel scales each bucket by a double factor to 2^-40 of
//    the row. (In 2^-38 of m's and an fp32 factor a round, the cumulative
//    masses were up to 1.0e-7 off against 64 bits, and 9.7e-8 with each
//    entry's mass cut to the row's 2^-40; so at most 4.6e-8.)
//    For top-k the buckets past one (the cut) whose entries up to it number k
//    are left out (at least k entries of this round are larger; for k <= 256
//    first those past one whose thread maxima number k, before the atomics);
//  * the candidate list: (z, index) of its entries up to bucket `last`, the
//    largest that leaves at most lmax of them, in index order.
// Then one workgroup per row (SPLIT: more) takes the row's statistics, brings
// the histograms to the row's buckets and masses, finds the threshold's
// bucket, takes that bucket's entries (top-k: and those above it) from the
// lists (from the row, for a round whose list ends before it), finds the
// threshold among them, and draws: top-k over the kept entries
// (draw_candidates), top-p by the rounds' kept masses (the buckets above the
// threshold's, plus its kept entries), then inside the round u falls in; with
// at most 64 entries up to the threshold's bucket one wave does all of it.
// Two launches where there were three (top-k <= 64), eight (larger) and six
// (top-p): 64 rows of 151936 at top-p 0.9 95 -> 28 us, one row at top-k 40 +
// top-p 28.6 -> 18.1 us, at top-k 1000 34.7 -> 26.9.
enum : int { SEL_SELECT = 0, SEL_ALL = 1, SEL_DEGEN = 2 };
struct RowSel {
    int mode;
    uint32_t zb, tau;
    int tie_lim;
    float zmax, S, inv1;  // inv1: 1 / the nucleus mass
    uint32_t arrived;     // workgroups whose part of a gather has landed
};
constexpr int ROW_PART = 256;  // then (a split gather) the bucket's entries: value, index
constexpr int CBITS = 13;      // count bits of a packed bucket (a round holds 4096 entries)
// Entries of bucket b below m have b - 1 < 8 (m - z) < b + 1 (b < 255), so
// exp(z - m) 2^mass_exp(b) lies in 2^29 .. 2^31 (46 / 256 is just below
// log2(e) / 8): its 24 bits are a whole number.
__device__ __forceinline__ int mass_exp(int b) { return (46 * b + 31 * 256 - 46) >> 8; }
struct ListHead {
    int n;    // entries
    int cut;  // the round's last bucket in its histogram
    float m;  // the round's maximum
    int pad;
};

template <bool COUNT>
__global__ __launch_bounds__(CNT) void chunk_hist_kernel(const float *__restrict__ L, int V, float invT, int top_k,
                                                         SpreadWs ws) {
    __shared__ unsigned long long s_h[CNW][256];
    __shared__ uint32_t s_tm[256];
    __shared__ float s_m[CNW], s_red[SNW];
    __shared__ int s_wn[CNW];
    const int c = blockIdx.x, row = blockIdx.y, t = threadIdx.x, wave = t >> 6, lane = t & 63;
    float z[CR][4];
    load_chunk(L + (size_t)row * V, V, c, invT, z);
#pragma unroll
    for (int w = 0; w < CNW; w++) s_h[w][t] = 0;
    s_tm[t] = 0;
    const int n = V - c * SROUND;  // entries of the row from this round on
    float tm = -__builtin_huge_valf();
#pragma unroll
    for (int r = 0; r < CR; r++)
#pragma unroll
        for (int e = 0; e < 4; e++) tm = fmaxf(tm, z[r][e]);
    float m = wave_max(tm);
    if (lane == 0) s_m[wave] = m;
    __syncthreads();
    m = s_m[0];
#pragma unroll
    for (int w = 1; w < CNW; w++) m = fmaxf(m, s_m[w]);
    // the buckets 4 lane .. 4 lane + 3 of a wave: how many leading buckets
    // hold at most `most` entries together (every wave by itself)
    auto leading = [&](const uint32_t (&h)[4], uint32_t most) {
        uint32_t cum[4], run = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            run += h[j];
            cum[j] = run;
        }
        const uint32_t inc = wave_scan_u(run);
        int k = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) k += __popcll(__ballot(inc - run + cum[j] <= most));
        return k;
    };
    uint32_t bcut = 255u;  // (top-k: buckets past it are left out)
    if (COUNT && top_k <= CNT) {
        if (chunk_entry(0) < n) atomicAdd(&s_tm[zbin(tm, m)], 1u);
        __syncthreads();
        const uint32_t h[4] = {s_tm[4 * lane], s_tm[4 * lane + 1], s_tm[4 * lane + 2], s_tm[4 * lane + 3]};
        bcut = min(255, leading(h, (uint32_t)top_k - 1));  // (the first bucket whose prefix reaches k)
    }
    // the statistics (chunk_stats_kernel's sums; top-k: only whether a NaN is there) and the histogram
    uint32_t bk[CR][4];
    bool in[CR][4];
#pragma unroll
    for (int r = 0; r < CR; r++) {
        float sw = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float x = z[r][e];
            float p = 0.f;
            if (x != x) sw = __builtin_nanf("");  // (flags the row even when m is -Inf)
            else if (!COUNT && m > -__builtin_huge_valf()) {
                p = pexp(x - m);
                sw += p;
            }
            bk[r][e] = zbin(x, m);
            in[r][e] = chunk_entry(r) + e < n && bk[r][e] <= bcut;
            if (in[r][e])
                atomicAdd(&s_h[wave][bk[r][e]],
                          COUNT ? 1ull
                                : ((unsigned long long)(uint32_t)__builtin_amdgcn_ldexpf(p, mass_exp(bk[r][e])) << CBITS) + 1ull);
        }
        sw = wave_sum(sw);
        if (lane == 0) s_red[CR * wave + r] = sw;
    }
    __syncthreads();
    unsigned long long hs = s_h[0][t];
#pragma unroll
    for (int w = 1; w < CNW; w++) hs += s_h[w][t];
    if (wave == 0) {
        const float sum = wave_sum(lane < SNW ? s_red[lane] : 0.f);
        if (lane == 0) ws.part[(size_t)row * ws.nround + c] = make_float2(m, sum);
    }
    s_tm[t] = (uint32_t)hs & ((1u << CBITS) - 1u);
    __syncthreads();
    const uint32_t h[4] = {s_tm[4 * lane], s_tm[4 * lane + 1], s_tm[4 * lane + 2], s_tm[4 * lane + 3]};
    int last = leading(h, ws.lmax) - 1;
    if (COUNT) {  // (the first bucket whose prefix reaches k ends both)
        bcut = min(bcut, (uint32_t)leading(h, (uint32_t)top_k - 1));
        last = min(last, (int)bcut);
        if ((uint32_t)t > bcut) hs = 0;
    }
    ((unsigned long long *)ws.slot(row, c))[t] = hs;
    // places in index order: (wave, group, lane, entry)
    int pos[CR], wn = 0;
#pragma unroll
    for (int r = 0; r < CR; r++) {
        int before = 0, all = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            in[r][e] = in[r][e] && (int)bk[r][e] <= last;
            const uint64_t mk = __ballot(in[r][e]);
            before += __builtin_amdgcn_mbcnt_hi((uint32_t)(mk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk, 0u));
            all += __popcll(mk);
        }
        pos[r] = wn + before;
        wn += all;
    }
    if (lane == 0) s_wn[wave] = wn;
    __syncthreads();
    int base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < CNW; w++) {
        base += w < wave ? s_wn[w] : 0;
        total += s_wn[w];
    }
    uint8_t *ls = ws.list(row, c);
    if (t == 0) {
        *(ListHead *)ls = ListHead{total, (int)bcut, m, 0};
        if (!COUNT && c == 0) ((RowSel *)ws.rowb(row))->arrived = 0;
    }
    float *lz = (float *)(ls + 16);
    uint16_t *li = (uint16_t *)(ls + 16 + 4 * ws.lmax);
#pragma unroll
    for (int r = 0; r < CR; r++) {
        int q = base + pos[r];
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (in[r][e]) {  // (total <= lmax)
                lz[q] = z[r][e];
                li[q] = (uint16_t)(chunk_entry(r) + e);
                q++;
            }
    }
}

// The gathers: entries lo <= z < hi that also(z, index) holds for, in index
// order, of the row's rounds c, round c's from place at(c) on: f(place, z,
// index). gather_lists takes them from the lists of the rounds need(c) holds
// for (the same in a wave), a wave a round, head and first entries in one
// load round. (64 entries after 64, after the head, a gather took 7 to 11 us,
// most of it latency; now 3 to 5. The lists of 2 or 3 rounds at a time are no
// faster: their code is longer, and one workgroup's time here is also that of
// fetching its code.) LONG: lists of more than LIST_MAX entries too.
constexpr int LE = (LIST_MAX + 63) / 64;
template <bool LONG, class N, class A, class K, class F>
__device__ __forceinline__ void gather_lists(const SpreadWs &ws, int row, float lo, float hi, N &&need, A &&at, K &&also,
                                             F &&f) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll 1
    for (int c = wave; c < ws.nround; c += SNW) {
        if (!need(c)) continue;
        const uint8_t *ls = ws.list(row, c);
        const float *lz = (const float *)(ls + 16);
        const uint16_t *li = (const uint16_t *)(ls + 16 + 4 * ws.lmax);
        const int nl = ((const ListHead *)ls)->n;
        uint32_t q = at(c);
        int n = 1;
#pragma unroll 1
        for (int i0 = 0; LONG ? i0 < n : i0 == 0; i0 += 64 * LE) {
            float z[LE];
            int j[LE];
#pragma unroll
            for (int e = 0; e < LE; e++) {  // (places past n: loaded, not used)
                const int i = min(i0 + 64 * e + lane, ws.lmax - 1);
                z[e] = lz[i];
                j[e] = li[i];
            }
            n = __builtin_amdgcn_readfirstlane(nl);
#pragma unroll
            for (int e = 0; e < LE; e++) {
                if (i0 + 64 * e >= n) break;
                const int id = c * SROUND + j[e];
                const bool k = i0 + 64 * e + lane < n && z[e] >= lo && z[e] < hi && also(z[e], id);
                const uint64_t m = __ballot(k);
                if (k)
                    f(q + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)), z[e],
                      id);
                q += __popcll(m);
            }
        }
    }
}

// gather_far reads the rounds whose bit is set in far (their lists end before
// the threshold's bucket) and that mine(c) holds for from the row, FB at a time by the whole workgroup,
// the next FB in flight, down to the round's cut (CUT): exactly the entries
// that its histogram counts. (Where the threshold's bucket is the row's last,
// 255, entries past the cut share that bucket, and each would take a place
// that the counts give to another round's.) s_w: 2 x 64 words. (A wave a
// round, one round of 4096 took 7 to 12 us; now 2.)
constexpr int FB = 4;
template <bool CUT, class M, class A, class K, class F>
__device__ __forceinline__ void gather_far(const SpreadWs &ws, int row, const float *__restrict__ Lr, int V, float invT,
                                           float lo, float hi, const uint32_t *far, uint32_t *s_w, M &&mine, A &&at,
                                           K &&also, F &&f) {
    static_assert(FB * SNW == 64, "a wave scans a batch's counts");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    auto next = [&](int c) {  // the first far round that is mine from c on (nround: none)
        while (c < ws.nround) {
            const uint32_t w = __builtin_amdgcn_readfirstlane(far[c >> 5]) >> (c & 31);
            if (w == 0u) {
                c = (c | 31) + 1;
                continue;
            }
            c += __ffs(w) - 1;
            if (mine(c)) return c;
            c++;
        }
        return ws.nround;
    };
    float x[FB][4], xl[FB];
    int xc[FB];
    auto load = [&](int c) {
#pragma unroll
        for (int b = 0; b < FB; b++) {
            xc[b] = c = next(c);
            xl[b] = lo;
            if (c >= ws.nround) continue;
            bool in;
            load_round(Lr, V, c, invT, x[b], in);
            if (CUT) {
                const ListHead hd = *(const ListHead *)ws.list(row, c);
                if (hd.cut < 255) xl[b] = fmaxf(lo, grid_lo(zq(hd.m) - hd.cut));
            }
            c++;
        }
    };
    load(0);
    for (int it = 0; xc[0] < ws.nround; it ^= 64) {
        float z[FB][4], lb[FB];
        int cb[FB];
#pragma unroll
        for (int b = 0; b < FB; b++) {
            cb[b] = xc[b];
            lb[b] = xl[b];
#pragma unroll
            for (int e = 0; e < 4; e++) z[b][e] = x[b][e];
        }
        load(cb[FB - 1] + 1);
        bool k[FB][4];
        uint32_t before[FB];
#pragma unroll
        for (int b = 0; b < FB; b++) {
            uint32_t all = 0;
            before[b] = 0;
            if (cb[b] < ws.nround) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int j = cb[b] * SROUND + 4 * (int)threadIdx.x + e;
                    k[b][e] = j < V && z[b][e] >= lb[b] && z[b][e] < hi && also(z[b][e], j);
                    const uint64_t m = __ballot(k[b][e]);
                    before[b] += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    all += __popcll(m);
                }
            }
            if (lane == 0) s_w[it + SNW * b + wave] = all;
        }
        __syncthreads();  // (the other half of s_w is free: every wave has passed its reads)
        const uint32_t v = s_w[it + lane];
        uint32_t inc = v;  // the scan within a round's 16 waves
        inc += __builtin_amdgcn_update_dpp(0, (int)inc, 0x111, 0xF, 0xF, true);
        inc += __builtin_amdgcn_update_dpp(0, (int)inc, 0x112, 0xF, 0xF, true);
        inc += __builtin_amdgcn_update_dpp(0, (int)inc, 0x114, 0xF, 0xF, true);
        inc += __builtin_amdgcn_update_dpp(0, (int)inc, 0x118, 0xF, 0xF, true);
#pragma unroll
        for (int b = 0; b < FB; b++) {
            if (cb[b] >= ws.nround) break;
            uint32_t q = at(cb[b]) + __builtin_amdgcn_readlane(inc - v, SNW * b + wave) + before[b];
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (k[b][e]) f(q++, z[b][e], cb[b] * SROUND + 4 * (int)threadIdx.x + e);
        }
    }
}

// Row blockIdx.x: its threshold and (draw) its token; otherwise the selection
// and the nucleus mass are left in the row's RowSel for a min-p after it. (A
// launch over the rounds for that mass: 5 us of 46 for one row.)
// SPLIT (top-p; grid y, 0: 1): every workgroup of a row finds the bucket by
// itself; where more than FB rounds' lists end before it, each takes the rounds
// c with c mod SPLIT = blockIdx.y into the row's workspace, and the last to
// arrive goes on with the bucket (no workgroup waits for another); everywhere
// else only the first goes on. The entries and the count cross XCDs through
// device-scope atomics, a wave's stores done before its workgroup counts in.
template <bool COUNT, int SPLIT>
__global__ __launch_bounds__(SNT) void row_threshold_kernel(const float *__restrict__ L, int V, float invT,
                                                            SampleArgs a, bool draw, SpreadWs ws,
                                                            const float *__restrict__ u, int32_t *__restrict__ out) {
    __shared__ float s_redf[2 * SNW];
    __shared__ uint32_t s_redu[SNW];
    __shared__ int s_redi[SNW];
    __shared__ uint32_t s_hist[256];
    __shared__ unsigned long long s_mass[256];
    __shared__ uint32_t s_sel[2];
    __shared__ unsigned long long s_selm[2];
    __shared__ int s_cnt;
    __shared__ unsigned long long s_cum[SMAX_ROUNDS];  // per round: the packed kept mass and count
    __shared__ uint32_t s_off[SMAX_ROUNDS];
    __shared__ uint32_t s_w[128];
    __shared__ uint32_t s_far[SMAX_ROUNDS / 32];  // rounds whose list ends before the threshold's bucket
    // the threshold bucket's keys, values and indices (top-k: the bucket's keys,
    // the values and indices of it and those above it); then (top-k) the sort
    // scratch, values and indices of the kept entries
    __shared__ uint32_t s_ck[SK_MAX];
    __shared__ float s_cz[COUNT ? 2 * SK_MAX : SK_MAX];
    __shared__ int s_ci[COUNT ? 2 * SK_MAX : SK_MAX];
    constexpr unsigned long long CMASK = (1ull << CBITS) - 1ull;
    const int row = blockIdx.x, t = threadIdx.x, wave = t >> 6, lane = t & 63, nround = ws.nround;
    const int g = SPLIT > 0 ? (int)blockIdx.y : 0;
    const float *Lr = L + (size_t)row * V;
    RowSel *rs = (RowSel *)ws.rowb(row);
    // the rounds' histograms, wave w those of rounds w, w + 16, ..: buckets
    // lane + 64 j of the round; the first HC of them stay in registers
    constexpr int HC = 4;
    unsigned long long hv[HC][4];
    auto load_hist = [&](int c, unsigned long long (&h)[4]) {
        const unsigned long long *p = (const unsigned long long *)ws.slot(row, c) + lane;
#pragma unroll
        for (int j = 0; j < 4; j++) h[j] = c < nround ? p[64 * j] : 0ull;
    };
#pragma unroll
    for (int i = 0; i < HC; i++) load_hist(wave + SNW * i, hv[i]);
    const float2 *pr = ws.part + (size_t)row * nround;
    const float ur = draw ? u[row] : 1.f;
    // the maxima of the rounds in hv, a round a lane
    const float ml = pr[min(wave + SNW * (lane & (HC - 1)), nround - 1)].x;
    float zmax, S;
    const bool ok = row_stats(pr, nround, zmax, S, COUNT);
    if (t < 256) {
        s_hist[t] = 0;
        s_mass[t] = 0;
    }
    if (t < SMAX_ROUNDS / 32) s_far[t] = 0;
    __syncthreads();
    if (!ok || ur != ur) {
        if (t == 0 && g == 0) {
            if (draw) out[row] = V - 1;
            else rs->mode = SEL_DEGEN;
        }
        return;
    }
    if (!(ur > 0.f)) {  // the reference's draw returns index 1 (here 0) when r <= 0
        if (t == 0 && g == 0) out[row] = 0;
        return;
    }
    const float invS = 1.0f / S;
    // a round of maximum m: its buckets' places in the row's count, and its
    // packed buckets with the mass in the row's 2^-40 (top-p; f: the round's
    // factor). (Shifts and factors of the rounds in hv: a round a lane.)
    const int zqm = zq(zmax);
    auto bucket_lo = [&](uint32_t b) { return b >= 255u ? -__builtin_huge_valf() : grid_lo(zqm - (int)b); };
    auto row_bucket = [&](int b, int sh) { return (uint32_t)min(b + min(sh, 255), 255); };
    auto factor = [&](float m) { return COUNT ? 0.0 : exp((double)m - (double)zmax) / (double)S; };
    auto to_row = [&](double f, unsigned long long (&h)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            h[j] = ((unsigned long long)__builtin_ldexp((double)(h[j] >> CBITS) * f, 40 - mass_exp(lane + 64 * j)) << CBITS) |
                   (h[j] & CMASK);
    };
    const int shl = zqm - zq(ml);
    const unsigned long long fl = __builtin_bit_cast(unsigned long long, factor(ml));
#pragma unroll
    for (int i = 0; i < HC; i++) {
        if (COUNT || wave + SNW * i >= nround) break;
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)fl, i);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(fl >> 32), i);
        to_row(__builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo), hv[i]);
    }
    // f(round, its shift, its buckets) over this wave's rounds
    auto rounds = [&](auto &&f) {
#pragma unroll
        for (int i = 0; i < HC; i++)
            if (wave + SNW * i < nround) f(wave + SNW * i, __builtin_amdgcn_readlane(shl, i), hv[i]);
#pragma unroll 1
        for (int c = wave + SNW * HC; c < nround; c += SNW) {
            unsigned long long h[4];
            load_hist(c, h);
            const float m = pr[c].x;
            if (!COUNT) to_row(factor(m), h);
            f(c, zqm - zq(m), h);
        }
    };
    rounds([&](int, int sh, const unsigned long long (&h)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if ((h[j] & CMASK) != 0) {
                const uint32_t b = row_bucket(lane + 64 * j, sh);
                atomicAdd(&s_hist[b], (uint32_t)(h[j] & CMASK));
                if (!COUNT) atomicAdd(&s_mass[b], h[j] >> CBITS);
            }
    });
    __syncthreads();
    const float tp = fmaxf(a.top_p, 0.f) * 1099511627776.0f;
    const unsigned long long target =
        COUNT ? (unsigned long long)a.top_k : tp < 1.0f ? 1ull : (unsigned long long)ceilf(tp);
    if (draw && nround <= 64) {
        // At most 64 entries up to the threshold's bucket (a top-k of tens, a
        // peaked row's nucleus): they are gathered in index order and one
        // wave ranks, keeps and draws. (Every wave finds the bucket by itself.)
        const uint32_t h[4] = {s_hist[4 * lane], s_hist[4 * lane + 1], s_hist[4 * lane + 2], s_hist[4 * lane + 3]};
        uint32_t cc[4], cr = 0;
        unsigned long long mc[4], mr = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            cr += h[j];
            cc[j] = cr;
            mr += COUNT ? (unsigned long long)h[j] : s_mass[4 * lane + j];
            mc[j] = mr;
        }
        const uint32_t ex = wave_scan_u(cr) - cr;
        unsigned long long mex = 0;
        if (COUNT) {
            mex = ex;
        } else {
            mex = mr;
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned long long y = __shfl_up(mex, o);
                if (lane >= o) mex += y;
            }
            mex -= mr;
        }
        const uint64_t hit = __ballot(mex < target && target <= mex + mr);
        if (hit != 0ull) {
            const int f = __ffsll((unsigned long long)hit) - 1;
            const int j = mex + mc[0] >= target ? 0 : mex + mc[1] >= target ? 1 : mex + mc[2] >= target ? 2 : 3;
            const uint32_t nle = __builtin_amdgcn_readlane(ex + (j == 0 ? cc[0] : j == 1 ? cc[1] : j == 2 ? cc[2] : cc[3]), f);
            const uint32_t zb = 4 * f + __builtin_amdgcn_readlane(j, f);
            if (nle <= 64u) {
                if (SPLIT > 0 && g != 0) return;
                rounds([&](int c, int sh, const unsigned long long (&x)[4]) {
                    uint32_t v = 0;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (row_bucket(lane + 64 * i, sh) <= zb) v += (uint32_t)x[i] & (uint32_t)CMASK;
                    v = wave_sum_u(v);
                    if (lane == 0) s_off[c] = v;
                });
                __syncthreads();
                const uint32_t n = lane < nround ? s_off[lane] : 0u, off = wave_scan_u(n) - n;
                gather_lists<false>(  // (at most 64 entries a round: every list reaches; top-k <= 64: none is long)
                    ws, row, bucket_lo(zb), __builtin_huge_valf(), [&](int c) { return __builtin_amdgcn_readlane(n, c) != 0; },
                    [&](int c) { return (uint32_t)__builtin_amdgcn_readlane(off, c); }, [&](float, int) { return true; },
                    [&](uint32_t p, float z, int id) {
                        s_cz[p & 63u] = z;  // (p < nle)
                        s_ci[p & 63u] = id;
                    });
                __syncthreads();
                if (wave != 0) return;
                const bool in = (uint32_t)lane < nle;
                const float z = in ? s_cz[lane] : 0.f;
                const int id = in ? s_ci[lane] : 0;
                const uint32_t key = in ? okey(z) : 0u;
                // the units (entries, or mass) ahead of this entry: larger
                // keys, and equal ones before it (slots are in index order);
                // kept while they are short of the target
                const unsigned long long mine = COUNT ? 1ull : mass_fx(z, zmax, invS);
                unsigned long long ahead = 0;
                for (uint32_t i = 0; i < nle; i++) {
                    const uint32_t ki = __builtin_amdgcn_readlane(key, i);
                    const uint32_t mhi = __builtin_amdgcn_readlane((uint32_t)(mine >> 32), i);  // (int: not widened as is)
                    const uint32_t mlo = __builtin_amdgcn_readlane((uint32_t)mine, i);
                    const unsigned long long mi = ((unsigned long long)mhi << 32) | mlo;
                    if (ki > key || (ki == key && i < (uint32_t)lane)) ahead += mi;
                }
                const bool keep = in && ahead < target;
                if constexpr (COUNT) {
                    const uint64_t km = __ballot(keep);
                    const uint32_t p = __builtin_amdgcn_mbcnt_hi((uint32_t)(km >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)km, 0u));
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    if (keep) {
                        s_cz[p] = z;
                        s_ci[p] = id;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    draw_candidates_wave(__popcll(km), a, ur, V, s_ci, s_cz, (int *)s_ck, out + row);
                } else {
                    unsigned long long cum = keep ? mine : 0ull;
                    for (int o = 1; o < 64; o <<= 1) {
                        const unsigned long long y = __shfl_up(cum, o);
                        if (lane >= o) cum += y;
                    }
                    const double goal = (double)ur * (double)__shfl(cum, 63);
                    const uint64_t got = __ballot(keep && goal <= (double)cum);
                    const int g = got ? __ffsll((unsigned long long)got) - 1 : 0;
                    const int tok = __shfl(id, g);
                    if (lane == 0) out[row] = got ? tok : V - 1;  // (none: u above 1)
                }
                return;
            }
        }
    }
    pick_bucket<!COUNT>(s_hist, s_mass, target, s_sel, s_selm, false);
    __syncthreads();
    Select R;
    R.all = s_selm[0] == ~0ull;
    R.zb = R.all ? 256u : s_sel[0];
    R.rem = R.all ? 0ull : target - s_selm[0];
    R.tau = 0u;
    R.cnt = 0;
    const int nzb = R.all ? 0 : (int)s_hist[R.zb];
    const bool gathered = nzb <= SK_MAX;
    const uint32_t zb = R.zb;
    const bool upto = COUNT && gathered && !R.all;
    // per round: the packed sum of the buckets above zb, and zb's count (upto:
    // theirs together)
    rounds([&](int c, int sh, const unsigned long long (&h)[4]) {
        unsigned long long v = 0;
        uint32_t q = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t b = row_bucket(lane + 64 * j, sh);
            if (b < zb) v += h[j];
            if (b == zb) q += (uint32_t)h[j] & (uint32_t)CMASK;
        }
        v = COUNT ? wave_sum_u((uint32_t)v) : wave_sum_u64(v);
        q = wave_sum_u(q);
        if (lane == 0) {
            s_cum[c] = v;
            s_off[c] = upto ? (uint32_t)v + q : q;
            if ((v & CMASK) + q > (unsigned long long)ws.lmax) atomicOr(&s_far[c >> 5], 1u << (c & 31));
        }
    });
    __syncthreads();
    bool split = false;
    if (SPLIT > 0) {
        if (gathered && !R.all) split = wave_sum_u64(lane < SMAX_ROUNDS / 32 ? __popc(s_far[lane]) : 0) > (unsigned long long)FB;
        if (!split && g != 0) return;
    }
    // from the bucket's lower bound to hi, each round at its s_off
    auto gather = [&](float hi, auto &&need, auto &&also, auto &&f) {
        auto at = [&](int c) { return s_off[c]; };
        auto mine = [&](int c) { return SPLIT == 0 || !split || (c & (SPLIT - 1)) == g; };
        gather_lists<COUNT>(ws, row, bucket_lo(zb), hi,
                            [&](int c) { return ((s_far[c >> 5] >> (c & 31)) & 1u) == 0u && need(c) && mine(c); }, at, also,
                            f);
        gather_far<COUNT>(ws, row, Lr, V, invT, bucket_lo(zb), hi, s_far, s_w, mine, at, also, f);
    };
    if (COUNT && upto) {
        // The entries up to the threshold's bucket (fewer than k above it, at
        // most SK_MAX in it) gathered once, in index order; the threshold among
        // the bucket's; then the candidates closed up in place. (A gather of
        // the bucket and another of the candidates: one row of 151936 at top-k
        // 200 27.9 us and 1000 31.5, 24.8 and 27.2 so.)
        constexpr int PT = 2 * SK_MAX / SNT;
        const int nle = (int)(target - R.rem) + nzb;
        const float hi = grid_lo(zqm - (int)zb + 1);
        uint32_t tot;
        const uint32_t off = block_excl_scan_u(t < nround ? s_off[t] : 0u, s_redu, tot);  // (nround <= SNT)
        if (t < nround) s_off[t] = off;
        if (t == 0) s_cnt = 0;
        __syncthreads();
        gather(
            __builtin_huge_valf(), [&](int c) { return c + 1 < nround ? s_off[c + 1] > s_off[c] : tot > s_off[c]; },
            [&](float, int) { return true; },
            [&](uint32_t p, float z, int j) {
                if (p < 2u * SK_MAX) {  // (p < nle: the entries chunk_hist_kernel counted)
                    s_cz[p] = z;
                    s_ci[p] = j;
                }
            });
        __syncthreads();
        for (int i = t; i < nle; i += SNT)
            if (s_cz[i] < hi) s_ck[atomicAdd(&s_cnt, 1)] = okey(s_cz[i]);  // (nzb of them)
        __syncthreads();
        refine_threshold<false>(Lr, V, nround, invT, zmax, 1.f, true, nzb, s_hist, s_mass, s_sel, s_selm, s_ck, s_cz, R);
        const uint32_t rem = (uint32_t)R.rem;  // elements equal to tau that are kept, lowest index first
        float z[PT];
        int id[PT];
        bool gt[PT], eq[PT];
        uint32_t ng = 0, nq = 0;
#pragma unroll
        for (int e = 0; e < PT; e++) {
            const int j = PT * t + e;
            const bool in = j < nle;
            z[e] = in ? s_cz[j] : 0.f;
            id[e] = in ? s_ci[j] : 0;
            const uint32_t k = okey(z[e]);  // (a bucket above zb has the larger keys)
            gt[e] = in && k > R.tau;
            eq[e] = in && k == R.tau;
            ng += gt[e];
            nq += eq[e];
        }
        const uint32_t ex = block_excl_scan_u(ng | (nq << 16), s_redu, tot);
        uint32_t er = ex >> 16, pos = (ex & 0xffffu) + min(rem, er);
#pragma unroll
        for (int e = 0; e < PT; e++) {
            if (gt[e] || (eq[e] && er < rem)) {
                s_cz[pos] = z[e];
                s_ci[pos] = id[e];
                pos++;
            }
            er += eq[e];
        }
        __syncthreads();
        draw_candidates((int)(tot & 0xffffu) + (int)min(rem, tot >> 16), a, ur, V, s_ci, s_cz, (int *)s_ck, s_redf, s_redi,
                        out + row);
        return;
    }
    int tie_lim = V, npart = -1;  // (npart >= 0: the threshold's part of the bucket is what was gathered)
    if (!R.all) {
        if (!COUNT && gathered) {
            uint32_t tot;
            const uint32_t cnt = t < nround ? s_off[t] : 0u;  // (nround <= SNT)
            const uint32_t off = block_excl_scan_u(cnt, s_redu, tot);
            if (t < nround) s_off[t] = off;
            __syncthreads();
            unsigned long long *gp = (unsigned long long *)(ws.rowb(row) + ROW_PART);
            auto keep1 = [&](uint32_t p, float z, int j) {
                s_ck[p] = okey(z);
                s_cz[p] = z;
                s_ci[p] = j;
            };
            gather(
                grid_lo(zqm - (int)zb + 1),
                [&](int c) { return c + 1 < nround ? s_off[c + 1] > s_off[c] : tot > s_off[c]; },
                [&](float, int) { return true; },
                [&](uint32_t p, float z, int j) {
                    if (p >= (uint32_t)SK_MAX) return;  // (p < nzb: the entries chunk_hist_kernel counted)
                    if (SPLIT > 0 && split)
                        __hip_atomic_store(gp + p, ((unsigned long long)(uint32_t)j << 32) | __float_as_uint(z), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    else
                        keep1(p, z, j);
                });
            if (SPLIT > 0 && split) {
                wait_stores_done();
                __syncthreads();
                if (t == 0)
                    s_cnt = (int)__hip_atomic_fetch_add(&rs->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __syncthreads();
                if (s_cnt != SPLIT - 1) return;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                for (int i = t; i < nzb; i += SNT) {
                    const unsigned long long v = __hip_atomic_load(gp + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    keep1(i, __uint_as_float((uint32_t)v), (int)(v >> 32));
                }
            }
            __syncthreads();
        } else if (!COUNT && zb < 255u) {
            // A flat row: the bucket's 256 parts in one pass, then the
            // threshold's part is gathered (in any order) in a second one,
            // in which the parts above it join their rounds' sums. (Key
            // passes over the row, 4 and one for the sums: 64 rows of
            // V = 151936 at sd 1, top-p 0.9: 191 us, 107 so. A top-k's
            // flat rows keep the key passes: this code cost its other rows 2 us.)
            if (t < 256) {
                s_hist[t] = 0;
                s_mass[t] = 0;
            }
            if (t == 0) s_cnt = 0;
            __syncthreads();
            const float lo = bucket_lo(zb), hi = grid_lo(zqm - (int)zb + 1);
            for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int) {
                bool q[4];
                uint32_t b[4];
                unsigned long long m[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    q[e] = in && z[e] >= lo && z[e] < hi;
                    b[e] = zpart(z[e]);
                    m[e] = q[e] ? mass_fx(z[e], zmax, invS) : 0ull;
                }
                hist_add4<true>(s_hist, s_mass, q, b, m);
            });
            __syncthreads();
            pick_bucket<true>(s_hist, s_mass, R.rem, s_sel, s_selm, true);
            __syncthreads();
            const uint32_t part = s_sel[0];
            const unsigned long long above = s_selm[0];
            if (above != ~0ull && s_hist[part] <= (uint32_t)SK_MAX) {  // (uniform)
                npart = (int)s_hist[part];
                R.rem -= above;
                unsigned long long vt = 0;
                for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
                    unsigned long long v = 0;
                    if (in)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (z[e] >= lo && z[e] < hi) {
                                const uint32_t b = zpart(z[e]);
                                if (b > part) v += (mass_fx(z[e], zmax, invS) << CBITS) + 1ull;
                                if (b == part) {
                                    const int p = atomicAdd(&s_cnt, 1);  // (p < npart: the predicate counted above)
                                    s_ck[p] = okey(z[e]);
                                    s_cz[p] = z[e];
                                    s_ci[p] = r * SROUND + 4 * t + e;
                                }
                            }
                    if (!draw) {  // (the row's sum alone is asked for)
                        vt += v >> CBITS;
                        return;
                    }
                    v = wave_sum_u64(v);
                    if (lane == 0 && v) atomicAdd(&s_cum[r], v);
                });
                vt = wave_sum_u64(vt);
                if (lane == 0 && vt) atomicAdd(&s_cum[0], vt << CBITS);
            }
            __syncthreads();
        }
        Select Q = R;  // (a copy: R, captured above, stays in registers)
        refine_threshold<!COUNT>(Lr, V, nround, invT, zmax, COUNT ? 1.f : S, !COUNT && (gathered || npart >= 0),
                                 !COUNT && gathered ? nzb : npart, s_hist, s_mass, s_sel, s_selm, s_ck, s_cz, Q);
        R = Q;
        if (R.all) {  // (the entries' masses a rounding short of the rounds': the whole bucket is kept)
            R.all = false;
            R.tau = 0u;
            R.cnt = 0;
            R.rem = 1;
        }
    }
    if (!R.all) {
        // ties at tau share one probability: keep the first n_eq of them
        unsigned long long n_eq = R.rem;
        if (!COUNT) {
            const float ptau = pexp(okey_inv(R.tau) - zmax) * (1.0f / S);
            const unsigned long long mt = (unsigned long long)(ptau * 1099511627776.0f);
            n_eq = mt ? (R.rem + mt - 1) / mt : (unsigned long long)R.cnt;
        }
        if (n_eq < 1) n_eq = 1;
        const uint32_t tau = R.tau;
        if (n_eq < R.cnt) {
            if (!COUNT && gathered) {  // the gather is in index order: slots 4 t .. 4 t + 3
                bool q[4];
                uint32_t nq = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int j = 4 * t + e;
                    q[e] = j < nzb && s_ck[j] == tau;
                    nq += q[e];
                }
                uint32_t tot;
                int cnum = (int)block_excl_scan_u(nq, s_redu, tot);
                int cand = INT_MAX;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (q[e]) {
                        cnum++;
                        if (cnum == (int)n_eq && cand == INT_MAX) cand = s_ci[4 * t + e] + 1;
                    }
                tie_lim = block_min_i(cand, s_redi);
            } else {
                int run = 0, lim = V;
                for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
                    bool q[4];
                    uint32_t nq = 0;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        q[e] = in && zbin(z[e], zmax) == zb && okey(z[e]) == tau;
                        nq += q[e];
                    }
                    uint32_t tot;
                    const uint32_t ex = block_excl_scan_u(nq, s_redu, tot);
                    int cand = INT_MAX;
                    int cc = run + (int)ex;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (q[e]) {
                            cc++;
                            if (cc == (int)n_eq && cand == INT_MAX) cand = r * SROUND + 4 * t + e + 1;
                        }
                    const int got = block_min_i(cand, s_redi);
                    if (lim == V && got != INT_MAX) lim = got;
                    run += (int)tot;
                });
                tie_lim = lim;
            }
        }
    }
    const bool all = R.all;
    const uint32_t tau = R.tau;
    // the kept entries of the threshold's bucket join their rounds' sums
    if (!all) {
        auto units = [&](float z, uint32_t k, int j) {
            return k > tau || (k == tau && j < tie_lim) ? COUNT ? 1ull : (mass_fx(z, zmax, invS) << CBITS) + 1ull : 0ull;
        };
        if (!COUNT && (gathered || npart >= 0)) {
            for (int i = t; i < (gathered ? nzb : npart); i += SNT) {
                const unsigned long long v = units(s_cz[i], s_ck[i], s_ci[i]);
                if (v) atomicAdd(&s_cum[s_ci[i] / SROUND], v);
            }
        } else {
            for_rounds(Lr, V, nround, invT, [&](const float (&z)[4], bool in, int r) {
                unsigned long long v = 0;
                if (in)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (zbin(z[e], zmax) == zb) v += units(z[e], okey(z[e]), r * SROUND + 4 * t + e);
                v = wave_sum_u64(v);
                if (lane == 0 && v) atomicAdd(&s_cum[r], v);
            });
        }
    }
    __syncthreads();
    if constexpr (COUNT) {
        uint32_t n;
        const uint32_t cnt = t < nround ? (uint32_t)(s_cum[t] & CMASK) : 0u;
        const uint32_t off = block_excl_scan_u(cnt, s_redu, n);
        for (int i = t; i < nround; i += SNT) s_off[i] = off;
        __syncthreads();  // (and the gathered bucket is no longer read)
        gather(
            __builtin_huge_valf(), [&](int c) { return (s_cum[c] & CMASK) != 0; },
            [&](float z, int j) {  // (a bucket above zb has the larger keys)
                const uint32_t k = okey(z);
                return k > tau || (k == tau && j < tie_lim);
            },
            [&](uint32_t p, float z, int j) {
                if (p < (uint32_t)SK_MAX) {
                    s_cz[p] = z;
                    s_ci[p] = j;
                }
            });
        __syncthreads();
        draw_candidates(min((int)n, SK_MAX), a, ur, V, s_ci, s_cz, (int *)s_ck, s_redf, s_redi, out + row);
        return;
    }
    // top-p: the round holding u of the kept mass (every wave by itself, 64
    // rounds at a time), then the entry inside it
    auto cum64 = [&](int b, unsigned long long carry) {
        unsigned long long inc = b + lane < nround ? s_cum[b + lane] >> CBITS : 0ull;
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long y = __shfl_up(inc, o);
            if (lane >= o) inc += y;
        }
        return carry + inc;
    };
    unsigned long long total = 0;
    for (int b = 0; b < nround; b += 64) total = __shfl(cum64(b, total), 63);
    if (!draw) {
        if (t == 0) {
            rs->mode = all ? SEL_ALL : SEL_SELECT;
            rs->zmax = zmax;
            rs->S = S;
            rs->zb = zb;
            rs->tau = tau;
            rs->tie_lim = tie_lim;
            rs->inv1 = total > 0 ? (float)(1099511627776.0 / (double)total) : 1.0f;
        }
        return;
    }
    const double goal = (double)ur * (double)total;
    unsigned long long below = 0;
    int rr = -1;
    for (int b = 0; b < nround && rr < 0; b += 64) {
        const unsigned long long cum = cum64(b, below);
        const uint64_t m = __ballot(b + lane < nround && goal <= (double)cum);
        const int f = m ? __ffsll((unsigned long long)m) - 1 : 64;
        if (f > 0) below = __shfl(cum, f - 1);
        if (f < 64) rr = b + f;
    }
    if (rr < 0) {  // (u above 1)
        if (t == 0) out[row] = V - 1;
        return;
    }
    const float inv = total > 0 ? (float)(1099511627776.0 / (double)total) : 1.0f;
    const float before = (float)((double)below * (total > 0 ? 1.0 / (double)total : 0.0));
    float z[4], v[4];
    bool in;
    load_round(Lr, V, rr, invT, z, in);
#pragma unroll
    for (int e = 0; e < 4; e++)
        v[e] = in && (all || above_threshold(z[e], rr * SROUND + 4 * t + e, zmax, zb, tau, tie_lim))
                   ? pexp(z[e] - zmax) * invS * inv
                   : 0.f;
    float tot;
    const int hit = first_cdf_hit(v, in ? 4 : 0, before, ur, s_redf, tot);
    const int local = block_min_i(hit, s_redi);
    // (the scan inside the round can end a rounding step below the mass that
    // selected it: then the round's last kept entry)
    int last = INT_MAX;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (v[e] > 0.f) last = INT_MAX - (4 * t + e);
    const int lastk = block_min_i(last, s_redi);
    if (t == 0) {
        const int tok =
            local != INT_MAX ? rr * SROUND + local : lastk != INT_MAX ? rr * SROUND + (INT_MAX - lastk) : V - 1;
        out[row] = min(tok, V - 1);
    }
}

// An entry's probability through the cuts of a min-p draw: p = exp(z - zmax)
// / S; after top-p 0 for what its selection drops, else divided by the nucleus
// mass (inv1 = 1 / it; 1 without top-p); 0 below thr = inv1 / S * min_p (the
// largest probability times min_p).
struct Keep {
    bool topp, all;
    uint32_t zb, tau;
    int tie_lim;
    float zmax, invS, inv1, thr;
    __device__ float p1(float z, int j) const {
        if (topp && !(all || above_threshold(z, j, zmax, zb, tau, tie_lim))) return 0.f;
        float p = pexp(z - zmax) * invS;
        if (topp) p = p * inv1;
        return p < thr ? 0.f : p;
    }
};

// 1 / the sum of the row's chunk values at SLOT_CSUM of their slots (a fixed
// order, as row_stats), or 1 when it is not positive.
__device__ float kept_inv(const SpreadWs &ws, int row) {
    const int l = threadIdx.x & 63;
    float acc = 0.f;
    for (int v = 0; 64 * v < ws.nround; v++) {
        const int i = 64 * v + l;
        const float sv = wave_sum(i < ws.nround ? *(const float *)(ws.slot(row, i) + SLOT_CSUM) : 0.f);
        if (l == v) acc = sv;
    }
    const float total = wave_sum(acc);
    return total > 0.f ? 1.0f / total : 1.0f;
}

// The row's statistics (after top-p those row_threshold_kernel stored) and
// cuts; false for a row without finite ones (no draw).
__device__ __forceinline__ bool load_keep(const SpreadWs &ws, int row, bool topp, float min_p, Keep &k) {
    float S;
    k.topp = topp;
    if (topp) {
        const RowSel *rs = (const RowSel *)ws.rowb(row);
        if (rs->mode == SEL_DEGEN) return false;
        k.zmax = rs->zmax;
        S = rs->S;
        k.all = rs->mode == SEL_ALL;
        k.zb = rs->zb;
        k.tau = rs->tau;
        k.tie_lim = rs->tie_lim;
        k.inv1 = rs->inv1;
    } else {
        if (!row_stats(ws.part + (size_t)row * ws.nround, ws.nround, k.zmax, S)) return false;
        k.all = false;
        k.zb = 256u;
        k.tau = 0u;
        k.tie_lim = 0;
        k.inv1 = 1.0f;
    }
    k.invS = 1.0f / S;
    k.thr = k.invS * k.inv1 * min_p;
    return true;
}

// Chunk blockIdx.x of row blockIdx.y: the sum of its kept probabilities at
// SLOT_CSUM.
__global__ __launch_bounds__(CNT) void chunk_keptsum_kernel(const float *__restrict__ L, int V, float invT, bool topp,
                                                            float min_p, SpreadWs ws) {
    __shared__ float s_red[SNW];
    const int c = blockIdx.x, row = blockIdx.y, t = threadIdx.x;
    float z[CR][4];
    load_chunk(L + (size_t)row * V, V, c, invT, z);
    Keep keep;
    if (!load_keep(ws, row, topp, min_p, keep)) return;
    float sum[CR];
#pragma unroll
    for (int r = 0; r < CR; r++) {
        sum[r] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) sum[r] += keep.p1(z[r][e], c * SROUND + chunk_entry(r) + e);
    }
    const float total = chunk_sum(sum, s_red);
    if (t == 0) *(float *)(ws.slot(row, c) + SLOT_CSUM) = total;
}

// Row blockIdx.x: the kept mass, each round's share of it, the round holding
// u, then the index inside it (as chunk_draw_kernel over the kept entries).
__global__ __launch_bounds__(SNT) void keep_draw_kernel(const float *__restrict__ L, int V, float invT, bool topp,
                                                        float min_p, SpreadWs ws, const float *__restrict__ u,
                                                        int32_t *__restrict__ out) {
    __shared__ float s_redf[2 * SNW];
    __shared__ int s_redi[SNW];
    __shared__ float s_round[SMAX_ROUNDS];
    __shared__ float s_before;
    __shared__ int s_rr;
    const int row = blockIdx.x, t = threadIdx.x, nround = ws.nround;
    const float ur = u[row];
    Keep keep;
    if (!load_keep(ws, row, topp, min_p, keep) || ur != ur) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    if (!(ur > 0.f)) {  // the reference's draw returns index 1 (here 0) when r <= 0
        if (t == 0) out[row] = 0;
        return;
    }
    const float inv = kept_inv(ws, row);
    for (int i = t; i < nround; i += SNT) s_round[i] = *(const float *)(ws.slot(row, i) + SLOT_CSUM) * inv;
    __syncthreads();
    if (t == 0) {
        float cum = 0.f;
        int rr = -1;
        for (int r = 0; r < nround; r++) {
            const float nc = cum + s_round[r];
            if (ur <= nc) {
                rr = r;
                break;
            }
            cum = nc;
        }
        s_rr = rr;
        s_before = cum;
    }
    __syncthreads();
    const int rr = s_rr;
    const float before = s_before;
    if (rr < 0) {
        if (t == 0) out[row] = V - 1;
        return;
    }
    float z[4], v[4];
    bool in;
    load_round(L + (size_t)row * V, V, rr, invT, z, in);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = in ? keep.p1(z[e], rr * SROUND + 4 * t + e) * inv : 0.f;
    float tot;
    const int hit = first_cdf_hit(v, in ? 4 : 0, before, ur, s_redf, tot);
    const int local = block_min_i(hit, s_redi);
    int last = INT_MAX;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (v[e] > 0.f) last = INT_MAX - (4 * t + e);
    const int lastk = block_min_i(last, s_redi);
    if (t == 0) {
        const int tok =
            local != INT_MAX ? rr * SROUND + local : lastk != INT_MAX ? rr * SROUND + (INT_MAX - lastk) : V - 1;
        out[row] = min(tok, V - 1);
    }
}

// In place on rows of logits: for every distinct id of the row's list in
// [0, V): x -= presence (if presence != 0), then x = x > 0 ? x / rep : x * rep
// (if rep != 1). A bitmap in LDS skips repeated ids; it covers a window of
// PEN_WINDOW ids, and a vocabulary past that is taken window by window
// (each reads the row's list once).
constexpr int PEN_NT = 256;
constexpr int PEN_WINDOW = 262144;
__global__ __launch_bounds__(PEN_NT) void penalty_kernel(float *__restrict__ L, int V, const int32_t *__restrict__ tok,
                                                          int n_tok, int64_t tok_stride, float presence,
                                                          float repetition) {
    __shared__ uint32_t seen[PEN_WINDOW / 32];
    const int row = blockIdx.x, t = threadIdx.x;
    const int32_t *ids = tok + (size_t)row * tok_stride;
    float *x = L + (size_t)row * V;
    for (int w0 = 0; w0 < V; w0 += PEN_WINDOW) {
        const int wn = min(PEN_WINDOW, V - w0);
        const int nw = (wn + 31) / 32;
        __syncthreads();  // (the previous window's bitmap is no longer read)
        for (int i = t; i < nw; i += PEN_NT) seen[i] = 0u;
        __syncthreads();
        for (int i = t; i < n_tok; i += PEN_NT) {
            const int id = ids[i] - w0;
            if (id < 0 || id >= wn) continue;
            const uint32_t bit = 1u << (id & 31);
            if (atomicOr(&seen[id >> 5], bit) & bit) continue;
            float v = x[w0 + id];
            if (presence != 0.f) v -= presence;
            if (repetition != 1.0f) v = v > 0.f ? v / repetition : v * repetition;
            x[w0 + id] = v;
        }
    }
}

}  // namespace

int sample_max_v() { return SMAX_ROUNDS * SROUND; }

hipError_t launch_sample(const float *L, int rows, int V, float T, int top_k, float top_p, float min_p, const float *u,
                         int32_t *out, hipStream_t st) {
    const SampleArgs a{T, top_k, top_p, min_p};
    draft_sample_kernel<<<rows, SNT, 0, st>>>(L, V, a, u, out);
    return hipGetLastError();
}

// A top-p's rows have 16 or 8 workgroups each while those of all rows are at
// most as many as there are CUs. V = 151936, top-p 0.9, by 1 workgroup and so:
// Gaussian sd 2 (38 rounds past their lists) 1 row 68.4 and 43.7 us, 16 rows
// 73.0 and 47.5, 32 rows 77.7 and 58.8; a language model's logits (no round past
// its list) 14.5 and 14.6, 19.0 and 19.2, 21.0 and 21.4 (by 16: 27.5).
constexpr int SPLIT_CU = 256;

size_t sample_spread_ws(int rows, int V) {
    const size_t rc = (size_t)rows * ((V + SROUND - 1) / SROUND);
    return rc * (sizeof(float2) + SLOT_BYTES) + (size_t)rows * ROW_BYTES;
}

// Rows spread over workgroups of one round each: plain draws (T > 0, no top-k,
// top-p or min-p): chunk statistics, then one workgroup per row merges them,
// picks the round and scans it (as draft_sample_kernel's draw); top-k up to
// SK_MAX (any top-p / min-p after it) and top-p: histograms and candidate
// lists, then the threshold and the draw per row; min-p, alone or after top-p:
// the chunks' kept sums, then the draw; T = 0: each chunk's argmax, then the
// row's. Rows over more than
// SMAX_ROUNDS rounds, and a larger top-k, run draft_sample_kernel.
// ws: sample_spread_ws bytes (8-byte aligned).
hipError_t launch_sample_spread(const float *L, int rows, int V, float T, int top_k, float top_p, float min_p,
                                const float *u, int32_t *out, void *ws, hipStream_t st) {
    const int nround = (V + SROUND - 1) / SROUND;
    if (T == 0.f && nround <= SMAX_ROUNDS) {
        float2 *part = (float2 *)ws;
        chunk_argmax_kernel<<<dim3(nround, rows), CNT, 0, st>>>(L, V, part);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        argmax_draw_kernel<<<rows, SNT, 0, st>>>(V, part, out);
        return hipGetLastError();
    }
    if (!(T > 0.f) || nround > SMAX_ROUNDS || top_k > SK_MAX)
        return launch_sample(L, rows, V, T, top_k, top_p, min_p, u, out, st);
    const bool topk = top_k > 0, topp = !topk && top_p < 1.0f, minp = !topk && min_p > 0.f;
    const float invT = 1.0f / T;
    const size_t rc = (size_t)rows * nround;
    uint8_t *w = (uint8_t *)ws;
    const SpreadWs W{(float2 *)w, w + rc * sizeof(float2), w + rc * (sizeof(float2) + SLOT_BYTES), nround, list_max(nround, topk ? top_k : 0)};
    const dim3 chunks(nround, rows);
    const SampleArgs a{T, top_k, top_p, min_p};
    hipError_t e;
    if (topk) {
        chunk_hist_kernel<true><<<chunks, CNT, 0, st>>>(L, V, invT, top_k, W);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        row_threshold_kernel<true, 0><<<rows, SNT, 0, st>>>(L, V, invT, a, true, W, u, out);
        return hipGetLastError();
    }
    if (topp) {
        chunk_hist_kernel<false><<<chunks, CNT, 0, st>>>(L, V, invT, 0, W);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (rows <= SPLIT_CU / 16)
            row_threshold_kernel<false, 16><<<dim3(rows, 16), SNT, 0, st>>>(L, V, invT, a, !minp, W, u, out);
        else if (rows <= SPLIT_CU / 8)
            row_threshold_kernel<false, 8><<<dim3(rows, 8), SNT, 0, st>>>(L, V, invT, a, !minp, W, u, out);
        else
            row_threshold_kernel<false, 0><<<rows, SNT, 0, st>>>(L, V, invT, a, !minp, W, u, out);
        if ((e = hipGetLastError()) != hipSuccess || !minp) return e;
    } else {
        chunk_stats_kernel<<<chunks, CNT, 0, st>>>(L, V, invT, W.part);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (!topp && !minp) {
        chunk_draw_kernel<<<rows, SNT, 0, st>>>(L, V, invT, W.part, u, out);
        return hipGetLastError();
    }
    chunk_keptsum_kernel<<<chunks, CNT, 0, st>>>(L, V, invT, topp, min_p, W);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    keep_draw_kernel<<<rows, SNT, 0, st>>>(L, V, invT, topp, min_p, W, u, out);
    return hipGetLastError();
}

hipError_t launch_penalties(float *L, int rows, int V, const int32_t *tok, int n_tok, int64_t tok_stride,
                            float presence, float repetition, hipStream_t st) {
    if (n_tok == 0 || (presence == 0.f && repetition == 1.0f)) return hipSuccess;
    penalty_kernel<<<rows, PEN_NT, 0, st>>>(L, V, tok, n_tok, tok_stride, presence, repetition);
    return hipGetLastError();
}
