// LM-head softmax statistics and speculative acceptance on gfx950.
//
// Softmax statistics are two-level: a grid of (V-chunk, row) workgroups
// writes a partial (max, sum exp(z - max)) per chunk of 4096 entries (each
// thread holds its 16 entries in registers: one round of loads); consumers
// merge the partials in chunk order (deterministic). z = L / T as the
// reference computes logits ./ temperature (src/ModelCPU.jl:1130-1132).
//
// Probabilities, their sums and every prefix sum of the draws are fp64 sums
// of per-entry fp32 exponentials whose argument is exact (ExpZ: relative
// error ~1e-7, independent across entries). A draw over 151936 entries of
// mass ~1e-5 each moves when the cumulative sum errs by a fraction of one
// entry's mass; fp32 sums err by ~1e-7 of the total, which moved ~0.4 % of
// residual draws against the exact prefix sums, fp64 ones by ~1e-15.
//
// Acceptance (src/SpeculativeDecoding.jl:75-104 with explicit uniforms) runs
// as three launches: statistics of every target and draft row; per (chunk,
// step) the ratio tests (every chunk's workgroup repeats them, the first
// publishes) and the chunk's sum of the sampling weights (residual or bonus
// distribution); and one workgroup per step that locates u * S by a chunk
// prefix and a scan inside the chunk. Every sum has one fixed order.
#include "common.h"

namespace {

constexpr int CHUNK = 4096;      // V elements per partial
constexpr int NT = 256;          // threads per workgroup

// exp(z - m) for an entry's probability: the difference rounded to fp32 plus
// its exact rounding error (two-sum), the accurate fp32 exp of the former
// times 1 + the latter (relative error ~1e-7, independent across entries;
// summed in double, such errors move a prefix sum by far less than one
// entry's mass). Non-finite differences give exp's own result.
__device__ __forceinline__ double dexp(float z, float m) {
    const float d = z - m;
    const float bz = d - z;
    const float err = (z - (d - bz)) + (-m - bz);
    const float e = expf(d);
    return (double)(e > 0.f && e < __builtin_huge_valf() ? fmaf(e, err, e) : e);
}

// The same over many entries of one row: exp(x / T - m) for m at or above
// every x / T, ~15 VALU instructions an entry where the division and dexp
// take ~45 (the statistics of 576 rows of 151936 took 191 us, bound by
// them). z = x / T by a reciprocal and two fma corrections (RN but for
// quotients within 2^-24 ulp of a rounding boundary); then z log2 e - M, M =
// m log2 e, without a rounding before the fraction: M = Mh + Ml with Mh on a
// grid g on which n + Mh is exact for every integer n in reach, so fma(z,
// log2 e, -(n + Mh)) rounds once, at a result below 1. An entry 230 below
// the maximum (-Inf among them) is clamped there: its exp is 0 in fp32
// either way. NaN stays NaN. Outside 2^-60 <= T <= 2^60 and |m| <= 2^20
// (fast false: a huge or infinite m has no such grid) the division and dexp
// are used.
struct ExpZ {
    float T, rT, m, xlim, Mh, Ml;
    bool fast;
    __device__ __forceinline__ ExpZ(float T_, float m_) : T(T_), m(m_) {
        fast = T >= 0x1p-60f && T <= 0x1p60f && fabsf(m) <= 0x1p20f;
        rT = 1.0f / T;
        xlim = (m - 230.0f) * T;
        const int il = fast ? ilogbf(fabsf(m) + 256.0f) : 8;
        const double Md = (double)m * 1.4426950408889634074;
        Mh = (float)ldexp(rint(ldexp(Md, 22 - il)), il - 22);  // (below 2^24 steps of g = 2^(il - 22))
        Ml = (float)(Md - (double)Mh);
    }
    // (only when fast)
    __device__ __forceinline__ float quick(float x) const {
        constexpr float L = 0x1.715476p+0f, LLO = 0x1.4ae0cp-26f;  // log2 e = L + LLO
        x = x < xlim ? xlim : x;
        const float q = x * rT;
        const float z = __builtin_fmaf(__builtin_fmaf(-q, T, x), rT, q);
        const float n = __builtin_rintf(__builtin_fmaf(z, L, -Mh));
        float f = __builtin_fmaf(z, L, -(n + Mh));
        f = __builtin_fmaf(z, LLO, f - Ml);
        return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
    }
    __device__ __forceinline__ double slow(float x) const { return dexp(x / T, m); }
};
// exp(m2 - m) in double for rescaling a partial sum (a few per row).
__device__ __forceinline__ double rescale(float m2, float m) { return exp((double)m2 - (double)m); }

// Partial softmax statistics: max z and sum exp(z - max) (16 bytes).
struct __align__(16) MS {
    float m, pad;
    double s;
};
__device__ __forceinline__ MS make_ms(float m, double s) {
    MS r;
    r.m = m;
    r.pad = 0.f;
    r.s = s;
    return r;
}

// Cross-lane moves on the VALU (DPP) and, across rows, one swizzle or
// bpermute: partner of lane l at butterfly level o (l ^ o for o = 1, 2, 16,
// 32; the mirror 7 - l within 8 for o = 4 and 15 - l within 16 for o = 8,
// which pair the same lanes' results once the lower levels have made every
// quad (octet) uniform).
template <int CTRL> __device__ __forceinline__ float dpp_mov(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
template <int O> __device__ __forceinline__ float partner(float v) {
    if constexpr (O == 1) return dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
    if constexpr (O == 2) return dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
    if constexpr (O == 4) return dpp_mov<0x141>(v);  // row_half_mirror
    if constexpr (O == 8) return dpp_mov<0x140>(v);  // row_mirror
    if constexpr (O == 16)                           // swizzle: xor 16 within 32
        return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
    return __shfl_xor(v, 32);
}
template <int O> __device__ __forceinline__ double partner_d(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_bit_cast(uint32_t, partner<O>(__builtin_bit_cast(float, (uint32_t)b)));
    const uint32_t hi = __builtin_bit_cast(uint32_t, partner<O>(__builtin_bit_cast(float, (uint32_t)(b >> 32))));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Butterfly sum / maximum over a wave (every lane gets the result).
__device__ __forceinline__ double wave_sum_d(double v) {
    v += partner_d<1>(v);
    v += partner_d<2>(v);
    v += partner_d<4>(v);
    v += partner_d<8>(v);
    v += partner_d<16>(v);
    v += partner_d<32>(v);
    return v;
}
__device__ __forceinline__ float wave_max_f(float v) {
    v = fmaxf(v, partner<1>(v));
    v = fmaxf(v, partner<2>(v));
    v = fmaxf(v, partner<4>(v));
    v = fmaxf(v, partner<8>(v));
    v = fmaxf(v, partner<16>(v));
    v = fmaxf(v, partner<32>(v));
    return v;
}

// A chunk's entries over the workgroup: wave w holds the 1024 entries from
// 1024 w, in PER / 4 rounds of 4 consecutive entries a lane (16-byte loads
// at any 4-byte alignment), so index order is (wave, round, lane, entry).
constexpr int PER = CHUNK / NT;  // 16 entries per thread
constexpr int PR = PER / 4;      // rounds
__device__ __forceinline__ int entry0(int r) {
    return (threadIdx.x >> 6) * (CHUNK / 4) + r * 256 + 4 * (threadIdx.x & 63);
}
// Entries past V read `fill`.
__device__ __forceinline__ void load_chunk(const float *__restrict__ src, int c, int V, float fill, float (&x)[PER]) {
    const int j0 = c * CHUNK;
    if (j0 + CHUNK <= V) {
#pragma unroll
        for (int r = 0; r < PR; r++) __builtin_memcpy(&x[4 * r], src + j0 + entry0(r), 16);
    } else {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int j = j0 + entry0(i / 4) + (i & 3);
            x[i] = j < V ? src[j] : fill;
        }
    }
}

// partial[row][chunk] = (max z, sum exp(z - max)). Rows [0, rows1) come from
// L1 at temperature T1, except every period-th row (r % period == period - 1,
// the bonus row of a verify step) at T_last; rows [rows1, ..) come from L2 at
// T2. With parent (a draft tree of rows1 nodes, target rows then draft rows)
// only the rows of nodes that are some node's parent are formed: the walk
// reads no others.
// One maximum over the workgroup's raw logits (the division by T > 0 keeps
// the order), then every exponential against it: no rescaling exp per thread
// and merge level. Bound by HBM and VALU together: 576 rows of 151936 (350
// MB) 191 -> 63 us (5.5 TB/s).
constexpr int TREE_FILTER = 4 * NT;  // (parents read per workgroup: at most 4 loads a thread)
__global__ __launch_bounds__(NT) void stats_partial_kernel(const float *__restrict__ L1, int rows1, float T1,
                                                           float T_last, int period, const float *__restrict__ L2,
                                                           float T2, int V, int nchunk,
                                                           const int32_t *__restrict__ parent,
                                                           MS *__restrict__ part) {
    __shared__ float sm[NT / 64];
    __shared__ double ss[NT / 64];
    const int chunk = blockIdx.x, row = blockIdx.y, wave = threadIdx.x >> 6;
    const bool first = row < rows1;
    if (parent != nullptr) {
        const int node = first ? row : row - rows1;
        bool used = false;
        for (int i = threadIdx.x; i < rows1; i += NT) used |= i > node && parent[i] == node;
        if (!__syncthreads_or(used)) return;
    }
    const float Tr = first ? ((period > 0 && row % period == period - 1) ? T_last : T1) : T2;
    const float *src = first ? L1 + (size_t)row * V : L2 + (size_t)(row - rows1) * V;
    float x[PER];
    load_chunk(src, chunk, V, -__builtin_huge_valf(), x);
    float m = x[0];
#pragma unroll
    for (int i = 1; i < PER; i++) m = fmaxf(m, x[i]);
    m = wave_max_f(m);
    if ((threadIdx.x & 63) == 0) sm[wave] = m;
    __syncthreads();
    m = sm[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) m = fmaxf(m, sm[w]);
    m = fmaxf(m, -__builtin_huge_valf()) / Tr;  // (all NaN: -Inf)
    double s = 0.0;
    if (m > -__builtin_huge_valf()) {
        const ExpZ E(Tr, m);
        if (E.fast) {
#pragma unroll
            for (int i = 0; i < PER; i++) s += (double)E.quick(x[i]);
        } else {
#pragma unroll 1
            for (int i = 0; i < PER; i++) {
                const int j = chunk * CHUNK + entry0(i / 4) + (i & 3);
                s += E.slow(j < V ? src[j] : -__builtin_huge_valf());
            }
        }
    }
    s = wave_sum_d(s);
    if ((threadIdx.x & 63) == 0) ss[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[(size_t)row * nchunk + chunk] = make_ms(m, ((ss[0] + ss[1]) + ss[2]) + ss[3]);
}

// A row's statistics from its chunk partials, by one wave: the maximum, then
// each partial's sum rescaled to it (one exp a partial). p0, p1: this lane's
// partials lane and lane + 64 (m = -Inf past the end); chunks past 128 are
// read here.
__device__ __forceinline__ MS wave_merge(const MS &p0, const MS &p1, const MS *__restrict__ part, int nchunk) {
    const int lane = threadIdx.x & 63;
    const float ninf = -__builtin_huge_valf();
    float m = fmaxf(p0.m, p1.m);
    for (int c = lane + 128; c < nchunk; c += 64) m = fmaxf(m, part[c].m);
    m = wave_max_f(m);
    double s = 0.0;
    if (p0.m > ninf) s = p0.s * rescale(p0.m, m);
    if (nchunk > 64 && p1.m > ninf) s += p1.s * rescale(p1.m, m);
    for (int c = lane + 128; c < nchunk; c += 64) {
        const MS p = part[c];
        if (p.m > ninf) s += p.s * rescale(p.m, m);
    }
    return make_ms(m, wave_sum_d(s));
}
__device__ __forceinline__ MS load_part(const MS *__restrict__ part, int c, int nchunk) {
    return c < nchunk ? part[c] : make_ms(-__builtin_huge_valf(), 0.0);
}

// The same by one thread, eight partials in flight.
__device__ MS thread_merge(const MS *__restrict__ part, int nchunk) {
    const float ninf = -__builtin_huge_valf();
    float m = ninf;
    double s = 0.0;
    for (int pass = 0; pass < 2; pass++)
        for (int c = 0; c < nchunk; c += 8) {
            MS v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = part[min(c + j, nchunk - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (c + j >= nchunk || !(v[j].m > ninf)) continue;
                if (pass == 0) m = fmaxf(m, v[j].m);
                else s += v[j].s * rescale(v[j].m, m);
            }
        }
    return make_ms(m, s);
}

// One wave per row.
__global__ __launch_bounds__(NT) void stats_merge_kernel(const MS *__restrict__ part, int rows, int nchunk,
                                                         float *__restrict__ zmax, float *__restrict__ zsum) {
    const int r = blockIdx.x * (NT / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= rows) return;  // (whole waves)
    const MS *p = part + (size_t)r * nchunk;
    const MS ms = wave_merge(load_part(p, lane, nchunk), load_part(p, lane + 64, nchunk), p, nchunk);
    if (lane == 0) {
        zmax[r] = ms.m;
        zsum[r] = (float)ms.s;
    }
}

// Sampling distribution of one draw of a verify step, set by the ratio
// tests:
//   kind 0: p_j (target row, temperature Tp)       bonus draw
//   kind 1: max(0, p_j - q_j)  (q: draft row)      standard residual
//   kind 2: max(0, p_j - qs)   (qs: scalar q_i)    reference residual
//   kind 3: the bonus token drawn beforehand by the filtered sampler
//           (top-k / top-p / min-p on target row k at T with u_bonus)
//   kind -1: invalid draft id (out_n = -1, nothing drawn)
//   kind -2: no draw in this slot
// fallback when the weights sum to 0: 1 = draw from p (standard mode),
// 2 = return V - 1 (the reference's all-NaN residual, length(probs)).
// pos: the index of the drawn token in the step's out_tok row. A step has
// one draw slot in the standard mode and two in the reference mode, whose
// second slot holds the bonus the reference appends after a rejection of
// the last draft (src/SpeculativeDecoding.jl:100: length(accepted) == gamma).
struct Decision {
    int kind, n, prow, qrow, fallback, pos;
    float Tp, mp, Tq, mq, u, pad;
    double isp, isq, qs;  // 1 / (sum of exp) of the p and q rows
};
__host__ __device__ constexpr int draw_slots(int mode) { return mode == 1 ? 2 : 1; }

// Inclusive scan over the 64 lanes of a wave (fixed association): a
// Hillis-Steele scan inside each row of 16 (DPP row shifts by 1, 2, 4, 8;
// lanes shifted in from outside the row read 0), then row r + 1 adds the
// total of row r (row broadcast of lane 15 into rows 1 and 3) and rows 2, 3
// add the total of rows 0, 1 (row broadcast of lane 31).
// A double moves as its two halves.
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_row(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xF, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_scan(double v) {
    v += dpp_row<0x111, 0xF>(v);  // row_shr:1
    v += dpp_row<0x112, 0xF>(v);  // row_shr:2
    v += dpp_row<0x114, 0xF>(v);  // row_shr:4
    v += dpp_row<0x118, 0xF>(v);  // row_shr:8
    v += dpp_row<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
    v += dpp_row<0x143, 0xC>(v);  // row_bcast:31 into rows 2, 3
    return v;
}

// Ratio tests of one verify step by a whole workgroup: the statistics of the
// step's 2k + 1 rows are merged first (row r by wave r % 4: the loads of
// all its rows in flight before any merge; kept in LDS), then lane i of wave
// 0 judges draft i (groups of 64 lanes for k > 64). The result is the
// decision of each draw slot (s_dec[0], s_dec[1]); with publish, the
// accepted drafts, out_n and the decisions are also written out. Every
// workgroup that calls it for the same step computes the same decision.
constexpr int DECIDE_MAX_ROWS = 255;  // 2k + 1, k <= 127
constexpr int DECIDE_WAVES = NT / 64;
__device__ void decide_block(const float *__restrict__ tgt, const float *__restrict__ drf,
                             const int32_t *__restrict__ draft_tok, int k, int V, float T,
                             const float *__restrict__ u_acc, const float *__restrict__ u_res,
                             const float *__restrict__ u_bonus, int mode, const MS *__restrict__ part,
                             int nchunk, int step, int steps, bool publish, const int32_t *__restrict__ bonus_pre,
                             int32_t *__restrict__ out_tok, int32_t *__restrict__ out_n,
                             Decision *__restrict__ dec, MS *ms, Decision *s_dec) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float *Lt = tgt + (size_t)step * (k + 1) * V;
    const float *Ld = drf + (size_t)step * k * V;
    const int32_t *dt = draft_tok + (size_t)step * k;
    const MS *Pt = part + (size_t)step * (k + 1) * nchunk;
    const MS *Pd = part + ((size_t)steps * (k + 1) + (size_t)step * k) * nchunk;
    const float Tr = mode == 0 ? T : 1.0f;
    // wave 0: the first 64 drafts' ids and uniforms, then (once the ids are
    // in) their two logits, issued before the merges
    const bool has0 = wave == 0 && lane < k;
    const int x0 = has0 ? dt[lane] : 0;
    const float ua0 = has0 ? u_acc[(size_t)step * k + lane] : 0.f;
    const int nrows = 2 * k + 1;
    float lx0 = 0.f, dx0 = 0.f;
    // rows wave, wave + W, ..: in batches of 8 per wave
    for (int r0 = wave; r0 < nrows; r0 += 8 * DECIDE_WAVES) {
        MS pv[8][2];
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int r = min(r0 + b * DECIDE_WAVES, nrows - 1);
            const MS *row = r <= k ? Pt + (size_t)r * nchunk : Pd + (size_t)(r - k - 1) * nchunk;
#pragma unroll
            for (int h = 0; h < 2; h++) pv[b][h] = load_part(row, lane + 64 * h, nchunk);
        }
        if (r0 == 0 && has0 && x0 >= 0 && x0 < V) {
            lx0 = Lt[(size_t)lane * V + x0];
            dx0 = Ld[(size_t)lane * V + x0];
        }
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int r = r0 + b * DECIDE_WAVES;
            if (r >= nrows) break;
            const MS v = wave_merge(pv[b][0], pv[b][1],
                                    r <= k ? Pt + (size_t)r * nchunk : Pd + (size_t)(r - k - 1) * nchunk, nchunk);
            if (lane == 0) ms[r] = v;
        }
    }
    __syncthreads();
    if (wave == 0) {
        int first = k;  // first draft that is invalid or rejected
        bool invalid = false;
        double f_q = 0.0;
        for (int base = 0; base < k && first == k; base += 64) {
            const int i = base + lane;
            bool bad = false, inv = false;
            double q = 0.0;
            if (i < k) {
                const bool pre = base == 0;  // the first 64 were fetched up front
                const int x = pre ? x0 : dt[i];
                if (x < 0 || x >= V) {
                    bad = inv = true;
                } else {
                    const MS pt = ms[i], pd = ms[k + 1 + i];
                    const double p = dexp((pre ? lx0 : Lt[(size_t)i * V + x]) / Tr, pt.m) / pt.s;
                    q = dexp((pre ? dx0 : Ld[(size_t)i * V + x]) / Tr, pd.m) / pd.s;
                    const double ratio = q > 0.0 ? fmin(1.0, p / q) : 1.0;
                    bad = !((double)(pre ? ua0 : u_acc[(size_t)step * k + i]) < ratio);
                }
            }
            const uint64_t m = __ballot(bad);
            if (m) {
                const int f = __ffsll((unsigned long long)m) - 1;
                first = base + f;
                invalid = __shfl(inv ? 1 : 0, f) != 0;
                f_q = __shfl(q, f);
            }
        }
        // accepted drafts
        if (publish)
            for (int i = lane; i < first; i += 64) out_tok[(size_t)step * (k + 1) + i] = dt[i];
        if (lane == 0) {
            const int nd = draw_slots(mode);
            Decision D{}, D2{};
            D2.kind = -2;
            if (invalid) {
                D.kind = -1;
                D.n = -1;
            } else {
                D.n = first;
                D.pos = first;
                if (first < k) {
                    const MS pt = ms[first], pd = ms[k + 1 + first];
                    D.kind = mode == 0 ? 1 : 2;
                    D.prow = first;
                    D.qrow = first;
                    D.Tp = Tr; D.mp = pt.m; D.isp = 1.0 / pt.s;
                    D.Tq = Tr; D.mq = pd.m; D.isq = 1.0 / pd.s;
                    D.qs = f_q;
                    D.u = u_res[step];
                    D.fallback = mode == 0 ? 1 : 2;
                    if (mode == 1 && first == k - 1) {  // the reference's bonus after the residual
                        const MS pk = ms[k];
                        D2.kind = bonus_pre ? 3 : 0;
                        D2.n = first;
                        D2.pos = first + 1;
                        D2.prow = k;
                        D2.Tp = T; D2.mp = pk.m; D2.isp = 1.0 / pk.s;
                        D2.Tq = T; D2.mq = 0.f; D2.isq = 1.0;
                        D2.u = u_bonus[step];
                        D2.fallback = 2;
                    }
                } else {
                    const MS pt = ms[k];
                    D.kind = bonus_pre ? 3 : 0;
                    D.prow = k;
                    D.qrow = 0;
                    D.Tp = T; D.mp = pt.m; D.isp = 1.0 / pt.s;
                    D.Tq = T; D.mq = 0.f; D.isq = 1.0; D.qs = 0.0;
                    D.u = u_bonus[step];
                    D.fallback = 2;
                }
            }
            s_dec[0] = D;
            s_dec[1] = D2;
            if (publish) {
                out_n[step] = D.n;
                dec[(size_t)step * nd] = D;
                if (nd > 1) dec[(size_t)step * nd + 1] = D2;
            }
        }
    }
    __syncthreads();
}

// Sampling weights of the thread's PER entries of chunk c (load_chunk's
// order): p (use_p, kind 0) or the residual.
__device__ __forceinline__ void chunk_weights(const Decision &D, const float *__restrict__ lt,
                                              const float *__restrict__ ld, int V, int c, bool use_p,
                                              double (&w)[PER]) {
    // (no fma of the two products: equal rows leave a residual of exactly 0)
#pragma clang fp contract(off)
    const bool need_q = !use_p && D.kind == 1;
    float x[PER], y[PER];
    load_chunk(lt, c, V, -__builtin_huge_valf(), x);
    if (need_q) load_chunk(ld, c, V, -__builtin_huge_valf(), y);
    const ExpZ P(D.Tp, D.mp);
    if (P.fast) {
#pragma unroll
        for (int i = 0; i < PER; i++) w[i] = (double)P.quick(x[i]) * D.isp;
    } else {
#pragma unroll
        for (int i = 0; i < PER; i++) w[i] = P.slow(x[i]) * D.isp;
    }
    if (need_q) {
        const ExpZ Q(D.Tq, D.mq);
        if (Q.fast) {
#pragma unroll
            for (int i = 0; i < PER; i++) w[i] = fmax(w[i] - (double)Q.quick(y[i]) * D.isq, 0.0);
        } else {
#pragma unroll
            for (int i = 0; i < PER; i++) w[i] = fmax(w[i] - Q.slow(y[i]) * D.isq, 0.0);
        }
    } else if (!use_p && D.kind == 2) {
#pragma unroll
        for (int i = 0; i < PER; i++) w[i] = fmax(w[i] - D.qs, 0.0);
    }
    if ((c + 1) * CHUNK > V) {  // (a scalar q or a NaN row would leave weights past the end)
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (c * CHUNK + entry0(i / 4) + (i & 3) >= V) w[i] = 0.0;
    }
}

// The chunk's sum of weights (sh: NT / 64 doubles; ends with the sum in
// every thread, sh free again).
__device__ __forceinline__ double chunk_sum(const double (&w)[PER], double *sh) {
    double s = 0.0;
#pragma unroll
    for (int r = 0; r < PR; r++) s += (w[4 * r] + w[4 * r + 1]) + (w[4 * r + 2] + w[4 * r + 3]);
    s = wave_sum_d(s);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    s = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return s;
}

// The chunk's sum of a draw slot's weights: csum[slot][c].
__device__ __forceinline__ void sum_chunk(const Decision &D, size_t slot, int step, int c,
                                          const float *__restrict__ tgt, const float *__restrict__ drf, int k, int V,
                                          int nchunk, double *sh, double *__restrict__ csum) {
    if (D.kind < 0 || D.kind == 3) return;
    const float *lt = tgt + ((size_t)step * (k + 1) + D.prow) * V;
    const float *ld = D.kind == 1 ? drf + ((size_t)step * k + D.qrow) * V : nullptr;
    double w[PER];
    chunk_weights(D, lt, ld, V, c, false, w);
    const double sw = chunk_sum(w, sh);
    if (threadIdx.x == 0) csum[slot * nchunk + c] = sw;
}

// The decision of verify step `step` (decide_block, computed by every
// workgroup; the first one publishes it), then csum[step][slot][c] = the
// sum of w over chunk c (grid: x chunk, y step, z draw slot).
__global__ __launch_bounds__(NT) void decide_sum_kernel(const float *__restrict__ tgt, const float *__restrict__ drf,
                                                        const int32_t *__restrict__ draft_tok, int k, int V, float T,
                                                        const float *__restrict__ u_acc,
                                                        const float *__restrict__ u_res,
                                                        const float *__restrict__ u_bonus, int mode,
                                                        const MS *__restrict__ part, int nchunk,
                                                        const int32_t *__restrict__ bonus_pre,
                                                        int32_t *__restrict__ out_tok, int32_t *__restrict__ out_n,
                                                        Decision *__restrict__ dec, double *__restrict__ csum) {
    __shared__ double sh[NT / 64];
    __shared__ MS ms[DECIDE_MAX_ROWS];
    __shared__ Decision s_dec[2];
    const int c = blockIdx.x, step = blockIdx.y;
    decide_block(tgt, drf, draft_tok, k, V, T, u_acc, u_res, u_bonus, mode, part, nchunk, step, gridDim.y,
                 c == 0 && blockIdx.z == 0, bonus_pre, out_tok, out_n, dec, ms, s_dec);
    sum_chunk(s_dec[blockIdx.z], (size_t)step * gridDim.z + blockIdx.z, step, c, tgt, drf, k, V, nchunk, sh, csum);
}

// The two halves as launches of their own, for more workgroups than run
// together: the decision once a step (grid: x step), then the chunk sums
// (decide_sum_kernel's grid), which read it.
__global__ __launch_bounds__(NT) void decide_kernel(const float *__restrict__ tgt, const float *__restrict__ drf,
                                                    const int32_t *__restrict__ draft_tok, int k, int V, float T,
                                                    const float *__restrict__ u_acc,
                                                    const float *__restrict__ u_res,
                                                    const float *__restrict__ u_bonus, int mode,
                                                    const MS *__restrict__ part, int nchunk,
                                                    const int32_t *__restrict__ bonus_pre,
                                                    int32_t *__restrict__ out_tok, int32_t *__restrict__ out_n,
                                                    Decision *__restrict__ dec) {
    __shared__ MS ms[DECIDE_MAX_ROWS];
    __shared__ Decision s_dec[2];
    decide_block(tgt, drf, draft_tok, k, V, T, u_acc, u_res, u_bonus, mode, part, nchunk, blockIdx.x, gridDim.x, true,
                 bonus_pre, out_tok, out_n, dec, ms, s_dec);
}
__global__ __launch_bounds__(NT) void sum_kernel(const float *__restrict__ tgt, const float *__restrict__ drf, int k,
                                                 int V, const Decision *__restrict__ dec, int nchunk,
                                                 double *__restrict__ csum) {
    __shared__ double sh[NT / 64];
    const size_t slot = (size_t)blockIdx.y * gridDim.z + blockIdx.z;
    sum_chunk(dec[slot], slot, blockIdx.y, blockIdx.x, tgt, drf, k, V, nchunk, sh, csum);
}

// First j with u * S <= C_j: the chunk by a prefix over the chunk sums (a
// wave scan, repeated by every wave: 64 chunks a round), then the entry by
// scans inside the chunk, C_j = before(chunk) + (the sums of the rounds
// before it in the chunk) + (the lanes before it, then its own entries).
// When the weights sum to zero the standard mode draws from p (its chunk
// sums are formed here), the reference mode returns V - 1; so does a u * S
// no chunk reaches (NaN weights, u above 1).
constexpr int MAX_CHUNKS = 1024;
__global__ __launch_bounds__(NT) void sample_kernel(const float *__restrict__ tgt, const float *__restrict__ drf,
                                                    int k, int V, const Decision *__restrict__ dec, int nchunk,
                                                    const double *__restrict__ csum,
                                                    const int32_t *__restrict__ bonus_pre,
                                                    int32_t *__restrict__ out_tok) {
    __shared__ double sh[PER];
    __shared__ double s_psum[MAX_CHUNKS];
    __shared__ int s_hit[NT / 64], s_last[NT / 64];
    const int step = blockIdx.x, t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const size_t slot = (size_t)step * gridDim.y + blockIdx.y;
    const double *cw = csum + slot * nchunk;
    double c0 = lane < nchunk ? cw[lane] : 0.0;  // (a slot without a draw: read, not used)
    const Decision D = dec[slot];
    if (D.kind < 0) return;
    int32_t *out = out_tok + (size_t)step * (k + 1) + D.pos;
    if (D.kind == 3) {
        if (t == 0) *out = bonus_pre[step];
        return;
    }
    const float *lt = tgt + ((size_t)step * (k + 1) + D.prow) * V;
    const float *ld = D.kind == 1 ? drf + ((size_t)step * k + D.qrow) * V : nullptr;
    const double *src = cw;
    bool usep = false;
    // the running sum through chunk b + lane, given the sum before chunk b
    auto round = [&](int b, double carry) {
        const int c = b + lane;
        return carry + wave_scan(b == 0 ? c0 : c < nchunk ? src[c] : 0.0);
    };
    auto total = [&]() {
        double carry = 0.0;
        for (int b = 0; b < nchunk; b += 64) carry = __shfl(round(b, carry), 63);
        return carry;
    };
    double w[PER];
    double S = total();
    if (!(S > 0.0)) {
        if (D.fallback != 1) {
            if (t == 0) *out = V - 1;
            return;
        }
        usep = true;
        for (int c = 0; c < nchunk; c++) {
            chunk_weights(D, lt, ld, V, c, true, w);
            const double sp = chunk_sum(w, sh);
            if (t == 0) s_psum[c] = sp;
        }
        __syncthreads();
        src = s_psum;
        c0 = lane < nchunk ? s_psum[lane] : 0.0;
        S = total();
    }
    const double target = (double)D.u * S;
    double before = 0.0;
    int c = -1;
    for (int b = 0; b < nchunk && c < 0; b += 64) {
        const double cum = round(b, before);
        const uint64_t hit = __ballot(b + lane < nchunk && target <= cum);
        const int f = hit ? __ffsll((unsigned long long)hit) - 1 : 64;
        if (f > 0) before = __shfl(cum, f - 1);
        if (f < 64) c = b + f;
    }
    if (c < 0) {
        if (t == 0) *out = V - 1;
        return;
    }
    chunk_weights(D, lt, ld, V, c, usep, w);
    double inc[PR];  // inclusive scans over the lanes of the rounds' sums
#pragma unroll
    for (int r = 0; r < PR; r++) {
        inc[r] = wave_scan((w[4 * r] + w[4 * r + 1]) + (w[4 * r + 2] + w[4 * r + 3]));
        if (lane == 63) sh[wave * PR + r] = inc[r];
    }
    __syncthreads();
    for (int i = 0; i < wave * PR; i++) before += sh[i];
    int hit = CHUNK, last = -1;
#pragma unroll
    for (int r = 0; r < PR; r++) {
        double run = __shfl_up(inc[r], 1);
        if (lane == 0) run = 0.0;
        const int j = entry0(r);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            run += w[4 * r + e];
            if (target <= before + run && hit == CHUNK) hit = j + e;
            if (w[4 * r + e] > 0.0) last = j + e;
        }
        before += sh[wave * PR + r];
    }
    for (int o = 32; o > 0; o >>= 1) {
        hit = min(hit, __shfl_xor(hit, o));
        last = max(last, __shfl_xor(last, o));
    }
    if (lane == 0) {
        s_hit[wave] = hit;
        s_last[wave] = last;
    }
    __syncthreads();
    if (t == 0) {
        // (the scan inside the chunk can end a rounding step below the sum
        // that selected it: then the chunk's last entry of positive weight)
        int h = CHUNK, l = -1;
        for (int i = 0; i < NT / 64; i++) {
            h = min(h, s_hit[i]);
            l = max(l, s_last[i]);
        }
        *out = min(c * CHUNK + (h < CHUNK ? h : l >= 0 ? l : CHUNK - 1), V - 1);
    }
}

// Julia's findmax order (the argmax of mtp_verify_step!): isless, the total
// order -Inf < ... < -0.0 < +0.0 < ... < +Inf < NaN; among equals (and among
// NaNs) the first index wins. `beats` is the strict order, `first_of` picks
// (value, index) pairs under it.
__device__ __forceinline__ bool beats(float a, float b) {
    if (isnan(a) || isnan(b)) return isnan(a) && !isnan(b);
    return a > b || (a == b && signbit(b) && !signbit(a));
}
__device__ __forceinline__ bool first_of(float v2, int i2, float bv, int bi) {
    return beats(v2, bv) || (!beats(bv, v2) && i2 < bi);
}

// Partial first-index argmax per (chunk, row). Every thread of a non-empty
// chunk holds a real index (a row of -Inf gives its first index).
__global__ __launch_bounds__(NT) void argmax_partial_kernel(const float *__restrict__ L, int V, int nchunk,
                                                            float2 *__restrict__ part) {
    __shared__ float sv[NT / 64];
    __shared__ int si[NT / 64];
    const int chunk = blockIdx.x, row = blockIdx.y;
    const float *src = L + (size_t)row * V;
    const int j0 = chunk * CHUNK, j1 = min(V, j0 + CHUNK);
    float bv = -__builtin_huge_valf();
    int bi = 0x7fffffff;
    for (int j = j0 + threadIdx.x; j < j1; j += NT) {
        const float v = src[j];
        if (first_of(v, j, bv, bi)) { bv = v; bi = j; }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float v2 = __shfl_xor(bv, o);
        const int i2 = __shfl_xor(bi, o);
        if (first_of(v2, i2, bv, bi)) { bv = v2; bi = i2; }
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sv[w] = bv; si[w] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < NT / 64; i++)
            if (first_of(sv[i], si[i], bv, bi)) { bv = sv[i]; bi = si[i]; }
        part[(size_t)row * nchunk + chunk] = make_float2(bv, __int_as_float(bi));
    }
}

// One wave per step: each row's first argmax over its chunks (lane l takes
// chunks l, l + 64, ..), then the matching prefix of the drafts.
__global__ __launch_bounds__(64) void greedy_kernel(const float2 *__restrict__ part, int nchunk,
                                                    const int32_t *__restrict__ draft_tok, int k,
                                                    int32_t *__restrict__ out_n, int32_t *__restrict__ out_argmax) {
    const int step = blockIdx.x, lane = threadIdx.x;
    int n = 0;
    bool go = true;
#pragma unroll 4
    for (int i = 0; i <= k; i++) {
        const float2 *p = part + ((size_t)step * (k + 1) + i) * nchunk;
        float bv = -__builtin_huge_valf();
        int bi = 0x7fffffff;
        for (int c = lane; c < nchunk; c += 64) {
            const float2 v = p[c];
            if (first_of(v.x, __float_as_int(v.y), bv, bi)) { bv = v.x; bi = __float_as_int(v.y); }
        }
        for (int o = 32; o > 0; o >>= 1) {
            const float v2 = __shfl_xor(bv, o);
            const int i2 = __shfl_xor(bi, o);
            if (first_of(v2, i2, bv, bi)) { bv = v2; bi = i2; }
        }
        if (out_argmax && lane == 0) out_argmax[(size_t)step * (k + 1) + i] = bi;
        if (i < k && go) {
            if (bi == draft_tok[(size_t)step * k + i]) n++;
            else go = false;
        }
    }
    if (lane == 0) out_n[step] = n;
}

// Tree walk by one workgroup: the statistics of every parent's target and
// draft row are merged (one wave a row) into ms, then every node is tested in
// parallel (the test of node i reads only its parent's rows and its own
// token: pass = u_i < min(1, p/q)), then its depth, or that it or an
// ancestor failed, comes from pointer jumping over the parents (parent[i] <
// i; log2 of the depth rounds): dep[i] sums 1 per node that passed and
// TREE_FAIL per failure from i to its ancestor anc[i]. The deepest accepted
// node, smallest index on ties, ends the path. Node state lives in LDS up to
// TREE_LDS nodes; a larger tree is walked by one thread from the workspace.
// (One thread walking 64 nodes in LDS, each row merged by one thread: 29 us;
// now 8 us. Above TREE_LDS nodes the rows are merged a thread each: a wave a
// row, 5000 nodes of V = 512 took 2.36 ms, 1.99 so.)
constexpr int TREE_NT = 1024;
constexpr int TREE_LDS = 4096;
constexpr int TREE_FAIL = -(1 << 24);
__global__ __launch_bounds__(TREE_NT) void tree_kernel(const float *__restrict__ tgt, const float *__restrict__ drf,
                                                       const int32_t *__restrict__ tok,
                                                       const int32_t *__restrict__ parent, int n, int V, float T,
                                                       const float *__restrict__ u, const MS *__restrict__ part,
                                                       int nchunk, MS *__restrict__ ms,
                                                       int32_t *__restrict__ out_path, int32_t *__restrict__ out_len,
                                                       int32_t *__restrict__ wsi) {
    constexpr int NPT = TREE_LDS / TREE_NT;
    __shared__ int32_t s_par[TREE_LDS], s_anc[TREE_LDS], s_dep[TREE_LDS];
    __shared__ uint8_t s_used[TREE_LDS];
    __shared__ int s_best[TREE_NT / 64];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const bool in_lds = n <= TREE_LDS;
    if (in_lds) {
        for (int i = t; i < n; i += TREE_NT) s_used[i] = 0;
        __syncthreads();
        for (int i = t; i < n; i += TREE_NT) {
            const int p = i > 0 ? parent[i] : 0;
            s_par[i] = p;
            if (i > 0 && p >= 0 && p < i) s_used[p] = 1;
        }
        __syncthreads();
    }
    if (in_lds) {
        for (int r = wave; r < 2 * n; r += TREE_NT / 64) {
            if (!s_used[r < n ? r : r - n]) continue;
            const MS *p = part + (size_t)r * nchunk;
            const MS v = wave_merge(load_part(p, lane, nchunk), load_part(p, lane + 64, nchunk), p, nchunk);
            if (lane == 0) ms[r] = v;
        }
    } else {  // (all rows, more than 8192: a thread each)
        for (int r = t; r < 2 * n; r += TREE_NT) ms[r] = thread_merge(part + (size_t)r * nchunk, nchunk);
    }
    __syncthreads();
    // 1 passed, 0 failed, -1 malformed
    auto test = [&](int i, int p) {
        if (i == 0) return 1;  // (the root is accepted)
        const int x = tok[i];
        if (p < 0 || p >= i || x < 0 || x >= V) return -1;
        const MS pt = ms[p];
        const MS pd = ms[n + p];
        const double pp = dexp(tgt[(size_t)p * V + x] / T, pt.m) / pt.s;
        const double qq = dexp(drf[(size_t)p * V + x] / T, pd.m) / pd.s;
        const double ratio = qq > 0.0 ? fmin(1.0, pp / qq) : 1.0;
        return (double)u[i] < ratio ? 1 : 0;
    };
    if (in_lds) {
        int dep[NPT], anc[NPT];
        bool bad = false, more = false;
#pragma unroll
        for (int j = 0; j < NPT; j++) {
            const int i = t + j * TREE_NT;
            dep[j] = 0;
            anc[j] = 0;
            if (i < n && i > 0) {
                const int p = s_par[i], r = test(i, p);
                bad |= r < 0;
                dep[j] = r > 0 ? 1 : TREE_FAIL;
                anc[j] = r < 0 ? 0 : p;
                more |= anc[j] != 0;
            }
        }
        if (__syncthreads_or(bad)) {
            if (t == 0) *out_len = -1;
            return;
        }
        while (__syncthreads_or(more)) {
#pragma unroll
            for (int j = 0; j < NPT; j++) {
                const int i = t + j * TREE_NT;
                if (i < n) {
                    s_dep[i] = dep[j];
                    s_anc[i] = anc[j];
                }
            }
            __syncthreads();
            more = false;
#pragma unroll
            for (int j = 0; j < NPT; j++) {
                const int a = anc[j];
                if (a != 0) {
                    dep[j] = max(dep[j] + s_dep[a], TREE_FAIL);
                    anc[j] = s_anc[a];
                    more |= anc[j] != 0;
                }
            }
        }
        int best = 0;  // depth * TREE_LDS + (TREE_LDS - 1 - index), at least the root's
#pragma unroll
        for (int j = 0; j < NPT; j++) {
            const int i = t + j * TREE_NT;
            if (i < n && dep[j] >= 0) best = max(best, dep[j] * TREE_LDS + (TREE_LDS - 1 - i));
        }
        for (int o = 32; o > 0; o >>= 1) best = max(best, __shfl_xor(best, o));
        if (lane == 0) s_best[wave] = best;
        __syncthreads();
        if (t != 0) return;
        for (int w = 1; w < TREE_NT / 64; w++) best = max(best, s_best[w]);
        const int len = best / TREE_LDS + 1;
        int v = TREE_LDS - 1 - best % TREE_LDS;
        for (int d = len - 1; d >= 0; d--) {
            out_path[d] = v;
            v = d > 0 ? s_par[v] : 0;
        }
        *out_len = len;
        return;
    }
    int32_t *par = wsi, *st = wsi + n;
    int8_t *pass = (int8_t *)(wsi + 2 * n);
    for (int i = t; i < n; i += TREE_NT) {
        const int p = parent[i];
        par[i] = p;
        pass[i] = (int8_t)test(i, p);
    }
    __syncthreads();
    if (t != 0) return;
    st[0] = 0;
    int best = 0;
    for (int i = 1; i < n; i++) {
        const int r = pass[i];
        if (r < 0) {
            *out_len = -1;
            return;
        }
        const int sp = st[par[i]];
        const int d = (sp >= 0 && r) ? sp + 1 : -1;
        st[i] = d;
        if (d > st[best]) best = i;
    }
    const int len = st[best] + 1;
    int v = best;
    for (int d = len - 1; d >= 0; d--) {
        out_path[d] = v;
        v = d > 0 ? par[v] : 0;
    }
    *out_len = len;
}

}  // namespace

int accept_nchunk(int V) { return (V + CHUNK - 1) / CHUNK; }

// Bytes of one softmax partial (MS) of a (row, chunk); a first-argmax
// partial (float2) fits in the same slot.
size_t accept_part_bytes() { return sizeof(MS); }

hipError_t launch_stats(const float *L, int rows, int V, float T, float T_last, int period, void *part,
                        hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    const int nc = accept_nchunk(V);
    stats_partial_kernel<<<dim3(nc, rows), NT, 0, st>>>(L, rows, T, T_last, period, L, T, V, nc, nullptr,
                                                             (MS *)part);
    return hipGetLastError();
}

hipError_t launch_stats_merge(const void *part, int rows, int V, float *zmax, float *zsum, hipStream_t st) {
    const int nc = accept_nchunk(V);
    stats_merge_kernel<<<(rows + NT / 64 - 1) / (NT / 64), NT, 0, st>>>((const MS *)part, rows, nc, zmax, zsum);
    return hipGetLastError();
}

size_t spec_accept_ws(int steps, int k, int V) {
    const size_t nc = accept_nchunk(V);
    return (size_t)steps * (2 * k + 1) * nc * sizeof(MS) + (size_t)steps * 2 * sizeof(Decision) +
           (size_t)steps * 2 * nc * sizeof(double) + 256;
}

// With more chunk-sum workgroups than CUs the decision has a launch of its
// own: a workgroup that decides first waits ~6 us for 2k + 1 rows' partials
// while its place on the CU could stream a chunk. Both ways
// measured at k = 4, V = 151936 (38 workgroups a step; a graph of 20 calls): 4
// steps 20.1 us in one launch, 21.0 in two; 8 steps 29.5 and 26.7; 64 steps
// 124.8 and 84.1; V = 32000 (8 a step): 32 steps 27.0 and 28.3, 64 steps 42.8
// and 36.9. Reference mode, two slots a step: 256 workgroups 19.9 and 21.5,
// 304 20.1 and 19.2.
constexpr size_t SPLIT_DECIDE = 256;

// ws: MS part[steps*(k+1) + steps*k][nchunk], Decision dec[steps][slots],
// double csum[steps][slots][nchunk] (slots = draw_slots(mode)). bonus_pre
// (nullptr: none): each step's bonus token, drawn beforehand from target row
// k by the filtered sampler; bonus draws then copy it.
hipError_t launch_spec_accept(const float *tgt, const float *drf, const int32_t *draft_tok, int steps, int k,
                              int V, float T, const float *u_acc, const float *u_res, const float *u_bonus,
                              int mode, const int32_t *bonus_pre, int32_t *out_tok, int32_t *out_n, void *ws,
                              hipStream_t st) {
    const int nc = accept_nchunk(V);
    const float Tr = mode == 0 ? T : 1.0f;
    const int nd = draw_slots(mode);
    MS *part = (MS *)ws;
    Decision *dec = (Decision *)(part + (size_t)steps * (2 * k + 1) * nc);
    double *csum = (double *)(dec + (size_t)steps * nd);
    stats_partial_kernel<<<dim3(nc, steps * (2 * k + 1)), NT, 0, st>>>(tgt, steps * (k + 1), Tr, T, k + 1,
                                                                      drf, Tr, V, nc, nullptr, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((size_t)steps * nc * nd > SPLIT_DECIDE) {
        decide_kernel<<<steps, NT, 0, st>>>(tgt, drf, draft_tok, k, V, T, u_acc, u_res, u_bonus, mode, part, nc,
                                            bonus_pre, out_tok, out_n, dec);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        sum_kernel<<<dim3(nc, steps, nd), NT, 0, st>>>(tgt, drf, k, V, dec, nc, csum);
    } else {
        decide_sum_kernel<<<dim3(nc, steps, nd), NT, 0, st>>>(tgt, drf, draft_tok, k, V, T, u_acc, u_res, u_bonus,
                                                              mode, part, nc, bonus_pre, out_tok, out_n, dec, csum);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    sample_kernel<<<dim3(steps, nd), NT, 0, st>>>(tgt, drf, k, V, dec, nc, csum, bonus_pre, out_tok);
    return hipGetLastError();
}

hipError_t launch_argmax_partial(const float *L, int rows, int V, float2 *part, hipStream_t st) {
    const int nc = accept_nchunk(V);
    argmax_partial_kernel<<<dim3(nc, rows), NT, 0, st>>>(L, V, nc, part);
    return hipGetLastError();
}

hipError_t launch_greedy(const float2 *part, int V, const int32_t *draft_tok, int steps, int k, int32_t *out_n,
                         int32_t *out_argmax, hipStream_t st) {
    const int nc = accept_nchunk(V);
    greedy_kernel<<<steps, 64, 0, st>>>(part, nc, draft_tok, k, out_n, out_argmax);
    return hipGetLastError();
}

// ws: MS part[2n][nchunk] (target rows then draft rows), MS ms[2n] (their
// merged statistics), then (above TREE_LDS nodes) int32 [2n] and int8 [n].
size_t tree_ws(int n, int V) {
    return ((size_t)2 * n * accept_nchunk(V) + 2 * (size_t)n) * sizeof(MS) + (size_t)n * 9 + 256;
}

hipError_t launch_tree(const float *tgt, const float *drf, const int32_t *tok, const int32_t *parent, int n, int V,
                       float T, const float *u, void *ws, int32_t *out_path, int32_t *out_len, hipStream_t st) {
    const int nc = accept_nchunk(V);
    MS *part = (MS *)ws;
    MS *ms = part + (size_t)2 * n * nc;
    int32_t *wsi = (int32_t *)(ms + 2 * n);
    stats_partial_kernel<<<dim3(nc, 2 * n), NT, 0, st>>>(tgt, n, T, T, 0, drf, T, V, nc,
                                                            n <= TREE_FILTER ? parent : nullptr, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    tree_kernel<<<1, TREE_NT, 0, st>>>(tgt, drf, tok, parent, n, V, T, u, part, nc, ms, out_path, out_len, wsi);
    return hipGetLastError();
}
