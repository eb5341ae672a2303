// Routers that pick several experts a token, and what surrounds their grouped products.
//
// router_topk: from the router's fp32 logits z [T, E] the `top` experts with the largest choice
// values are taken (the lowest index wins among equals), and each gets a weight.  Four ways of scoring:
//   sigmoid (mode 0): scores s = sigmoid(z); the choice goes by s + bias (bias may be null); an expert's
//     weight is its score s without the bias, divided by the sum of the taken scores if `renorm`;
//   softmax over the taken (mode 1): the choice goes by z + bias; the weights are the softmax of the taken
//     experts' logits z alone (they add up to one; `renorm` has nothing left to do);
//   softmax over the taken, bias inside (mode 3): z + bias are the logits themselves: the choice goes by them and the
//     weights are their softmax over the taken;
//   softmax over all (mode 2): scores s = softmax(z) over every expert; choice and weights as with sigmoid.
// With `n_groups` > 1 the experts form equal groups of neighbours and only those of the `keep_groups` groups whose
// largest choice value is largest can be taken (the lowest group among equals).  The logits' rows may lie `ld` apart.
// Outputs expert[t*top + j] and weight[t*top + j] in the order of choice:
// "virtual tokens" t*top + j that the expert plan (moe_plan with its fan) sorts by expert.  router_plan: both at once.
// moe_combine: out[t] = sum_j weight[t*top + j] * y[t*top + j] (+ extra[t]) in fp32, j in order (no weights: all 1);
// the extra row may come in `n_extra` parts, T rows apart, that are added first; with `gate` it is multiplied by
// sigmoid(gate[t*ldg]).
// gated_rows: g[t] = gelu_tanh(a[t]) * table[ids[t]][col0 .. col0 + n): a gate on a per-token row
// of a table (a second, small embedding that a layer mixes into the stream).
#include "common.h"

#define TOPK_MAX_PER_LANE 8      // up to 512 experts

// The largest and the smallest of a wave's values, by moves within the vector registers, the same in every lane.  (By six steps of shuffles of
// value, expert and score an expert that is taken was a chain of 0.6 us; us before and now, with the row list: one token, 4 of 16 experts 5.2 /
// 3.6, 2 of 16 3.7 / 2.9; 8 tokens, 8 of 128 11.2 / 8.2, 8 of 512 16.9 / 13.6; 1,531, 4 of 16 10.2 / 8.5.)
#define SP_TOPK_STEP(op, ctrl, rows) x = op(x, __builtin_bit_cast(decltype(x), __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), ctrl, rows, 0xf, false)))
#define SP_TOPK_STEPS(op) /* from one lane below within 16, two, four, eight; rows 0 and 2 to 1 and 3; row 1 to 2 and 3 */ \
    SP_TOPK_STEP(op, 0x111, 0xf); SP_TOPK_STEP(op, 0x112, 0xf); SP_TOPK_STEP(op, 0x114, 0xf); SP_TOPK_STEP(op, 0x118, 0xf); \
    SP_TOPK_STEP(op, 0x142, 0xa); SP_TOPK_STEP(op, 0x143, 0xc)
__device__ __forceinline__ float topk_max(float x) {
    SP_TOPK_STEPS(fmaxf);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}
__device__ __forceinline__ int topk_min(int x) {
    SP_TOPK_STEPS(min);
    return __builtin_amdgcn_readlane(x, 63);
}
#undef SP_TOPK_STEPS
#undef SP_TOPK_STEP

// One token's choice by one wave: lane j < min(top, 64) gets the j-th taken expert and its weight, and everything is
// written to expert[] and weight[].  NU: experts a lane, so that 64 * NU >= E.
template <int NU>
__device__ __forceinline__ int topk_of_token(const float* __restrict__ logits, const float* __restrict__ bias, int* __restrict__ expert,
                                             float* __restrict__ weight, int t, int lane, int E, int ld, int top, int renorm, int mode,
                                             int n_groups, int keep_groups) {
    float s[NU], c[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = lane + u * 64;
        s[u] = 0.f; c[u] = -INFINITY;
        if (e < E) {
            const float z = logits[(size_t)t * ld + e];
            s[u] = mode == 0 ? 1.0f / (1.0f + expf(-z)) : z;
            if (mode == 3 && bias) s[u] += bias[e];
        }
    }
    if (mode == 3) { bias = nullptr; mode = 1; }
    if (mode == 2) {
        float zm = -INFINITY, zs = 0.f;
#pragma unroll
        for (int u = 0; u < NU; ++u) if (lane + u * 64 < E) zm = fmaxf(zm, s[u]);
        zm = wave_max(zm);
#pragma unroll
        for (int u = 0; u < NU; ++u) if (lane + u * 64 < E) { s[u] = expf(s[u] - zm); zs += s[u]; }
        zs = 1.0f / wave_sum(zs);
#pragma unroll
        for (int u = 0; u < NU; ++u) s[u] *= zs;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = lane + u * 64;
        if (e < E) {
            c[u] = s[u] + (bias ? bias[e] : 0.f);
            if (!(c[u] == c[u])) c[u] = -INFINITY;          // a NaN is never chosen before a number
        }
    }
    if (n_groups > 1) {
        // the best group left is the group of the best expert of the groups left
        const int gs = E / n_groups;
        int grp[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) grp[u] = (lane + u * 64) / gs;
        unsigned open = 0;                                  // bit u: this lane's expert u is in a group that stays
        for (int j = 0; j < keep_groups; ++j) {
            float best = -INFINITY; int be = 0x7fffffff;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int e = lane + u * 64;
                if (e < E && !(open >> u & 1) && (c[u] > best || (c[u] == best && e < be))) { best = c[u]; be = e; }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const float ob = __shfl_xor(best, o, 64); const int oe = __shfl_xor(be, o, 64);
                if (ob > best || (ob == best && oe < be)) { best = ob; be = oe; }
            }
            const int gb = be / gs;
#pragma unroll
            for (int u = 0; u < NU; ++u) if (lane + u * 64 < E && grp[u] == gb) open |= 1u << u;
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) if (!(open >> u & 1)) c[u] = -INFINITY;
    }
    float sum = 0.f, top_z = -INFINITY;          // mode 1: the sum of exp(z - top_z) over the taken so far
    float mine_w = 0.f; int mine_e = 0;
    for (int j = 0; j < top; ++j) {
        float best = -INFINITY; int be = 0x7fffffff; float bs = 0.f;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int e = lane + u * 64;
            if (e < E && (c[u] > best || (c[u] == best && e < be))) { best = c[u]; be = e; bs = s[u]; }
        }
        // the lanes that hold the largest value, and of them the lowest expert (one lane but for ties)
        const float most = topk_max(best);
        unsigned long long who = __ballot(best == most && be != 0x7fffffff);      // (a lane without an expert has that one)
        if (NU > 1 && (who & (who - 1))) {
            const int lowest = topk_min(best == most ? be : 0x7fffffff);          // (every lane's)
            who = __ballot(best == most && be == lowest);
        }
        const int src = __ffsll(who) - 1;
        be = __builtin_amdgcn_readlane(be, src);
        bs = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(bs), src));
        // a taken expert leaves the contest: its mark lies below every score
#pragma unroll
        for (int u = 0; u < NU; ++u) if (lane + u * 64 == be) c[u] = -INFINITY;
        if (mode == 1) {
            const float nz = fmaxf(top_z, bs);
            sum = sum * expf(top_z - nz) + expf(bs - nz);        // (exp(-inf) = 0 at the first)
            top_z = nz;
        } else {
            sum += bs;
        }
        if (lane == j % 64 && j < 64) { mine_w = bs; mine_e = be; }
        if (j >= 64 && lane == 0) { expert[(size_t)t * top + j] = be; weight[(size_t)t * top + j] = bs; }
    }
    if (mode == 1) {
        const float inv = 1.0f / sum;
        if (lane < top && lane < 64) { expert[(size_t)t * top + lane] = mine_e; weight[(size_t)t * top + lane] = expf(mine_w - top_z) * inv; }
        if (top > 64 && lane == 0) for (int j = 64; j < top; ++j) weight[(size_t)t * top + j] = expf(weight[(size_t)t * top + j] - top_z) * inv;
        return mine_e;
    }
    const float inv = renorm ? 1.0f / (sum + 1e-20f) : 1.0f;
    if (lane < top && lane < 64) { expert[(size_t)t * top + lane] = mine_e; weight[(size_t)t * top + lane] = mine_w * inv; }
    if (renorm && top > 64 && lane == 0) for (int j = 64; j < top; ++j) weight[(size_t)t * top + j] *= inv;
    return mine_e;
}

template <int NU>
__global__ __launch_bounds__(256)
void router_topk_kernel(const float* __restrict__ logits, const float* __restrict__ bias, int* __restrict__ expert,
                        float* __restrict__ weight, int T, int E, int ld, int top, int renorm, int mode,
                        int n_groups, int keep_groups) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    topk_of_token<NU>(logits, bias, expert, weight, t, threadIdx.x & 63, E, ld, top, renorm, mode, n_groups, keep_groups);
}

// The choice and the row list of the grouped products (moe_plan with a fan of `top` and `shared` groups that every token
// visits) of a step of a few tokens by one workgroup, a wave a token: two kernels become one.  Both are a chain of
// latencies: the logits' load, then a maximum over the wave for every expert that is taken.  Measured on an
// MI355X, one launch against two, us: 1 token, 1 of 16 experts 2.4 / 3.5, 4 of 64 3.3 / 4.4; 8 tokens, 2 of 16 3.4 / 4.6, 8 of
// 128 7.5 / 8.6, 8 of 512 12.6 / 14.6.  No second token a wave: its choice would wait for the first one's, which
// router_topk's further workgroups do not (when the maximum was six steps of shuffles: 16 tokens, 8 of 64 17.8 / 12.9; 64 tokens, 8 of 128 72 /
// 16; 512 tokens, 1 of 16 95 / 9.7).  The entries' experts stay in LDS in between; ranks are counted as moe_plan_kernel counts them.
#define RP_NT 512
#define RP_MAX (RP_NT / 64 * 64)       // entries: a token a wave, up to 64 experts each; a thread ranks one
template <int NU>
__global__ __launch_bounds__(RP_NT)
void router_plan_kernel(const float* __restrict__ logits, const float* __restrict__ bias, int* __restrict__ expert,
                        float* __restrict__ weight, int T, int E, int ld, int top, int renorm, int mode, int n_groups,
                        int keep_groups, int* __restrict__ src, float* __restrict__ scale, int* __restrict__ dst,
                        int* __restrict__ offsets, int shared) {
    __shared__ unsigned short e_of[RP_MAX];
    const int lane = threadIdx.x & 63, n = T * top;
    const int t = threadIdx.x >> 6;
    if (t < T) {
        const int e = topk_of_token<NU>(logits, bias, expert, weight, t, lane, E, ld, top, renorm, mode, n_groups, keep_groups);
        if (lane < top) e_of[t * top + lane] = (unsigned short)e;
    }
    __syncthreads();                                        // (the weights of this workgroup's waves are visible to it, too)
    const int i = threadIdx.x;
    if (i < n) {
        const int me = e_of[i];
        int rank = 0;
        for (int j = 0; j < n; ++j) {
            const int ej = e_of[j];
            rank += (ej < me) || (ej == me && j < i);
        }
        src[rank] = i / top; scale[rank] = weight[i]; dst[rank] = i;
    }
    for (int j = i; j < shared * T; j += RP_NT) { src[n + j] = j % T; scale[n + j] = 1.0f; dst[n + j] = n + j; }
    for (int g = i; g <= E + shared; g += RP_NT) {
        int c = 0;
        if (g <= E) for (int j = 0; j < n; ++j) c += e_of[j] < g;
        else c = n + (g - E) * T;
        offsets[g] = c;
    }
}

static int topk_check(int T, int E, int ld, int top, int mode, int n_groups, int keep_groups) {
    SP_REQUIRE(mode >= 0 && mode <= 3, "router_topk: scoring %d", mode);
    SP_REQUIRE(ld >= E, "router_topk: rows of %d logits for %d experts", ld, E);
    SP_REQUIRE(n_groups >= 1 && E > 0 && E % n_groups == 0 && keep_groups >= 1 && keep_groups <= n_groups, "router_topk: %d of %d groups of %d experts",
               keep_groups, n_groups, E);
    SP_REQUIRE(top <= keep_groups * (E / n_groups), "router_topk: %d experts out of %d groups of %d", top, keep_groups, E / n_groups);
    SP_REQUIRE(T >= 0 && E > 0 && E <= 64 * TOPK_MAX_PER_LANE, "router_topk: %d experts, at most %d", E, 64 * TOPK_MAX_PER_LANE);
    SP_REQUIRE(top > 0 && top <= E, "router_topk: %d of %d experts", top, E);
    return 0;
}
#define SP_BY_EXPERTS(GO) do { if (E <= 64) GO(1); else if (E <= 128) GO(2); else if (E <= 256) GO(4); else GO(TOPK_MAX_PER_LANE); } while (0)

extern "C" int spite_router_topk(const float* logits, const float* bias, int* expert, float* weight, int T, int E, int ld, int top,
                                 int renorm, int mode, int n_groups, int keep_groups, hipStream_t st) {
    if (int rc = topk_check(T, E, ld, top, mode, n_groups, keep_groups)) return rc;
    if (T == 0) return 0;
#define SP_RT(NU) router_topk_kernel<NU><<<(T + 3) / 4, 256, 0, st>>>(logits, bias, expert, weight, T, E, ld, top, renorm, mode, n_groups, keep_groups)
    SP_BY_EXPERTS(SP_RT);
#undef SP_RT
    SP_LAUNCH_CHECK("router_topk");
    return 0;
}

extern "C" int spite_moe_plan(int* expert, float* weight, const float* logits, int* src, float* scale, int* dst,
                              int* offsets, int T, int E, int shared, int fan, hipStream_t st);

// Whether router_plan makes choice and row list in one launch.
extern "C" int spite_router_plan_is_one_launch(int T, int top) { return T > 0 && T <= RP_NT / 64 && top <= 64; }

// router_topk, then moe_plan over its T * top entries with `shared` groups of T rows behind the experts'; in one launch
// for a few tokens.
extern "C" int spite_router_plan(const float* logits, const float* bias, int* expert, float* weight, int T, int E, int ld, int top,
                                 int renorm, int mode, int n_groups, int keep_groups, int* src, float* scale, int* dst,
                                 int* offsets, int shared, hipStream_t st) {
    if (int rc = topk_check(T, E, ld, top, mode, n_groups, keep_groups)) return rc;
    SP_REQUIRE(shared >= 0 && shared <= 64, "router_plan: %d shared groups", shared);
    if (!spite_router_plan_is_one_launch(T, top)) {
        if (int rc = spite_router_topk(logits, bias, expert, weight, T, E, ld, top, renorm, mode, n_groups, keep_groups, st)) return rc;
        return spite_moe_plan(expert, weight, nullptr, src, scale, dst, offsets, T * top, E, shared, top, st);
    }
#define SP_RP(NU) router_plan_kernel<NU><<<1, RP_NT, 0, st>>>(logits, bias, expert, weight, T, E, ld, top, renorm, mode, n_groups, \
                                                              keep_groups, src, scale, dst, offsets, shared)
    SP_BY_EXPERTS(SP_RP);
#undef SP_RP
    SP_LAUNCH_CHECK("router_plan");
    return 0;
}

// VEC elements a thread (4 where rows are a multiple of four floats and 16-byte aligned); every element is summed in
// the same order either way.
template <int VEC>
__global__ __launch_bounds__(256)
void moe_combine_kernel(const float* __restrict__ y, const float* __restrict__ weight, const float* __restrict__ extra,
                        const float* __restrict__ gate, int ldg, float* __restrict__ out, int T, int d, int top, int n_extra) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int dv = d / VEC;
    if (i >= (size_t)T * dv) return;
    const size_t t = i / dv, c = (i - t * dv) * VEC;
    vec acc;
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    for (int j = 0; j < top; ++j) {
        const float w = weight ? weight[t * top + j] : 1.0f;
        const vec v = *(const vec*)(y + (t * top + j) * d + c);
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = fmaf(w, v[e], acc[e]);
    }
    if (extra) {
        vec x = *(const vec*)(extra + t * d + c);
        for (int j = 1; j < n_extra; ++j) x += *(const vec*)(extra + ((size_t)j * T + t) * d + c);
        const float g = gate ? 1.0f / (1.0f + expf(-gate[t * ldg])) : 1.0f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += g * x[e];
    }
    *(vec*)(out + t * d + c) = acc;
}

extern "C" int spite_moe_combine(const float* y, const float* weight, const float* extra, const float* gate, int ldg, float* out,
                                 int T, int d, int top, int n_extra, hipStream_t st) {
    SP_REQUIRE(T >= 0 && d > 0 && top > 0 && n_extra >= 1, "moe_combine: bad sizes T=%d d=%d top=%d, %d extra rows", T, d, top, n_extra);
    SP_REQUIRE(!gate || (extra && ldg >= 1), "moe_combine: a gate without the row that it gates");
    if (T == 0) return 0;
    auto al = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    const bool v4 = d % 4 == 0 && al(y) && al(extra) && al(out);
    const size_t n = (size_t)T * (v4 ? d / 4 : d);
    SP_REQUIRE((n + 255) / 256 < (1u << 31), "moe_combine: too many elements");
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (v4) moe_combine_kernel<4><<<grid, 256, 0, st>>>(y, weight, extra, gate, ldg, out, T, d, top, n_extra);
    else moe_combine_kernel<1><<<grid, 256, 0, st>>>(y, weight, extra, gate, ldg, out, T, d, top, n_extra);
    SP_LAUNCH_CHECK("moe_combine");
    return 0;
}

template <typename TA, typename TT>
__global__ __launch_bounds__(256)
void gated_rows_kernel(const TA* __restrict__ a, const int* __restrict__ ids, const TT* __restrict__ table, int ld_table,
                       int col0, TA* __restrict__ g, int T, int n, int fast) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * n) return;
    const size_t t = i / n, c = i - t * n;
    const float z = to_f32<TA>(a[i]);
    const float act = 0.5f * z * (1.0f + (fast ? 1.0f - 2.0f / (__expf(2.0f * 0.7978845608028654f * (z + 0.044715f * z * z * z)) + 1.0f)
                                              : tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z))));
    g[i] = from_f32<TA>(act * to_f32<TT>(table[(size_t)ids[t] * ld_table + col0 + c]));
}

extern "C" int spite_gated_rows(const void* a, int dtype, const int* ids, const void* table, int table_dtype, int ld_table,
                                int col0, void* g, int T, int n, hipStream_t st) {
    SP_REQUIRE(T >= 0 && n > 0 && col0 >= 0 && col0 + n <= ld_table, "gated_rows: columns %d..%d of %d", col0, col0 + n, ld_table);
    if (T == 0) return 0;
    const unsigned grid = (unsigned)(((size_t)T * n + 255) / 256);
    if (dtype == SP_F32 && table_dtype == SP_F32)
        gated_rows_kernel<float, float><<<grid, 256, 0, st>>>((const float*)a, ids, (const float*)table, ld_table, col0, (float*)g, T, n, 0);
    else if (dtype == SP_BF16 && table_dtype == SP_BF16)
        gated_rows_kernel<bf16, bf16><<<grid, 256, 0, st>>>((const bf16*)a, ids, (const bf16*)table, ld_table, col0, (bf16*)g, T, n, 1);
    else if (dtype == SP_BF16 && table_dtype == SP_F32)
        gated_rows_kernel<bf16, float><<<grid, 256, 0, st>>>((const bf16*)a, ids, (const float*)table, ld_table, col0, (bf16*)g, T, n, 1);
    else return sp_fail("gated_rows: dtypes %d and %d", dtype, table_dtype);
    SP_LAUNCH_CHECK("gated_rows");
    return 0;
}
