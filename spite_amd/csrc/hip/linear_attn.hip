// Linear attention: a recurrent state per head instead of a cache of keys and values.
//
//   S_t = diag(a_t) S_(t-1) + k_t v_t^T        (S: D x V per head; a_t decays the rows, one per key channel)
//   o_t = S_t^T q_t
//
// The decay a_t is either a number per key channel that the token decides (`decay` fp32 [T, H*D]) or a
// constant per head (`head_decay` fp32 [H]).  The state lives in fp32 in a row per request slot,
// [slots, H, D, V]; every sum and product of the recurrence is fp32 whatever the type of q, k and v.
//
// Options of the recurrence: `qk_heads` < H: several heads share one q and one k head (head h reads q/k head
// h / (H / qk_heads)); `v_scale` fp32 [T, H]: the token's value row of a head is multiplied by a number in fp32 before it
// enters the state (a step size); `bonus` fp32 [H, D]: the result is read off the state *before* the token enters it, and the
// token's own outer product counts with a weight per key channel instead:
//   o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t,   S_t = diag(a_t) S_(t-1) + k_t v_t^T.
//
// channel_decay:      z -> sigmoid(z + b)^(1/tau) in place, through its logarithm; or z -> exp(-exp(z + b)).
// linear_attn_scan:   the recurrence token by token, in fp32 FMAs, with the tokens' rows staged through LDS in
//                     blocks; its bits do not depend on how a request's tokens are cut into steps.
// gated_group_norm:   y = rmsnorm(o over groups of `group` elements) * w * act(gate), the step between the
//                     recurrence and the output projection.
#include "common.h"
#include <type_traits>

// ------------------------------------------------------------------ decay per channel
// a = sigmoid(z + b)^(1/tau) = exp(log sigmoid(z + b) / tau), log sigmoid(x) = -(max(-x, 0) + log1p(exp(-|x|))).
__global__ __launch_bounds__(256)
void channel_decay_kernel(float* __restrict__ z, const float* __restrict__ bias, size_t n, int width, float inv_tau, int mode) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const float x = z[i] + (bias ? bias[i % width] : 0.f);
        if (mode == 1) { z[i] = expf(-expf(x)); continue; }
        const float ls = -(fmaxf(-x, 0.f) + log1pf(expf(-fabsf(x))));
        z[i] = expf(ls * inv_tau);
    }
}

extern "C" int spite_channel_decay(float* z, const float* bias, int T, int width, float inv_tau, int mode, hipStream_t st) {
    SP_REQUIRE(mode == 0 || mode == 1, "channel_decay: mode %d", mode);
    SP_REQUIRE(T >= 0 && width > 0 && inv_tau > 0.f, "channel_decay: bad sizes T=%d width=%d 1/tau=%g", T, width, (double)inv_tau);
    const size_t n = (size_t)T * width;
    if (n == 0) return 0;
    const int blocks = (int)((n + 255) / 256 < 16384 ? (n + 255) / 256 : 16384);
    channel_decay_kernel<<<blocks, 256, 0, st>>>(z, bias, n, width, inv_tau, mode);
    SP_LAUNCH_CHECK("channel_decay");
    return 0;
}

// ------------------------------------------------------------------ the recurrence, token by token
// A workgroup of 512 threads takes 16 value columns of one head of one entry of the step and walks the
// entry's tokens in order.  Thread (vc, dg) = (tid / 32, tid % 32) holds, in registers, the state's elements
// S[d][v0 + vc] for D / 32 key channels d (four consecutive ones at 4 dg, and again 128
// further on for the widest heads; two at 2 dg for heads up to 64): 32 lanes read 512 consecutive bytes of a
// token's q, k or decay row from LDS in one wide read without bank conflicts.  The tokens' q, k, decay and value slice go
// through LDS a block of tokens at a time, two buffers: the next block's loads are in flight while this block is computed,
// and nothing looks at a loaded value before that (the places of what lies outside the head are cleared once).  A whole
// block is one stretch of code: only the state's FMA waits for the token before.  The sums over the key channels are taken
// for the tokens of a block together (la_sums).  The state tile goes through LDS on the way in and out, so that its rows
// are read and written 64 bytes at a time.
// Bound by the instructions that a wave issues: at D = 128, 12 a token for the state and 17 around them (the reads from LDS,
// the sums, the fetches), 180 cycles a token with two waves a SIMD.  So a fetch is set up once and costs a compare, a select
// and an add a block; k, and what lies outside a head, take no product or select on the way into LDS, tokens past the last none at all;
// and no store is waited for (an asm statement below pins where the loads are waited for: with the loads in branches the compiler
// also waited at the head of each block, for the block's stores with them).  At the start, what is the same for a
// workgroup is asked for at once, then the state, then the first tokens.  128 registers, so that two workgroups fit a CU, for
// the widest heads too (their rows are read one token ahead where there is a decay per channel).
// us, and in brackets before a fetch was set up once: 1,531 tokens, one request, V = D = 128: 107 for 16 heads
// and 108 for 32 (126 and 127), decay per channel 135 (159) and 218 for 40 heads (248); heads of 64: 93 (104);
// 800 tokens, 8 heads of 256: 102 (122), decay per channel 124 (146); 3 requests of 700 tokens, 40 heads of 256 with a decay
// per channel: 363 (406; 453 with 153 registers); 32 of 17 tokens, 16 heads: 64 (83; 102).  1,000 tokens of fp32,
// 16 heads: 83 (121).  Tried: two columns a lane, which halves the reads of q and k (168 us with 16 columns a workgroup);
// half the columns a workgroup where 128 workgroups leave CUs idle (122, 77 for heads of 64); loads two blocks ahead (124); addresses
// from one scalar base and 32-bit offsets (fp32 5 to 14 % slower, short entries no faster).
// The order of every sum is fixed by D alone: the bits do not depend on how a request's tokens are cut.
#define LA_VC 16        // value columns a workgroup
#define LA_NT 512       // threads a workgroup: 16 columns x 32 lanes
#define LA_DG 32        // lanes that share a column's key channels
#define LA_MAXD 256

template <int RR> struct la_block { static constexpr int tokens = RR == 16 ? 8 : 16; };

// The sum over 32 lanes (two rows of 16) of each of TB values: lane l against l ^ 16, ^ 15, ^ 7, ^ 2 and ^ 1 in turn.  As
// long as there are two values left, the lanes with the step's bit clear (4, 3, 2, 1 and 0) go on with the first half of
// them and the others with the second half, so that a step halves the values instead of repeating itself for each: 38
// instructions for 16 values, against 96 and a wait between most of them.  The pairs that are added do not depend on TB.
// Lane l ends with value la_owner<TB>(l)'s sum.
template <int CTRL> __device__ __forceinline__ float la_from(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int CTRL, int BIT, int N> __device__ __forceinline__ void la_halve(float* x, int l) {
    if constexpr (N > 1) {
        const bool up = l & BIT;
#pragma unroll
        for (int j = 0; j < N / 2; ++j) {
            const float keep = up ? x[j + N / 2] : x[j], give = up ? x[j] : x[j + N / 2];
            x[j] = keep + la_from<CTRL>(give);
        }
    } else x[0] += la_from<CTRL>(x[0]);
}
template <int TB> __device__ __forceinline__ float la_sums(float* x, int l) {
    constexpr int H = TB > 1 ? TB / 2 : 1;
#pragma unroll
    for (int j = 0; j < H; ++j) {                    // (the swap exchanges the first's odd rows with the second's even ones)
        const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[j]), __float_as_uint(x[TB > 1 ? j + H : j]), false, false);
        x[j] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    }
    la_halve<0x140, 8, H>(x, l);                     // row_mirror
    la_halve<0x141, 4, (H > 1 ? H / 2 : 1)>(x, l);   // row_half_mirror
    la_halve<0x4e, 2, (H > 2 ? H / 4 : 1)>(x, l);    // quad_perm 2 3 0 1
    la_halve<0xb1, 1, (H > 4 ? H / 8 : 1)>(x, l);    // quad_perm 1 0 3 2
    return x[0];
}
template <int TB> __device__ __forceinline__ int la_owner(int l) { return TB == 16 ? l >> 1 : TB == 8 ? l >> 2 : 0; }

#define LA_OWN(r) (PR >= 4 ? ((r) / 4) * 128 + dg * 4 + ((r) % 4) : dg * PR + (r))    // the thread's r-th key channel

// The workgroup's columns of the state, in and out through LDS (D rows of LA_VC + 1): a thread's PR loads are all asked for
// before the first is waited for (one
// after another, a step of single tokens of 8 requests with 16 heads of 128 took 7.5 us for 7.0, of 32 requests 21.3 for 18.4).
template <int PR> __device__ __forceinline__ void la_state_ask(float* x, const float* srow, int D, int V, int v0) {
    const int tid = threadIdx.x, c = tid % LA_VC;
#pragma unroll
    for (int u = 0; u < PR; ++u) {
        const int d = tid / LA_VC + u * (LA_NT / LA_VC);
        x[u] = srow[d < D && v0 + c < V ? (size_t)d * V + v0 + c : 0];
    }
}
template <int PR> __device__ __forceinline__ void la_state_in(float* S, const float* x, float* sm, int D, int V, int v0) {
    const int tid = threadIdx.x, vc = tid / LA_DG, dg = tid % LA_DG, c = tid % LA_VC;
#pragma unroll
    for (int u = 0; u < PR; ++u) {
        const int d = tid / LA_VC + u * (LA_NT / LA_VC);
        sm[d * (LA_VC + 1) + c] = d < D && v0 + c < V ? x[u] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PR; ++r) S[r] = sm[LA_OWN(r) * (LA_VC + 1) + vc];
    __syncthreads();
}
template <int PR> __device__ __forceinline__ void la_state_out(const float* S, float* srow, float* sm, int D, int V, int v0) {
    const int tid = threadIdx.x, vc = tid / LA_DG, dg = tid % LA_DG, c = tid % LA_VC;
#pragma unroll
    for (int r = 0; r < PR; ++r) sm[LA_OWN(r) * (LA_VC + 1) + vc] = S[r];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PR; ++u) {
        const int d = tid / LA_VC + u * (LA_NT / LA_VC);
        if (d < D && v0 + c < V) srow[(size_t)d * V + v0 + c] = sm[d * (LA_VC + 1) + c];
    }
}

// VEC: q, k, v (bfloat16) and the decay rows start on 16 bytes and D and V are multiples of 8: a fetch is
// 16 bytes.  Otherwise one element.  (Every loop over the arrays below is unrolled and both lambdas are inlined, so that
// the arrays stay in registers.)
// TB: tokens a block: 16 (8 for the widest heads).
template <typename T, int RR, bool CH, bool VEC, bool PRE>
__global__ __launch_bounds__(LA_NT) __attribute__((amdgpu_waves_per_eu(VEC ? 4 : 1, VEC ? 4 : 2)))
void linear_attn_scan_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int ldq, int ldk, int ldv,
                             const float* __restrict__ decay, const float* __restrict__ head_decay, float q_scale,
                             float* __restrict__ state, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slots,
                             float* __restrict__ out, int H, int D, int V, int keep, int qk_rep,
                             const float* __restrict__ v_scale, const float* __restrict__ bonus) {
    constexpr int TB = la_block<RR>::tokens;
    constexpr int Dp = 16 * RR;                     // key channels, padded
    constexpr int PR = RR / 2;                      // key channels a thread
    constexpr int NQ = CH ? 3 : 2;                  // rows of Dp a token: q, k and, per channel, the decay
    constexpr int per = NQ * Dp + LA_VC;
    // A fetch is one load and no branch around it.  Three lists of fetches a block: q and k, the value slice (elements
    // of type T) and the decay rows (fp32).
    constexpr int WA = VEC ? 8 : 1, WB = VEC ? 4 : 1;               // elements a fetch
    constexpr int NQF = TB * Dp / WA, CV = LA_VC / WA, CB = Dp / WB;   // fetches: q's of a block; of v's slice and of the decay a token
    constexpr int UQ = (2 * NQF + LA_NT - 1) / LA_NT, UB = CH ? (TB * CB + LA_NT - 1) / LA_NT : 0;      // fetches a thread and block
    static_assert(TB * CV <= LA_NT, "linear_attn_scan: the value slice is one fetch a thread");
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int PV = PR < 4 ? PR : 4;             // key channels an LDS read
    constexpr int LOOK = RR == 16 ? (CH && VEC ? 1 : 2) : CH && RR == 8 ? 3 : 4;            // tokens whose rows are on their way from LDS
    typedef float vec __attribute__((ext_vector_type(PV)));
    using RawA = typename std::conditional<VEC, u32x4, T>::type;
    using RawB = typename std::conditional<VEC, f32x4, float>::type;
    extern __shared__ __attribute__((aligned(16))) float sm[];      // max(2 * TB * per, Dp * (LA_VC + 1)) floats
    const int e = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * LA_VC;
    const int tid = threadIdx.x, vc = tid / LA_DG, dg = tid % LA_DG;
    // (all that is the same for the workgroup at once: left where they are used, these loads are five more waits in a row,
    // half a microsecond that an entry of few tokens cannot hide)
    asm volatile("" :: "s"(q), "s"(k), "s"(v), "s"(decay), "s"(state), "s"(out), "s"(v_scale), "s"(H), "s"(D), "s"(V), "s"(keep), "s"(qk_rep),
                 "s"(ldq), "s"(ldk), "s"(ldv), "s"(q_scale));
    int t_lo = cu_seqlens[e], t_hi = cu_seqlens[e + 1], slot = seq_slots[e];
    float hd = CH ? 1.f : head_decay[h];
    asm volatile("" : "+s"(t_lo), "+s"(t_hi), "+s"(slot), "+s"(hd));
    if (t_lo >= t_hi) return;
    float* srow = state + ((size_t)slot * H + h) * (size_t)D * V;
    float S[PR], x[PR];
    la_state_ask<PR>(x, srow, D, V, v0);                    // (on its way while the fetches are set up)
    const int hq = qk_rep == 1 ? h : h / qk_rep;            // the head of q and k that this head reads
    // The thread's fetches: where the next block's lie, what one block further is, whether they are part of the head, and
    // their place in a block's buffer.
    const T* pq[UQ]; size_t sq[UQ]; int jq[UQ], wq[UQ]; float mq[UQ]; bool iq[UQ];
    const float* pb[UB > 0 ? UB : 1]; int jb[UB > 0 ? UB : 1], wb[UB > 0 ? UB : 1]; bool ib[UB > 0 ? UB : 1];
    const int jv0 = tid / CV, cv = (tid % CV) * WA, wv = jv0 * per + NQ * Dp + cv;
    const bool iv = jv0 < TB && v0 + cv < V;
    int jv = t_lo + jv0;
    const T *pv = v + (size_t)jv * ldv + h * V + v0 + cv, *some = q + (size_t)t_lo * ldq + hq * D;   // (some: for fetches outside the head or past the last token)
#pragma unroll
    for (int u = 0; u < UQ; ++u) {
        const int x = tid + u * LA_NT, part = x / NQF, j = x % NQF / (Dp / WA), d = x % (Dp / WA) * WA;
        const int ld = part ? ldk : ldq;
        iq[u] = part < 2 && d < D;
        jq[u] = t_lo + j; wq[u] = j * per + part * Dp + d; mq[u] = part ? 1.f : q_scale; sq[u] = (size_t)TB * ld;
        pq[u] = (part ? k : q) + (size_t)(t_lo + j) * ld + hq * D + d;
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
        const int x = tid + u * LA_NT, j = x / CB, d = (x % CB) * WB;
        ib[u] = j < TB && d < D;
        jb[u] = t_lo + j; wb[u] = j * per + 2 * Dp + d;
        pb[u] = decay + ((size_t)(t_lo + j) * H + h) * D + d;
    }
    RawA nq[UQ], nv;
    float fv = 1.f;                                          // the factor on the value fetch
    asm volatile("" : "+v"(fv));                             // (written here: behind a load it would wait for it)
    RawB nb[UB > 0 ? UB : 1];
    bool gq[UQ], gv = false, gb[UB > 0 ? UB : 1];            // which of the fetches asked for last there are
    auto ask = [&]() __attribute__((always_inline)) {        // asks for the next block in order
#pragma unroll
        for (int u = 0; u < UQ; ++u) {
            const bool ok = iq[u] && jq[u] < t_hi;
            gq[u] = VEC ? ok : iq[u];
            nq[u] = *(const RawA*)(ok ? pq[u] : some);
            pq[u] += sq[u]; jq[u] += TB;
        }
        gv = iv && jv < t_hi;
        nv = *(const RawA*)(gv ? pv : some);
        if (v_scale) fv = v_scale[(size_t)(gv ? jv : t_lo) * H + h];
        pv += (size_t)TB * ldv; jv += TB;
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const bool ok = ib[u] && jb[u] < t_hi;
            gb[u] = VEC ? ok : ib[u];
            nb[u] = *(const RawB*)(ok ? pb[u] : decay);
            pb[u] += (size_t)TB * H * D; jb[u] += TB;
        }
    };
    ask();
    la_state_in<PR>(S, x, sm, D, V, v0);
    if (D < Dp || v0 + LA_VC > V) {                            // the places of what lies outside the head, in both buffers: never written again
        auto clear = [&](int at, int n) __attribute__((always_inline)) {
            for (int i = 0; i < n; ++i) sm[at + i] = sm[TB * per + at + i] = 0.f;
        };
#pragma unroll
        for (int u = 0; u < UQ; ++u) if (!iq[u] && tid + u * LA_NT < 2 * NQF) clear(wq[u], WA);
        if (jv0 < TB && !iv) clear(wv, WA);
#pragma unroll
        for (int u = 0; u < UB; ++u) if (!ib[u] && tid + u * LA_NT < TB * CB) clear(wb[u], WB);
    }
    float ub[PRE ? PR : 1];
    if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r < PR; ++r) { const int d = LA_OWN(r); ub[r] = d < D ? bonus[(size_t)h * D + d] : 0.f; }
    }
    const int own = la_owner<TB>(dg);                        // the token of a block whose result the thread stores
    const bool stores = dg % (LA_DG / TB) == 0 && v0 + vc < V;
    float* po = out + ((size_t)(t_lo + own) * H + h) * V + v0 + vc;
    // Turn `it` computes block `it` from buffer it & 1 while block it + 1 is on its way into the other one;
    // turn -1 only fetches.
    const int n_blocks = (t_hi - t_lo + TB - 1) / TB;
    for (int it = -1; it < n_blocks; ++it) {
        const int t0 = t_lo + it * TB;                              // this block's first token
        const bool more = it + 1 < n_blocks;
        float accs[TB];
        const float* cur = sm + (it & 1) * (TB * per);
        const int n_tok = t_hi - t0 < TB ? t_hi - t0 : TB;
        // A whole block is one stretch of code, its tokens' rows read LOOK tokens ahead of their use (the barriers keep
        // the compiler from moving the reads back to it): only the state's FMA waits for the token before.
        vec q4[LOOK][PR / PV], k4[LOOK][PR / PV], a4[CH ? LOOK : 1][PR / PV];
        float vv[LOOK];
        auto read = [&](int j) {
            const float* row = cur + j * per;
            vv[j % LOOK] = row[NQ * Dp + vc];
#pragma unroll
            for (int r = 0; r < PR; r += PV) {
                q4[j % LOOK][r / PV] = *(const vec*)(row + LA_OWN(r));
                k4[j % LOOK][r / PV] = *(const vec*)(row + Dp + LA_OWN(r));
                if constexpr (CH) a4[j % LOOK][r / PV] = *(const vec*)(row + 2 * Dp + LA_OWN(r));
            }
        };
        auto token = [&](int j) {                               // the state moves on; the thread's part of the result
            accs[j] = 0.f;
#pragma unroll
            for (int r = 0; r < PR; ++r) {
                float a = hd;
                if constexpr (CH) a = a4[j % LOOK][r / PV][r % PV];
                const float qr = q4[j % LOOK][r / PV][r % PV], kv = k4[j % LOOK][r / PV][r % PV] * vv[j % LOOK];
                if (PRE) accs[j] = fmaf(fmaf(ub[PRE ? r : 0], kv, S[r]), qr, accs[j]);
                S[r] = fmaf(a, S[r], kv);
                if (!PRE) accs[j] = fmaf(S[r], qr, accs[j]);
            }
        };
        if (it >= 0) {
#pragma unroll
            for (int j = 0; j < LOOK; ++j) read(j);
            __builtin_amdgcn_sched_barrier(0x7);
            if (!VEC) ask();
            if (n_tok == TB) {
                if (VEC) ask();
#pragma unroll
                for (int j = 0; j < TB; ++j) {
                    __builtin_amdgcn_sched_barrier(0x7);
                    token(j);
                    if (j + LOOK < TB) read(j + LOOK);
                }
                __builtin_amdgcn_sched_barrier(0x7);
            } else {                                            // (the last block: nothing left to ask for)
#pragma unroll
                for (int j = 0; j < TB; ++j) {
                    accs[j] = 0.f;
                    if (j < n_tok) { read(j); token(j); }
                }
            }
        }
        // The loads are waited for here, whatever the branches below do: what the compiler holds for pending at the head of the
        // loop it waits for there, and for this block's stores with it.
#pragma unroll
        for (int u = 0; u < UQ; ++u) asm volatile("" : "+v"(nq[u]));
        asm volatile("" : "+v"(nv), "+v"(fv));
#pragma unroll
        for (int u = 0; u < UB; ++u) asm volatile("" : "+v"(nb[u]));
        if (more) {
            float* buf = sm + ((it + 1) & 1) * (TB * per);
            auto put = [&](float* dst, const RawA& got, float m) __attribute__((always_inline)) {
                if constexpr (VEC) {
                    const u32x4 w = got;
                    f32x4 lo, hi;
                    lo.x = __builtin_bit_cast(float, w.x << 16) * m, lo.y = __builtin_bit_cast(float, w.x & 0xffff0000u) * m;
                    lo.z = __builtin_bit_cast(float, w.y << 16) * m, lo.w = __builtin_bit_cast(float, w.y & 0xffff0000u) * m;
                    hi.x = __builtin_bit_cast(float, w.z << 16) * m, hi.y = __builtin_bit_cast(float, w.z & 0xffff0000u) * m;
                    hi.z = __builtin_bit_cast(float, w.w << 16) * m, hi.w = __builtin_bit_cast(float, w.w & 0xffff0000u) * m;
                    *(f32x4*)dst = lo;
                    *(f32x4*)(dst + 4) = hi;
                } else dst[0] = to_f32<T>(got) * m;
            };
#pragma unroll
            for (int u = 0; u < UQ; ++u) if (gq[u]) put(buf + wq[u], nq[u], u * LA_NT >= NQF ? 1.f : mq[u]);   // (known for k: no product)
            if (gv) put(buf + wv, nv, fv);
#pragma unroll
            for (int u = 0; u < UB; ++u) if (gb[u]) *(RawB*)(buf + wb[u]) = nb[u];
        }
        if (it < 0) { __syncthreads(); continue; }
        const float mine = la_sums<TB>(accs, dg);
        // the block's results leave after the next block's rows are in LDS: waiting for those loads does not wait for these stores
        if (stores && t0 + own < t_hi) *po = mine;
        po += (size_t)TB * H * V;
        __syncthreads();
    }
    if (keep) la_state_out<PR>(S, srow, sm, D, V, v0);
}

// Steps of single tokens: workgroups that hold little LDS and few registers, so that many are resident and their round
// trips to memory overlap (the scan, 32 requests of a token, 16 heads of 128: 26.7 us for 18.4).  The same sums in the same order; an
// entry of more tokens is right too, a token at a time.
template <typename T, int RR, bool CH, bool VEC, bool PRE>
__global__ __launch_bounds__(LA_NT) __attribute__((amdgpu_waves_per_eu(1, 4)))
void linear_attn_single_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int ldq, int ldk, int ldv,
                             const float* __restrict__ decay, const float* __restrict__ head_decay, float q_scale,
                             float* __restrict__ state, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slots,
                             float* __restrict__ out, int H, int D, int V, int keep, int qk_rep,
                             const float* __restrict__ v_scale, const float* __restrict__ bonus) {
    constexpr int Dp = 16 * RR;                     // key channels, padded
    constexpr int PR = RR / 2;                      // key channels a thread
    constexpr int NQ = CH ? 3 : 2;                  // rows of Dp a token: q, k and, per channel, the decay
    constexpr int per = NQ * Dp + LA_VC;
    // Two lists of fetches: A from q, k and the value slice (elements of type T), B from the decay rows (fp32).
    constexpr int WA = VEC ? 8 : 1, WB = VEC ? 4 : 1;               // elements a fetch
    constexpr int CA = (2 * Dp + LA_VC) / WA, CB = CH ? Dp / WB : 1; // fetches a token
    constexpr int UA = (CA + LA_NT - 1) / LA_NT, UB = CH ? (CB + LA_NT - 1) / LA_NT : 0;     // fetches a thread
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int PV = PR < 4 ? PR : 4;             // key channels an LDS read
    typedef float vec __attribute__((ext_vector_type(PV)));
    using RawA = typename std::conditional<VEC, u32x4, T>::type;
    using RawB = typename std::conditional<VEC, f32x4, float>::type;
    extern __shared__ __attribute__((aligned(16))) float sm[];      // max(2 * per, Dp * (LA_VC + 1)) floats
    const int e = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * LA_VC;
    const int tid = threadIdx.x, vc = tid / LA_DG, dg = tid % LA_DG;
    const int t_lo = cu_seqlens[e], t_hi = cu_seqlens[e + 1];
    if (t_lo >= t_hi) return;
    const int vcol = v0 + vc;
    const bool vok = vcol < V;
    float* srow = state + ((size_t)seq_slots[e] * H + h) * (size_t)D * V;
    float S[PR];
    float x[PR];
    la_state_ask<PR>(x, srow, D, V, v0);
    la_state_in<PR>(S, x, sm, D, V, v0);
    const float hd = CH ? 1.f : head_decay[h];
    const int hq = h / qk_rep;
    float ub[PRE ? PR : 1];
    if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r < PR; ++r) { const int d = LA_OWN(r); ub[r] = d < D ? bonus[(size_t)h * D + d] : 0.f; }
    }
    RawA na[UA];
    float ns[UA];                                            // the factor on a fetch's elements
    RawB nb[UB > 0 ? UB : 1];
    for (int t = t_lo - 1; t < t_hi; ++t) {                 // (turn t_lo - 1 only fetches)
        const int tn = t + 1;
        const bool more = tn < t_hi;
        if (more) {
#pragma unroll
            for (int u = 0; u < UA; ++u) {
                const int e0 = (tid + u * LA_NT) * WA, part = e0 / Dp, d = e0 % Dp;
                // q and k: channel d of the head; the value slice: column v0 + e0 - 2 Dp
                const T* base = part == 0 ? q : part == 1 ? k : v;
                const int ld = part == 0 ? ldq : part == 1 ? ldk : ldv;
                const int col = part < 2 ? hq * D + d : h * V + v0 + (e0 - 2 * Dp);
                const bool ok = e0 < CA * WA && (part < 2 ? d < D : v0 + (e0 - 2 * Dp) < V);
                na[u] = *(const RawA*)(base + (size_t)(ok ? tn : t_lo) * ld + (ok ? col : 0));
                ns[u] = part == 0 ? q_scale : (part == 2 && v_scale) ? v_scale[(size_t)(ok ? tn : t_lo) * H + h] : 1.f;
            }
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const int d = (tid + u * LA_NT) * WB;
                const bool ok = d < D;
                nb[u] = *(const RawB*)(decay + ((size_t)(ok ? tn : t_lo) * H + h) * D + (ok ? d : 0));
            }
        }
        float mine = 0.f;
        if (t >= t_lo) {
            const float* row = sm + ((t - t_lo) & 1) * per;
            const float vv = row[NQ * Dp + vc];
#pragma unroll
            for (int r = 0; r < PR; r += PV) {
                const vec q4 = *(const vec*)(row + LA_OWN(r)), k4 = *(const vec*)(row + Dp + LA_OWN(r));
                vec a4;
                if constexpr (CH) a4 = *(const vec*)(row + 2 * Dp + LA_OWN(r));
#pragma unroll
                for (int x = 0; x < PV; ++x) {
                    float a = hd;
                    if constexpr (CH) a = a4[x];
                    const float kv = k4[x] * vv;
                    if (PRE) mine = fmaf(fmaf(ub[PRE ? r + x : 0], kv, S[r + x]), q4[x], mine);
                    S[r + x] = fmaf(a, S[r + x], kv);
                    if (!PRE) mine = fmaf(S[r + x], q4[x], mine);
                }
            }
            mine = la_sums<1>(&mine, dg);
        }
        if (more) {
            float* buf = sm + ((tn - t_lo) & 1) * per;
#pragma unroll
            for (int u = 0; u < UA; ++u) {
                const int e0 = (tid + u * LA_NT) * WA, part = e0 / Dp;
                if (e0 < CA * WA) {
                    float* dst = buf + (part < 2 ? e0 : e0 + (NQ - 2) * Dp);
                    const float m = ns[u];
                    const bool in = ((part < 2) & (e0 % Dp < D)) | ((part >= 2) & (v0 + (e0 - 2 * Dp) < V));
                    const RawA got = in ? na[u] : RawA{};
                    if constexpr (VEC) {
                        const u32x4 w = got;
                        f32x4 lo, hi;
                        lo.x = __builtin_bit_cast(float, w.x << 16) * m, lo.y = __builtin_bit_cast(float, w.x & 0xffff0000u) * m;
                        lo.z = __builtin_bit_cast(float, w.y << 16) * m, lo.w = __builtin_bit_cast(float, w.y & 0xffff0000u) * m;
                        hi.x = __builtin_bit_cast(float, w.z << 16) * m, hi.y = __builtin_bit_cast(float, w.z & 0xffff0000u) * m;
                        hi.z = __builtin_bit_cast(float, w.w << 16) * m, hi.w = __builtin_bit_cast(float, w.w & 0xffff0000u) * m;
                        *(f32x4*)dst = lo;
                        *(f32x4*)(dst + 4) = hi;
                    } else dst[0] = to_f32<T>(got) * m;
                }
            }
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const int d = (tid + u * LA_NT) * WB;
                if (d < Dp) *(RawB*)(buf + 2 * Dp + d) = d < D ? nb[u] : RawB{};
            }
        }
        if (t >= t_lo && dg == 0 && vok) out[((size_t)t * H + h) * V + vcol] = mine;
        __syncthreads();
    }
    if (keep) la_state_out<PR>(S, srow, sm, D, V, v0);
}

// Heads of up to 64 where instructions and not round trips are what a workgroup waits for (the rule is in spite_linear_attn_scan): one
// fetch a thread covers q, k and the value slice of a block of 16 tokens, its address is found again for each block, what lies outside a head
// goes to LDS as zeros: some 40 instructions less than the scan before the first token, and fewer loads a block.  bfloat16 in pieces of
// 16 bytes.  The same sums in the same order.
template <bool CH, bool PRE>
__global__ __launch_bounds__(LA_NT) __attribute__((amdgpu_waves_per_eu(1, 2)))
void linear_attn_blocks_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v, int ldq, int ldk, int ldv,
                               const float* __restrict__ decay, const float* __restrict__ head_decay, float q_scale,
                               float* __restrict__ state, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slots,
                               float* __restrict__ out, int H, int D, int V, int keep, int qk_rep,
                               const float* __restrict__ v_scale, const float* __restrict__ bonus) {
    constexpr int TB = 16, Dp = 64, PR = 2, LOOK = 4;               // tokens a block; key channels, padded, and a thread's; tokens read ahead
    constexpr int NQ = CH ? 3 : 2, per = NQ * Dp + LA_VC;           // rows of Dp a token, its floats in LDS
    constexpr int CA = (2 * Dp + LA_VC) / 8, CB = Dp / 4;           // fetches a token: q, k and the value slice; the decay
    static_assert(TB * CA <= LA_NT && TB * CB <= LA_NT && la_block<4>::tokens == TB, "linear_attn_blocks: a fetch of each kind a thread");
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    extern __shared__ __attribute__((aligned(16))) float sm[];      // 2 * TB * per floats
    const int e = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * LA_VC;
    const int tid = threadIdx.x, vc = tid / LA_DG, dg = tid % LA_DG;
    const int t_lo = cu_seqlens[e], t_hi = cu_seqlens[e + 1];
    if (t_lo >= t_hi) return;
    float* srow = state + ((size_t)seq_slots[e] * H + h) * (size_t)D * V;
    float S[PR], x[PR];
    la_state_ask<PR>(x, srow, D, V, v0);
    la_state_in<PR>(S, x, sm, D, V, v0);
    const float hd = CH ? 1.f : head_decay[h];
    float ub[PR];
    if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r < PR; ++r) { const int d = LA_OWN(r); ub[r] = d < D ? bonus[(size_t)h * D + d] : 0.f; }
    }
    // the thread's fetches: token ja of a block and elements ea .. + 7 of its row of q, k and value slice; token jb and channels db .. + 3
    const int ja = tid / CA, ea = tid % CA * 8, part = ea / Dp, hq = h / qk_rep;
    const bf16* base = part == 0 ? q : part == 1 ? k : v;
    const int ld = part == 0 ? ldq : part == 1 ? ldk : ldv, col = part < 2 ? hq * D + ea % Dp : h * V + v0 + (ea - 2 * Dp);
    const bool in = part < 2 ? ea % Dp < D : v0 + (ea - 2 * Dp) < V;
    const int jb = tid / CB, db = tid % CB * 4;
    u32x4 na;
    f32x4 nb;
    float ns;                                                // the factor on the fetch's elements
    const int n_blocks = (t_hi - t_lo + TB - 1) / TB;
    for (int it = -1; it < n_blocks; ++it) {                 // (turns as in the scan)
        const int t0 = t_lo + it * TB, tn = t0 + TB;                // this block's first token, the next block's
        const bool more = it + 1 < n_blocks;
        if (more) {
            const bool ok = ja < TB && tn + ja < t_hi && in;
            na = *(const u32x4*)(base + (size_t)(ok ? tn + ja : t_lo) * ld + (ok ? col : 0));
            ns = part == 0 ? q_scale : (part == 2 && v_scale) ? v_scale[(size_t)(ok ? tn + ja : t_lo) * H + h] : 1.f;
            if constexpr (CH) {
                const bool okb = jb < TB && tn + jb < t_hi && db < D;
                nb = *(const f32x4*)(decay + ((size_t)(okb ? tn + jb : t_lo) * H + h) * D + (okb ? db : 0));
            }
        }
        float mine = 0.f;                                           // one token's result (la_owner)
        if (it >= 0) {
            const float* cur = sm + (it & 1) * (TB * per);
            const int n_tok = t_hi - t0 < TB ? t_hi - t0 : TB;
            float accs[TB], vv[LOOK];
            f32x2 q2[LOOK], k2[LOOK], a2[CH ? LOOK : 1];
            auto read = [&](int j) {
                const float* row = cur + j * per;
                vv[j % LOOK] = row[NQ * Dp + vc];
                q2[j % LOOK] = *(const f32x2*)(row + LA_OWN(0));
                k2[j % LOOK] = *(const f32x2*)(row + Dp + LA_OWN(0));
                if constexpr (CH) a2[j % LOOK] = *(const f32x2*)(row + 2 * Dp + LA_OWN(0));
            };
            auto token = [&](int j) {
                accs[j] = 0.f;
#pragma unroll
                for (int r = 0; r < PR; ++r) {
                    float a = hd;
                    if constexpr (CH) a = a2[j % LOOK][r];
                    const float qr = q2[j % LOOK][r], kv = k2[j % LOOK][r] * vv[j % LOOK];
                    if (PRE) accs[j] = fmaf(fmaf(ub[r], kv, S[r]), qr, accs[j]);
                    S[r] = fmaf(a, S[r], kv);
                    if (!PRE) accs[j] = fmaf(S[r], qr, accs[j]);
                }
            };
            if (n_tok == TB) {
#pragma unroll
                for (int j = 0; j < LOOK; ++j) read(j);
#pragma unroll
                for (int j = 0; j < TB; ++j) {
                    __builtin_amdgcn_sched_barrier(0x7);
                    token(j);
                    if (j + LOOK < TB) read(j + LOOK);
                }
                __builtin_amdgcn_sched_barrier(0x7);
            } else {
#pragma unroll
                for (int j = 0; j < TB; ++j) {
                    accs[j] = 0.f;
                    if (j < n_tok) { read(j); token(j); }
                }
            }
            mine = la_sums<TB>(accs, dg);
        }
        if (more) {
            float* buf = sm + ((it + 1) & 1) * (TB * per);
            if (ja < TB && tn + ja < t_hi) {
                float* dst = buf + ja * per + (part < 2 ? ea : ea + (NQ - 2) * Dp);
                const u32x4 w = in ? na : u32x4{0, 0, 0, 0};
                f32x4 lo, hi;
                lo.x = __builtin_bit_cast(float, w.x << 16) * ns, lo.y = __builtin_bit_cast(float, w.x & 0xffff0000u) * ns;
                lo.z = __builtin_bit_cast(float, w.y << 16) * ns, lo.w = __builtin_bit_cast(float, w.y & 0xffff0000u) * ns;
                hi.x = __builtin_bit_cast(float, w.z << 16) * ns, hi.y = __builtin_bit_cast(float, w.z & 0xffff0000u) * ns;
                hi.z = __builtin_bit_cast(float, w.w << 16) * ns, hi.w = __builtin_bit_cast(float, w.w & 0xffff0000u) * ns;
                *(f32x4*)dst = lo;
                *(f32x4*)(dst + 4) = hi;
            }
            if constexpr (CH) {
                if (jb < TB && tn + jb < t_hi) *(f32x4*)(buf + jb * per + 2 * Dp + db) = db < D ? nb : f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        if (it >= 0 && dg % (LA_DG / TB) == 0) {
            const int t = t0 + la_owner<TB>(dg);
            if (t < t_hi && v0 + vc < V) out[((size_t)t * H + h) * V + v0 + vc] = mine;
        }
        __syncthreads();
    }
    if (keep) la_state_out<PR>(S, srow, sm, D, V, v0);
}
#undef LA_OWN

enum la_form { LA_SCAN, LA_BLOCKS, LA_SINGLE };
struct la_args {
    dim3 grid; hipStream_t st; const void *q, *k, *v; int ldq, ldk, ldv; const float *decay, *head_decay; float q_scale;
    float* state; const int *cu_seqlens, *seq_slots; float* out; int H, D, V, keep, qk_rep; const float *v_scale, *bonus;
};

template <typename T, int RR, bool CH, bool VEC, bool PRE>
static void la_launch(const la_args& a, la_form form) {
    const int TB = form == LA_SINGLE ? 1 : la_block<RR>::tokens;
    constexpr int Dp = 16 * RR, per = (CH ? 3 : 2) * Dp + LA_VC;
    constexpr size_t tile = (size_t)Dp * (LA_VC + 1);
    static_assert(sizeof(float) * 2 * la_block<RR>::tokens * per <= 64 * 1024, "linear_attn_scan: the token blocks must fit the default LDS limit");
    const size_t blocks = (size_t)2 * TB * per, bytes = (blocks > tile ? blocks : tile) * sizeof(float);
    auto* kernel = form == LA_SINGLE ? linear_attn_single_kernel<T, RR, CH, VEC, PRE> : linear_attn_scan_kernel<T, RR, CH, VEC, PRE>;
    if constexpr (RR == 4 && VEC) if (form == LA_BLOCKS) kernel = linear_attn_blocks_kernel<CH, PRE>;
    kernel<<<a.grid, LA_NT, bytes, a.st>>>(
        (const T*)a.q, (const T*)a.k, (const T*)a.v, a.ldq, a.ldk, a.ldv, a.decay, a.head_decay, a.q_scale, a.state, a.cu_seqlens,
        a.seq_slots, a.out, a.H, a.D, a.V, a.keep, a.qk_rep, a.v_scale, a.bonus);
}

template <typename T, bool VEC, int RR>
static void la_pick_decay(const la_args& a, la_form form) {
    if (a.bonus) la_launch<T, RR, true, VEC, true>(a, form);      // (the caller has made sure that a bonus comes with a decay per channel)
    else if (a.decay) la_launch<T, RR, true, VEC, false>(a, form);
    else la_launch<T, RR, false, VEC, false>(a, form);
}

template <typename T, bool VEC>
static void la_pick(const la_args& a, la_form form) {
    if (a.D <= 64) la_pick_decay<T, VEC, 4>(a, form);
    else if (a.D <= 128) la_pick_decay<T, VEC, 8>(a, form);
    else la_pick_decay<T, VEC, 16>(a, form);
}

extern "C" int spite_linear_attn_scan(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv, int dtype,
                                      const float* decay, const float* head_decay, float q_scale, float* state, int n_slots,
                                      const int* cu_seqlens, const int* seq_slots, int n_seqs, float* out,
                                      int H, int D, int V, int keep, int longest, int qk_heads, const float* v_scale,
                                      const float* bonus, hipStream_t st) {
    if (qk_heads <= 0) qk_heads = H;
    SP_REQUIRE(H % qk_heads == 0, "linear_attn_scan: %d heads over %d heads of q and k", H, qk_heads);
    SP_REQUIRE(!bonus || decay, "linear_attn_scan: the bonus form goes with a decay per channel");
    SP_REQUIRE(n_seqs >= 0 && H > 0 && D > 0 && V > 0 && n_slots > 0, "linear_attn_scan: bad sizes");
    SP_REQUIRE(D <= LA_MAXD, "linear_attn_scan: %d key channels a head (at most %d)", D, LA_MAXD);
    SP_REQUIRE(ldq >= qk_heads * D && ldk >= qk_heads * D && ldv >= H * V, "linear_attn_scan: rows shorter than the heads");
    SP_REQUIRE((decay != nullptr) != (head_decay != nullptr), "linear_attn_scan: a decay per channel or one per head, one of them");
    SP_REQUIRE(H <= 65535 && (V + LA_VC - 1) / LA_VC <= 65535, "linear_attn_scan: too many heads or value columns");
    SP_REQUIRE(dtype == SP_F32 || dtype == SP_BF16, "linear_attn_scan: unknown dtype %d", dtype);
    if (n_seqs == 0) return 0;
    const la_args a{dim3(n_seqs, H, (V + LA_VC - 1) / LA_VC), st, q, k, v, ldq, ldk, ldv, decay, head_decay, q_scale, state,
                    cu_seqlens, seq_slots, out, H, D, V, keep, H / qk_heads, v_scale, bonus};
    auto on16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    const bool vec = dtype == SP_BF16 && D % 8 == 0 && V % 8 == 0 && ldq % 8 == 0 && ldk % 8 == 0 && ldv % 8 == 0
                     && on16(q) && on16(k) && on16(v) && on16(decay);
    // Which kernel (the same bits from each): single tokens their own; heads of up to 64 in blocks where instructions and not
    // round trips are what a workgroup waits for: with a decay per head and more than two workgroups a compute unit (16 requests, 40
    // heads of 64, us with the scan / in blocks: 5 tokens 15.8 / 13.5, 33 26.9 / 24.8, 500 242 / 233; but 4 requests, 16 heads, 256
    // workgroups, 500 tokens 34.3 / 38.3), and for heads of less than 64, which the scan pads, with no more tokens than a
    // block (8 requests, 16 heads of 32, a decay per channel, 5 tokens: 5.8 / 5.2).
    const long groups = (long)n_seqs * H * ((V + LA_VC - 1) / LA_VC);
    const bool blocks = D <= 64 && ((!decay && groups > 2L * sp_cu_count()) || (D < 64 && longest > 0 && longest <= la_block<4>::tokens));
    const la_form form = longest == 1 ? LA_SINGLE : vec && blocks ? LA_BLOCKS : LA_SCAN;      // (longest 0: not known)
    if (dtype == SP_F32) la_pick<float, false>(a, form);
    else if (vec) la_pick<bf16, true>(a, form);
    else la_pick<bf16, false>(a, form);
    SP_LAUNCH_CHECK("linear_attn_scan");
    return 0;
}

// ------------------------------------------------------------------ norm over groups, weight, gate
// One wave a (token, group): y[c] = o[c] / sqrt(mean over the group (o^2) + eps) * w[c % n_w] * act(gate[c]),
// act: 1 silu, 2 sigmoid (0: no gate).  o fp32 [T, n]; gate rows `ldg` apart, in y's type.
// `pre_gate`: the gate comes before the norm, y = rmsnorm(o * act(gate)) * w.  `skip` (rows `lds` apart, in y's type)
// with `skip_w` fp32 [n / skip_group]: o[c] + skip_w[c / skip_group] * skip[c] stands for o[c] (a direct path from
// the recurrence's input to its result, one weight a head).
#define GGN_KEEP 8            // values a lane keeps: groups of up to 512 elements are read once
// (the wide form reads its values twice: holding up to 24 of them a thread was measured slower, 40 against 30 us)
struct ggn_extra { const void* skip; int lds; const float* skip_w; int skip_group; int pre_gate; };
template <typename TO>
__device__ __forceinline__ float ggn_value(const float* orow, const TO* gate, int ldg, size_t t, int c0, int c, int act, const ggn_extra& ex) {
    float x = orow[c];
    if (ex.skip) x = fmaf(ex.skip_w[(c0 + c) / ex.skip_group], to_f32<TO>(((const TO*)ex.skip)[t * ex.lds + c0 + c]), x);
    if (ex.pre_gate && act) {
        const float g = to_f32<TO>(gate[t * ldg + c0 + c]);
        const float sg = 1.0f / (1.0f + expf(-g));
        x *= act == 1 ? g * sg : sg;
    }
    return x;
}
template <typename TO>
__global__ __launch_bounds__(256)
void gated_group_norm_kernel(const float* __restrict__ o, const TO* __restrict__ gate, int ldg, const float* __restrict__ w,
                             int n_w, TO* __restrict__ y, int T, int n, int group, float eps, int act, ggn_extra ex) {
    const int lane = threadIdx.x & 63;
    const int groups = n / group;
    const size_t item = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= (size_t)T * groups) return;
    const size_t t = item / groups;
    const int c0 = (int)(item % groups) * group;
    const float* orow = o + t * n + c0;
    float ss = 0.f;
    float kept[GGN_KEEP];                             // a lane's first values stay in registers between the two passes
#pragma unroll
    for (int k = 0; k < GGN_KEEP; ++k) {
        const int c = lane + k * 64;
        kept[k] = c < group ? ggn_value<TO>(orow, gate, ldg, t, c0, c, act, ex) : 0.f;
        ss = fmaf(kept[k], kept[k], ss);
    }
    for (int c = lane + GGN_KEEP * 64; c < group; c += 64) { const float x = ggn_value<TO>(orow, gate, ldg, t, c0, c, act, ex); ss = fmaf(x, x, ss); }
    const float sc = 1.0f / sqrtf(wave_sum(ss) / (float)group + eps);
#pragma unroll
    for (int k = 0; k < GGN_KEEP; ++k) {
        const int c = lane + k * 64;
        if (c >= group) continue;
        float x = kept[k] * sc * w[(c0 + c) % n_w];
        if (act && !ex.pre_gate) {
            const float g = to_f32<TO>(gate[t * ldg + c0 + c]);
            const float sg = 1.0f / (1.0f + expf(-g));
            x *= act == 1 ? g * sg : sg;
        }
        y[t * n + c0 + c] = from_f32<TO>(x);
    }
    for (int c = lane + GGN_KEEP * 64; c < group; c += 64) {
        float x = ggn_value<TO>(orow, gate, ldg, t, c0, c, act, ex) * sc * w[(c0 + c) % n_w];
        if (act && !ex.pre_gate) {
            const float g = to_f32<TO>(gate[t * ldg + c0 + c]);
            const float sg = 1.0f / (1.0f + expf(-g));
            x *= act == 1 ? g * sg : sg;
        }
        y[t * n + c0 + c] = from_f32<TO>(x);
    }
}

// The same for bfloat16 rows in groups of up to 256 that a lane moves eight elements at a time: 16 lanes a group.
__global__ __launch_bounds__(256)
void gated_group_norm_vec_kernel(const float* __restrict__ o, const bf16* __restrict__ gate, int ldg, const float* __restrict__ w, int n_w,
                                 bf16* __restrict__ y, int T, int n, int group, float eps, int act) {
    const int l = threadIdx.x & 15, groups = n / group;
    const size_t item = (size_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (item >= (size_t)T * groups) return;
    const size_t t = item / groups;
    const int c0 = (int)(item - t * groups) * group;
    const float* orow = o + t * n + c0;
    f32x4 x[2][2];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = l * 8 + i * 128;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            x[i][p] = c < group ? *(const f32x4*)(orow + c + 4 * p) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(x[i][p][e], x[i][p][e], ss);
        }
    }
    const float sc = 1.0f / sqrtf(row16_sum(ss) / (float)group + eps);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = l * 8 + i * 128;
        if (c >= group) continue;
        const float* wr = w + (c0 + c) % n_w;                  // (a multiple of eight: n_w is one, or a group's multiple)
        bf16x8 g, out;
        if (act) g = *(const bf16x8*)(gate + t * ldg + c0 + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = x[i][e >> 2][e & 3] * sc * wr[e];
            if (act) {
                const float z = (float)g[e], sg = 1.0f / (1.0f + expf(-z));
                v *= act == 1 ? z * sg : sg;
            }
            out[e] = (bf16)v;
        }
        *(bf16x8*)(y + t * n + c0 + c) = out;
    }
}

// The same for wide groups (the heads normed together): a workgroup a (token, group), the sum of squares across
// its four waves through LDS.
template <typename TO>
__global__ __launch_bounds__(256)
void gated_group_norm_wide_kernel(const float* __restrict__ o, const TO* __restrict__ gate, int ldg, const float* __restrict__ w,
                                  int n_w, TO* __restrict__ y, int n, int group, float eps, int act, ggn_extra ex) {
    __shared__ float part[4];
    const int groups = n / group;
    const size_t t = blockIdx.x / groups;
    const int c0 = (int)(blockIdx.x % groups) * group;
    const float* orow = o + t * n + c0;
    float ss = 0.f;
#pragma unroll 8
    for (int c = threadIdx.x; c < group; c += 256) { const float x = ggn_value<TO>(orow, gate, ldg, t, c0, c, act, ex); ss = fmaf(x, x, ss); }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float sc = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)group + eps);
    const bool whole = n_w >= n;                      // a weight for every element of the row: no wrapping
#pragma unroll 4
    for (int c = threadIdx.x; c < group; c += 256) {
        float x = ggn_value<TO>(orow, gate, ldg, t, c0, c, act, ex) * sc * w[whole ? c0 + c : (c0 + c) % n_w];
        if (act && !ex.pre_gate) {
            const float g = to_f32<TO>(gate[t * ldg + c0 + c]);
            const float sg = 1.0f / (1.0f + expf(-g));
            x *= act == 1 ? g * sg : sg;
        }
        y[t * n + c0 + c] = from_f32<TO>(x);
    }
}

// The same without a gate before the sum or a skip, for groups of up to 256 * V: a thread keeps its elements, and what it loads (the row, the
// gate and the weights) is asked for at once, where the kernel above waits for memory in each of its loops, twice.  The same elements a thread
// and the same order of sums: the same bits.  us, above and here: one row of 2,048 5.2 / 3.3, of 5,120 10.0 / 5.1, of 8,192 14.1 / 6.9;
// 1,531 rows of 2,048 9.2 / 7.0.  Elements a thread come in steps of 8, 20 and 32: what a group has less is its last element again, from the cache
// (one row of 512 3.2 / 2.6, of 2,304 4.3 / 3.2, of 5,632 7.2 / 4.1; 1,531 of 512 5.3 / 4.7, of 2,304 8.1 / 7.0; of 18 widths none is slower).
template <typename TO, int V>
__global__ __launch_bounds__(256)
void gated_group_norm_rows_kernel(const float* __restrict__ o, const TO* __restrict__ gate, int ldg, const float* __restrict__ w,
                                  int n_w, TO* __restrict__ y, int n, int group, float eps, int act) {
    __shared__ float part[4];
    const int groups = n / group;
    const size_t t = blockIdx.x / groups;
    const int c0 = (int)(blockIdx.x % groups) * group, tid = threadIdx.x;
    const float* orow = o + t * n + c0;
    const bool whole = n_w >= n;                      // a weight for every element of the row: no wrapping
    float x[V], ww[V];
    TO g[V];
    int at[V];                                        // elements past the group: its last one again
#pragma unroll
    for (int k = 0; k < V; ++k) at[k] = tid + 256 * k < group ? tid + 256 * k : group - 1;
#pragma unroll
    for (int k = 0; k < V; ++k) x[k] = orow[at[k]];
    if (act)
#pragma unroll
        for (int k = 0; k < V; ++k) g[k] = gate[t * ldg + c0 + at[k]];
#pragma unroll
    for (int k = 0; k < V; ++k) ww[k] = w[whole ? c0 + at[k] : (c0 + at[k]) % n_w];
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < V; ++k) ss = tid + 256 * k < group ? fmaf(x[k], x[k], ss) : ss;
    ss = wave_sum(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    const float sc = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)group + eps);
#pragma unroll
    for (int k = 0; k < V; ++k) {
        if (tid + 256 * k >= group) break;
        float v = x[k] * sc * ww[k];
        if (act) {
            const float z = to_f32<TO>(g[k]);
            const float sg = 1.0f / (1.0f + expf(-z));
            v *= act == 1 ? z * sg : sg;
        }
        y[t * n + c0 + at[k]] = from_f32<TO>(v);
    }
}

extern "C" int spite_gated_group_norm(const float* o, const void* gate, int ldg, const float* w, int n_w, void* y, int y_dtype,
                                      int T, int n, int group, float eps, int act, int pre_gate, const void* skip, int lds,
                                      const float* skip_w, int skip_group, hipStream_t st) {
    SP_REQUIRE(!skip || (skip_w && skip_group > 0 && n % skip_group == 0 && lds >= n), "gated_group_norm: skip rows of %d in heads of %d", lds, skip_group);
    const ggn_extra ex{skip, lds, skip_w, skip_group > 0 ? skip_group : 1, pre_gate};
    SP_REQUIRE(T >= 0 && n > 0 && group > 0 && n % group == 0, "gated_group_norm: rows of %d in groups of %d", n, group);
    SP_REQUIRE(n_w > 0 && n % n_w == 0 && (n_w % group == 0 || group % n_w == 0), "gated_group_norm: %d weights for groups of %d", n_w, group);
    SP_REQUIRE(act >= 0 && act <= 2 && (act == 0 || (gate && ldg >= n)), "gated_group_norm: gate");
    SP_REQUIRE(eps > 0.f, "gated_group_norm: the norm needs an eps");
    if (T == 0) return 0;
    const size_t items = (size_t)T * (n / group);
    SP_REQUIRE((items + 3) / 4 < (1u << 31), "gated_group_norm: too many groups");
    if (group >= 512 && group <= 8192 && !skip && !pre_gate && items < (1u << 31)) {
        SP_REQUIRE(y_dtype == SP_F32 || y_dtype == SP_BF16, "gated_group_norm: unknown dtype %d", y_dtype);
#define SP_GGN(V) do { if (y_dtype == SP_F32) gated_group_norm_rows_kernel<float, V><<<(unsigned)items, 256, 0, st>>>(o, (const float*)gate, ldg, w, n_w, (float*)y, n, group, eps, act); \
                       else gated_group_norm_rows_kernel<bf16, V><<<(unsigned)items, 256, 0, st>>>(o, (const bf16*)gate, ldg, w, n_w, (bf16*)y, n, group, eps, act); } while (0)
        if (group <= 2048) SP_GGN(8);
        else if (group <= 5120) SP_GGN(20);
        else SP_GGN(32);
#undef SP_GGN
        SP_LAUNCH_CHECK("gated_group_norm");
        return 0;
    }
    if (group >= 512 && items < (1u << 31)) {
        if (y_dtype == SP_F32)
            gated_group_norm_wide_kernel<float><<<(unsigned)items, 256, 0, st>>>(o, (const float*)gate, ldg, w, n_w, (float*)y, n, group, eps, act, ex);
        else if (y_dtype == SP_BF16)
            gated_group_norm_wide_kernel<bf16><<<(unsigned)items, 256, 0, st>>>(o, (const bf16*)gate, ldg, w, n_w, (bf16*)y, n, group, eps, act, ex);
        else return sp_fail("gated_group_norm: unknown dtype %d", y_dtype);
        SP_LAUNCH_CHECK("gated_group_norm");
        return 0;
    }
    auto on16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    if (y_dtype == SP_BF16 && !skip && !pre_gate && group % 8 == 0 && group <= 256 && n_w % 8 == 0 && on16(o) && on16(y)
        && (act == 0 || (ldg % 8 == 0 && on16(gate)))) {
        gated_group_norm_vec_kernel<<<(unsigned)((items + 15) / 16), 256, 0, st>>>(o, (const bf16*)gate, ldg, w, n_w, (bf16*)y, T, n, group, eps, act);
        SP_LAUNCH_CHECK("gated_group_norm");
        return 0;
    }
    const unsigned grid = (unsigned)((items + 3) / 4);
    if (y_dtype == SP_F32)
        gated_group_norm_kernel<float><<<grid, 256, 0, st>>>(o, (const float*)gate, ldg, w, n_w, (float*)y, T, n, group, eps, act, ex);
    else if (y_dtype == SP_BF16)
        gated_group_norm_kernel<bf16><<<grid, 256, 0, st>>>(o, (const bf16*)gate, ldg, w, n_w, (bf16*)y, T, n, group, eps, act, ex);
    else return sp_fail("gated_group_norm: unknown dtype %d", y_dtype);
    SP_LAUNCH_CHECK("gated_group_norm");
    return 0;
}
