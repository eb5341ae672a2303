// fp32 attention over row-major pages (head sizes in multiples of 16 up to 128, pages in multiples of 4 keys): the true
// 32-bit path at the sizes that models have; attn_generic.hip keeps the others.
//
// A workgroup of W waves per (token, query head), or per token and several query heads of one key head (af_heads): eight, or fewer
// where a window or a chunk never shows a query that many tiles.  Keys are walked in tiles of 32 that start at multiples of 32 positions, the tiles dealt to the waves in turn, each
// wave with its own running maximum, sum and output; they meet in LDS at the end, in their order.  So the order of every
// sum depends on the layer and the query's position alone, as in the plain kernel: a token gives the same bits whether it
// comes in a whole prompt, a portion or alone.
//
// Bound by latency (decode: a chain of loads, table entry - keys - values, over few workgroups) or by the loads' path
// (prompts).  Hence tiles of 32 over eight waves, so that 256 keys are one such chain; 16-byte loads over whole lines,
// for the scores a key's row by four lanes, for the output 32 consecutive keys of a value row by eight; a lane keeps the
// partial sums of its four keys until the end instead of summing across lanes in every tile.
#include "common.h"

#define AF_KEYS 32

// Sums and maxima over lanes in the order of a butterfly, without the trip through the LDS crossbar that a shuffle is: lanes l ^ 1 and
// l ^ 2 by a permutation of each four; once four lanes agree, the mirror image of eight is as good as l ^ 4, and once eight do, that of
// sixteen as l ^ 8.
#define AF_DPP(x, ctl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (float)(x)), ctl, 0xf, 0xf, false))
__device__ __forceinline__ float af_quad_sum(float x) {
    x += AF_DPP(x, 0xB1);
    x += AF_DPP(x, 0x4E);
    return x;
}
__device__ __forceinline__ float af_eight_sum(float x) { x = af_quad_sum(x); return x + AF_DPP(x, 0x141); }
// over the sixteen quads, whose lanes agree
__device__ __forceinline__ float af_quads_sum(float x) {
    x += AF_DPP(x, 0x141);
    x += AF_DPP(x, 0x140);
    return rows4_sum(x);
}
__device__ __forceinline__ float af_quads_max(float x) {
    x = fmaxf(x, AF_DPP(x, 0x141));
    x = fmaxf(x, AF_DPP(x, 0x140));
    return rows4_max(x);
}

// NI: the head size in units of 16, at most.  NQ: query heads of one key head that a workgroup serves, each with a wave's loads of
// keys and values shared by them all and sums of its own.  Every rounding is written out: the instantiations agree bit for bit.
template <int NI, int W, int NQ>
__global__ __launch_bounds__(64 * W)
void attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                     float* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                     const int* __restrict__ block_table, int max_blocks, int H, int G, int hd, int ps, int vis, int span,
                     float scale, float softcap, const float* __restrict__ slopes) {
    __shared__ __align__(16) float p_sh[W][NQ][AF_KEYS];
    __shared__ __align__(16) float q_sh[NQ][NI * 16];
    __shared__ float o_sh[W][NQ][NI * 16];
    __shared__ float ml_sh[W][NQ][2], f_sh[NQ][W + 1];
    const int t = blockIdx.x, h0 = blockIdx.y * NQ, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h0 / (H / G), ni = hd >> 4;
    const int p = positions[t];
    const int* bt = block_table + (size_t)seq_of_token[t] * max_blocks;
    const int lo = sp_first_visible(p, vis, span);
    const float* qr = q + ((size_t)t * H + h0) * hd;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // scores: lane (kr, cq) takes elements 16 i + 4 cq .. + 3 of keys kr and kr + 16 of a tile
    const int kr = lane >> 2, cq = (lane & 3) * 4;
    f32x4 qv[NI];
    if constexpr (NQ == 1) {
#pragma unroll
        for (int i = 0; i < NI; ++i) qv[i] = i < ni ? *(const f32x4*)(qr + i * 16 + cq) : zero;
    } else {
        for (int c = threadIdx.x; c < NQ * NI * 16; c += 64 * W) q_sh[c / (NI * 16)][c % (NI * 16)] = c % (NI * 16) < hd ? qr[c / (NI * 16) * hd + c % (NI * 16)] : 0.f;
        __syncthreads();
    }
    // output: lane (cr, kq) takes elements 8 i + cr of keys 4 kq .. + 3
    const int cr = lane >> 3, kq = (lane & 7) * 4;
    float o[NQ][NI * 2], m[NQ], l[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
#pragma unroll
        for (int i = 0; i < NI * 2; ++i) o[n][i] = 0.f;
        m[n] = -INFINITY;
        l[n] = 0.f;
    }

    for (int j0 = (lo & ~(AF_KEYS - 1)) + wave * AF_KEYS; j0 <= p; j0 += AF_KEYS * W) {
        // the table entries of this tile's keys and values, then every row of keys, before anything waits for them
        int page[2];
        bool seen[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int j = j0 + n * 16 + kr;
            seen[n] = j >= lo && j <= p;
            page[n] = seen[n] ? bt[j / ps] : -1;
        }
        const int jv = j0 + kq;
        const int vpage = jv + 3 >= lo && jv <= p ? bt[jv / ps] : -1;
        f32x4 kv[2][NI];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const float* row = page[n] >= 0 ? k_pages + ((size_t)page[n] * G + g) * hd * ps + (size_t)((j0 + n * 16 + kr) % ps) * hd : qr;
#pragma unroll
            for (int i = 0; i < NI; ++i) kv[n][i] = *(const f32x4*)(row + (i < ni ? i : 0) * 16 + cq);
        }
        float s[NQ][2];
#pragma unroll
        for (int nq = 0; nq < NQ; ++nq) {
            const float slope = slopes ? slopes[h0 + nq] : 0.f;
            f32x4 a[2] = {zero, zero};
#pragma unroll
            for (int i = 0; i < NI; ++i) {             // (the query is zero beyond the head)
                const f32x4 x = NQ == 1 ? qv[i] : *(const f32x4*)&q_sh[nq][i * 16 + cq];
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[n][e] = fmaf(x[e], kv[n][i][e], a[n][e]);
            }
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                float x = (a[n][0] + a[n][1]) + (a[n][2] + a[n][3]);
                x = af_quad_sum(x);
                x = fmaf(x, scale, slope * (float)(j0 + n * 16 + kr - p));
                if (softcap > 0.f) x = softcap * tanhf(x / softcap);
                s[nq][n] = !seen[n] ? -INFINITY : page[n] >= 0 ? x : NAN;    // a page that was given back is asked for: poison the result
            }
        }
        const float* vp = vpage >= 0 ? v_pages + ((size_t)vpage * G + g) * hd * ps + (jv % ps) : nullptr;
        f32x4 v[NI * 2];
#pragma unroll
        for (int i = 0; i < NI * 2; ++i) v[i] = vp ? *(const f32x4*)(vp + (size_t)((i < ni * 2 ? i : 0) * 8 + cr) * ps) : zero;
        float alpha[NQ];
#pragma unroll
        for (int nq = 0; nq < NQ; ++nq) {
            const float mx = af_quads_max(fmaxf(s[nq][0], s[nq][1]));
            const float m_new = fmaxf(m[nq], mx);
            alpha[nq] = expf(m[nq] - m_new);
            float sum = 0.f;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                s[nq][n] = expf(s[nq][n] - m_new);     // 0 where the key is not seen
                sum += s[nq][n];
                if ((lane & 3) == n) p_sh[wave][nq][n * 16 + kr] = s[nq][n];
            }
            l[nq] = fmaf(l[nq], alpha[nq], af_quads_sum(sum));
            m[nq] = m_new;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (j0 < lo || j0 + AF_KEYS - 1 > p) {         // some keys of the tile are not seen: what their places hold must not count
#pragma unroll
            for (int i = 0; i < NI * 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][e] = jv + e >= lo && jv + e <= p ? v[i][e] : 0.f;
        }
#pragma unroll
        for (int nq = 0; nq < NQ; ++nq) {
            const f32x4 pv = *(const f32x4*)&p_sh[wave][nq][kq];
#pragma unroll
            for (int i = 0; i < NI * 2; ++i) {
                float a = o[nq][i] * alpha[nq];
#pragma unroll
                for (int e = 0; e < 4; ++e) a = fmaf(pv[e], v[i][e], a);
                o[nq][i] = a;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // the waves' records meet in LDS; a wave without tiles leaves none (its sum is zero: one whose every score was poisoned has NaN)
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq) {
        if (l[nq] != 0.f)
#pragma unroll
            for (int i = 0; i < NI * 2; ++i) {
                const float a = af_eight_sum(o[nq][i]);
                if ((lane & 7) == (i & 7)) o_sh[wave][nq][i * 8 + cr] = a;
            }
        if (lane == 0) { ml_sh[wave][nq][0] = m[nq]; ml_sh[wave][nq][1] = l[nq]; }
    }
    __syncthreads();
    // a wave's weight exp(its maximum - the largest), and one over the sum: of one head by every thread for itself, of more by as many
    // threads as there are heads (one barrier more: 32 tokens, 4 heads of 16, 4.8 us with it, 4.6 without)
    auto weights = [&](int nq, float* f) {
        float mm = ml_sh[0][nq][0];
#pragma unroll
        for (int w = 1; w < W; ++w) mm = fmaxf(mm, ml_sh[w][nq][0]);
        float ll = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            f[w] = ml_sh[w][nq][0] == -INFINITY ? 0.f : expf(ml_sh[w][nq][0] - mm);
            ll = fmaf(ml_sh[w][nq][1], f[w], ll);
        }
        f[W] = 1.0f / fmaxf(ll, 1e-30f);
    };
    if constexpr (NQ > 1) {
        if (threadIdx.x < NQ) weights(threadIdx.x, f_sh[threadIdx.x]);
        __syncthreads();
    }
    for (int c = threadIdx.x; c < NQ * NI * 16; c += 64 * W) {
        const int nq = c / (NI * 16), e = c % (NI * 16);
        if (e >= hd) continue;
        float f[W + 1];
        if constexpr (NQ == 1) weights(0, f);
        else
#pragma unroll
            for (int w = 0; w <= W; ++w) f[w] = f_sh[nq][w];
        float a = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w)
            if (ml_sh[w][nq][1] != 0.f) a = fmaf(o_sh[w][nq][e], f[w], a);
        out[((size_t)t * H + h0 + nq) * hd + e] = a * f[W];
    }
}

// Query heads a workgroup (one, two or four of those that read a key head): what takes the fewest rounds over the compute units, each at
// its cost.  A workgroup of two heads takes a quarter longer than one of one, of four four fifths (16 tokens, 16 heads of 128 over 4, one
// round: 5.5, 6.5 and 8.7 us); how many a unit holds follows from their registers.  Alone a token of a request is served by a
// workgroup a head, a prompt by one for four: 301 tokens, 16 heads of 128 over 4, 95.6 us with one, 62.0 with two, 47.1 with four (114 with one and
// shuffles in place of the lanes' permutations), 40 13.5 / 11.6 / 8.8, 64 behind 1,000 57 / 35 / 26; 8 heads of 32 over 1, 150 tokens 7.8 / 6.8 / 7.6.
static int af_heads(int T, int H, int sharing, int hd, int waves) {
    static const int held[4][3] = {{4, 4, 3}, {4, 3, 2}, {2, 2, 1}, {1, 1, 1}};       // workgroups of eight waves a compute unit
    const int* units = held[hd <= 16 ? 0 : hd <= 32 ? 1 : hd <= 64 ? 2 : 3];
    int best = 1;
    double least = 0.0;
    for (int i = 0; i < 3 && sharing % (1 << i) == 0; ++i) {
        const long slots = (long)sp_cu_count() * units[i] * 8 / waves;
        const double cost = (double)(((long)T * (H >> i) + slots - 1) / slots) * (i == 0 ? 1.0 : i == 1 ? 1.26 : 1.8);
        if (i == 0 || cost < least) { best = 1 << i; least = cost; }
    }
    return best;
}

// The attention if it is of this kernel's shape (returns 0, or an error), else 1: the plain kernel's.
int sp_attn_f32(const float* q, const float* k_pages, const float* v_pages, float* out, const int* positions,
                const int* seq_of_token, const int* block_table, int max_blocks, int T, int H, int G, int hd, int page_size,
                int vis, int span, float scale, float softcap, const float* slopes, hipStream_t st) {
    if (hd % 16 || hd > 128 || page_size % 4 || ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16) return 1;
    // Waves for no more tiles than a query sees, lanes for no more of the head than there is: 3,000 tokens of a prompt, 4 heads
    // of 16 behind a window of 64 keys, 23 us (46 with eight waves and heads padded to 64, 60 for the plain kernel); of 16 heads of 128
    // over 4, 190.  Windows of up to eight keys only where two heads share a workgroup's loads and the head fills its lanes (1,000 tokens, 16
    // heads of 128 over 4, windows of one and eight keys: 37 and 42 us, the plain kernel's wave a row 48 and 97; 0.45 to 0.9 over
    // heads of 16 to 64 and 128); else the plain kernel's, which makes no tile of 32 keys for each head (700 tokens, two keys:
    // 40 heads of 128 over 8 94 / 109, 12 of 96 over 4 23 / 34, 6 of 80 over 2 12 / 20).  By the layer alone: a token's bits do not depend on the step.
    if (sp_vis_has_span(vis) && span <= 8 && !(H / G % 2 == 0 && (hd <= 64 || hd == 128))) return 1;
    const long tiles = sp_vis_has_span(vis) ? ((long)span + 30) / 32 + 1 : 8;      // that a query sees at most
    const int waves = tiles <= 2 ? 2 : tiles <= 4 ? 4 : 8, nq = af_heads(T, H, H / G, hd, waves);
#define AF_GO(NI, W, NQ) attn_f32_kernel<NI, W, NQ><<<dim3(T, H / NQ), 64 * W, 0, st>>>(q, k_pages, v_pages, out, positions, seq_of_token, block_table, \
        max_blocks, H, G, hd, page_size, vis, span, scale, softcap, slopes)
#define AF_HEADS(NI, W) do { if (nq == 4) AF_GO(NI, W, 4); else if (nq == 2) AF_GO(NI, W, 2); else AF_GO(NI, W, 1); } while (0)
#define AF_HEAD(W) do { if (hd <= 16) AF_HEADS(1, W); else if (hd <= 32) AF_HEADS(2, W); else if (hd <= 64) AF_HEADS(4, W); else AF_HEADS(8, W); } while (0)
    if (waves == 2) AF_HEAD(2);
    else if (waves == 4) AF_HEAD(4);
    else AF_HEAD(8);
#undef AF_HEAD
#undef AF_HEADS
#undef AF_GO
    SP_LAUNCH_CHECK("attn_f32");
    return 0;
}
