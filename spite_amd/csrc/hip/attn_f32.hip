// fp32 attention over row-major pages (head sizes in multiples of 16 up to 128, pages in multiples of 4 keys): the true
// 32-bit path at the sizes that models have; attn_generic.hip keeps the others.
//
// A workgroup of W waves per (token, query head): eight, or fewer where a window or a chunk never shows a query that many
// tiles.  Keys are walked in tiles of 32 that start at multiples of 32 positions, the tiles dealt to the waves in turn, each
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

template <int NI, int W>     // NI: the head size in units of 16, at most
__global__ __launch_bounds__(64 * W)
void attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                     float* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                     const int* __restrict__ block_table, int max_blocks, int H, int G, int hd, int ps, int vis, int span,
                     float scale, float softcap, const float* __restrict__ slopes) {
    __shared__ __align__(16) float p_sh[W][AF_KEYS];
    __shared__ float o_sh[W][NI * 16];
    __shared__ float ml_sh[W][2];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h / (H / G), ni = hd >> 4;
    const int p = positions[t];
    const int* bt = block_table + (size_t)seq_of_token[t] * max_blocks;
    const int lo = sp_first_visible(p, vis, span);
    const float slope = slopes ? slopes[h] : 0.f;
    const float* qr = q + ((size_t)t * H + h) * hd;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // scores: lane (kr, cq) takes elements 16 i + 4 cq .. + 3 of keys kr and kr + 16 of a tile
    const int kr = lane >> 2, cq = (lane & 3) * 4;
    f32x4 qv[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) qv[i] = i < ni ? *(const f32x4*)(qr + i * 16 + cq) : zero;
    // output: lane (cr, kq) takes elements 8 i + cr of keys 4 kq .. + 3
    const int cr = lane >> 3, kq = (lane & 7) * 4;
    float o[NI * 2];
#pragma unroll
    for (int i = 0; i < NI * 2; ++i) o[i] = 0.f;
    float m = -INFINITY, l = 0.f;

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
        float s[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            f32x4 a = zero;
#pragma unroll
            for (int i = 0; i < NI; ++i)               // (qv is zero beyond the head)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = fmaf(qv[i][e], kv[n][i][e], a[e]);
            float x = (a[0] + a[1]) + (a[2] + a[3]);
            x += __shfl_xor(x, 1, 64);
            x += __shfl_xor(x, 2, 64);
            x = x * scale + slope * (float)(j0 + n * 16 + kr - p);
            if (softcap > 0.f) x = softcap * tanhf(x / softcap);
            s[n] = !seen[n] ? -INFINITY : page[n] >= 0 ? x : NAN;    // a page that was given back is asked for: poison the result
        }
        const float* vp = vpage >= 0 ? v_pages + ((size_t)vpage * G + g) * hd * ps + (jv % ps) : nullptr;
        f32x4 v[NI * 2];
#pragma unroll
        for (int i = 0; i < NI * 2; ++i) v[i] = vp ? *(const f32x4*)(vp + (size_t)((i < ni * 2 ? i : 0) * 8 + cr) * ps) : zero;
        float mx = fmaxf(s[0], s[1]);
#pragma unroll
        for (int d = 4; d < 64; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
        const float m_new = fmaxf(m, mx), alpha = expf(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            s[n] = expf(s[n] - m_new);                 // 0 where the key is not seen
            sum += s[n];
            if ((lane & 3) == n) p_sh[wave][n * 16 + kr] = s[n];
        }
#pragma unroll
        for (int d = 4; d < 64; d <<= 1) sum += __shfl_xor(sum, d, 64);
        l = l * alpha + sum;
        m = m_new;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const f32x4 pv = *(const f32x4*)&p_sh[wave][kq];
        if (j0 < lo || j0 + AF_KEYS - 1 > p) {         // some keys of the tile are not seen: what their places hold must not count
#pragma unroll
            for (int i = 0; i < NI * 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][e] = jv + e >= lo && jv + e <= p ? v[i][e] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NI * 2; ++i) {
            float a = o[i] * alpha;
#pragma unroll
            for (int e = 0; e < 4; ++e) a = fmaf(pv[e], v[i][e], a);
            o[i] = a;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
#pragma unroll
    for (int i = 0; i < NI * 2; ++i) {
        float a = o[i];
        a += __shfl_xor(a, 1, 64);
        a += __shfl_xor(a, 2, 64);
        a += __shfl_xor(a, 4, 64);
        if ((lane & 7) == (i & 7)) o_sh[wave][i * 8 + cr] = a;
    }
    if (lane == 0) { ml_sh[wave][0] = m; ml_sh[wave][1] = l; }
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= hd) return;
    float mm = ml_sh[0][0];
#pragma unroll
    for (int w = 1; w < W; ++w) mm = fmaxf(mm, ml_sh[w][0]);
    float ll = 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const float f = ml_sh[w][0] == -INFINITY ? 0.f : expf(ml_sh[w][0] - mm);   // a wave without tiles
        ll += ml_sh[w][1] * f;
        a += o_sh[w][c] * f;
    }
    out[((size_t)t * H + h) * hd + c] = a * (1.0f / fmaxf(ll, 1e-30f));
}

// The attention if it is of this kernel's shape (returns 0, or an error), else 1: the plain kernel's.
int sp_attn_f32(const float* q, const float* k_pages, const float* v_pages, float* out, const int* positions,
                const int* seq_of_token, const int* block_table, int max_blocks, int T, int H, int G, int hd, int page_size,
                int vis, int span, float scale, float softcap, const float* slopes, hipStream_t st) {
    if (hd % 16 || hd > 128 || page_size % 4 || ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16) return 1;
    // Waves for no more tiles than a query sees, lanes for no more of the head than there is: 3,000 tokens of a prompt, 4 heads
    // of 16 behind a window of 64 keys, 25 us (46 with eight waves and heads padded to 64, 60 for the plain kernel); 1,000 tokens,
    // 16 heads of 128, 170 (332, 751).  A few keys are the plain kernel's, a wave a row: a window of one, 1,000 tokens, 16 heads
    // of 128, 47 against 82 us; of eight, 4 heads of 16, 3,000 tokens, 17 against 27; of 33 35 against 16.
    if (sp_vis_has_span(vis) && span <= 8) return 1;
    dim3 grid(T, H);
    const long tiles = sp_vis_has_span(vis) ? ((long)span + 30) / 32 + 1 : 8;      // that a query sees at most
#define AF_GO(NI, W) attn_f32_kernel<NI, W><<<grid, 64 * W, 0, st>>>(q, k_pages, v_pages, out, positions, seq_of_token, block_table, \
        max_blocks, H, G, hd, page_size, vis, span, scale, softcap, slopes)
#define AF_HEAD(W) do { if (hd <= 16) AF_GO(1, W); else if (hd <= 32) AF_GO(2, W); else if (hd <= 64) AF_GO(4, W); else AF_GO(8, W); } while (0)
    if (tiles <= 2) AF_HEAD(2);
    else if (tiles <= 4) AF_HEAD(4);
    else AF_HEAD(8);
#undef AF_HEAD
#undef AF_GO
    SP_LAUNCH_CHECK("attn_f32");
    return 0;
}
