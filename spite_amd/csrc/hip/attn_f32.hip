// fp32 attention over row-major pages (head sizes in multiples of 16 up to 128, pages in multiples of 4 keys): the true
// 32-bit path at the sizes that models have; attn_generic.hip keeps the others.
//
// A workgroup of four waves per (token, query head).  Keys are walked in tiles of 64 that start at multiples of 64
// positions, tile t by wave t % 4, each wave with its own running maximum, sum and output; the four meet in LDS at the
// end, in their order.  So the order of every sum depends on the query's position alone, as in the plain kernel: a token
// gives the same bits whether it comes in a whole prompt, a portion or alone.
//
// Bound by latency (decode: a chain of loads over few workgroups) or by the loads' path (prompts).  Hence 16-byte loads
// over whole runs: for the scores a key's row is read by four lanes, 64 bytes a load and key, all loads of 16 keys
// in flight; for the output 16 lanes read 64 consecutive keys of a value row, and a lane keeps the partial sums of its
// four keys until the end instead of summing across lanes in every tile.
#include "common.h"

#define AF_WAVES 4

template <int NI>     // the head size in units of 16, at most
__global__ __launch_bounds__(64 * AF_WAVES)
void attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                     float* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                     const int* __restrict__ block_table, int max_blocks, int H, int G, int hd, int ps, int vis, int span,
                     float scale, float softcap, const float* __restrict__ slopes) {
    __shared__ __align__(16) float p_sh[AF_WAVES][64];
    __shared__ float o_sh[AF_WAVES][NI * 16];
    __shared__ float ml_sh[AF_WAVES][2];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h / (H / G), ni = hd >> 4;
    const int p = positions[t];
    const int* bt = block_table + (size_t)seq_of_token[t] * max_blocks;
    const int lo = sp_first_visible(p, vis, span);
    const float slope = slopes ? slopes[h] : 0.f;
    const float* qr = q + ((size_t)t * H + h) * hd;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // scores: lane (kr, cq) takes elements 16 i + 4 cq .. + 3 of keys kr, kr + 16, ... of a tile
    const int kr = lane >> 2, cq = (lane & 3) * 4;
    f32x4 qv[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) qv[i] = i < ni ? *(const f32x4*)(qr + i * 16 + cq) : zero;
    // output: lane (cr, kq) takes elements 4 i + cr of keys 4 kq .. + 3
    const int cr = lane >> 4, kq = (lane & 15) * 4;
    float o[NI * 4];
#pragma unroll
    for (int i = 0; i < NI * 4; ++i) o[i] = 0.f;
    float m = -INFINITY, l = 0.f;

    for (int j0 = (lo & ~63) + wave * 64; j0 <= p; j0 += 64 * AF_WAVES) {
        float s[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int j = j0 + n * 16 + kr;
            const bool seen = j >= lo && j <= p;
            const int page = seen ? bt[j / ps] : -1;
            const float* row = page >= 0 ? k_pages + ((size_t)page * G + g) * hd * ps + (size_t)(j % ps) * hd : qr;
            f32x4 a = zero;
#pragma unroll
            for (int i = 0; i < NI; ++i)
                if (i < ni) {
                    const f32x4 kv = *(const f32x4*)(row + i * 16 + cq);
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[e] = fmaf(qv[i][e], kv[e], a[e]);
                }
            float x = (a[0] + a[1]) + (a[2] + a[3]);
            x += __shfl_xor(x, 1, 64);
            x += __shfl_xor(x, 2, 64);
            x = x * scale + slope * (float)(j - p);
            if (softcap > 0.f) x = softcap * tanhf(x / softcap);
            s[n] = !seen ? -INFINITY : page >= 0 ? x : NAN;    // a page that was given back is asked for: poison the result
        }
        float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
#pragma unroll
        for (int d = 4; d < 64; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
        const float m_new = fmaxf(m, mx), alpha = expf(m - m_new);
        float ps_ = 0.f;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            s[n] = expf(s[n] - m_new);                 // 0 where the key is not seen
            ps_ += s[n];
            if ((lane & 3) == n) p_sh[wave][n * 16 + kr] = s[n];
        }
#pragma unroll
        for (int d = 4; d < 64; d <<= 1) ps_ += __shfl_xor(ps_, d, 64);
        l = l * alpha + ps_;
        m = m_new;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const f32x4 pv = *(const f32x4*)&p_sh[wave][kq];
        const int jv = j0 + kq;
        const int page = jv + 3 >= lo && jv <= p ? bt[jv / ps] : -1;
        const bool edge = j0 < lo || j0 + 63 > p;      // some keys of the tile are not seen: what their places hold must not count
        const float* vp = page >= 0 ? v_pages + ((size_t)page * G + g) * hd * ps + (jv % ps) : nullptr;
#pragma unroll
        for (int i = 0; i < NI * 4; ++i)
            if (i < ni * 4) {
                f32x4 v = vp ? *(const f32x4*)(vp + (size_t)(i * 4 + cr) * ps) : zero;
                if (edge) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = jv + e >= lo && jv + e <= p ? v[e] : 0.f;
                }
                float a = o[i] * alpha;
#pragma unroll
                for (int e = 0; e < 4; ++e) a = fmaf(pv[e], v[e], a);
                o[i] = a;
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
#pragma unroll
    for (int i = 0; i < NI * 4; ++i)
        if (i < ni * 4) {
            const float a = row16_sum(o[i]);
            if ((lane & 15) == (i & 15)) o_sh[wave][i * 4 + cr] = a;
        }
    if (lane == 0) { ml_sh[wave][0] = m; ml_sh[wave][1] = l; }
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= hd) return;
    float mm = ml_sh[0][0];
#pragma unroll
    for (int w = 1; w < AF_WAVES; ++w) mm = fmaxf(mm, ml_sh[w][0]);
    float ll = 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
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
    dim3 grid(T, H);
#define AF_GO(NI) attn_f32_kernel<NI><<<grid, 64 * AF_WAVES, 0, st>>>(q, k_pages, v_pages, out, positions, seq_of_token, block_table, \
        max_blocks, H, G, hd, page_size, vis, span, scale, softcap, slopes)
    if (hd <= 64) AF_GO(4); else AF_GO(8);
#undef AF_GO
    SP_LAUNCH_CHECK("attn_f32");
    return 0;
}
