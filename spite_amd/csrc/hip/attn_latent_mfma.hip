// Latent attention on the matrix units (bfloat16): query rows [Dk] against cache rows [Dk] of one
// shared kv head, the value of a key being the first R elements of its row (see latent.hip).
//
// Because all heads read the same rows, the heads are the kernel's batch: query row t*H + h is
// one column of a 16-column MFMA tile, so a decoded token alone fills tiles with its heads, and a
// prompt's portion fills them with (token, head) pairs.  A workgroup of eight waves takes up to 128 consecutive
// query rows of one request (the list `wg`, built on the host from the step's entries: first row
// and number of rows), one wave per 16 rows.  All waves walk the same blocks of 32 keys, from the
// first key that the first row may read to the last row's own position.  Every row masks by its own position.
//
// A block's rows go straight from the pages to LDS (loads with the lds bit, an eighth of a block a wave), two blocks ahead in
// three buffers: one barrier a block, no register and no wave waits for them.  They lie there once, row by row, and serve both products:
//   S^T = K Q^T    reads 16 bytes of a row a lane;
//   O^T = V^T P^T  reads its operand, the same rows' elements turned, by transposing reads (four rows x 16 columns to 16 lanes).
// The 16-byte pieces of a row are exchanged by XOR with half its number, so that either read spreads over the banks.
// A block of rows of 576 takes eight waves 3.0 us, 6,700 cycles: some 2,200 of products, 4,400 and more of reads of LDS (36 KB a
// wave for the first product, 32 for the second) and the softmax between them, which the waves reach together.  Two tiles of
// rows a wave would halve the reads, but their output and queries fill the register file (240 spilled).  Before, a block was staged in
// two layouts, the turned one by 2-byte stores, and prompts had no load in flight: 40 heads of 576 / 512, two prompts of 1,021 and
// 765 tokens 294 us, now 174; 2,048 tokens 680 / 345; 700 behind a window of 4,096 796 / 485; two tokens of 1,024 keys 25.7 / 20.4, 64 of 500
// 41.9 / 32.0; rows of 320 and 192 0.43 to 0.88 of the time.
//
// Tiles: S^T tile tt (of 2) holds the keys (r/4)*8 + tt*4 + r%4 of the block in its rows r, so the
// eight scores a lane holds are eight consecutive keys: P^T is the next product's operand without a
// shuffle.  Scores, maximum, sum and the output are fp32; a score less the maximum goes into the exponent's units, base 2, and
// not the score: rounded there, scores of some thousands would each be off by more than their difference is.
//
// Few workgroups with many keys (decoded tokens of a few requests over long contexts): the blocks
// of keys are dealt to `n_splits` workgroups a work item (grid.y), each leaves a record (output not
// yet divided, maximum, sum) per query row, and a second kernel joins the records.
#include "common.h"

#define LM_ROWS 128        // query rows per workgroup at most (8 waves of 16)
#define LM_TABLE 64        // blocks of keys whose cache rows are looked up ahead, a half at a time
#define LM_BUFS 3

typedef short s16x4 __attribute__((ext_vector_type(4)));
static __device__ __attribute__((aligned(16))) const unsigned lm_zeros[4] = {0, 0, 0, 0};      // what a row that is not read holds

// A scaled score, rounded: the maximum is taken off it afterwards, not in the same operation, with masks or without.
static __device__ __forceinline__ float lm_scaled(float s, float scale) {
#pragma clang fp contract(off)
    return s * scale;
}

template <int KQ, int NV>   // Dk <= 32*KQ, R <= 16*NV
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(KQ > 6 ? 2 : 4)))
void attn_latent_mfma_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kv_pages, bf16* __restrict__ out,
                             const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                             const int* __restrict__ block_table, int max_blocks, const int* __restrict__ wg,
                             int H, int Dk, int R, int ps, int vis, int span, float scale,
                             float* __restrict__ part, int n_splits) {
    constexpr int PP = KQ * 4, BUF = 32 * PP * 16;                  // 16-byte pieces of a staged row; bytes of a block
    constexpr int XI = (PP / 2 + 7) / 8;                            // loads of a kilobyte a wave and block
    static_assert(PP % 8 == 0 && PP / 8 % 2 == 1, "an odd number of 128 bytes: neighbouring rows start 32 banks apart");
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    int* krow = (int*)(lds + LM_BUFS * BUF);                        // [LM_TABLE * 32] cache rows; -1: page given back, -2: not read
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g4 = lane >> 4;
    const int item = gridDim.x - 1 - blockIdx.x;                    // an entry's last rows, which read the most keys, start first
    const int row0 = wg[2 * item], nrows = wg[2 * item + 1];
    const int t_first = row0 / H, t_last = (row0 + nrows - 1) / H;
    const int* bt = block_table + (size_t)seq_of_token[t_first] * max_blocks;
    const int key_lo = sp_first_visible(positions[t_first], vis, span), key_hi = positions[t_last];

    // this workgroup's share of the blocks of keys
    int blk_first = key_lo >> 5, blk_end = (key_hi >> 5) + 1;
    if (n_splits > 1) {
        const int per = (blk_end - blk_first + n_splits - 1) / n_splits;
        blk_first += (int)blockIdx.y * per;
        blk_end = blk_first + per < blk_end ? blk_first + per : blk_end;
    }
    const int n_blk = blk_end - blk_first;

    // this lane's query row: a column of every tile
    const int my = wave * 16 + c;
    const bool row_ok = my < nrows;
    const int row = row0 + (row_ok ? my : 0);
    const int my_p = positions[row / H];
    const int my_lo = sp_first_visible(my_p, vis, span);
    // what this wave's rows read at all, and what all of them read (positions grow with the rows)
    const bool has_rows = wave * 16 < nrows;
    const int w_last = wave * 16 + 15 < nrows ? wave * 16 + 15 : nrows - 1;
    const int p_first = has_rows ? positions[(row0 + wave * 16) / H] : -1, p_last = has_rows ? positions[(row0 + w_last) / H] : -1;
    const int wave_lo = sp_first_visible(p_first, vis, span), wave_lo_all = sp_first_visible(p_last, vis, span);

    bf16x8 qf[KQ];
#pragma unroll
    for (int k = 0; k < KQ; ++k) {
        const int f = k * 32 + g4 * 8;
        bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        if (f < Dk) z = *(const bf16x8*)(q + (size_t)row * Dk + f);
        qf[k] = z;
    }
    // (there before the first block is asked for: a wait for them later would be one for the blocks too)
#pragma unroll
    for (int k = 0; k < KQ; ++k) asm volatile("" : "+v"(qf[k]));

    // the cache rows of 32 blocks from b0 on, to their half of the table; whether a key of them lies in a page that was given back
    auto look_up = [&](int b0) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = u * 512 + tid, j = ((blk_first + b0) << 5) + i;
            int r = -2;
            if (j >= key_lo && j <= key_hi) { const int page = bt[j / ps]; r = page >= 0 ? page * ps + j % ps : -1; }
            krow[((b0 & (LM_TABLE - 1)) << 5) + i] = r;
        }
        __syncthreads();
    };
    // this lane's pieces of a block, which key's and which piece of its row: kept in LDS, since the registers are full
    int* mine = krow + LM_TABLE * 32 + tid;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int at = i * 8 + wave < PP / 2 ? i * 8 + wave : PP / 2 - 1;           // (loads past the block's last: that one again)
        const int l = at * 64 + lane, r = l / PP, pc = (l % PP) ^ ((r >> 1) & 7);
        const int key = (((r & 15) >> 2) << 3) + ((r >> 4) << 2) + (r & 3);
        mine[i * 512] = pc * 8 < Dk ? key | pc << 8 : -1;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    auto ask = [&](int b, int buf) {
        const int* tab = krow + ((b & (LM_TABLE - 1)) << 5);
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int at = i * 8 + wave < PP / 2 ? i * 8 + wave : PP / 2 - 1;
            const int what = mine[i * 512], r = what < 0 ? -2 : tab[what & 255];
            const bf16* src = r >= 0 ? kv_pages + ((size_t)r * Dk + (what >> 8) * 8) : (const bf16*)lm_zeros;
            const unsigned to = lds0 + buf * BUF + at * 1024;
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                         :: "v"(src), "s"(__builtin_amdgcn_readfirstlane(to)) : "memory", "m0");
        }
    };

    float m_run = -INFINITY, l_run = 0.f;
    f32x4 o[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) o[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    // operands' places in a block: S^T rows c and c + 16, piece 4 k + g4; V^T rows 4 g4 + c / 4 and 16 further on, 8 bytes of piece 2 a + ..
    const int kx = (c >> 1) & 7, vr = g4 * 4 + (c >> 2), vx = (vr >> 1) & 7;
    const int kat = c * PP * 16 + ((g4 ^ kx) << 4);                // (pieces 8 n + g4; 8 n + 4 + g4: bit 6 the other way)
    const int vat = vr * PP * 16 + ((((c >> 1) & 1) ^ (vx & 1)) << 4) + ((c & 1) << 3), vxor = (vx & 6) << 4;

    if (n_blk > 0) {
        look_up(0);
        ask(0, 0);
        if (n_blk > 1) ask(1, 1);
    }
    for (int b = 0, buf = 0; b < n_blk; ++b, buf = buf + 1 < LM_BUFS ? buf + 1 : 0) {
        if (b + 1 < n_blk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(XI) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                               // the block is there, and the one before is no longer read
        asm volatile("" ::: "memory");
        if (b + 2 < n_blk) {
            if (((b + 2) & (LM_TABLE / 2 - 1)) == 0) look_up(b + 2);
            ask(b + 2, buf ? buf - 1 : LM_BUFS - 1);
        }
        const int blk0 = (blk_first + b) << 5;
        if (blk0 + 31 < wave_lo || blk0 > p_last) continue;         // nothing here for this wave's rows

        const unsigned char* kb = lds + buf * BUF;
        f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int k = 0; k < KQ; ++k)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
                s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(kb + (kat ^ (k & 1) << 6) + (k >> 1) * 128 + tt * 16 * PP * 16), qf[k], s[tt], 0, 0, 0);
        // the keys' rows, to see whether a page was given back, and masks, where some row does not read the whole block
        float mx = -INFINITY;
        const int* tab = krow + ((b & (LM_TABLE - 1)) << 5) + g4 * 8;
        int gone = tab[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) gone = min(gone, tab[i]);
        if (blk0 >= wave_lo_all && blk0 + 31 <= p_first && !__any(gone < 0)) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) { s[tt][i] = lm_scaled(s[tt][i], scale); mx = fmaxf(mx, s[tt][i]); }
        } else {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = blk0 + g4 * 8 + tt * 4 + i;
                    s[tt][i] = row_ok && j >= my_lo && j <= my_p ? (tab[tt * 4 + i] == -1 ? NAN : lm_scaled(s[tt][i], scale)) : -INFINITY;
                    mx = fmaxf(mx, s[tt][i]);
                }
        }
        mx = rows4_max(mx);
        const float m_new = fmaxf(m_run, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;       // (a row that has seen no key yet: weights of zero)
        const float alpha = __expf(m_run - m_use);
        float sum = 0.f;
        bf16x8 pf;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float e = __expf(s[tt][i] - m_use);
                sum += e;
                pf[tt * 4 + i] = (bf16)e;
            }
        sum = rows4_sum(sum);
        l_run = l_run * alpha + sum;
        m_run = m_new;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int a = 0; a < NV; ++a) o[a] = o[a] * alpha;
        }
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            const unsigned char* vp = kb + vat + (((a & 7) << 5) ^ vxor) + (a >> 3) * 256;
            typedef __attribute__((address_space(3))) s16x4* lds4;
            const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)vp);
            const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vp + 16 * PP * 16));
            const bf16x8 v = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
            o[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf, o[a], 0, 0, 0);
        }
    }
    if (!row_ok) return;
    if (m_run == -INFINITY && max(my_lo, blk_first << 5) <= min(my_p, (blk_end << 5) - 1)) {
        // every key that the row reads here has the score -inf: no weights to divide by
        l_run = NAN;
#pragma unroll
        for (int a = 0; a < NV; ++a) o[a] = f32x4{NAN, NAN, NAN, NAN};
    }
    // o[a][i] of lane (c, g4) is O[row c][a*16 + g4*4 + i]
    if (n_splits > 1) {
        float* rec = part + ((size_t)row * n_splits + blockIdx.y) * (R + 2);
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            const int col = a * 16 + g4 * 4;
            if (col < R) {
#pragma unroll
                for (int i = 0; i < 4; ++i) rec[col + i] = o[a][i];
            }
        }
        if (g4 == 0) { rec[R] = m_run; rec[R + 1] = l_run; }
        return;
    }
    const float inv = 1.0f / fmaxf(l_run, 1e-30f);
    bf16* orow = out + (size_t)row * R;
#pragma unroll
    for (int a = 0; a < NV; ++a) {
        const int col = a * 16 + g4 * 4;
        if (col < R) {
            bf16x4 w;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (bf16)(o[a][i] * inv);
            *(bf16x4*)(orow + col) = w;
        }
    }
}

// Joins the records [row][split][R + 2] of a split call: one workgroup a query row.
__global__ __launch_bounds__(256)
void attn_latent_join_kernel(const float* __restrict__ part, bf16* __restrict__ out, int R, int n_splits) {
    __shared__ float wsh[1024];          // weight of every split: exp(m_s - M) / L
    __shared__ float red[8];
    const size_t row = blockIdx.x;
    const float* rec = part + row * n_splits * (R + 2);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the first 1024 splits' maxima and sums, four a thread
    float ms[4], ls[4], M = -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int s = tid + u * 256;
        ms[u] = s < n_splits ? rec[(size_t)s * (R + 2) + R] : -INFINITY;
        ls[u] = s < n_splits ? rec[(size_t)s * (R + 2) + R + 1] : 0.f;
        M = fmaxf(M, ms[u]);
    }
    M = wave_max(M);
    if (lane == 0) red[wave] = M;
    __syncthreads();
    M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float L = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int s = tid + u * 256;
        const float w = ms[u] == -INFINITY ? 0.f : __expf(ms[u] - M);
        if (s < n_splits) wsh[s] = w;
        L += w * ls[u];
    }
    L = wave_sum(L);
    if (lane == 0) red[4 + wave] = L;
    __syncthreads();
    const float inv = 1.0f / fmaxf(red[4] + red[5] + red[6] + red[7], 1e-30f);
    // (a split without keys left zeros and the weight 0: its record is read like the others', so that the loads follow
    // each other without waiting; two columns a thread, R is a multiple of 8)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    for (int c = tid * 2; c < R; c += 512) {
        f32x2 acc = {0.f, 0.f};
#pragma unroll 8
        for (int s = 0; s < n_splits; ++s) {
            const f32x2 v = *(const f32x2*)(rec + (size_t)s * (R + 2) + c);
            acc[0] += wsh[s] * v[0];
            acc[1] += wsh[s] * v[1];
        }
        bf16* o = out + row * R + c;
        o[0] = (bf16)(acc[0] * inv);
        o[1] = (bf16)(acc[1] * inv);
    }
}

// `wg`: int32 pairs (first query row, rows <= 128) on the device, `n_wg` of them, each within one
// request's rows of the step; `max_rows`: the most rows of any pair (it sizes the workgroups).
// `n_splits` > 1: the keys of every pair are dealt to that many workgroups; `part` (fp32,
// rows * n_splits * (R + 2) floats, rows = T * H) holds their records.
extern "C" int spite_attn_latent_mfma(const void* q, const void* kv_pages, void* out, const int* positions,
                                      const int* seq_of_token, const int* block_table, int max_blocks, const int* wg,
                                      int n_wg, int max_rows, int H, int Dk, int R, int page_size, int vis, int span,
                                      float scale, float* part, int n_splits, int n_rows, hipStream_t st) {
    SP_REQUIRE(H > 0 && n_wg >= 0 && max_rows >= 0 && max_rows <= LM_ROWS, "latent attention: %d rows a workgroup, at most %d", max_rows, LM_ROWS);
    SP_REQUIRE(Dk > 0 && Dk % 8 == 0 && R > 0 && R % 8 == 0 && R <= Dk && Dk <= 576 && R <= 512,
               "latent attention (MFMA): rows of %d with a latent of %d: multiples of 8, at most 576 and 512", Dk, R);
    SP_REQUIRE(page_size > 0 && max_blocks > 0, "latent attention: bad page size %d or table width %d", page_size, max_blocks);
    SP_REQUIRE(vis >= 0 && vis < SP_VIS_COUNT && (!sp_vis_has_span(vis) || span > 0), "latent attention: chunk or window of %d", span);
    SP_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)kv_pages & 15) == 0 && ((uintptr_t)out & 7) == 0, "latent attention: operands must be 16-byte aligned");
    SP_REQUIRE(n_splits >= 1 && n_splits <= 1024 && (n_splits == 1 || part), "latent attention: %d splits", n_splits);
    if (n_wg == 0 || max_rows == 0) return 0;
    const int kq = (Dk + 31) / 32, nv = (R + 15) / 16;
#define SP_LM(KQV, NVV) do { \
        auto kern = attn_latent_mfma_kernel<KQV, NVV>; \
        constexpr size_t sh = LM_BUFS * 32 * KQV * 64 + (LM_TABLE * 32 + (KQV * 2 + 7) / 8 * 512) * sizeof(int); \
        static bool allowed = false; \
        if (!allowed) { hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh); \
            if (e != hipSuccess) return sp_fail("latent attention: %zu bytes of LDS refused: %s", sh, hipGetErrorString(e)); allowed = true; } \
        kern<<<dim3(n_wg, n_splits), 512, sh, st>>>((const bf16*)q, (const bf16*)kv_pages, (bf16*)out, positions, seq_of_token, \
                                        block_table, max_blocks, wg, H, Dk, R, page_size, vis, span, scale, part, n_splits); } while (0)
    if (kq <= 6 && nv <= 8) SP_LM(6, 8);
    else if (kq <= 10 && nv <= 16) SP_LM(10, 16);
    else SP_LM(18, 32);
#undef SP_LM
    SP_LAUNCH_CHECK("attn_latent_mfma");
    if (n_splits > 1) {
        attn_latent_join_kernel<<<n_rows, 256, 0, st>>>(part, (bf16*)out, R, n_splits);
        SP_LAUNCH_CHECK("attn_latent_join");
    }
    return 0;
}
