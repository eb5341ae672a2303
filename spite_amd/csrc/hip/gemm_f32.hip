// fp32 matrix product Y = A . W^T on the matrix units (v_mfma_f32_16x16x4_f32: fp32 operands, fp32 FMAs, no narrower
// step anywhere), the true 32-bit path of every projection whose rows can be read 16 bytes at a time.
//
// The order of every sum depends on K alone.  k is cut into eight runs of `seg` (K / 8 rounded up to 64); inside a
// run the products are added in steps of 16 k, four MFMAs a step (MFMA e takes k0 + 4q + e of its four rows of lanes
// q); the runs' sums are then added in their order, ((0 + s0) + s1) + ... + s7.  Both kernels below keep this order, so
// a row has the same bits whether it comes alone or among many, and shorter chains round less than one ascending
// chain over K.
//
//  gemm_f32_rows: few rows.  Bound by the stream of W (one row of X makes 0.5 FLOP a byte).  A workgroup takes 16
//    rows of W (GLU: 16 of each half) and gives one run of k to each of its eight waves, so that a product with
//    2,048 output rows has 1,024 waves in flight; the runs' sums meet in LDS.  A wave's next 32 k are on their way while 32 are multiplied, so
//    that a wave needs 54 registers and three and four workgroups fit a compute unit (us, with 128 k asked for behind conditions and waited for
//    together / now: 1 row x 3,072 x 2,048 8.4 / 7.5, x 32,768 54.8 / 50.6, two groups of a row gated 2 x 3,072 x 2,048 24.4 / 19.1, 17 groups
//    of 16 rows and of one 107.5 / 97.7, 64 x 3,072 x 2,048 25.8 / 23.8).
//  gemm_f32_tile: many rows, bound by the MFMAs (256 FLOP a clock and compute unit).  TM (64 or 32) rows of X times 64 rows of
//    W a workgroup: X through double-buffered LDS, a step ahead, read by all four waves; a wave's 16 rows of W straight into
//    registers, two steps ahead.  One workgroup a compute unit reaches 70 % of the units' rate at K = 2,048, its start and end included.
//
// Which one, and its tile: see f32_variant.
#include "common.h"


// sum of one step of 16 k: the lane's four k of each operand
__device__ __forceinline__ void f32_step(f32x4& acc, f32x4 w, f32x4 x) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[0], x[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[1], x[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[2], x[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[3], x[3], acc, 0, 0, 0);
}

__device__ __forceinline__ int f32_seg(int K) { return (K + 511) / 512 * 64; }

// A lane of a result tile holds W rows n0 + 4q .. + 3 of X row `s`.
__device__ __forceinline__ void f32_store(float* __restrict__ Y, size_t row, int ldy, int n, int N, f32x4 v, bool vec) {
    float* y = Y + row * ldy + n;
    if (vec && n + 3 < N) *(f32x4*)y = v;
    else
#pragma unroll
        for (int r = 0; r < 4; ++r) if (n + r < N) y[r] = v[r];
}

// HALVES (GLU, N a multiple of 8): a workgroup takes eight rows of each half, in one MFMA operand: twice as many workgroups, where
// those of sixteen are few or some compute units have one more than others (2 x 3,072 x 2,048, two groups of a row 27.3 -> 23.9 us, three 36.1 ->
// 31.5; five, 3.75 a unit, 46.2 with either).
template <int MT, int GLU, bool HALVES = false>
__global__ __launch_bounds__(512)
void gemm_f32_rows_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, long w_group_stride,
                          float* __restrict__ Y, int ldy, int M, int N, int K, const int* __restrict__ offsets, int n_groups,
                          const int* __restrict__ a_rows, const float* __restrict__ a_scale, const int* __restrict__ y_rows,
                          int act, float act_limit, int vec_y) {
    constexpr int NB = GLU && !HALVES ? 2 : 1;
    __shared__ f32x4 red[8][MT * NB][64];
    asm volatile("" :: "s"(A), "s"(lda), "s"(W), "s"(w_group_stride), "s"(Y), "s"(ldy), "s"(M), "s"(N), "s"(K), "s"(offsets), "s"(n_groups), "s"(a_rows),
                 "s"(a_scale), "s"(y_rows), "s"(act), "s"(act_limit), "s"(vec_y));      // (every argument at once)
    int g = 0, row0 = 0, row_end = M;
    if (offsets) {
        if (!sp_find_tile_scalar(offsets, n_groups, MT * 16, blockIdx.y, g, row0, row_end)) return;
    } else {
        row0 = blockIdx.y * (MT * 16);
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * (HALVES ? 8 : 16);
    const float* Wg = W + (size_t)g * w_group_stride;
    const int wn = n0 + r < N ? n0 + r : N - 1;
    const float* wp[NB];
    wp[0] = Wg + (size_t)(HALVES ? n0 + (r & 7) + (r < 8 ? 0 : N) : wn) * K;
    if (NB == 2) wp[NB - 1] = Wg + (size_t)(N + wn) * K;
    const float* xp[MT];
    float sc[MT];
    bool live[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int s = row0 + m * 16 + r;
        live[m] = s < row_end;
        const int ss = live[m] ? s : row0;             // a row that exists: its products are not stored
        xp[m] = A + (size_t)(a_rows ? a_rows[ss] : ss) * lda;
        sc[m] = a_scale ? a_scale[ss] : 1.0f;
    }
    const int seg = f32_seg(K);
    const int k_lo = wave * seg, k_hi = k_lo + seg < K ? k_lo + seg : K;
    f32x4 acc[MT][NB];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[m][b] = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 2, KU = 16 * U;                   // steps of 16 k a piece (four: one or two rows 3 to 6 % slower, tall tables 3 % faster)
    f32x4 w[2][U][NB], x[2][U][MT];
    auto load = [&](int to, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 16 + q * 4;
#pragma unroll
            for (int b = 0; b < NB; ++b) w[to][u][b] = *(const f32x4*)(wp[b] + k);
#pragma unroll
            for (int m = 0; m < MT; ++m) x[to][u][m] = *(const f32x4*)(xp[m] + k);
        }
    };
    auto mul = [&](int to) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const f32x4 xs = x[to][u][m] * sc[m];
#pragma unroll
                for (int b = 0; b < NB; ++b) f32_step(acc[m][b], w[to][u][b], xs);
            }
    };
    // A piece is multiplied while the next one is on its way.  No load stands behind a condition, where the compiler would wait at the
    // next product for every load there may be.
    const int whole = k_hi > k_lo ? (k_hi - k_lo) / KU : 0;
    if (whole >= 2) {
        load(0, k_lo);
        load(1, k_lo + KU);
        int i = 0;
        for (; i + 4 <= whole; i += 2) {
            mul(0);
            load(0, k_lo + (i + 2) * KU);
            mul(1);
            load(1, k_lo + (i + 3) * KU);
        }
        mul(0);
        if (i + 2 == whole) mul(1);
        else {
            load(0, k_lo + (i + 2) * KU);
            mul(1);
            mul(0);
        }
    } else if (whole == 1) {
        load(0, k_lo);
        mul(0);
    }
    if (k_lo + whole * KU < k_hi) {                    // the run's end: zeros past it (K is a multiple of 4, a run's end of 4)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k_lo + whole * KU + u * 16 + q * 4;
            const bool in = k < k_hi;
#pragma unroll
            for (int b = 0; b < NB; ++b) w[0][u][b] = in ? *(const f32x4*)(wp[b] + k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < MT; ++m) x[0][u][m] = in ? *(const f32x4*)(xp[m] + k) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        mul(0);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) red[wave][m * NB + b][lane] = acc[m][b];
    __syncthreads();
    if (wave >= MT) return;
    const int m = wave, s = row0 + m * 16 + r;
    f32x4 t[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        t[b] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i) t[b] += red[i][m * NB + b][lane];
    }
    if (HALVES)                                        // rows 8 to 15, the up half's: 32 lanes further on
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float up = __shfl_down(t[0][e], 32, 64);
            t[0][e] = sp_gated(t[0][e], up, act, act_limit, false);
        }
    if (s >= row_end || (HALVES && q >= 2)) return;
    if (GLU && !HALVES)
#pragma unroll
        for (int e = 0; e < 4; ++e) t[0][e] = sp_gated(t[0][e], t[NB - 1][e], act, act_limit, false);
    f32_store(Y, y_rows ? (size_t)y_rows[s] : (size_t)s, ldy, n0 + q * 4, N, t[0], vec_y);
}

#define F32_TK 64                 // k a step through LDS
#define F32_LD (F32_TK + 4)       // LDS row: 16 bytes more than a step, so that 16 rows' reads spread over the banks

// The loop over k for a tile whose first LIVE groups of 16 rows hold rows (an expert's last tile is seldom full).  X goes through
// LDS a step ahead, its operands are read from there a piece of 16 k ahead of their products (read at their use, each piece waited
// for LDS some 150 of its 256 to 512 cycles of products), and a chain of four MFMAs is spread over the accumulators.  A wave's W lies
// in sets of registers:
//  * two, each piece asked for again, two steps on, as soon as its products are issued, and the next step's rows put into LDS before
//    the last piece's products;
//  * BURST, groups of few rows, bound by the stream of W from memory: three, a whole step's pieces asked for at once at the start of the
//    step two before, the rows put into LDS last, since waiting for them is waiting for the W asked for before them.
// Before and now (us): 200 rows x 2,048 x 3,072 55 / 34, 301 x 3,072 x 2,048 54 / 44, 301 x 32,768 x 2,048 380 / 365, gated 301 x 3,072
// x 2,048 100 / 78; 16 groups and one of all of 301 rows, gated 2 x 3,072 x 2,048, 271 / 245, and 2,048 x 3,072 144 / 139 (with two sets 150).
// Groups' last steps, whose loads would pass the end, are not in the whole steps' loop nor guarded one by one (they were, and short sums spent
// most of their time there: 128 groups and one of all of 150 rows, 2,048 x 512, 73 us before / 76 with guards / 68 now; 800 rows of 128
// groups x 768 x 512 38.7 / 41.5 / 38.6).  64 groups of a few rows x 2,048 x 3,072 take 3 % more than before (317 / 308), at 5.1 TB/s of W.
template <int TM, int NB, int LIVE, bool BURST>
__device__ __forceinline__ void f32_tile_loop(float* xs, const float* const* wp, const float* const* xp, const float* sc, int K,
                                              int seg, int lr, int lk, int r, int q, f32x4 (&tot)[TM / 16][NB]) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = F32_TK / 16, XL = TM * F32_TK / 1024;      // pieces of 16 k, 16-byte pieces of X a thread
    constexpr int S = BURST ? 3 : 2;                              // sets of W
    f32x4 acc[LIVE][NB], w[S][U][NB], xv[XL], x0[LIVE], x1[LIVE];
#pragma unroll
    for (int m = 0; m < LIVE; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[m][b] = zero;
    const float* wl[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) wl[b] = wp[b] + q * 4;
    const float* xl = xs + r * F32_LD + q * 4;
    float* xw = xs + lr * F32_LD + lk;
    int buf = 0, k0 = 0, flush = seg;
    // (whole: every k that the step asks for exists; else k past the end takes the last four's address, and zeros in their place)
    auto load_w = [&](f32x4 (&w)[NB], int k, bool whole) {
        const int kc = whole || k + q * 4 < K ? k : K - 4 - q * 4;
#pragma unroll
        for (int b = 0; b < NB; ++b) w[b] = *(const f32x4*)(wl[b] + kc);
    };
    auto load_x = [&](int k, bool whole) {
        const int kc = whole || k + lk < K ? k + lk : K - 4;
#pragma unroll
        for (int i = 0; i < XL; ++i) xv[i] = *(const f32x4*)(xp[i] + kc);
    };
    auto put_x = [&](int to, int k, bool whole) {
        const bool in = whole || k + lk < K;
#pragma unroll
        for (int i = 0; i < XL; ++i) *(f32x4*)(xw + to * (TM * F32_LD) + i * (TM / XL) * F32_LD) = in ? xv[i] * sc[i] : zero;
    };
    auto read_x = [&](f32x4 (&x)[LIVE], int u) {
#pragma unroll
        for (int m = 0; m < LIVE; ++m) x[m] = *(const f32x4*)(xl + buf * (TM * F32_LD) + m * 16 * F32_LD + u * 16);
    };
    auto step = [&](f32x4 (&w)[U][NB], f32x4 (&w2)[U][NB], bool whole) {
        __syncthreads();                               // this step's rows are in LDS, the other buffer is free
        if (k0 == flush) {
#pragma unroll
            for (int m = 0; m < LIVE; ++m)
#pragma unroll
                for (int b = 0; b < NB; ++b) { tot[m][b] += acc[m][b]; acc[m][b] = zero; }
            flush += seg;
        }
        read_x(x0, 0);
        load_x(k0 + F32_TK, whole);
        if (BURST)
#pragma unroll
            for (int u = 0; u < U; ++u) load_w(w2[u], k0 + 2 * F32_TK + u * 16, whole);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            f32x4 (&x)[LIVE] = u & 1 ? x1 : x0;
            if (u + 1 < U) read_x(u & 1 ? x0 : x1, u + 1);
            else if (!BURST) put_x(buf ^ 1, k0 + F32_TK, whole);
            if (!whole && k0 + u * 16 + 16 > K) {
                const bool in = k0 + u * 16 + q * 4 < K;
#pragma unroll
                for (int b = 0; b < NB; ++b) w[u][b] = in ? w[u][b] : zero;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int m = 0; m < LIVE; ++m)
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][b][e], x[m][e], acc[m][b], 0, 0, 0);
            if (!BURST) load_w(w[u], k0 + S * F32_TK + u * 16, whole);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (BURST) put_x(buf ^ 1, k0 + F32_TK, whole);
        buf ^= 1;
        k0 += F32_TK;
    };
    load_x(0, false);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u) load_w(w[i][u], i * F32_TK + u * 16, false);
    put_x(0, 0, false);
    while (k0 + (S + 2) * F32_TK <= K) {
#pragma unroll
        for (int i = 0; i < S; ++i) step(w[i], w[(i + 2) % S], true);
    }
    if constexpr (BURST) {
        while (k0 + 2 * F32_TK < K) {
#pragma unroll
            for (int i = 0; i < S; ++i) step(w[i], w[(i + 2) % S], false);
        }
        if (k0 < K) step(w[0], w[2 % S], false);
        if (k0 < K) step(w[1], w[0], false);
    } else
    while (k0 < K) {
#pragma unroll
        for (int i = 0; i < S; ++i)
            if (k0 < K) step(w[i], w[(i + 2) % S], false);
    }
#pragma unroll
    for (int m = 0; m < LIVE; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) tot[m][b] += acc[m][b];
}

template <int TM, int GLU, bool BURST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(GLU ? (TM == 64 || BURST ? 2 : 3) : TM == 64 ? 3 : 4)))
void gemm_f32_tile_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, long w_group_stride,
                          float* __restrict__ Y, int ldy, int M, int N, int K, const int* __restrict__ offsets, int n_groups,
                          const int* __restrict__ a_rows, const float* __restrict__ a_scale, const int* __restrict__ y_rows,
                          int act, float act_limit, int vec_y) {
    constexpr int NB = GLU ? 2 : 1;
    __shared__ __align__(16) float xs[2 * TM * F32_LD];
    int g = 0, row0 = 0, row_end = M;
    if (offsets) {
        // the last groups' tiles start first: a group that every row visits comes last and has the full ones, an expert's
        // hold a few rows and fill the end (17 groups, 301 rows over 16 and all of them, 2 x 3,072 x 2,048 gated: 264 / 287 us; 16 x 20 rows 208 / 252)
        if (!sp_find_tile(offsets, n_groups, TM, gridDim.y - 1 - blockIdx.y, g, row0, row_end)) return;
    } else {
        row0 = blockIdx.y * TM;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 64 + wave * 16;
    const float* Wg = W + (size_t)g * w_group_stride;
    const int wn = n0 + r < N ? n0 + r : N - 1;
    const float* wp[NB];
    wp[0] = Wg + (size_t)wn * K;
    if (GLU) wp[NB - 1] = Wg + (size_t)(N + wn) * K;
    // the loader: a thread brings 4 k of every XL-th part of the rows
    constexpr int XL = TM * F32_TK / 1024, PIECES = F32_TK / 4;
    const int lk = (threadIdx.x % PIECES) * 4, lr = threadIdx.x / PIECES;
    const float* xp[XL];
    float sc[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int s = row0 + lr + i * (TM / XL), ss = s < row_end ? s : row0;
        xp[i] = A + (size_t)(a_rows ? a_rows[ss] : ss) * lda;
        sc[i] = a_scale ? a_scale[ss] : 1.0f;
    }
    f32x4 tot[TM / 16][NB];
#pragma unroll
    for (int m = 0; m < TM / 16; ++m)
#pragma unroll
        for (int b = 0; b < NB; ++b) tot[m][b] = {0.f, 0.f, 0.f, 0.f};
    const int rows = row_end - row0, seg = f32_seg(K);
    bool done = false;
    if constexpr (TM == 64) {
        if (rows > 48) f32_tile_loop<TM, NB, 4, false>(xs, wp, xp, sc, K, seg, lr, lk, r, q, tot);
        else if (rows > 32) f32_tile_loop<TM, NB, 3, false>(xs, wp, xp, sc, K, seg, lr, lk, r, q, tot);
        done = rows > 32;
    }
    if (done) {}
    else if (rows > 16) f32_tile_loop<TM, NB, 2, BURST>(xs, wp, xp, sc, K, seg, lr, lk, r, q, tot);
    else f32_tile_loop<TM, NB, 1, BURST>(xs, wp, xp, sc, K, seg, lr, lk, r, q, tot);
#pragma unroll
    for (int m = 0; m < TM / 16; ++m) {
        const int s = row0 + m * 16 + r;
        if (s >= row_end) continue;
        f32x4 t = tot[m][0];
        if (GLU)
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = sp_gated(t[e], tot[m][NB - 1][e], act, act_limit, false);
        f32_store(Y, y_rows ? (size_t)y_rows[s] : (size_t)s, ldy, n0 + q * 4, N, t, vec_y);
    }
}

// Rows of X a workgroup takes: of gemm_f32_rows (16, 32 or 64; 8: 16 rows, eight columns), or minus those of gemm_f32_tile (32 or
// 64).  `n_groups` 0: no groups.
//
// Both kernels take a time that follows from the most workgroups that a compute unit gets, c: for 2,048 of K, on an MI355X (us), the
// stream of 16 rows 7 c (gated 11.5 c), tiles of 32 rows 7 + 19 c (5 + 41 c), of 64 9 + 29 c (10 + 56 c); the stream gives each
// of its eight waves a run of 64 k and more, so that shorter sums than 512 leave some idle.  Most lines lie where 14,900 products (1
// to 1,500 tokens, up to 128 groups of 1 to 8 a token, K of 128 to 8,192) were timed with every variant when tiles took
// 14 + 19.5 c (14 + 47 c) and 17 + 36 c (19 + 82 c); those of 17 to 64 rows, and the figures here, are of the tiles as they are (1,428
// products, 9 to 1,200 tokens, up to 129 groups, K of 512 to 5,120: the choice is 4 % off the best variant on average, 17 to 64 rows 1 in
// groups and 4 without, where the lines before were 70 and 18 off; groups of few rows 6 to 9, which tiles have gained most on).  The stream has become 8 to 22 % faster since (see the top); by 260 products with
// every variant as it is the choice is off the best by 1.5 % for groups of few rows, 4 up to 16 rows (gated: sixteen columns a workgroup
// instead of eight), 5 and 7 at 17 to 64 without groups and with, and 16 to 18 beyond, where narrow W, which leaves tiles too few, would be
// the stream's (4 groups, 119 rows x 256 x 1,024 17.1 us, by the stream 6.8):
//  * groups of up to eight rows on average: the stream of every group's W, 16 rows a workgroup (16 groups and one of all t rows, 2 x
//    3,072 x 2,048 gated: t = 17 114, with 32 rows a workgroup 170, tiles 131; t = 64 184 / tiles 171), but tiles of 32 rows where sums are
//    short and tiles enough (K <= 512 and more than one a compute unit; plain K < 2,048 and more than two: 129 groups x 4,096 x 1,536,
//    400 rows, 465 / stream 634; 2,048 x 2,048 stays, 500 rows, 396 / tiles 344).
//  * 17 to 64 rows, no groups or larger ones: over three to seven groups the stream, 16 rows a workgroup, up to four of them a compute unit
//    (c of 2.8: 5 groups, 48 rows x 2,048 x 2,048, 25.5, tiles of 32 28.9, 64 rows a workgroup 48; over the line: x 3,072 x 2,048, 4.1,
//    36 / 30 / 63, gated 59 / 51 / 100; 64 rows, gated 6,144 x 768, 9.8, 48 / 38 / 103).  Over one or two and without groups three and a half,
//    where W is taller than a workgroup of any rows a unit (64 rows x 5,120 x 5,120, c = 5, 96 / 55 / 106; 52 x 4,096 x 1,536 stays, 18 / 20);
//    below, 16 rows up to one workgroup a unit (64 x 1,024 x 1,024 7.9, all rows in one 13.8), then as many rows a workgroup as there are, which
//    reads W once (33 x 3,072 x 2,048 19.3, with 16 rows 21.6).  W of fewer than 256 columns over groups was not timed and has the rows it had.
//  * up to 16 rows: the stream, unless W is tall enough for two workgroups of tiles a compute unit (32,768 x 2,048: 9 rows
//    55 with the stream, 46 with tiles of 32).
//  * more rows: tiles of 32 up to three of them a compute unit, gated two, with groups two and a quarter (3,072 x 2,048, 101 rows: 26
//    / 43, 301, near the line, 45 / 45; gated, 380, over it, 119 / 148), and where groups hold up to 20 rows, plain ones 160 (17 groups, 2 x
//    3,072 x 2,048, t = 150 177 / 174, t = 301, over the line, 238 / 230); none past 128 a compute unit, more than was timed.
//  * eight columns: up to a workgroup of sixteen a compute unit, up to three for K of 2,048 and more (3,072 x 2,048, two groups of a
//    row 23.9 / 27.3; 5 rows x 6,144 x 768, over the line, 16.9 / 15.3).
static int f32_variant(int M, int N, int K, int n_groups, int glu) {
    const long cus = sp_cu_count(), cols = (N + 63) / 64, live = n_groups ? (n_groups < M ? n_groups : M) : 1, streams = (N + 15) / 16 * live;
    const bool halves = glu && N % 8 == 0 && (streams <= cus || (streams <= 3 * cus && K >= 2048));
    const bool few = n_groups && M > 16 && M <= 8L * n_groups;
    const bool short_sum = (K <= 512 && live * cols > cus) || (!glu && K < 2048 && live * cols > 2 * cus);
    if (few && !short_sum && M / 16L + n_groups <= 65535) return halves ? 8 : 16;      // (the grid's limit)
    if (!few && M > 16 && M <= 64 && (!n_groups || N >= 256)) {
        const double c = ((N + 15) / 16) * (n_groups ? M / 16.0 + 0.5 * live : (M + 15) / 16) / cus;      // workgroups of 16 rows a compute unit
        if (n_groups > 2 ? c > 4.0 : c > 3.5 && (N + 15) / 16 > cus) return -32;
        if (n_groups > 2 || c <= 1.0) return 16;
    }
    if (!few && M <= 64 && (n_groups || M <= 8 || cols * ((M + 31) / 32) < 2 * cus)) return M > 32 ? 64 : M > 16 ? 32 : halves ? 8 : 16;
    const double tiles = (n_groups ? M / 32.0 + 0.5 * live : (M + 31) / 32) * cols / cus;         // of 32 rows, a compute unit
    if (tiles <= (!glu ? 3.0 : n_groups ? 2.25 : 2.0) || (!n_groups && M <= 64)) return -32;
    return tiles <= 128.0 && (M <= 20L * n_groups || (!glu && M <= 160L * n_groups)) ? -32 : -64;
}
extern "C" int spite_gemm_f32_choice(int M, int N, int K, int n_groups, int glu) { return f32_variant(M, N, K, n_groups, glu); }
// Gated, K = 2,048: the rows alone.
extern "C" int spite_gemm_f32_variant(int M, int N, int n_groups) { const int v = f32_variant(M, N, 2048, n_groups, 1); return v == 8 ? 16 : v; }

// The product if its rows can be read 16 bytes at a time (returns 0, or an error), else 1: the plain kernel's.
int sp_gemm_f32(const float* A, int lda, const float* W, long w_group_stride, float* Y, int ldy, int M, int N, int K,
                const int* offsets, int n_groups, const int* a_rows, const float* a_scale, const int* y_rows, int glu,
                float act_limit, hipStream_t st) {
    if (K % 4 || lda % 4 || w_group_stride % 4 || ((uintptr_t)A | (uintptr_t)W) % 16) return 1;
    const int vec_y = ldy % 4 == 0 && (uintptr_t)Y % 16 == 0;
    const int variant = f32_variant(M, N, K, offsets ? n_groups : 0, glu), tile = variant == 8 ? 16 : variant > 0 ? variant : -variant;
    const int m_tiles = offsets ? M / tile + (n_groups < M ? n_groups : M) : (M + tile - 1) / tile;
    SP_REQUIRE(m_tiles <= 65535, "gemm: too many row tiles (%d)", m_tiles);
#define SP_F32_ARGS A, lda, W, w_group_stride, Y, ldy, M, N, K, offsets, n_groups, a_rows, a_scale, y_rows, glu, act_limit, vec_y
    if (variant < 0) {
        dim3 grid((N + 63) / 64, m_tiles);
#define SP_F32_TILE(TM, GLU) do { if (offsets) gemm_f32_tile_kernel<TM, GLU, true><<<grid, 256, 0, st>>>(SP_F32_ARGS); \
                                  else gemm_f32_tile_kernel<TM, GLU, false><<<grid, 256, 0, st>>>(SP_F32_ARGS); } while (0)
        if (tile == 32 && glu) SP_F32_TILE(32, 1);
        else if (tile == 32) SP_F32_TILE(32, 0);
        else if (glu) SP_F32_TILE(64, 1);
        else SP_F32_TILE(64, 0);
#undef SP_F32_TILE
        SP_LAUNCH_CHECK("gemm_f32_tile");
        return 0;
    }
    dim3 grid((N + 15) / 16, m_tiles);
#define SP_F32_ROWS(MT) do { if (glu) gemm_f32_rows_kernel<MT, 1><<<grid, 512, 0, st>>>(SP_F32_ARGS); \
                             else gemm_f32_rows_kernel<MT, 0><<<grid, 512, 0, st>>>(SP_F32_ARGS); } while (0)
    if (variant == 8)
        gemm_f32_rows_kernel<1, 1, true><<<dim3(N / 8, m_tiles), 512, 0, st>>>(SP_F32_ARGS);
    else if (tile == 16) SP_F32_ROWS(1);
    else if (tile == 32) SP_F32_ROWS(2);
    else SP_F32_ROWS(4);
#undef SP_F32_ROWS
#undef SP_F32_ARGS
    SP_LAUNCH_CHECK("gemm_f32_rows");
    return 0;
}
