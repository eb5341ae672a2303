// Tiled bf16 product for many rows with both operands in LDS: Y[M,N] = X[M,K] . W[N,K]^T, fp32 accumulation on MFMA
// 16x16x32, W in MFMA operand order (see gemm_tiled.hip), K a multiple of 64.
//
// A workgroup of eight waves owns 256 rows of W (GLU: 128 gate rows and the matching 128 up rows) and 32 * NB rows of X
// ("slots"), NB = 3 .. 8; a wave owns 64 of the one and 16 * NB of the other.  What bounds such a product on this chip is
// first the path from L2 into a compute unit and then, near 1.3 PFLOP/s, the power limit, which lowers the clock.  The
// tile asks for 32 KB of operands per 256 x 256 x 32 products, as 512 x 160 through registers would, but as the operands go
// straight to LDS (buffer loads with the lds bit) no register waits for them and they are asked for three to five
// phases of 32 k ahead; and the tile may be as tall as the group of rows needs, in steps of 32.
//
//  * W: four buffers of a phase (16 tiles of one kilobyte, copied as they lie in memory).  X: three buffers of a unit of
//    64 k, eight lanes to the 128 bytes of a row (whole cache lines), the 16-byte pieces of row r exchanged by XOR with
//    r / 2 mod 8, so that the sixteen rows an operand read touches spread over all banks (measured: no conflicts).
//  * A phase multiplies the operands that were read from LDS during the phase before, while it reads the next phase's,
//    two MFMAs to a read.  One barrier a phase: behind it, every wave's loads for the next phase are there (each waits
//    for its own before it) and the buffers of this phase are free, so the loads that refill them go out.
//  * Groups (experts): each group takes as few tiles as 256 rows allow, of the smallest NB that then covers its rows; the
//    tiles of one column follow each other, tall ones of a group that every token visits beside the experts' short
//    ones, whose time is the stream of their W: compute and memory are busy together.
//  * Plain products: NB by the rounds that the tiles make on the chip: see lds_time.
//
// Measured on an MI355X beside gemm_tiled (us): 2,048 x 5,120 x 5,120 91 / 101, 1,786 x 5,120 x 8,192 126 / 155, 1,547 x 7,168 x
// 5,120 98 / 103, 1,547 x 2 x 16,384 x 5,120 gated 452 / 480, 8,192^3 848 / 890 (1.30 PFLOP/s).
#include "common.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));

#define GL_BN 256
#define GL_WB (GL_BN * 64)             // bytes of W a phase

// A buffer over everything from p on (the offsets are checked on the host).
__device__ __forceinline__ i32x4 gl_buffer(const void* p) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    i32x4 r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xffff));
    r[2] = -1;
    r[3] = 0x00020000;
    return r;
}

struct gl_args {
    const bf16* X; int ldx; const bf16* W; long w_group_stride; void* Y; int ldy, M, N, K;
    const int* offsets; int n_groups; const int* a_rows; const float* a_scale; const int* y_rows;
    int m_tiles, n_tiles, nb, act; float act_limit;
};

// One tile: rows row0 .. of the group whose rows end at row_end, W rows (columns of the result) from n0 on.
template <int NB, bool GLU, typename TY>
__device__ __forceinline__ void gl_tile(const gl_args& a, unsigned char* lds, const bf16* Wg, int row0, int row_end, int n0) {
    constexpr int BM = 32 * NB, XB = BM * 128;                   // bytes of a unit of X
    constexpr int XI = (BM + 63) / 64, WI = 2;                   // load instructions a wave: a unit of X, a phase of W
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4, wn = wave & 3, wm = wave >> 2;
    const int nu = a.K / 64, kt = a.K / 32, N = a.N;
    const i32x4 xbuf = gl_buffer(a.X), wbuf = gl_buffer(Wg);
    // X: instruction i brings eight rows (blocks past the tile's last: that one again); rows past the group its last row
    int xoff[XI], xblk[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        xblk[i] = i * 8 + wave < BM / 8 ? i * 8 + wave : BM / 8 - 1;
        const int row = xblk[i] * 8 + (lane >> 3);
        int s = row0 + row;
        s = s < row_end ? s : row_end - 1;
        xoff[i] = (a.a_rows ? a.a_rows[s] : s) * a.ldx * 2 + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    // W: a wave's four bands lie together in LDS: 64 columns, or 32 gate and the matching 32 up rows; bands past N the last one
    constexpr int TG = GLU ? 2 : 4;
    int wbase[WI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int t = wave * WI + i, x = t & 3;
        int band = n0 / 16 + (t >> 2) * TG + x % TG;
        band = band < N / 16 ? band : N / 16 - 1;
        if (GLU && x >= TG) band += N / 16;
        wbase[i] = band * kt * 1024;
    }
    const int wvoff = lane * 16;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    auto load_x = [&](int v, int xb) {
        const int k = (v < nu ? v : nu - 1) * 128;
#pragma unroll
        for (int i = 0; i < XI; ++i) sp_load_lds(xbuf, xoff[i], k, lds0 + xb * XB + xblk[i] * 1024);
    };
    auto load_w = [&](int t) {
        const int k = (t < kt ? t : kt - 1) * 1024;
#pragma unroll
        for (int i = 0; i < WI; ++i) sp_load_lds(wbuf, wvoff, wbase[i] + k, lds0 + 3 * XB + (t & 3) * GL_WB + (wave * WI + i) * 1024);
    };
    f32x4 acc[4][NB];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[x][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 wa[2][4], xa[2][NB];
    const int xrow = wm * 16 * NB + r, swz = (xrow >> 1) & 7;    // (rows 16 further on are exchanged alike)
    const int xl0 = xrow * 128 + ((q ^ swz) * 16), xl1 = xrow * 128 + (((4 + q) ^ swz) * 16);
    const int wl = 3 * XB + wn * 4096 + lane * 16;
#define GL_READ(set, xb, t, kk) do { \
        const unsigned char* wp_ = lds + wl + ((t) & 3) * GL_WB; \
        const unsigned char* xp_ = lds + ((kk) ? xl1 : xl0) + (xb) * XB; \
        _Pragma("unroll") for (int x = 0; x < 4; ++x) wa[set][x] = *(const bf16x8*)(wp_ + x * 1024); \
        _Pragma("unroll") for (int b = 0; b < NB; ++b) xa[set][b] = *(const bf16x8*)(xp_ + b * 2048); } while (0)
#define GL_MUL(set) do { \
        _Pragma("unroll") for (int b = 0; b < NB; ++b) \
        _Pragma("unroll") for (int x = 0; x < 4; ++x) \
            acc[x][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[set][x], xa[set][b], acc[x][b], 0, 0, 0); \
        _Pragma("unroll") for (int i = 0; i < 4 + NB; ++i) { \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); __builtin_amdgcn_sched_group_barrier(0x008, 2, 0); } } while (0)
    // the wave's loads in the order in which they were asked for: a phase needs all but the last XI + 2 WI of them (an odd
    // phase asks for a unit of X and then a phase of W, an even one for W)
#define GL_MEET(pending) do { \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(pending) : "memory"); \
        __builtin_amdgcn_s_barrier(); \
        __builtin_amdgcn_sched_barrier(0); } while (0)
    load_x(0, 0); load_w(0); load_x(1, 1); load_w(1); load_w(2); load_x(2, 2); load_w(3);
    GL_MEET(2 * XI + 3 * WI);
    GL_READ(0, 0, 0, 0);
    int xb = 0;                                                  // the unit's buffer
    for (int u = 0; u < nu; ++u) {
        const int xn = xb == 2 ? 0 : xb + 1, t = 2 * u;
        GL_MEET(XI + 2 * WI);                                    // phase 2u: reads the second half of the unit
        load_w(t + 4);
        __builtin_amdgcn_sched_barrier(0);
        GL_READ(1, xb, t + 1, 1);
        GL_MUL(0);
        __builtin_amdgcn_sched_barrier(0);
        GL_MEET(XI + 2 * WI);                                    // phase 2u + 1: reads the next unit, this one is free
        load_x(u + 3, xb);
        load_w(t + 5);
        __builtin_amdgcn_sched_barrier(0);
        GL_READ(0, xn, t + 2, 0);
        GL_MUL(1);
        __builtin_amdgcn_sched_barrier(0);
        xb = xn;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no load into LDS outlives the workgroup
#undef GL_READ
#undef GL_MUL
#undef GL_MEET

    // acc[x][b][i] of lane (r, q): column n0 + (wn * TG + x) * 16 + q * 4 + i, slot row0 + wm * 16 NB + b * 16 + r
    TY* Y = (TY*)a.Y;
    const bool vec_ok = (a.ldy & 3) == 0 && (((uintptr_t)Y) & 15) == 0;          // (N is a multiple of 16)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int s = row0 + wm * 16 * NB + b * 16 + r;
        if (s >= row_end) continue;
        const float sc = a.a_scale ? a.a_scale[s] : 1.0f;
        TY* yrow = Y + (a.y_rows ? (size_t)a.y_rows[s] : (size_t)s) * a.ldy;
#pragma unroll
        for (int x = 0; x < TG; ++x) {
            const int n = n0 + (wn * TG + x) * 16 + q * 4;
            if (n >= N) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[x][b][i] * sc;
                if constexpr (GLU) v[i] = sp_gated(v[i], acc[x + 2][b][i] * sc, a.act, a.act_limit, true);
                else if (a.act < 0) v[i] = sp_unary(v[i], -a.act, true);         // a plain product with an activation of its own
            }
            TY* dst = yrow + n;
            if (vec_ok) {
                if constexpr (sizeof(TY) == 2) {
                    bf16x4 o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (bf16)v[i];
                    *(bf16x4*)dst = o;
                } else {
                    *(f32x4*)dst = f32x4{v[0], v[1], v[2], v[3]};
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) dst[i] = from_f32<TY>(v[i]);
            }
        }
    }
}

// The tiles of a group of `rows` rows: as few as 256 rows each allow, all of the height, in units of 32 rows, that
// covers it then.
__device__ __forceinline__ int gl_group_tiles(int rows, int& nb) {
    const int tiles = (rows + 255) / 256, each = tiles ? (rows + tiles - 1) / tiles : 0;
    nb = each > 192 ? 8 : each > 160 ? 6 : each > 128 ? 5 : each > 96 ? 4 : 3;
    return tiles;
}

template <bool GLU, typename TY, bool GROUPED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_lds_kernel(gl_args a) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    constexpr int NCOLS = GLU ? GL_BN / 2 : GL_BN;
    // workgroups go to the eight XCDs in turn, each with an L2 of its own: XCD x takes the x-th eighth of the tiles
    const int units = a.m_tiles * a.n_tiles, per_xcd = (units + 7) / 8;
    const int unit = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if ((int)(blockIdx.x / 8) >= per_xcd || unit >= units) return;
    if constexpr (GROUPED) {
        // the row tile runs fastest: the tiles of one column of W of every group
        int mt = unit % a.m_tiles, g = 0, b = 0, e = 0, nb = 8;
        for (; g < a.n_groups; ++g) {                            // (uniform: scalar loads)
            b = a.offsets[g];
            e = a.offsets[g + 1];
            const int tiles = gl_group_tiles(e - b, nb);
            if (mt < tiles) break;
            mt -= tiles;
        }
        if (g == a.n_groups) return;
        const bf16* Wg = a.W + (size_t)g * a.w_group_stride;
        const int row0 = b + mt * 32 * nb, n0 = unit / a.m_tiles * NCOLS;
        if (nb == 8) gl_tile<8, GLU, TY>(a, lds, Wg, row0, e, n0);
        else if (nb == 6) gl_tile<6, GLU, TY>(a, lds, Wg, row0, e, n0);
        else if (nb == 5) gl_tile<5, GLU, TY>(a, lds, Wg, row0, e, n0);
        else if (nb == 4) gl_tile<4, GLU, TY>(a, lds, Wg, row0, e, n0);
        else gl_tile<3, GLU, TY>(a, lds, Wg, row0, e, n0);
    } else {
        // bands of eight row tiles, inside a band the row tile runs fastest: what an XCD works on at a time is about as
        // many row tiles as columns
        const int band_sz = 8 * a.n_tiles, band = unit / band_sz, in = unit % band_sz;
        const int bm = a.m_tiles - band * 8 < 8 ? a.m_tiles - band * 8 : 8;
        const int row0 = (band * 8 + in % bm) * 32 * a.nb, n0 = in / bm * NCOLS;
        if (a.nb == 8) gl_tile<8, GLU, TY>(a, lds, a.W, row0, a.M, n0);
        else if (a.nb == 6) gl_tile<6, GLU, TY>(a, lds, a.W, row0, a.M, n0);
        else if (a.nb == 5) gl_tile<5, GLU, TY>(a, lds, a.W, row0, a.M, n0);
        else gl_tile<4, GLU, TY>(a, lds, a.W, row0, a.M, n0);
    }
}

// Which NB suits a plain product, and what it takes then, in us: a round of tiles over the compute units takes (4.3 + 1.95 NB)
// ns a k (measured at NB = 4, 5, 6, 8 and K = 5,120: 62, 71, 81 and 102 us), and every round but the first 10 us for its
// tiles' start and end, which short sums over k do not hide (448 k, 18 rounds: 401 us).
static double lds_time(int M, int N, int K, bool glu, int* nb_out) {
    const long cus = sp_cu_count(), cols = (N + (glu ? 127 : 255)) / (glu ? 128 : 256);
    double least = -1.0, further = 0.0;
    for (int nb : {8, 6, 5, 4}) {
        const long tiles = (M + 32 * nb - 1) / (32 * nb) * cols, rounds = (tiles + cus - 1) / cus;
        const double t = (double)rounds * K * (4.3e-3 + 1.95e-3 * nb);
        if (least < 0.0 || t < least) { *nb_out = nb; least = t; further = 10.4 * (double)(rounds - 1); }
    }
    return least + further;
}
extern "C" double spite_gemm_lds_time(int M, int N, int K, int glu) { int nb; return lds_time(M, N, K, glu != 0, &nb); }

// Arguments as spite_gemm_tiled's; `nb`: the plain product's tile height in units of 32 rows (4, 5, 6 or 8), 0 the library's choice;
// `x_rows`: how many rows X has, which a row list's entries stay below (0 without one: M).
extern "C" int spite_gemm_lds(const void* X, int ldx, const void* W, long w_group_stride, void* Y, int y_dtype, int ldy, int M,
                              int N, int K, const int* offsets, int n_groups, const int* a_rows, const float* a_scale,
                              const int* y_rows, int glu, float act_limit, int nb, int x_rows, hipStream_t st) {
    SP_REQUIRE(M >= 0 && N > 0 && K > 0 && ldx >= K && ldy >= N, "gemm_lds: bad sizes M=%d N=%d K=%d", M, N, K);
    SP_REQUIRE(K % 64 == 0 && N % 16 == 0, "gemm_lds: operand order needs K=%d a multiple of 64 and N=%d of 16", K, N);
    SP_REQUIRE(ldx % 8 == 0, "gemm_lds: the row stride %d must be a multiple of 8", ldx);
    SP_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_lds: operands must be 16-byte aligned");
    SP_REQUIRE(y_dtype == SP_BF16 || y_dtype == SP_F32, "gemm_lds: output dtype %d", y_dtype);
    SP_REQUIRE(!offsets || n_groups > 0, "gemm_lds: grouped call without groups");
    SP_REQUIRE(nb == 0 || nb == 4 || nb == 5 || nb == 6 || nb == 8, "gemm_lds: tile of %d rows", 32 * nb);
    const int unary = glu >> 4;
    glu &= 15;
    SP_REQUIRE(!(glu && unary) && unary <= SP_UNARY_TANH, "gemm_lds: activation code %d", glu | (unary << 4));
    SP_REQUIRE(glu <= SP_ACT_LAST && (glu != SP_ACT_CLAMPED || act_limit > 0.f), "gemm_lds: activation code %d with bound %g", glu, act_limit);
    SP_REQUIRE(!a_rows || x_rows > 0, "gemm_lds: a row list over %d rows of X", x_rows);
    // the loads' offsets are 32-bit: rows of X and a group's W
    SP_REQUIRE((size_t)(a_rows ? x_rows : M) * ldx * 2 < ((size_t)1 << 31) && (size_t)(glu ? 2 : 1) * N * K * 2 < ((size_t)1 << 31),
               "gemm_lds: operands of 2 GiB and more (M=%d, %d rows of X, N=%d K=%d)", M, x_rows, N, K);
    if (M == 0) return 0;
    gl_args a{(const bf16*)X, ldx, (const bf16*)W, w_group_stride, Y, ldy, M, N, K, offsets, n_groups, a_rows, a_scale, y_rows,
              0, 0, 0, glu ? glu : -unary, act_limit};
    a.nb = offsets ? 8 : nb;
    if (!a.nb) lds_time(M, N, K, glu != 0, &a.nb);
    a.n_tiles = (N + (glu ? 127 : 255)) / (glu ? 128 : 256);
    // a group of r rows has ceil(r / 256) tiles: at most r / 256 + 1
    a.m_tiles = offsets ? M / 256 + (n_groups < M ? n_groups : M) : (M + 32 * a.nb - 1) / (32 * a.nb);
    SP_REQUIRE((long)a.m_tiles * a.n_tiles < (1L << 30), "gemm_lds: too many tiles");
    const int grid = (a.m_tiles * a.n_tiles + 7) / 8 * 8;
    const size_t sh = (size_t)3 * 32 * a.nb * 128 + 4 * GL_WB;
#define SP_GL(GLUV, TY, GROUPEDV) do { \
        auto kern = gemm_lds_kernel<GLUV, TY, GROUPEDV>; \
        static bool allowed = false; \
        if (!allowed) { hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
            if (e != hipSuccess) return sp_fail("gemm_lds: 160 KB of LDS refused: %s", hipGetErrorString(e)); allowed = true; } \
        kern<<<grid, 512, sh, st>>>(a); } while (0)
#define SP_GL2(GROUPEDV) do { \
        if (glu) { if (y_dtype == SP_BF16) SP_GL(true, bf16, GROUPEDV); else SP_GL(true, float, GROUPEDV); } \
        else { if (y_dtype == SP_BF16) SP_GL(false, bf16, GROUPEDV); else SP_GL(false, float, GROUPEDV); } } while (0)
    if (offsets) SP_GL2(true); else SP_GL2(false);
#undef SP_GL2
#undef SP_GL
    SP_LAUNCH_CHECK("gemm_lds");
    return 0;
}
