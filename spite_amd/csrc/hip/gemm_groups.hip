// Products over groups of rows (experts) for many rows: Y[M,N] = X[M,K] . W[g][N,K]^T, bf16 in, fp32 accumulation on MFMA
// 16x16x32, W in MFMA operand order (see gemm_tiled.hip), plain or gated with silu.
//
// A step's groups differ: a router gives each expert a few rows or a few hundred, a shared expert takes every one.  A tile
// of one height for all multiplies padding for the small groups and reads W again for the large ones; here every group
// takes as few tiles as `cap` rows (128 or 160) allow, all of the height, in units of 16 rows, that then covers it.
//
// A workgroup of NW waves (eight or four) owns 16 * A * NW rows of W (GLU: half of them gate rows, the others the matching up rows) and
// one tile of 16 * NB rows of X; a wave owns A bands of 16 rows of W and every row of X: A x NB accumulator tiles.  A is four, or five for
// plain products whose tiles of 320 columns fit the chip where those of 256 and 512 do not (one wave a SIMD, its accumulators in AGPRs).
//  * W never touches LDS: S rotating sets of operand registers (six up to 96 rows, four above), each asked for again as soon as
//    its products are issued, S - 1 half steps of 32 k ahead.  A group of one tile reads its W once: non-temporal loads.
//  * X goes straight to LDS (buffer loads with the lds bit), four buffers of 64 k, asked for three steps ahead: no register
//    waits for it, and waiting for it (loads are counted in order) waits for no younger W.  The 16-byte pieces of a row are
//    exchanged by XOR with half its number, so that an operand read spreads over all banks.  One barrier per 64 k.
//  * Rows past the group and steps past K (K is cut into rounds of S / 2 steps of 64) are loads beyond the buffer's end, which
//    give zeros: no branch in the loop, and products of zeros cost the matrix units less power, which is what bounds the
//    clock here.
//  * Workgroups go to the eight XCDs in turn, an eighth of the tiles each, in an order by which those that run at a time share what they
//    read (gemm_groups_kernel).
// The sum over k runs in the order of gemm_tiled and gemm_lds: the same bits.
//
// Measured on an MI355X against gemm_tiled's best tile (us; 16 experts of which a token takes `top`, beside them one or two
// groups of every token): 2,048 tokens x 2 x 8,192 x 5,120 gated 640 / 718, 1,547 579 / 630, 330 444 / 481; 1,786, top 2,
// 2 x 4,096 x 5,120 550 / 590; 1,531, top 4, 2 x 1,024 x 2,048 79 / 108; 1,200 x 2,048 x 3,072 59 / 74; but 1,512 x 3,072 x 2,048, which
// stays with gemm_tiled, 67 / 60.  At 2,048 tokens what bounds it is the power limit (the clock falls to 1.6 GHz with the matrix units
// half busy), at 330 the stream of W (6.4 TB/s).
#include <math.h>
#include "common.h"

struct gg_args {
    const bf16* X; int ldx; const bf16* W; long w_group_stride; void* Y; int ldy, M, N, K;
    const int* offsets; int n_groups; const int* a_rows; const float* a_scale; const int* y_rows;
    int m_tiles, n_tiles, cap;
    int per_xcd; int* others;              // tiles an XCD may have, and where the groups go that have more (see gemm_groups_kernel)
};
#define GG_PAST ((int)0x80000000)      // an offset beyond every buffer's end: loads give zeros

// A buffer of 2 GiB from p on (the operands' offsets are checked on the host), p the same in every lane.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gg_buffer(const void* p) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    const uint64_t u = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
    return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)u, 0, 0x7fffffff, 0x00020000);
}

// One tile: rows row0 .. of the group g whose rows end at row_end, columns of the result from n0 on.
template <int NW, int A, int NB, int S, bool GLU, typename TY, bool NTW>
__device__ __forceinline__ void gg_tile(const gg_args& p, unsigned char* lds, int g, int row0, int row_end, int n0, int u_first, int nu, TY* Y) {
    constexpr int XB = 16 * NB * 128;                            // bytes of a step of X
    constexpr int XI = (2 * NB + NW - 1) / NW;                   // load instructions a wave: a step of X (eight rows each)
    constexpr int TG = GLU ? A / 2 : A;                          // bands that name distinct columns
    static_assert(S % 2 == 0, "whole steps a round");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4, N = p.N, kt = 2 * nu;
    const __amdgpu_buffer_rsrc_t xbuf = gg_buffer(p.X), wbuf = gg_buffer(p.W + (size_t)g * p.w_group_stride);
    int xoff[XI], xblk[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        xblk[i] = i * NW + wave < 2 * NB ? i * NW + wave : 2 * NB - 1;       // blocks past the tile's last: that one again
        const int row = xblk[i] * 8 + (lane >> 3), s = row0 + row;
        const int at = s < row_end ? s : row_end - 1;
        xoff[i] = (p.a_rows ? p.a_rows[at] : at) * p.ldx * 2 + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
        if (s >= row_end) xoff[i] = GG_PAST;
    }
    int wband[A];
#pragma unroll
    for (int a = 0; a < A; ++a) {
        int band = n0 / 16 + wave * TG + a % TG;
        band = band < N / 16 ? band : N / 16 - 1;                // bands past N read the last one again
        if (GLU && a >= TG) band += N / 16;
        wband[a] = (band * (p.K / 32) + 2 * u_first) * 1024;
    }
    const int wlane = lane * 16;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    auto load_x = [&](int u) {
        const int k0 = (u_first + (u < nu ? u : 0)) * 128, past = u < nu ? 0 : GG_PAST;
#pragma unroll
        for (int i = 0; i < XI; ++i) sp_load_lds(xbuf, xoff[i] | past, __builtin_amdgcn_readfirstlane(k0), lds0 + (u & 3) * XB + xblk[i] * 1024);
    };
    auto load_w = [&](bf16x8 (&ws)[A], int t) {
        const int at = (t < kt ? t : 0) * 1024, past = t < kt ? 0 : GG_PAST;
#pragma unroll
        for (int a = 0; a < A; ++a)          // (2: non-temporal)
            ws[a] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wlane | past, wband[a] + at, NTW ? 2 : 0));
    };
    f32x4 acc[A][NB];          // [W band a][slot tile b]
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int swz = (r >> 1) & 7, xl0 = r * 128 + ((q ^ swz) * 16), xl1 = r * 128 + (((4 + q) ^ swz) * 16);
    auto mul = [&](bf16x8 (&ws)[A], int buf, int kk) {
        const unsigned char* xs = lds + buf * XB + (kk ? xl1 : xl0);
        constexpr int NX = NB == 9 ? 3 : 4;                      // slot tiles read from LDS at a time
#pragma unroll
        for (int b0 = 0; b0 < NB; b0 += NX) {
            bf16x8 xf[NX];
#pragma unroll
            for (int b = 0; b < NX; ++b)
                if (b0 + b < NB) xf[b] = *(const bf16x8*)(xs + (b0 + b) * 2048);
#pragma unroll
            for (int a = 0; a < A; ++a)
#pragma unroll
                for (int b = 0; b < NX; ++b)
                    if (b0 + b < NB)
                        acc[a][b0 + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[a], xf[b], acc[a][b0 + b], 0, 0, 0);
        }
    };
    // Step u: half steps 2u and 2u + 1 with the X of buffer u % 4, while X of step u + 3 goes to the buffer that step u - 1 has
    // left (every wave has passed the barrier behind it).  Before the barrier each wave waits until its own loads of X for
    // step u + 1 are there: younger than those are two steps of X and the W asked for since, three steps of eight loads or,
    // with fewer sets, at least the sets of the start and one step.
    constexpr int PENDING = 2 * XI + (2 + S < 6 ? 2 + S : 6) * A;
    static_assert(PENDING < 64, "a wait for more loads than the counter holds");
#define GG_MEET(pending) do { \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(pending) : "memory"); \
        __builtin_amdgcn_s_barrier(); \
        __builtin_amdgcn_sched_barrier(0); } while (0)
    bf16x8 w[S][A];
    load_x(0);
    load_x(1);
    load_x(2);
#pragma unroll
    for (int s = 0; s < S; ++s) load_w(w[s], s);
    GG_MEET(2 * XI + A * S);
    auto step = [&](bf16x8 (&wa)[A], bf16x8 (&wb)[A], int u) {
        load_x(u + 3);
        __builtin_amdgcn_sched_barrier(0);
        mul(wa, u & 3, 0);
        load_w(wa, 2 * u + S);
        __builtin_amdgcn_sched_barrier(0);
        mul(wb, u & 3, 1);
        load_w(wb, 2 * u + S + 1);
        __builtin_amdgcn_sched_barrier(0);
        GG_MEET(PENDING);
    };
    for (int u = 0; u < nu; u += S / 2) {
#pragma unroll
        for (int j = 0; j < S / 2; ++j) step(w[2 * j], w[2 * j + 1], u + j);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no load into LDS outlives the workgroup
#undef GG_MEET

    // acc[a][b][i] of lane (r, q): column n0 + (wave * TG + a) * 16 + q * 4 + i, slot row0 + b * 16 + r; four columns a store
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int s = row0 + b * 16 + r;
        if (s >= row_end) continue;
        const float sc = p.a_scale ? p.a_scale[s] : 1.0f;
        TY* yrow = Y + (p.y_rows ? (size_t)p.y_rows[s] : (size_t)s) * p.ldy;
#pragma unroll
        for (int a = 0; a < TG; ++a) {
            const int n = n0 + (wave * TG + a) * 16 + q * 4;
            if (n >= N) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[a][b][i] * sc;
                if constexpr (GLU) v[i] = sp_gated(v[i], acc[a + TG][b][i] * sc, SP_ACT_SILU, 0.f, true);
            }
            if constexpr (sizeof(TY) == 2) {
                bf16x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (bf16)v[i];
                *(bf16x4*)(yrow + n) = o;
            } else {
                *(f32x4*)(yrow + n) = f32x4{v[0], v[1], v[2], v[3]};
            }
        }
    }
}

// The tiles of a group of `rows` rows, and their height in units of 16 rows (2, 4 and every one from 5 to 10).
__device__ __host__ __forceinline__ int gg_group_tiles(int rows, int cap, int& nb) {
    const int tiles = (rows + cap - 1) / cap, each = tiles ? (rows + tiles - 1) / tiles : 0;
    nb = (each + 15) / 16;
    nb = nb <= 2 ? 2 : nb <= 4 ? 4 : nb;
    return tiles;
}

// Groups from which on four waves' tiles of 64 columns go to the XCDs by group too.
#define GG_BY_GROUP 64

template <int NW, int A, bool GLU, typename TY>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(A == 4 ? 2 : 1, A == 4 ? 2 : 1)))
void gemm_groups_kernel(gg_args p) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    // The groups' tiles, 64 groups at a time: a prefix sum over the lanes (one after another the loads of the offsets cost half a
    // microsecond a group); what it finds is kept in scalar registers.  The launch is as large as the rows allow, up to a tile a group more than there are.
    // Those that there are are dealt evenly to the XCDs and go to their first workgroups: with empty ones among them an XCD got
    // more than its eighth, and two tiles met on one compute unit while others had none (126 rows of 4 of 4 experts and of one more x 2 x
    // 5,120 x 16,384 gated, 200 tiles of four waves, 506 -> 292 us; 1,483 of 8 of 32 x 768 x 16,384, eight waves, 846 -> 483; over 559 sizes 0.96).
    const int lane = threadIdx.x & 63;
    int b = 0, e = 0, h = 0, nt = 0;                     // the lane's group: its rows, their tiles and these tiles' height
    int g = -1, row0 = 0, row_end = 0, nb = 8, tiles = 1, col = 0;
    if (A == 4 && (NW == 8 || p.n_groups < GG_BY_GROUP)) {     // row tiles of all groups run fastest
        int incl = 0, all = 0;
        auto scan = [&](int c) {
            b = e = 0;
            if (c + lane < p.n_groups) { b = p.offsets[c + lane]; e = p.offsets[c + lane + 1]; }
            nt = incl = gg_group_tiles(e - b, p.cap, h);
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(incl, o, 64); if (lane >= o) incl += v; }
            return __builtin_amdgcn_readlane(incl, 63);
        };
        for (int c = 0; c < p.n_groups; c += 64) all += scan(c);
        const int units = all * p.n_tiles, per_xcd = (units + 7) / 8;
        const int unit = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
        if ((int)(blockIdx.x / 8) >= per_xcd || unit >= units) return;
        const int mt = __builtin_amdgcn_readfirstlane(unit % all);
        int base = 0;
        for (int c = 0; c < p.n_groups; c += 64) {
            const int total = p.n_groups <= 64 ? all : scan(c);
            if (mt < base + total) {
                const bool mine = mt >= base + incl - nt && mt < base + incl;
                const int src = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)__ballot(mine)) - 1);
                g = c + src;
                nb = __builtin_amdgcn_readlane(h, src);
                tiles = __builtin_amdgcn_readlane(nt, src);
                row_end = __builtin_amdgcn_readlane(e, src);
                row0 = __builtin_amdgcn_readlane(b, src) + (mt - base - __builtin_amdgcn_readlane(incl - nt, src)) * 16 * nb;
                break;
            }
            base += total;
        }
        col = __builtin_amdgcn_readfirstlane(unit / all);
    } else {
        // (80 columns a wave, or four waves and 64 groups and more.  With eight waves a gated product beside a shared expert lost 3 to 5 %.  With
        // four and fewer groups, products in a row are 2 to 3 % faster by it, but within a step, where the rows of X come from the product before or
        // by a row list, they are not: 1,531 rows of 4 of 16 experts and of two more x 2 x 1,024 x 2,048 gated 91.2 us, by this order 94.8, x 2,048 x
        // 1,024 66.3 / 65.8, latent attention's over its heads 49.7 / 50.9; and where the fullest of a few groups has 1.6 times the average an XCD
        // waits for another: 903 rows of 8 experts x 2 x 3,072 x 1,024 32 / 38.  Over 64 and more the XCDs' shares even out: nine products, rows spread
        // by chance and by lognormal loads of 0.2 to 0.8, 4 % faster on average, none slower; serving 128 experts, a step 44.4 ms / 43.6.)
        //  * groups of up to four tiles and no more than twice the average (experts): all columns of a group go to one XCD, row tiles of a column
        //    next to each other, so that what runs there at a time reads the group's rows of X once from memory and its W once;
        //  * larger ones (a shared expert): row tiles of all of them running fastest, an eighth of the columns an XCD.
        // An XCD has an eighth of either kind, in turn: the first wait for the stream of W, the second for the matrix units.  (One tile a
        // compute unit, 2,048 rows of 16 experts x 5,120 x 8,192, 242 -> 223 us, with 1.38 GB read instead of 1.61; 36 products of 8 to 128 experts
        // 5 % faster on average.)
        int few = 0, many = 0, limit = 0;      // tiles of either kind up to and with the lane's group; the first kind's most
        auto look = [&](int c) {
            b = e = 0;
            if (c + lane < p.n_groups) { b = p.offsets[c + lane]; e = p.offsets[c + lane + 1]; }
            nt = gg_group_tiles(e - b, p.cap, h);
        };
        auto scan = [&](int c) {
            if (c > 0 || p.n_groups > 64) look(c);
            few = sp_wave_scan(nt <= limit ? nt : 0);
            many = sp_wave_scan(nt <= limit ? 0 : nt);
        };
        int all = 0, live = 0;
        for (int c = 0; c < p.n_groups; c += 64) {
            look(c);
            all += __builtin_amdgcn_readlane(sp_wave_scan(nt), 63);
            live += __popcll(__ballot(nt > 0));
        }
        limit = all ? min(4, 2 * all / live) : 0;
        int all_few = 0, all_many = 0;
        for (int c = 0; c < p.n_groups; c += 64) {
            scan(c);
            all_few += __builtin_amdgcn_readlane(few, 63);
            all_many += __builtin_amdgcn_readlane(many, 63);
        }
        const int xcd = blockIdx.x % 8, at = blockIdx.x / 8;     // the XCD's workgroups in turn
        const int units_few = all_few * p.n_tiles, units_many = all_many * p.n_tiles, per_few = (units_few + 7) / 8, per_many = (units_many + 7) / 8;
        const int n_few = min(max(units_few - xcd * per_few, 0), per_few), n_all = n_few + min(max(units_many - xcd * per_many, 0), per_many);
        if (p.others) {
            // The host knows the groups' sizes on average alone, and a tile more than fits the rounds that it reckoned with costs a round (a tile
            // of 320 columns has a compute unit to itself).  So the tiles that there are decide: where they do not fit, this launch does
            // nothing and leaves the groups to the product behind it, which walks `others`, empty groups otherwise.
            const bool fits = per_few + per_many <= p.per_xcd;
            if (blockIdx.x == 0)
                for (int i = threadIdx.x; i <= p.n_groups; i += NW * 64) p.others[i] = fits ? 0 : p.offsets[i];
            if (!fits) return;
        }
        if (at >= n_all) return;
        const int before = __builtin_amdgcn_readfirstlane((int)((long)at * n_few / n_all));
        const bool is_few = __builtin_amdgcn_readfirstlane((int)((long)(at + 1) * n_few / n_all)) > before;
        const int unit = is_few ? xcd * per_few + before : xcd * per_many + at - before;
        const int mt = is_few ? 0 : __builtin_amdgcn_readfirstlane(unit % all_many);
        int base = 0;
        for (int c = 0; c < p.n_groups; c += 64) {
            if (p.n_groups > 64) scan(c);
            const int first = base + (is_few ? few - (nt <= limit ? nt : 0) : many - (nt <= limit ? 0 : nt));      // tiles of its kind before the lane's group
            const bool mine = (nt <= limit) == is_few && (is_few ? unit >= first * p.n_tiles && unit < (first + nt) * p.n_tiles : mt >= first && mt < first + nt);
            const unsigned long long who = __ballot(mine);
            if (who) {
                const int src = __builtin_amdgcn_readfirstlane(__ffsll(who) - 1);
                const int first_tile = __builtin_amdgcn_readlane(first, src);
                g = c + src;
                nb = __builtin_amdgcn_readlane(h, src);
                tiles = __builtin_amdgcn_readlane(nt, src);
                row_end = __builtin_amdgcn_readlane(e, src);
                const int j = unit - first_tile * p.n_tiles;
                col = __builtin_amdgcn_readfirstlane(is_few ? j / tiles : unit / all_many);
                row0 = __builtin_amdgcn_readlane(b, src) + (is_few ? __builtin_amdgcn_readfirstlane(j % tiles) : mt - first_tile) * 16 * nb;
                break;
            }
            base += __builtin_amdgcn_readlane(is_few ? few : many, 63);
        }
    }
    if (g < 0) return;
    const int n0 = col * (GLU ? 8 : 16) * A * NW;
#define GG_TILE(NB, S, NT) gg_tile<NW, A, NB, S, GLU, TY, NT>(p, lds, g, row0, row_end, n0, 0, p.K / 64, (TY*)p.Y)
#define GG_TILES(NT) switch (nb) { \
        case 2: GG_TILE(2, 6, NT); break; \
        case 4: GG_TILE(4, 6, NT); break; \
        case 5: GG_TILE(5, 6, NT); break; \
        case 6: GG_TILE(6, 6, NT); break; \
        case 7: GG_TILE(7, A == 5 ? 6 : 4, NT); break; \
        case 8: GG_TILE(8, A == 5 ? 6 : 4, NT); break; \
        case 9: GG_TILE(9, A == 5 ? 6 : 4, NT); break; \
        default: GG_TILE(10, A == 5 ? 6 : 4, NT); }
    if (tiles == 1) GG_TILES(true) else GG_TILES(false)
#undef GG_TILES
#undef GG_TILE
}

template <int NW, int A, bool GLU, typename TY>
static int gg_launch(gg_args p, hipStream_t st) {
    const int cols = (GLU ? 8 : 16) * A * NW;
    p.n_tiles = (p.N + cols - 1) / cols;
    // row tiles: a group of r rows has ceil(r / cap): at most r / cap + 1
    p.m_tiles = p.M / p.cap + (p.n_groups < p.M ? p.n_groups : p.M);
    SP_REQUIRE((long)p.m_tiles * p.n_tiles < (1L << 30), "gemm_groups: too many tiles");
    int grid = ((p.m_tiles * p.n_tiles + 7) / 8 + 1) * 8;      // (an eighth of either kind, rounded up)
    if (p.others && grid > 8 * p.per_xcd) grid = 8 * p.per_xcd;
    static bool allowed = false;
    if (!allowed) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_groups_kernel<NW, A, GLU, TY>, hipFuncAttributeMaxDynamicSharedMemorySize, 4 * 160 * 128);
        SP_REQUIRE(e == hipSuccess, "gemm_groups: 80 KB of LDS refused: %s", hipGetErrorString(e));
        allowed = true;
    }
    gemm_groups_kernel<NW, A, GLU, TY><<<grid, NW * 64, (size_t)4 * p.cap * 128, st>>>(p);
    SP_LAUNCH_CHECK("gemm_groups");
    return 0;
}

// Plain products of some tens to some hundreds of rows, by the same tiles: four waves and 256 rows of W a workgroup, tiles of
// 16 * NB rows, the sum over k cut into `runs` runs, each a workgroup of its own that writes its partial sums to Y + run * M * N
// (one run: the result).  The chip takes one workgroup a compute unit at a time: what bounds these sizes is the stream of W
// and, since a workgroup's waits are filled by no other, the number of its steps; so as many runs as make up to one
// workgroup a unit, and no more (rounds of them cost twice: 330 x 7,168 x 5,120 in 3 runs of 7 x 16 rows 39 us, in 6 54).
//
// Measured on an MI355X against the best of gemm_tiled (its runs of 128 x 512), gemm_lds and, up to 64 rows, gemm_skinny, launches in
// a row over weights that the caches do not hold, with the sum of the runs (us): 64 x 32,768 x 5,120 62 / 119, 64 x 5,120 x 8,192
// 26 / 34, 80 x 7,168 x 5,120 26 / 34, 330 39 / 55, 500 x 5,120 x 5,120 39 / 55, 500 x 2,048 x 2,048 23 / 30, 1,531 x 576 x 5,120 27 / 37.
// (W's loads are non-temporal however many row tiles read it; cached ones were not timed there.)
template <int NB, int S, typename TY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_runs_kernel(gg_args p, int runs) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int units = p.m_tiles * p.n_tiles * runs, per_xcd = (units + 7) / 8;
    const int unit = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if ((int)(blockIdx.x / 8) >= per_xcd || unit >= units) return;
    const int tile = unit / p.m_tiles, ks = tile % runs, all = p.K / 64;
    // (quotients: in scalar registers again)
    const int mt = __builtin_amdgcn_readfirstlane(unit % p.m_tiles), n0 = __builtin_amdgcn_readfirstlane(tile / runs) * 256;
    const int each = __builtin_amdgcn_readfirstlane((all + runs - 1) / runs), first = __builtin_amdgcn_readfirstlane(ks) * each;
    gg_tile<4, 4, NB, S, false, TY, true>(p, lds, 0, mt * 16 * NB, p.M, n0, first, all - first < each ? all - first : each,
                                       (TY*)p.Y + (size_t)ks * p.M * p.N);
}

template <int NB, int S, typename TY>
static int gr_launch(gg_args p, int runs, hipStream_t st) {
    constexpr int SH = 4 * NB * 16 * 128;
    p.n_tiles = (p.N + 255) / 256;
    p.m_tiles = (p.M + 16 * NB - 1) / (16 * NB);
    static bool allowed = false;
    if (!allowed) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_runs_kernel<NB, S, TY>, hipFuncAttributeMaxDynamicSharedMemorySize, SH);
        SP_REQUIRE(e == hipSuccess, "gemm_runs: %d bytes of LDS refused: %s", SH, hipGetErrorString(e));
        allowed = true;
    }
    SP_REQUIRE((long)p.m_tiles * p.n_tiles * runs < (1L << 30), "gemm_runs: too many tiles");
    gemm_runs_kernel<NB, S, TY><<<(p.m_tiles * p.n_tiles * runs + 7) / 8 * 8, 256, SH, st>>>(p, runs);
    SP_LAUNCH_CHECK("gemm_runs");
    return 0;
}
template <typename TY>
static int gr_launch_nb(const gg_args& p, int runs, int nb, hipStream_t st) {
    switch (nb) {
        case 2: return gr_launch<2, 6, TY>(p, runs, st);
        case 4: return gr_launch<4, 6, TY>(p, runs, st);
        case 5: return gr_launch<5, 6, TY>(p, runs, st);
        case 6: return gr_launch<6, 6, TY>(p, runs, st);
        case 7: return gr_launch<7, 4, TY>(p, runs, st);
        case 8: return gr_launch<8, 4, TY>(p, runs, st);
        case 9: return gr_launch<9, 4, TY>(p, runs, st);
        case 10: return gr_launch<10, 4, TY>(p, runs, st);
        default: return sp_fail("gemm_runs: tiles of %d rows", 16 * nb);
    }
}

int sp_add_runs(const float* part, int runs, void* Y, int y_dtype, int ldy, int M, int N, hipStream_t st);       // gemm_tiled.hip

// Y[M,N] = X[M,K] . W[N,K]^T, W in operand order.  `nb`: a tile's rows in units of 16 (2, 4 .. 10); `part`: [runs][M][N] floats where there
// is more than one run (aligned to 16 bytes, as rows of Y are where there is one).
extern "C" int spite_gemm_runs(const void* X, int ldx, const void* W, void* Y, int y_dtype, int ldy, int M, int N, int K, int runs, int nb,
                               float* part, hipStream_t st) {
    SP_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && ldy >= N, "gemm_runs: bad sizes M=%d N=%d K=%d", M, N, K);
    SP_REQUIRE(K % 64 == 0 && N % 16 == 0, "gemm_runs: operand order needs K=%d a multiple of 64 and N=%d of 16", K, N);
    SP_REQUIRE(ldx % 8 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_runs: operands must be 16-byte aligned");
    SP_REQUIRE(y_dtype == SP_BF16 || y_dtype == SP_F32, "gemm_runs: output dtype %d", y_dtype);
    const int all = K / 64;
    SP_REQUIRE(runs >= 1 && runs <= 64 && (all + runs - 1) / runs * (runs - 1) < all, "gemm_runs: %d runs over %d steps leave a run empty", runs, all);
    SP_REQUIRE(runs == 1 ? ldy % 4 == 0 && ((uintptr_t)Y & 15) == 0 : part && ((uintptr_t)part & 15) == 0, "gemm_runs: rows of the result must be 16-byte aligned");
    // the loads' offsets are 32-bit
    SP_REQUIRE((size_t)M * ldx * 2 < ((size_t)1 << 31) && (size_t)N * K * 2 < ((size_t)1 << 31), "gemm_runs: operands of 2 GiB and more (M=%d N=%d K=%d)", M, N, K);
    gg_args p{(const bf16*)X, ldx, (const bf16*)W, 0, Y, ldy, M, N, K, nullptr, 1, nullptr, nullptr, nullptr, 0, 0, 0, 0, nullptr};
    if (runs == 1) return y_dtype == SP_BF16 ? gr_launch_nb<bf16>(p, 1, nb, st) : gr_launch_nb<float>(p, 1, nb, st);
    p.Y = part;
    p.ldy = N;
    const int rc = gr_launch_nb<float>(p, runs, nb, st);
    return rc ? rc : sp_add_runs(part, runs, Y, y_dtype, ldy, M, N, st);
}

// The runs and tile (runs * 16 + nb) that suit a plain product, and what it takes then, in us; 0 if the tiles alone are more than one a
// compute unit.  A step of 64 k takes 0.457 + 0.038 nb us, or what the stream of W needs for 32 KB a workgroup (8.3 TB/s: row
// tiles share it); more than one run a launch, and the passes over the partial sums at 6.8 TB/s.  Fitted to 296 sizes (20 to 3,000
// rows, N and K of 128 to 20,000), each with several choices; the choice is within 1 % of the best of them on average.
extern "C" int spite_gemm_runs_choice(int M, int N, int K, double* us) {
    const long cus = sp_cu_count(), cols = (N + 255) / 256;
    const int steps = K / 64;
    int best = 0;
    *us = 0.0;
    for (int rt = (M + 159) / 160; rt <= (M + 63) / 64 && rt * cols <= cus; ++rt) {
        int nb = ((M + rt - 1) / rt + 15) / 16;
        nb = nb <= 2 ? 2 : nb <= 4 ? 4 : nb;
        if ((M + 16 * nb - 1) / (16 * nb) != rt) continue;
        long most = cus / (rt * cols) < 16 ? cus / (rt * cols) : 16;
        if (most > steps / 2) most = steps / 2;
        while (most > 1 && (steps + most - 1) / most * (most - 1) >= steps) --most;      // no run may be empty
        for (long runs : {most, 1L}) {
            if (runs < 1) continue;
            const double step = fmax(0.457 + 0.038 * nb, 0.0328 * (double)(cols * runs) / 8.27);
            const double t = 9.2 + (double)((steps + runs - 1) / runs) * step
                           + (runs > 1 ? 1.7 + (2.0 * runs + 1.0) * M * N * 4e-6 / 6.76 : 0.0);
            if (best == 0 || t < *us) { best = (int)runs * 16 + nb; *us = t; }
        }
    }
    return best;
}

// Arguments as spite_gemm_lds's (`x_rows`: how many rows X has); `waves` 4 or 8, or 5 for four waves of 80 columns (plain only), `cap` 128 or 160.  Gated with silu
// (`glu` SP_ACT_SILU) or plain (0); rows of Y that 16-byte stores can take.  `others` (with waves 5; n_groups + 1 offsets, or none): only where
// the groups' tiles fit `rounds` of a tile a compute unit, others then all 0; else nothing is computed and others is a copy of offsets.
extern "C" int spite_gemm_groups(const void* X, int ldx, const void* W, long w_group_stride, void* Y, int y_dtype, int ldy, int M,
                                 int N, int K, const int* offsets, int n_groups, const int* a_rows, const float* a_scale,
                                 const int* y_rows, int glu, int waves, int cap, int x_rows, int rounds, int* others, hipStream_t st) {
    SP_REQUIRE(M >= 0 && N > 0 && K > 0 && ldx >= K && ldy >= N, "gemm_groups: bad sizes M=%d N=%d K=%d", M, N, K);
    SP_REQUIRE(offsets && n_groups > 0, "gemm_groups: no groups");
    SP_REQUIRE(K % 64 == 0 && N % 16 == 0, "gemm_groups: operand order needs K=%d a multiple of 64 and N=%d of 16", K, N);
    SP_REQUIRE(ldx % 8 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0, "gemm_groups: operands must be 16-byte aligned");
    SP_REQUIRE(ldy % 4 == 0 && ((uintptr_t)Y & 15) == 0, "gemm_groups: rows of Y must be 16-byte aligned");
    SP_REQUIRE(y_dtype == SP_BF16 || y_dtype == SP_F32, "gemm_groups: output dtype %d", y_dtype);
    SP_REQUIRE(glu == 0 || glu == SP_ACT_SILU, "gemm_groups: activation code %d", glu);
    SP_REQUIRE(((waves == 4 || waves == 8) && (cap == 128 || cap == 160)) || (waves == 5 && !glu && (cap == 128 || cap == 160)), "gemm_groups: %d waves, tiles of %d rows", waves, cap);
    SP_REQUIRE(x_rows > 0 && (a_rows || x_rows >= M), "gemm_groups: %d rows of X", x_rows);
    SP_REQUIRE(!others || (waves == 5 && rounds > 0 && rounds < (1 << 16) && others != offsets), "gemm_groups: %d rounds of tiles for others, with %d waves", rounds, waves);
    // the loads' offsets are 32-bit: rows of X and a group's W
    SP_REQUIRE((size_t)x_rows * ldx * 2 < ((size_t)1 << 31) && (size_t)(glu ? 2 : 1) * N * K * 2 < ((size_t)1 << 31),
               "gemm_groups: operands of 2 GiB and more (%d rows of X, N=%d K=%d)", x_rows, N, K);
    if (M == 0) return 0;
    const gg_args p{(const bf16*)X, ldx, (const bf16*)W, w_group_stride, Y, ldy, M, N, K, offsets, n_groups, a_rows, a_scale, y_rows, 0, 0, cap, rounds * (sp_cu_count() / 8), others};
    if (waves == 5) return y_dtype == SP_BF16 ? gg_launch<4, 5, false, bf16>(p, st) : gg_launch<4, 5, false, float>(p, st);
    if (waves == 8) {
        if (glu) return y_dtype == SP_BF16 ? gg_launch<8, 4, true, bf16>(p, st) : gg_launch<8, 4, true, float>(p, st);
        return y_dtype == SP_BF16 ? gg_launch<8, 4, false, bf16>(p, st) : gg_launch<8, 4, false, float>(p, st);
    }
    if (glu) return y_dtype == SP_BF16 ? gg_launch<4, 4, true, bf16>(p, st) : gg_launch<4, 4, true, float>(p, st);
    return y_dtype == SP_BF16 ? gg_launch<4, 4, false, bf16>(p, st) : gg_launch<4, 4, false, float>(p, st);
}

// What a product over groups takes, in us: `routed` groups that hold `mean` rows each on average (sizes taken as normal about it)
// beside `whole` groups that take all `tokens` rows.
//
// The tiles to expect go to eight XCDs and, in turn, to the four shader engines of each; gemm_tiled and gemm_lds have a
// launch's empty tiles among the others, so that an engine may get more than its share of real ones.  A tile takes `tile` us and, for
// every 5,120 of K, `w` and `x` for each 16 rows (gemm_lds: 32) of its height; where none waits for another `alone` of that; rounds of
// them, of which a last one that is not full counts for `part` and what fills it.  Beside it the stream of the weights of the
// groups that hold rows; the two together between their maximum and their sum.  A gated product takes `gated` of it, one whose bands of
// W lie multiples of 64 KB apart `aligned` (they meet in the same memory channels), and the result is written at `out` TB/s.
// Fitted to 3,600 products (4 to 128 groups of 1 to 8 a token, 65 to 6,000 tokens, N of 512 to 8,192, K of 512 to 16,384, gated in
// bfloat16 and plain in fp32), each timed with every kernel: 7 to 9 % off (gemm_lds 11), much of it alike for all of one size.
// (Four waves over 64 groups and more have become 4 % faster since, by the order of their tiles.)
struct gg_fit { int rows, cols; double start, tile, w, x, tbs, power, part, alone, gated, out, aligned; };
// (The last two, four waves of 80 columns, are fitted to 205 plain products of 8 to 64 experts: 5 % off.)
static const gg_fit GG_FITS[10] = {      // gemm_groups with four waves and tiles of up to 128 and 160 rows, and eight; gemm_tiled's three; gemm_lds; four waves of 80 columns
    {128, 256, 7.15, 2.46, 73.6, 6.2, 9, 1.3, 0.32, 0.444, 0.957, 4.77, 1.03},
    {160, 256, 6.86, 3.15, 86.8, 6.28, 8.58, 1.49, 0.334, 0.45, 0.962, 4.54, 1.02},
    {128, 512, 3.56, 7.1, 99, 2.34, 9, 1.56, 0.784, 0.892, 0.971, 6.32, 1.06},
    {160, 512, 4.23, 7.44, 105, 2.87, 9, 1.71, 0.764, 0.846, 0.98, 5.19, 1.05},
    {128, 512, 6.34, 6.22, 74.1, 6.16, 9, 1.67, 0.654, 0.821, 1.01, 5.73, 0.992},
    {160, 512, 11.1, 5.39, 80.7, 6.63, 7.06, 2.33, 0.659, 0.792, 1.02, 5.3, 1},
    {64, 512, 1.25, 6.7, 72.8, 6.27, 8.59, 1.65, 0.896, 0.922, 1.02, 2, 0.987},
    {256, 256, 2.24, 12.1, 12.9, 12.9, 7.19, 1.47, 0.75, 0.827, 0.979, 6.65, 1.01},
    {128, 320, 6.37, 2.26, 57.5, 5.01, 8.93, 1.89, 0.786, 0.827, 1, 4.83, 1.04},
    {160, 320, 5.88, 2.12, 63.2, 4.83, 7.89, 2.62, 0.828, 0.851, 1, 4.49, 1.03}
};
static int gg_fit_tiles(int kind, int rows, int& nb) {
    if (kind < 4 || kind >= 8) return gg_group_tiles(rows, GG_FITS[kind].rows, nb);
    const int height = GG_FITS[kind].rows, tiles = (rows + height - 1) / height;
    nb = height / 16;
    if (kind == 7) {                     // as gemm_lds takes them
        const int each = tiles ? (rows + tiles - 1) / tiles : 0;
        nb = each > 192 ? 8 : each > 160 ? 6 : each > 128 ? 5 : each > 96 ? 4 : 3;
    }
    return tiles;
}
static double gg_estimate(int kind, int tokens, int routed, double mean, int whole, int N, int K, int glu, int rounds = 0) {
    static const double Z[11] = {-1.6, -1.0, -0.67, -0.43, -0.2, 0.0, 0.2, 0.43, 0.67, 1.0, 1.6};
    const gg_fit& f = GG_FITS[kind];
    const double share = mean / tokens < 1.0 ? mean / tokens : 1.0, sd = sqrt(tokens * share * (1.0 - share));
    double n = 0.0, sum = 0.0;
    int most = 2, nb;
    for (double z : Z) {
        const int rows = (int)(mean + z * sd + 0.5);
        if (rows <= 0) continue;
        const int t = gg_fit_tiles(kind, rows, nb);
        n += t; sum += (double)t * nb;
        most = nb > most ? nb : most;
    }
    n *= routed / 11.0; sum *= routed / 11.0;
    if (whole) {
        const int t = gg_fit_tiles(kind, tokens, nb);
        n += (double)whole * t; sum += (double)whole * t * nb;
        most = nb > most ? nb : most;
    }
    if (n <= 0.0) return 0.0;
    const long cols = (N + f.cols / (glu ? 2 : 1) - 1) / (f.cols / (glu ? 2 : 1));
    const double rows = (double)routed * mean + (double)whole * tokens, cus = sp_cu_count();
    double u;                            // rounds of tiles
    if (kind < 4 || kind >= 8) {
        u = ceil(n * cols / 8.0) / (cus / 8.0 * (kind < 2 ? 2.0 : 1.0));
        if (rounds) u = fmin(fmax(u, rounds - 1 + cols / cus), rounds);      // (one tile of a group more than fits the rounds before, at the least)
    } else {
        const long real = n > 1.0 ? (long)(n + 0.5) : 1, groups = routed + whole;
        long launched = (long)(rows / f.rows) + (groups < (long)rows ? groups : (long)rows), most_tiles = 0;
        if (launched < real) launched = real;
        const long units = launched * cols, per = (units + 7) / 8;
        for (long first = 0; first < units; first += per)
            for (long engine = 0; engine < 4; ++engine) {
                long c = 0;
                for (long unit = first + engine; unit < first + per && unit < units; unit += 4) c += unit % launched < real;
                most_tiles = c > most_tiles ? c : most_tiles;
            }
        u = most_tiles / (cus / 32.0);
    }
    const double tile = f.tile + K / 5120.0 * (f.w + f.x * sum / n), tallest = f.tile + K / 5120.0 * (f.w + f.x * most);
    double work = f.alone * tallest;
    if (kind < 2 && u > 0.5) work = u <= 1.0 ? fmax(tile, work) : tile * (u + f.part * (ceil(u - 1e-9) - u));
    if (kind >= 2 && u > 1.0) work = tile * (u + f.part * (ceil(u - 1e-9) - u));
    const double live = routed * (1.0 - pow(1.0 - share, tokens));
    const double stream = (live + whole) * N * K * (glu ? 4e-6 : 2e-6) / f.tbs;
    const double us = f.start + pow(pow(work, f.power) + pow(stream, f.power), 1.0 / f.power);
    return us * (glu ? f.gated : 1.0) * (K % 2048 == 0 ? f.aligned : 1.0) + rows * N * (glu ? 2e-6 : 4e-6) / f.out;
}

// Which waves and cap suit it: waves * 256 + cap, or 0 where the other product, gemm_lds (`lds`) or gemm_tiled with its tile `shape`, is
// estimated within 2 % of the best of them.  us[0]: what the taken one is estimated to take.  Over those products the choice is 18 %
// faster than the others on average; at 93 it is 2 % and more slower, at 43 of them by 5 % and more (a quarter of those where one
// group took a quarter of the rows, which the estimate cannot know).  16 experts and a shared one: 1,547 tokens x 2 x 8,192 x 5,120
// gated tiles of eight waves (579 us, gemm_tiled 630), 1,512 x 3,072 x 2,048 stays (gemm_groups 67, gemm_tiled 60).
extern "C" int spite_gemm_groups_choice(int tokens, int routed, double mean, int whole, int N, int K, int glu, int shape, int lds, double* us) {
    *us = 0.0;
    if (tokens <= 0 || routed <= 0 || mean <= 0.0) return 0;
    const double other = gg_estimate(lds ? 7 : shape == 3 ? 5 : shape == 4 || shape == 5 ? 6 : 4, tokens, routed, mean, whole, N, K, glu);
    int best = 0;
    for (int kind = 0; kind < 4; ++kind) {
        const double t = gg_estimate(kind, tokens, routed, mean, whole, N, K, glu);
        if (best == 0 || t < *us) { best = (kind < 2 ? 4 : 8) * 256 + GG_FITS[kind].rows; *us = t; }
    }
    if (*us < 0.98 * other) return best;
    *us = other;
    return 0;
}

// How likely the tiles of `cap` rows of all groups are no more than `budget`: a group's rows taken as normal, and the sum of their tiles too.
static double gg_chance(int cap, int tokens, int routed, double mean, int whole, long budget) {
    const double share = mean / tokens < 1.0 ? mean / tokens : 1.0, sd = sqrt(tokens * share * (1.0 - share)) + 1e-9;
    double m = 0.0, sq = 0.0;                // a group's tiles, and their square: the sums over k of P(more than k tiles) and of 2 k + 1 times that
    for (int k = 0; (double)k * cap <= tokens; ++k) {
        const double more = 0.5 * erfc(((double)k * cap + 0.5 - mean) / (sd * M_SQRT2));
        if (more < 1e-12) break;
        m += more; sq += (2 * k + 1) * more;
    }
    const double sum = routed * m + (double)whole * ((tokens + cap - 1) / cap), spread = sqrt(routed * (sq - m * m > 0.0 ? sq - m * m : 0.0)) + 1e-9;
    return 0.5 * erfc((sum - (budget + 0.5)) / (spread * M_SQRT2));
}

// The same for a plain product by tiles of four waves of 80 columns (waves code 5), against whichever of the others would run: 0, or 5 * 256 +
// cap, and in `rounds` those of a tile a compute unit that the groups' tiles have to fit.  A plain product back has few columns: 5,120 make ten
// tiles of 512 for each of 16 experts, 160 for 256 compute units, and 320 of 256, of which 64 units have two; sixteen of 320 are one each, but
// with one expert of more than `cap` rows they are 272, in two rounds: 2,048 rows x 5,120 x 8,192 273 us by tiles of 512 columns, 237 by one round of
// these, 350 by two.  Routers do not spread their rows as evenly as chance would, which the estimate cannot know, so that the device decides
// by the tiles that there are (gemm_groups_kernel).  Of the two launches one finds nothing to do: 2 to 5 us, which products
// of 120 us and more make up for where the tiles can be expected to fit.  (79 products of 8 to 128 experts that are
// taken, rows spread as by chance / by lognormal loads of 0.2 / 0.4 / 0.8 besides: 0.90 / 0.94 / 0.96 / 0.97 of what ran otherwise on average, four of
// the 316 times more than 3 % slower, the worst 13; without the device's decision 0.90 / 0.97 / 0.98 / 1.02, 63 times, 65.  16 experts, 5,120 x
// 8,192, 2,048 rows by chance, the fullest expert 143, 445 / 244; unevenly, 186 to 353, 288 / 290, 299 / 302, 282 / 283.)
extern "C" int spite_gemm_groups_wide_choice(int tokens, int routed, double mean, int whole, int N, int K, int shape, int lds, int* rounds) {
    double us;
    *rounds = 0;
    spite_gemm_groups_choice(tokens, routed, mean, whole, N, K, 0, shape, lds, &us);
    if (us < 120.0) return 0;
    int best = 0;
    double least = 0.95 * us;
    const long cols = (N + 319) / 320, cus = sp_cu_count();
    for (int kind = 8; kind < 10; ++kind) {
        const int cap = GG_FITS[kind].rows;
        int r = 1;
        double chance;
        while ((chance = gg_chance(cap, tokens, routed, mean, whole, r * cus / cols)) < 0.5) ++r;
        const double t = chance * gg_estimate(kind, tokens, routed, mean, whole, N, K, 0, r) + (1.0 - chance) * us + 3.0;
        if (t < least) {
            best = 5 * 256 + cap;
            *rounds = r;
            // the taller tiles: where groups are of one shorter tile on average, for those that are not (the others' are the same); else
            // theirs differ more in height, and have to be the faster ones
            least = fmin(0.95 * us, (mean <= cap ? 1.02 : 0.98) * t);
        }
    }
    return best;
}
