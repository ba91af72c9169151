// Y[M, N] = X[M, K] . W[N, K]^T, float32 throughout, by the matrix cores' bfloat16 instruction.
//
// A float32 number is the sum of three bfloat16 numbers (8 bits of mantissa each, rounded to nearest, so that the rest is
// what the next one holds): x = x1 + x2 + x3, |x2| <= 2^-8 |x|, |x3| <= 2^-17 |x|.  Both operands are taken 2^24 times
// as large, so that the third part of the smallest normal number is one too: exact for all numbers below 2^104, subnormal
// ones among them; the sums are scaled back.  Beyond, and where a sum passes 2^80, it is no finite number and is taken
// again (below).  Of the nine products of two such sums the six largest are taken, each exact in the instruction's float32
// sum; what is left out is at most 2^-24 of a product, what one float32 rounding of it may lose.  Against 64 bits, in
// units of 2^-24 (here / the float32 instruction): normal operands, K = 64 / 512 / 4,096, root mean square 0.8 / 2.2 / 2.5
// against 2.4 / 6.8 / 19; positive ones, largest 1.0 / 8.3 / 5.4 against 9.0 / 23 / 70; operands whose left-out products are
// the largest and of one sign 0.99 against 0.99.
//
// What bounds it: the matrix cores (six products at 16 times the rate of the float32 instruction), and from 17 to 64
// rows W's bytes.  W comes straight into registers, each wave its own rows, and is parted beside the products (13
// vector instructions a pair, between MFMAs); X's parts, made once by a small kernel in the order of the operands, go
// straight into LDS and serve the four waves.  The largest product of each stage has a sum of its own, so that a sum
// is rounded once a stage at its full size: 2.6 times closer to 64 bits than six roundings, for no vector work.
// Against the float32 instruction (256 rows, us): 4096 x 4096 84 -> 57, 12288 x 4096 232 -> 155 (192 blocks of 128 rows of W
// for 256 compute units), 22016 x 4096 436 -> 263 (1.05 PFLOP/s of bfloat16 products; 688 blocks of 64 for 512 places), 4096 x
// 11008 227 -> 126; 2,048 rows of 22016 x 4096 2,850 -> 1,590 (1.4 PFLOP/s).
// (Published as bf16x6 and the like: Henry, Tang, Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", 2019.)
#include "api.h"
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define SP_K 32                                   // k a stage
#define SP_UP 0x1p24f                             // operands' scale
#define SP_DOWN 0x1p-48f

// two float32, scaled, as their three bfloat16 parts, each pair packed
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
    a *= SP_UP;
    b *= SP_UP;
    p1 = pack_bf16x2(a, b);
    a -= __uint_as_float(p1 << 16);
    b -= __uint_as_float(p1 & 0xffff0000u);
    p2 = pack_bf16x2(a, b);
    a -= __uint_as_float(p2 << 16);
    b -= __uint_as_float(p2 & 0xffff0000u);
    p3 = pack_bf16x2(a, b);
}

// The 8 k of a lane: 4 q .. 4 q + 3 and 16 + 4 q .. 16 + 4 q + 3 of a stage's 32 (both operands alike), so that
// a load of 16 bytes a lane reads 64 neighbouring bytes of a row.
__device__ __forceinline__ void split8(f32x4_t lo, f32x4_t hi, illm_u32x4_t (&p)[3]) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const f32x4_t v = h < 2 ? lo : hi;
        uint32_t a, b, c;
        split_pair(v[2 * (h & 1)], v[2 * (h & 1) + 1], a, b, c);
        p[0][h] = a;
        p[1][h] = b;
        p[2][h] = c;
    }
}

// X's parts in the order that the product's blocks bring them into LDS: [stage of 32 k][16 rows][part][lane].
// Rows beyond M are zeros.
__global__ void __launch_bounds__(256)
f32_split_rows_kernel(const float* __restrict__ X, illm_u32x4_t* __restrict__ P, int M, int K, int tiles) {
    const int lane = threadIdx.x & 63, tile = blockIdx.y;
    const int stage = blockIdx.x * 4 + threadIdx.x / 64;
    if (stage >= K / SP_K) return;
    const int row = tile * 16 + (lane & 15);
    f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    if (row < M) {
        const float* at = X + (size_t)row * K + stage * SP_K + 4 * (lane >> 4);
        lo = *(const f32x4_t*)at;
        hi = *(const f32x4_t*)(at + 16);
    }
    illm_u32x4_t p[3];
    split8(lo, hi, p);
    illm_u32x4_t* to = P + ((size_t)stage * tiles + tile) * 192 + lane;
#pragma unroll
    for (int i = 0; i < 3; ++i) to[64 * i] = p[i];
}

// A block of NW waves takes MT * 16 rows of X and 16 * NW * NT of W; a wave all those rows and 16 * NT of W's.  K is summed in
// parts of `per` stages, and the parts' sums are added in order: by whoever reads the planes, a part a block (grid y), or in
// here (FOLD, per a multiple of 6), one part after the other.  Both ways give the same bits.
template <int MT, int NT, int NS, bool FOLD, int NW = 4>
__global__ void __launch_bounds__(64 * NW, 2)
gemm_f32_split_kernel(const illm_u32x4_t* __restrict__ P, const float* __restrict__ X, const float* W,
                      void* __restrict__ Y, int y_dt, int M, int N, int K, int m_tiles, int per) {
    constexpr int UNITS = MT * 3;                                              // KB of X a stage
    constexpr int LX = (UNITS + NW - 1) / NW, L = LX + 2 * NT;                       // loads a wave a stage
    __shared__ illm_u32x4_t st0[UNITS * 64], st1[UNITS * 64], st2[UNITS * 64];
    __shared__ illm_u32x4_t st3[NS > 3 ? UNITS * 64 : 1], st4[NS > 3 ? UNITS * 64 : 1], st5[NS > 3 ? UNITS * 64 : 1];
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int r = lane & 15, q = lane >> 4;
    // the blocks that share rows of W run next to each other on one XCD (block ids go round the 8)
    const int xcd = blockIdx.x & 7, j8 = blockIdx.x >> 3;
    const int mt = j8 % m_tiles, n0 = ((j8 / m_tiles) * 8 + xcd) * (16 * NW * NT);
    if (n0 >= N) return;
    const int every = K / SP_K;
    const int first = FOLD ? 0 : blockIdx.y * per, last = FOLD ? every - 1 : min(first + per, every) - 1;

    const __amdgpu_buffer_rsrc_t xr = illm_buffer(P, (size_t)every * m_tiles * UNITS * 1024);
    const uint32_t x_stage = (uint32_t)m_tiles * UNITS * 1024, x_lane = (uint32_t)mt * UNITS * 1024 + lane * 16;
    auto load_x = [&](illm_u32x4_t* b, int s) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)min(s, last) * x_stage;
#pragma unroll
        for (int i = 0; i < LX; ++i) {
            const int u = min(i * NW + wave, UNITS - 1);
            ld16_lds(xr, b + u * 64, x_lane + u * 1024, at);
        }
    };
    struct Raw { f32x4_t lo[NT], hi[NT]; };
    struct Parts { illm_u32x4_t w[NT][3]; };
    uint32_t wo[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) wo[i] = (uint32_t)(min(n0 + (wave * NT + i) * 16 + r, N - 1) - n0) * (uint32_t)K * 4u + 16u * q;
    const char* const wbase = (const char*)(W + (size_t)n0 * K);
    auto load_w = [&](Raw& g, int s) __attribute__((always_inline)) {
        const char* const at = wbase + (size_t)min(s, last) * (SP_K * 4);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            g.lo[i] = *(const f32x4_t*)(at + wo[i]);
            g.hi[i] = *(const f32x4_t*)(at + wo[i] + 64);
        }
    };
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // The large products have a sum of their own (one rounding a stage at its size), the five small ones another.
    f32x4_t low[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) low[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    auto split_part = [&](const Raw& g, Parts& p, int e) __attribute__((always_inline)) {     // the e-th pair of a lane
        const f32x4_t v = e % 4 < 2 ? g.lo[e / 4] : g.hi[e / 4];
        uint32_t a, b, c;
        split_pair(v[2 * (e & 1)], v[2 * (e & 1) + 1], a, b, c);
        p.w[e / 4][0][e % 4] = a;
        p.w[e / 4][1][e % 4] = b;
        p.w[e / 4][2][e % 4] = c;
    };
    auto multiply = [&](const illm_u32x4_t* b, const Parts& p, const Raw& next, Parts& pn) __attribute__((always_inline)) {
        constexpr int PW[6] = {2, 0, 1, 0, 1, 0}, PX[6] = {0, 0, 1, 2, 0, 1};
        constexpr int E = (4 * NT + MT - 1) / MT;                              // pairs of W split beside 16 rows of X
        illm_u32x4_t xf[2][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) xf[0][c] = b[c * 64 + lane];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            if (j + 1 < MT) {
#pragma unroll
                for (int c = 0; c < 3; ++c) xf[(j + 1) & 1][c] = b[((j + 1) * 3 + c) * 64 + lane];
            }
#pragma unroll
            for (int e = j * E; e < (j + 1) * E; ++e)
                if (e < 4 * NT) split_part(next, pn, e);
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    f32x4_t& to = t == 1 ? acc[i][j] : low[i][j];
                    to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&p.w[i][PW[t]],
                                                                 *(const bf16x8_t*)&xf[j & 1][PX[t]], to, 0, 0, 0);
                }
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
            for (int t = 0; t < 6 * NT; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 2 * E / NT + 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    Raw g0, g1, g2, g3, g4, g5;
    Parts p0, p1;
    // Turn s: stage s of X stands in LDS and stage s + 1 of W in registers when every wave's loads of NS - 1 turns
    // ago have arrived; those of the turns since may still be under way.  Nobody reads stage s - 1 any more.
    auto turn = [&](illm_u32x4_t* cur, illm_u32x4_t* after, const Parts& p, Parts& pn, const Raw& next, Raw& ask,
                    int s) __attribute__((always_inline)) {
        constexpr int VM = (NS - 2) * L;
        static_assert(VM < 64, "the wait count");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070 | (VM & 15) | ((VM >> 4) << 14));    // vmcnt(VM), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load_x(after, s + NS - 1);
        load_w(ask, s + NS);
        if (s <= last) multiply(cur, p, next, pn);
    };
    // The counted waits need the loads in this order: what a wave has under way behind the wait of turn 0 must be later than
    // stage 0 of X, which other waves read behind the barrier.  (The scheduler is held by the barriers here and in `turn`;
    // selection is since W's pointer is not __restrict__: loads of memory that nothing writes float to any place.)
    auto ask_ahead = [&](Raw& g, illm_u32x4_t* b, int s) __attribute__((always_inline)) {
        load_w(g, s);
        load_x(b, s);
        __builtin_amdgcn_sched_barrier(0);
    };
    ask_ahead(g0, st0, first);
    ask_ahead(g1, st1, first + 1);
    if constexpr (NS > 3) {
        ask_ahead(g2, st2, first + 2);
        ask_ahead(g3, st3, first + 3);
        ask_ahead(g4, st4, first + 4);
        load_w(g5, first + 5);
    } else {
        load_w(g2, first + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 4 * NT; ++e) split_part(g0, p0, e);
    // A part's sums, left in `low`: [i][j][v] is row (wave * NT + i) * 16 + 4 q + v of W's, row 16 j + r of X's.  Those that are
    // no finite numbers (an infinity has no parts) are taken again by the wave on the float32 instruction: all of its tiles
    // at once, so that data full of NaN takes the time of both instructions and no more (256 rows of 4096 x 4096,
    // us alone: finite 71, all of X NaN 162, one number of it 158; a lane's own multiply-adds had taken 7,922 and 724).
    auto odd = [](float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; };
    auto part_sums = [&](int s0, int s1) __attribute__((always_inline)) {
        bool again = false;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                low[i][j] = (acc[i][j] + low[i][j]) * SP_DOWN;
                acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) again |= odd(low[i][j][e]);
            }
        if (!__any(again)) return;
        const char* const xb = (const char*)(X + (size_t)mt * MT * 16 * K);
        uint32_t xo[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) xo[j] = (uint32_t)min(j * 16 + r, M - 1 - mt * MT * 16) * (uint32_t)K * 4u + 16u * q;
#pragma unroll 1
        for (int k = s0 * SP_K; k < (s1 + 1) * SP_K; k += 16) {
            f32x4_t xv[MT], wv[NT];
#pragma unroll
            for (int i = 0; i < NT; ++i) wv[i] = *(const f32x4_t*)(wbase + (size_t)k * 4 + wo[i]);
#pragma unroll
            for (int j = 0; j < MT; ++j) xv[j] = *(const f32x4_t*)(xb + (size_t)k * 4 + xo[j]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i][e], xv[j][e], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (odd(low[i][j][e])) low[i][j][e] = acc[i][j][e];
                acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            }
    };
    f32x4_t tot[FOLD ? NT : 1][FOLD ? MT : 1];
    int part = first;                               // FOLD: where the part under way began
    for (int s = first; s <= last; s += 6) {
        if constexpr (NS == 3) {
            turn(st0, st2, p0, p1, g1, g0, s);
            turn(st1, st0, p1, p0, g2, g1, s + 1);
            turn(st2, st1, p0, p1, g0, g2, s + 2);
            turn(st0, st2, p1, p0, g1, g0, s + 3);
            turn(st1, st0, p0, p1, g2, g1, s + 4);
            turn(st2, st1, p1, p0, g0, g2, s + 5);
        } else {
            turn(st0, st5, p0, p1, g1, g0, s);
            turn(st1, st0, p1, p0, g2, g1, s + 1);
            turn(st2, st1, p0, p1, g3, g2, s + 2);
            turn(st3, st2, p1, p0, g4, g3, s + 3);
            turn(st4, st3, p0, p1, g5, g4, s + 4);
            turn(st5, st4, p1, p0, g0, g5, s + 5);
        }
        if constexpr (FOLD) {
            if (s + 6 - part < per && s + 6 <= last) continue;
            part_sums(part, min(s + 5, last));
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    tot[i][j] = part == 0 ? low[i][j] : tot[i][j] + low[i][j];
                    low[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
            part = s + 6;
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);             // no load into LDS outlives the block
    if constexpr (!FOLD) part_sums(first, last);

#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = (mt * MT + j) * 16 + r;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int n = n0 + (wave * NT + i) * 16 + 4 * q;
            f32x4_t v;
            if constexpr (FOLD) v = tot[i][j];
            else v = low[i][j];
            if (m >= M) continue;
            const size_t at = ((size_t)blockIdx.y * M + m) * N + n;
            if (n + 3 < N && (N & 3) == 0 && y_dt == ILLM_F32) {
                *(f32x4_t*)((float*)Y + at) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) st_f(Y, y_dt, at + e, v[e]);
            }
        }
    }
}

// Y = the planes' sum, in order; four elements a thread, n4 of them.
__global__ void __launch_bounds__(256)
f32_planes_sum_kernel(const float* __restrict__ planes, void* __restrict__ Y, int y_dt, int S, size_t n4) {
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < n4; i += gridDim.x * 256ull) {
        f32x4_t v = ((const f32x4_t*)planes)[i];
        for (int s = 1; s < S; ++s) v += ((const f32x4_t*)planes)[s * n4 + i];
        st_f4(Y, y_dt, i, make_float4(v[0], v[1], v[2], v[3]));
    }
}

struct SplitTiles { int mt, nt, m_tiles, blocks, waves; };

// Rows in equal tiles of at most 128.  Along W a block takes 64 or 128: a compute unit works through its blocks
// in rounds of 256, and one of 128 takes 1.8 times one of 64 (245 rows, us with 128 / with 64: 12288 x 4096
// 146 / 164, 22016 x 4096 263 / 252; 64 rows: 94 / 70 and 112 / 129; 900 rows of 22016 x 4096 789 / 850).  A block of a part
// takes 128, one that adds up its parts 64 (their sums need the registers).  Up to 16 rows, where W's bytes bound it, 32 from
// more than 256 blocks of 64 on (9 rows, us with 128 / 64 / 32: 32000 x 4096 138 / 123 / 122, 22016 x 4096 - / 105 / 91, 12288 x
// 4096 - / 55 / 62).
static SplitTiles split_tiles(int M, int N, bool planes, bool fold) {
    const int tiles = (M + 15) / 16, m_tiles = (tiles + 7) / 8, need = (tiles + m_tiles - 1) / m_tiles;
    const int mt = need <= 2 ? need : need <= 4 ? 4 : need <= 6 ? 6 : 8;
    const int b1 = (N + 63) / 64 * m_tiles, b2 = (N + 127) / 128 * m_tiles;
    if (mt == 1 && !planes && !fold) return b1 > 256 ? SplitTiles{1, 1, 1, (N + 31) / 32, 2} : SplitTiles{1, 1, 1, b1, 4};
    const bool wide = !fold && (planes || 10 * 23 * ((b2 + 255) / 256) <= 10 * 13 * ((b1 + 255) / 256));
    return {mt, wide ? 2 : 1, m_tiles, wide ? b2 : b1, 4};
}

// Stages of 32 k in a part of K, 0 where K is one part.  A row's bits hang on them, so they are the same for all numbers
// of rows up to 128 and for all above: parts for about one block a compute unit at 128 and at 256 rows where the tiles are
// fewer (than 160 of 64 columns), at most 8, each of at least 16 stages; a multiple of 6 (a round of the kernel's loop).
extern "C" int illm_gemm_f32_split_per(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K < SP_K) return 0;
    const int m_tiles = M <= 128 ? 1 : 2, blocks = (N + 127) / 128 * m_tiles;
    if ((N + 63) / 64 * m_tiles >= 160) return 0;
    const int every = K / SP_K, s = max(1, min(min(256 / blocks, 8), every / 16)), per = ((every + s - 1) / s + 5) / 6 * 6;
    return per >= every ? 0 : per;
}

// Whether the parts of so many rows are taken by a block each (planes that somebody adds) and not one after the other by the
// same blocks: up to 128 MB of planes and 256 MB of X's parts (us, planes and their sum / in one: 245 / 1,024 / 2,048 rows of 4096 x 4096 60 / 177 /
// 346 against 95 / 180 / 364, of 4096 x 11008 124 / 430 / 841 against 240 / 457 / 909, of 2048 x 2048 33 / 61 / 107 against
// 51 / 56 / 97; all of K in one part, as it had been from 257 rows on, 4096 x 4096 163 / 314 at 1,024 / 2,048).
extern "C" int illm_gemm_f32_split_planes(int M, int N, int K) {
    const int per = illm_gemm_f32_split_per(M, N, K);
    if (!per || N % 4) return 0;
    return (long long)((K / SP_K + per - 1) / per) * M * N <= 1 << 25 && 6LL * M * K <= 1 << 28;
}

// Rows of X as its parts are laid out (M filled up to whole tiles): 6 bytes of scratch for each of their K.
extern "C" int illm_gemm_f32_split_rows(int M) {
    if (M <= 0) return 0;
    const SplitTiles t = split_tiles(M, 64, false, true);
    return t.m_tiles * t.mt * 16;
}

// float32 X [M, K] and W [N, K] on 16-byte addresses, K % 32 == 0; P: scratch of 6 K illm_gemm_f32_split_rows(M) bytes
// (at most 4 GiB).  per: stages of 32 k in a part of K, 0 for one part.  planes 0: Y [M, N], float32 or bfloat16, per a
// multiple of 6; else the parts' float32 planes [ceil(K / 32 per)][M][N].
extern "C" int illm_gemm_f32_split(const float* X, const float* W, void* P, size_t p_bytes, void* Y, int y_dt, int M,
                                   int N, int K, int per, int planes, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % SP_K || K >= 1 << 22 || !illm_dtype_ok(y_dt) || !X || !W || !Y || !P ||
        per < 0 || (planes && y_dt != ILLM_F32) || ((uintptr_t)X | (uintptr_t)W | (uintptr_t)P | (uintptr_t)Y) % 16)
        return ILLM_ERR_ARG;
    const int every = K / SP_K;
    if (per == 0 || per >= every) per = every;
    const bool fold = !planes && per < every;
    const int parts = planes ? (every + per - 1) / per : 1;
    const SplitTiles t = split_tiles(M, N, parts > 1, fold);
    const size_t need = (size_t)t.m_tiles * t.mt * 16 * K * 6;
    const long long grid_x = ((long long)(t.blocks / t.m_tiles) + 7) / 8 * 8 * t.m_tiles;
    if ((fold && per % 6) || parts > 65535 || need > p_bytes || need > 0xffffffffu || grid_x > 0x7fffffff ||
        t.m_tiles * t.mt > 65535)
        return ILLM_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(f32_split_rows_kernel, dim3((every + 3) / 4, t.m_tiles * t.mt), dim3(256), 0, st, X,
                       (illm_u32x4_t*)P, M, K, t.m_tiles * t.mt);
    const dim3 grid((unsigned)grid_x, parts);
#define ILLM_SPLIT(MT, NT, NS, FOLD, IF, ...)                                                                        \
    if (t.mt == MT && t.nt == NT && fold == FOLD && IF)                                                                \
        hipLaunchKernelGGL((gemm_f32_split_kernel<MT, NT, NS, FOLD __VA_OPT__(,) __VA_ARGS__>), grid, dim3(64 * t.waves), 0, \
                           st, (const illm_u32x4_t*)P, X, W, Y, y_dt, M, N, K, t.m_tiles, per)
#define ILLM_SPLIT_ROWS(MT, NS) ILLM_SPLIT(MT, 1, NS, false, t.waves == 4); ILLM_SPLIT(MT, 2, NS, false, true); ILLM_SPLIT(MT, 1, NS, true, true)
    ILLM_SPLIT(1, 1, 6, false, t.waves == 2, 2);
    ILLM_SPLIT_ROWS(1, 6);
    ILLM_SPLIT_ROWS(2, 6); ILLM_SPLIT_ROWS(4, 6); ILLM_SPLIT_ROWS(6, 3); ILLM_SPLIT_ROWS(8, 3);
#undef ILLM_SPLIT_ROWS
#undef ILLM_SPLIT
    return illm_launch_status();
}

// Y [n], float32 or bfloat16, from float32 planes [S][n]; n a multiple of 4, all on 16-byte addresses.
extern "C" int illm_f32_planes_sum(const float* planes, void* Y, int y_dt, int S, size_t n, void* stream) {
    if (!planes || !Y || S < 1 || n % 4 || !illm_dtype_ok(y_dt) || ((uintptr_t)planes | (uintptr_t)Y) % 16) return ILLM_ERR_ARG;
    if (n == 0) return ILLM_OK;
    const size_t blocks = (n / 4 + 255) / 256;
    hipLaunchKernelGGL(f32_planes_sum_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                       (hipStream_t)stream, planes, Y, y_dt, S, n / 4);
    return illm_launch_status();
}
