// Products of up to 256 bfloat16 rows with a thin matrix, both operands row-major, float32 accumulation
// on the matrix cores (MFMA 16x16x32), K cut over blockIdx.y: float32 planes [splits][M][N] that
// `add_rmsnorm` adds in order (the o and down projections of 129 to 256 rows).
//
// The vendor GEMM finds too few tiles for these (192 rows of the 7B shape: o 32 us, down 49 with its rows
// filled up to 256).  Here a block takes all rows, 64 or 128 columns (`tiles_columns`) and its part of K, about one
// block a compute unit: a part of K is what keeps the chip busy and X small.  Both operands go straight from memory into
// LDS, 64 k (a row's 128 bytes) a stage, two or three stages ahead, one barrier a stage.  Measured with
// the norm behind it at 192 rows, matrices cold: o 39 -> 21 us, down 61 -> 37.  What is left: with W's
// lines taken from L2 a stage takes 60 % of the time, so the blocks wait for memory (up to 96 KB a
// compute unit are under way); an extra wave that asks for W's lines 8 or 16 stages ahead gained nothing.
// The same loop with whole K (q|k|v with its rotation 47 -> 42 us, gate|up 61 -> 60, 73 -> 78 at the 8B
// shape) does not beat the vendor's by enough to stand beside it.
#include "api.h"
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define GT_K 64                                   // k a stage

// TM x TN: rows of X and of W a block takes; WM x WN waves; NS stages in LDS.
template <int TM, int TN, int WM, int WN, int NS>
__global__ void __launch_bounds__(64 * WM * WN, 1)
gemm_tiles_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, float* __restrict__ Y,
                  int M, int N, int K, int splits) {
    constexpr int WAVES = WM * WN, MT = TM / WM / 16, NT = TN / WN / 16;
    constexpr int LX = TM / 8 / WAVES, LW = TN / 8 / WAVES, L = LX + LW;       // loads a wave a stage
    static_assert(LX * 8 * WAVES == TM && LW * 8 * WAVES == TN, "whole loads");
    constexpr int UNITS = (TM + TN) * 8;                                       // 16-byte units of a stage
    // (arrays of their own: the compiler then knows that a stage's reads do not touch what is being loaded)
    __shared__ illm_u32x4_t st0[UNITS], st1[UNITS], st2[UNITS], st3[NS > 3 ? UNITS : 1];
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int r = lane & 15, q = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;
    const int every = K / GT_K, per = (every + splits - 1) / splits;
    const int first = blockIdx.y * per, last = min(first + per, every) - 1;    // stages of this part of K
    const int n0 = blockIdx.x * TN;

    // A load instruction brings 8 rows of 128 bytes; 16-byte piece c of row t stands at place c ^ (t % 8)
    // of the row, so that the 16 rows an MFMA operand reads at once lie in different banks.
    const __amdgpu_buffer_rsrc_t xr = illm_buffer(X, (size_t)M * K * 2);
    const __amdgpu_buffer_rsrc_t wr = illm_buffer(W, (size_t)N * K * 2);
    uint32_t xo[LX], wo[LW];
    const int lr = lane >> 3, lc = (lane & 7) ^ lr;
#pragma unroll
    for (int i = 0; i < LX; ++i) xo[i] = (uint32_t)((i * WAVES + wave) * 8 + lr) * (uint32_t)K * 2u + lc * 16;
#pragma unroll
    for (int i = 0; i < LW; ++i) wo[i] = (uint32_t)(n0 + (i * WAVES + wave) * 8 + lr) * (uint32_t)K * 2u + lc * 16;
    auto load = [&](illm_u32x4_t* b, int s) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)min(s, last) * (GT_K * 2);               // (past the end: not used)
#pragma unroll
        for (int i = 0; i < LW; ++i) ld16_lds(wr, b + (TM + (i * WAVES + wave) * 8) * 8, wo[i], at);
#pragma unroll
        for (int i = 0; i < LX; ++i) ld16_lds(xr, b + (i * WAVES + wave) * 64, xo[i], at);
    };
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int w_at = (TM + wn * (TN / WN) + r) * 8, x_at = (wm * (TM / WM) + r) * 8;
    auto multiply = [&](const illm_u32x4_t* b) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int c = (kk * 4 + q) ^ (r & 7);
            illm_u32x4_t wf[NT], xf[MT];
#pragma unroll
            for (int i = 0; i < NT; ++i) wf[i] = b[w_at + i * 128 + c];
#pragma unroll
            for (int j = 0; j < MT; ++j) xf[j] = b[x_at + j * 128 + c];
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&wf[i], *(const bf16x8_t*)&xf[j],
                                                                        acc[i][j], 0, 0, 0);
        }
    };
    // Stage s stands in its buffer when every wave's loads of it have arrived: each wave waits for its own
    // (those of the NS - 2 stages behind it may still be under way) and meets the others.  By then nobody
    // reads the buffer of stage s - 1 any more (a wave waits for its LDS reads too), so stage s + NS - 1
    // goes there.
    auto turn = [&](illm_u32x4_t* cur, illm_u32x4_t* next, int s) __attribute__((always_inline)) {
        constexpr int VM = (NS - 2) * L;
        static_assert(VM < 64, "the wait count");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070 | (VM & 15) | ((VM >> 4) << 14));    // vmcnt(VM), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load(next, s + NS - 1);
        if (s <= last) multiply(cur);
    };
    load(st0, first);
    load(st1, first + 1);
    if constexpr (NS > 3) load(st2, first + 2);
    for (int s = first; s <= last; s += NS) {
        if constexpr (NS == 3) {
            turn(st0, st2, s);
            turn(st1, st0, s + 1);
            turn(st2, st1, s + 2);
        } else {
            turn(st0, st3, s);
            turn(st1, st0, s + 1);
            turn(st2, st1, s + 2);
            turn(st3, st2, s + 3);
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);             // no load into LDS outlives the block

    // acc[i][j][v]: tile row wn * (TN / WN) + 16 i + 4 q + v of W, row wm * (TM / WM) + 16 j + r of X
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = wm * (TM / WM) + 16 * j + r;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int n = n0 + wn * (TN / WN) + 16 * i + 4 * q;
            if (n < N)                               // (N is a multiple of 4)
                *(f32x4_t*)(Y + ((size_t)blockIdx.y * M + m) * N + n) = acc[i][j];
        }
    }
}

// Columns a block takes.  X (from L2) costs a block as much as W (see gemm_short.hip): of 128 columns X is read half as often,
// for twice the planes, which pays where a part of K is then at least 16 stages long.  us with the norm that
// adds the planes, matrices cold, 160 / 256 rows, 64 -> 128 columns: 4096 x 11008 37.5 / 46.2 -> 34.9 / 43.4, 4096 x 14336
// 43.6 / 53.6 -> 39.4 / 48.6, 8192 x 28672 155 / 192 -> 124 / 146; with parts of 8 stages 4096 x 4096 19.4 / 25.3 -> 21.6 / 27.6,
// 2048 x 8192 19.4 / 24.9 -> 22.0 / 27.5.  (Within the 4 GiB of a load's offset.)
static int tiles_columns(int N, int K) {
    const int blocks = (N + 127) / 128;
    return K / GT_K >= 16 * max(1, 256 / blocks) && (N + 127LL) * K * 2 < 0xffffffffLL ? 128 : 64;
}

// Parts of K for about one block a compute unit, each at least 8 stages long and none empty.
extern "C" int illm_gemm_tiles_splits(int N, int K) {
    if (N <= 0 || K < GT_K) return 1;
    const int columns = tiles_columns(N, K), blocks = (N + columns - 1) / columns, every = K / GT_K;
    const int s = max(1, min(256 / blocks, every / 8)), per = (every + s - 1) / s;
    return (every + per - 1) / per;
}

// X [M <= 256, K], W [N, K], K % 64 == 0, N % 4 == 0, planes Y float32 [splits][M][N], no part of K empty; X
// and W each within the 4 GiB that a load's 32-bit offset reaches; X, W and Y on 16-byte addresses (a lane brings or
// stores 16 bytes at a time).  Else ILLM_ERR_ARG.
extern "C" int illm_gemm_tiles_planes(const void* X, const void* W, float* Y, int M, int N, int K, int splits,
                                      void* stream) {
    if (!X || !W || !Y || M <= 0 || M > 256 || N <= 0 || K <= 0 || K % GT_K || N % 4 || splits < 1 || splits > 65535 ||
        (long long)(N + 63) * K * 2 >= 0xffffffffLL || 256LL * K * 2 >= 0xffffffffLL ||
        ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16)
        return ILLM_ERR_ARG;
    const int every = K / GT_K, per = (every + splits - 1) / splits;
    if ((long long)(splits - 1) * per >= every) return ILLM_ERR_ARG;
    const int columns = tiles_columns(N, K);
    const dim3 grid((N + columns - 1) / columns, splits);
#define ILLM_TILES(TM, TN, NS)                                                                                        \
    hipLaunchKernelGGL((gemm_tiles_kernel<TM, TN, 4, 2, NS>), grid, dim3(512), 0, (hipStream_t)stream, (const bf16_t*)X, \
                       (const bf16_t*)W, Y, M, N, K, splits)
    if (columns == 64) {
        if (M <= 192) ILLM_TILES(192, 64, 4);
        else ILLM_TILES(256, 64, 3);
    } else {
        if (M <= 192) ILLM_TILES(192, 128, 3);
        else ILLM_TILES(256, 128, 3);
    }
#undef ILLM_TILES
    return illm_launch_status();
}
