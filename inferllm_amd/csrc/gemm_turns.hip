// Gate and up products of many bfloat16 rows (prompts) with their activation in one kernel, Y[M, F] = act(X . Wg^T, X . Wu^T)
// with W = [Wg | Wu], by the loop of gemm_turns.h; the activation acts on the float32 sums, as in the kernels for few rows.
//
// A block works through tiles, its loads running ahead from one to the next, so that only the results lie between a tile's
// last product and the next one's first.  Block ids go round the 8 XCDs: an XCD takes a stretch of the tiles, in groups of
// 8 along X, so that the 32 under way share 8 panels of X and 4 of W in its L2.
// Against the vendor GEMM (cut along the columns where that was faster) and the activation behind it, which wrote and read
// both products (us, in turn on one card, weights from memory): 2 x 14336 x 4096 of 9,061 rows 1,547 -> 1,495, of 512 108 -> 97;
// 2 x 11008 x 4096 of 9,061 / 2,048 / 500 rows 1,283 / 289 / 99 -> 1,178 / 276 / 90 (1.34 PFLOP/s, 688 tiles or 2.7 rounds of 256,
// one round of 172); 2 x 5376 x 2048 of 2,964 rows 119 -> 105.  What bounds the large ones is the chip's power.
#include <algorithm>

#include "api.h"
#include "gemm_turns.h"

// g / (1 + e^-(alpha g)), off by at most 4.1 x 2^-24 of it wherever the result is a normal number (expf and a division
// 3.1): e^x as 2^(x log2 e) with the product's rounding and log2 e's taken along, and the denominator's quarter, so that
// the reciprocal of a sum of up to 2^128 is no subnormal number, which the hardware makes zero.  Nothing is under way on the
// matrix cores while a tile's results are formed: us of 2 x 11008 x 4096, 500 / 2,048 rows, by expf and a division 92.2 / 279,
// by this 89.3 / 271, by a plain product, exponential and reciprocal (18 x 2^-24 down to -20, 65 to -87, zero below -87.3)
// 87.8 / 266.
__device__ __forceinline__ float turns_gated(float g, float alpha) {
    const float z = fminf(fmaxf(alpha * g, -128.0f), 128.0f);          // (beyond: e^-z is infinite or nothing beside 1)
    const float h = -1.44269502f * z;
    const float rest = fmaf(-1.44269502f, z, -h) - 1.92596299e-8f * z;
    const float d = 0.25f + 0.25f * (__builtin_amdgcn_exp2f(h) * fmaf(rest, 0.693147182f, 1.0f));
    return (0.25f * g) * __builtin_amdgcn_rcpf(d);
}

struct TileAt { int m, n; };
__device__ __forceinline__ TileAt turns_tile(int t, int tiles, int mts, int nts) {
    const int xcd = t & 7, at = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (t >> 3);
    const int group = at / (8 * nts), in = at - group * 8 * nts, gm = min(8, mts - group * 8);
    return {group * 8 + in % gm, in / gm};
}

// limit > 0: g sigmoid(alpha g) (u + 1), g = min(gate, limit), u = clamp(up, -limit, limit); else silu(gate) up (alpha 1).
// K % 128 == 0, F % 8 == 0.
template <int MT0, int MT1, int NTH>
__global__ void __launch_bounds__(512, 2)
gemm_turns_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, bf16_t* __restrict__ Y, int M, int F, int K,
                  float limit, float alpha) {
    using T = Turns<MT0, MT1, NTH, NTH>;
    constexpr int COLS = T::BN / 2;
    __shared__ illm_u32x4_t x0a[T::UX0], x1a[T::UX1], w0a[T::UW0], w1a[T::UW1];
    __shared__ illm_u32x4_t x0b[T::UX0], x1b[T::UX1], w0b[T::UW0], w1b[T::UW1];
    const int mts = (M + T::BM - 1) / T::BM, nts = (F + COLS - 1) / COLS, tiles = mts * nts, stages = K / 64;
    T t;
    t.begin();
    struct Loads {
        const T& t;
        const bf16_t *X, *W;
        int M, F, K, mts, nts, tiles, stages, tile, stage;
        __amdgpu_buffer_rsrc_t rx, rw0, rw1, rx1;              // of stage s + 2; rx1: of stage s + 1
        uint32_t at, at1, ox0[T::CX0], ox1[T::CX1], ow0[T::CW0], ow1[T::CW1];
        // (rows past the matrices and stages past the last tile: zeros, read from nowhere)
        __device__ __forceinline__ void aim() {
            const bool on = tile < tiles;
            const TileAt a = turns_tile(on ? tile : 0, tiles, mts, nts);
            const size_t row = (size_t)K * 2, n0 = (size_t)a.n * COLS, w_rows = on ? (size_t)min(COLS, F - a.n * COLS) : 0;
            rx = illm_buffer(X + (size_t)a.m * T::BM * K, on ? (size_t)min(T::BM, M - a.m * T::BM) * row : 0);
            rw0 = illm_buffer(W + n0 * K, w_rows * row);
            rw1 = illm_buffer(W + ((size_t)F + n0) * K, w_rows * row);
            at = 0;
        }
        __device__ __forceinline__ void advance() {
            rx1 = rx;
            at1 = at;
            at += 128;
            if (++stage == stages) {
                stage = 0;
                tile += gridDim.x;
                aim();
            }
        }
        __device__ __forceinline__ void x1(illm_u32x4_t* to) const { t.load(to, rx1, ox1, at1); }
        __device__ __forceinline__ void w0(illm_u32x4_t* to) const { t.load(to, rw0, ow0, at); }
        __device__ __forceinline__ void x0(illm_u32x4_t* to) const { t.load(to, rx, ox0, at); }
        __device__ __forceinline__ void w1(illm_u32x4_t* to) { t.load(to, rw1, ow1, at); advance(); }
    } ld = {t, X, W, M, F, K, mts, nts, tiles, stages, (int)blockIdx.x, 0};
    const uint32_t K2 = (uint32_t)K * 2u;
#pragma unroll
    for (int i = 0; i < T::CX0; ++i) ld.ox0[i] = t.template x_row<MT0>(i, 0) * K2 + t.lc;
#pragma unroll
    for (int i = 0; i < T::CX1; ++i) ld.ox1[i] = t.template x_row<MT1>(i, MT0 * 16) * K2 + t.lc;
#pragma unroll
    for (int i = 0; i < NTH; ++i) {                            // (part 0 gate rows, part 1 the up rows of the same columns)
        const typename T::WAt w = t.template w_row<NTH>(i);
        ld.ow0[i] = ld.ow1[i] = (uint32_t)(w.wave * NTH * 16 + turns_column<NTH>(w.tile, w.row)) * K2 + t.lc;
    }
    ld.aim();
    ld.w0(w0a); ld.x0(x0a); ld.w1(w1a);
    ld.x1(x1a);
    ld.w0(w0b); ld.x0(x0b); ld.w1(w1b);
    t.start(w0a);
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        t.clear();
        for (int s = 0; s < stages; s += 2) {
            t.template stage<0>(x0a, x1a, w0a, w1a, x1b, w0b, ld);
            t.template stage<1>(x0b, x1b, w0b, w1b, x1a, w0a, ld);
        }
        const TileAt a = turns_tile(tile, tiles, mts, nts);
#pragma unroll
        for (int j = 0; j < T::MT; ++j) {
            const int m = a.m * T::BM + t.wm * T::MT * 16 + 16 * j + t.r;
            const int n = a.n * COLS + t.wn * NTH * 16 + t.q * 4 * NTH;
            if (m >= M || n >= F) continue;
            uint32_t o[2 * NTH];
#pragma unroll
            for (int i = 0; i < NTH; ++i) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float g = t.acc[i][j][e], u = t.acc[NTH + i][j][e];
                    const float gc = limit > 0.f ? fminf(g, limit) : g;
                    const float uc = limit > 0.f ? fminf(fmaxf(u, -limit), limit) + 1.0f : u;
                    v[e] = turns_gated(gc, alpha) * uc;
                }
                o[2 * i] = pack_bf16x2(v[0], v[1]);
                o[2 * i + 1] = pack_bf16x2(v[2], v[3]);
            }
            bf16_t* const to = Y + (size_t)m * F + n;
            if constexpr (NTH == 2) *(uint4*)to = make_uint4(o[0], o[1], o[2], o[3]);
            else *(uint2*)to = make_uint2(o[0], o[1]);
        }
    }
    t.end();
}

static const struct { int m, n, cost; } TURNS_SHAPES[4] = {{256, 256, 88}, {192, 256, 73}, {128, 256, 59}, {256, 128, 58}};

static long long turns_tiles(int M, int F, int shape) {
    const auto s = TURNS_SHAPES[shape];
    return ((long long)M + s.m - 1) / s.m * ((2LL * F + s.n - 1) / s.n);
}

// Tiles of 256 x 256, 192 x 256, 128 x 256 or 256 x 128 rows of X and of W: the least of rounds of 256 blocks times a
// round's time (K = 4,096, us: 88, 73, 59 and 58; with the gate as it is now about 1 more each).
static int turns_shape(int M, int F) {
    int best = 0;
    long long least = -1;
    for (int i = 0; i < 4; ++i) {
        const long long cost = (turns_tiles(M, F, i) + 255) / 256 * TURNS_SHAPES[i].cost;
        if (least < 0 || cost < least) { best = i; least = cost; }
    }
    return best;
}

extern "C" int illm_gemm_turns_tiles(int M, int F, int* shape) {
    const int s = turns_shape(M, F);
    if (shape) *shape = s;
    return (int)std::min(turns_tiles(M, F, s), 0x7fffffffLL);
}

// X [M, K], W [2 F, K] = [gate | up], Y [M, F], bfloat16 on 16-byte addresses, K % 128 == 0, F % 8 == 0.
extern "C" int illm_gemm_turns_gate_up(const void* X, const void* W, void* Y, int M, int F, int K, float limit, float alpha,
                                       void* stream) {
    if (!X || !W || !Y || M <= 0 || F <= 0 || F > 1 << 29 || K < 128 || K % 128 || K > 1 << 22 || F % 8 || limit < 0.f ||
        ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16)
        return ILLM_ERR_ARG;
    if (!(limit > 0.f)) alpha = 1.0f;
#define ILLM_TURNS(I, MT0, MT1, NTH)                                                                                     \
    case I:                                                                                                              \
        hipLaunchKernelGGL((gemm_turns_kernel<MT0, MT1, NTH>), dim3((unsigned)(tiles < 256 ? tiles : 256)), dim3(512), 0, \
                           (hipStream_t)stream, (const bf16_t*)X, (const bf16_t*)W, (bf16_t*)Y, M, F, K, limit, alpha);  \
        break
    const int shape = turns_shape(M, F);
    const long long tiles = turns_tiles(M, F, shape);
    if (tiles > 0x3fffffff) return ILLM_ERR_ARG;
    switch (shape) {
        ILLM_TURNS(0, 4, 4, 2);
        ILLM_TURNS(1, 4, 2, 2);
        ILLM_TURNS(2, 2, 2, 2);
        ILLM_TURNS(3, 4, 4, 1);
    }
#undef ILLM_TURNS
    return illm_launch_status();
}
