// Products of up to 256 rows (prompts) with the wide matrices of a block, X[M, K] . W[N, K]^T from the tiled copy of W (see
// gemm_rows.hip), bfloat16, sums in float32 on the matrix cores (MFMA 16x16x32) as planes of parts of K, and what follows them in
// the kernel that adds the planes:
//   gate|up  tiles of 8 gate rows and the same 8 up rows: Y[M, F] = act(gate) up;
//   q|k|v    tiles of 8 rows of a q or k head and their rotation partners, then of 16 rows of v: q and k rotated by the row's
//            position, all three into Y[M, N], k and v into the paged cache too.
// A block takes all rows, up to 14 tiles of W and a part of K, 64 k a stage, two or three stages ahead, one barrier a stage.  X and W
// go straight from memory into LDS, W in operand order.  The rows are two groups of waves', the tiles WN waves' of each.
//
// X (from L2) costs a block as much as W (from memory), so a part of K is what keeps X small, and its planes are paid for it: 160
// rows, us, whole K a block with rotation or activation behind the sums / K in two with the planes' kernel / the vendor GEMM with
// theirs: 12288 x 4096 50 / 35.5 / 43.3, 22016 x 4096 54 / 49.6 / 57.9.
// What a stage waits for is open.  It takes as long as its bytes of X and W at some 38 GB/s a compute unit, with two or three stages under
// way; that is neither memory's rate nor L2's (loads alone bring 120 to 146 GB/s from L2 into LDS, and in gemm_tiles.hip 60 % of a
// stage remains with W in L2).
#include <math.h>

#include "api.h"
#include "common.h"

typedef __bf16 gs_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float gs_f32x4_t __attribute__((ext_vector_type(4)));

// MT: tiles of 16 rows a group of waves; NT: tiles of W a wave.
template <int MT, int NT, int WN, int NS>
__global__ void __launch_bounds__(128 * WN, 1)
gemm_short_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ Wt, float* __restrict__ Y, int M, int K, int tiles,
                  int tb, int splits) {
    constexpr int WAVES = 2 * WN, SLOTS = NT * WN, XL = 4 * MT, WL = 2 * SLOTS;          // loads a stage
    constexpr int L = (XL + WL + WAVES - 1) / WAVES, UNITS = (XL + WL) * 64;
    // (arrays of their own: the compiler then knows that a stage's reads do not touch what is being loaded)
    __shared__ illm_u32x4_t st0[UNITS], st1[UNITS], st2[UNITS], st3[NS > 3 ? UNITS : 1];
    const int lane = threadIdx.x & 63, wave = wave_index(), r = lane & 15, q = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const int t0 = blockIdx.x * tb, last_tile = min(t0 + tb, tiles) - 1;
    const int every = K / 64, per = (every + splits - 1) / splits, first = blockIdx.y * per, last = min(first + per, every) - 1;

    // X: a load brings 8 rows of 128 bytes, 16-byte piece c of row t to place c ^ (t % 8).  W: 16 rows of 32 k, lane l's piece
    // to place l.  Rows past M are zeros; slots past the block's tiles bring its last again.
    const __amdgpu_buffer_rsrc_t xr = illm_buffer(X, (size_t)M * K * 2), wr = illm_buffer(Wt, (size_t)tiles * 16 * K * 2);
    uint32_t off[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int n = min(i * WAVES + wave, XL + WL - 1), w = n - XL;
        off[i] = n < XL ? (uint32_t)(n * 8 + (lane >> 3)) * (uint32_t)K * 2u + ((lane & 7) ^ (lane >> 3)) * 16u
                        : ((uint32_t)min(t0 + (w >> 1), last_tile) * (uint32_t)(K / 32) + (w & 1)) * 1024u + (r * 4 + q) * 16u;
    }
    auto load = [&](illm_u32x4_t* to, int s) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)min(s, last) * 128u;               // (past the end: not used)
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int n = min(i * WAVES + wave, XL + WL - 1);
            if (n < XL) ld16_lds(xr, to + n * 64, off[i], at);
            else ld16_lds(wr, to + n * 64, off[i], at * 16);
        }
    };
    gs_f32x4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (gs_f32x4_t){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const illm_u32x4_t* b) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int c = (kk * 4 + q) ^ (r & 7);
            illm_u32x4_t wf[NT], xf[MT];
#pragma unroll
            for (int i = 0; i < NT; ++i) wf[i] = b[(XL + (wn * NT + i) * 2 + kk) * 64 + lane];
#pragma unroll
            for (int j = 0; j < MT; ++j) xf[j] = b[((wm * MT + j) * 16 + r) * 8 + c];
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const gs_bf16x8_t*)&wf[i], *(const gs_bf16x8_t*)&xf[j],
                                                                        acc[i][j], 0, 0, 0);
        }
    };
    // Stage s stands in its buffer when every wave's loads of it have arrived: each wave waits for its own (those of the NS - 2
    // stages behind it may be under way) and meets the others.  By then nobody reads the buffer of stage s - 1 any more (a wave
    // waits for its LDS reads too), so stage s + NS - 1 goes there.
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

    // acc[i][j][e]: row 4 q + e of tile t0 + wn NT + i, row (wm MT + j) 16 + r of X
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = (wm * MT + j) * 16 + r;
        if (m >= M) continue;
        float* const to = Y + (((size_t)blockIdx.y * M + m) * tiles + t0 + wn * NT) * 16 + 4 * q;
#pragma unroll
        for (int i = 0; i < NT; ++i)
            if (wn * NT + i < tb && t0 + wn * NT + i < tiles) *(gs_f32x4_t*)(to + i * 16) = acc[i][j];
    }
}

struct GsQkv {
    const float* cos_sin;        // [max_pos][hd / 2][2]
    const int32_t *row_pos, *row_slot, *slot_len;
    bf16_t *kcache, *vcache;
    const int32_t* page_table;
    int table_stride, page_size, ring, nh, nkv, hd;
};

// 16 sums of a tile's row: the planes' in order.
__device__ __forceinline__ void planes_tile(const float* at, size_t plane, int S, float (&v)[16]) {
    gs_f32x4_t a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = ((const gs_f32x4_t*)at)[i];
    for (int s = 1; s < S; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] += ((const gs_f32x4_t*)(at + s * plane))[i];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = a[i / 4][i % 4];
}

// grid (ceil(tiles / 256), M): a thread a tile of a row, 8 results.  F % 8 == 0.  limit > 0: g sigmoid(alpha g) (u + 1), g = min(gate,
// limit), u = clamp(up, +- limit); else silu(gate) up.
__global__ void __launch_bounds__(256)
gate_up_planes_kernel(const float* __restrict__ P, bf16_t* __restrict__ Y, int S, int M, int tiles, float limit, float alpha) {
    const int tile = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (tile >= tiles) return;
    float v[16], y[8];
    planes_tile(P + ((size_t)m * tiles + tile) * 16, (size_t)M * tiles * 16, S, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float g = v[e], u = v[8 + e];
        if (limit > 0.f) {
            const float gc = fminf(g, limit), uc = fminf(fmaxf(u, -limit), limit);
            y[e] = gc / (1.0f + expf(-alpha * gc)) * (uc + 1.0f);
        } else {
            y[e] = (g / (1.0f + expf(-g))) * u;
        }
    }
    ((uint4*)Y)[(size_t)m * tiles + tile] = make_uint4(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]),
                                                       pack_bf16x2(y[6], y[7]));
}

// grid (ceil(tiles / 256), M): a thread a tile of a row.
__global__ void __launch_bounds__(256)
qkv_planes_kernel(const float* __restrict__ P, bf16_t* __restrict__ Y, int S, int M, int tiles, GsQkv t) {
    const int tile = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (tile >= tiles) return;
    const int pos = t.row_pos[m], slot = t.row_slot[m], per_head = t.hd / 16, turned = (t.nh + t.nkv) * per_head;
    const bool turn = tile < turned;
    const int head = tile / per_head, in = tile - head * per_head;          // (of v: the heads behind those of q and k)
    gs_f32x4_t c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = ((const gs_f32x4_t*)(t.cos_sin + (size_t)pos * t.hd + 16 * (turn ? in : 0)))[i];
    const bool over = t.ring > 0 && t.slot_len;
    const int last_page = over ? (t.slot_len[slot] - 1) / t.page_size : 0;
    float v[16];
    planes_tile(P + ((size_t)m * tiles + tile) * 16, (size_t)M * tiles * 16, S, v);
    int a = 16 * in, b = a + 8;                                // where the two halves of the 16 belong
    if (turn) {
        a = 8 * in;
        b = a + t.hd / 2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = v[e], y = v[8 + e], cs = c[e / 2][2 * (e & 1)], sn = c[e / 2][2 * (e & 1) + 1];
            v[e] = x * cs - y * sn;
            v[8 + e] = x * sn + y * cs;
        }
    }
    const uint4 lo = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    const uint4 hi = make_uint4(pack_bf16x2(v[8], v[9]), pack_bf16x2(v[10], v[11]), pack_bf16x2(v[12], v[13]), pack_bf16x2(v[14], v[15]));
    bf16_t* const row = Y + ((size_t)m * (t.nh + 2 * t.nkv) + head) * t.hd;
    *(uint4*)(row + a) = lo;
    *(uint4*)(row + b) = hi;
    // (a later row of this step lands on the same ring page: this one is already outside)
    if (head < t.nh || (over && pos / t.page_size + t.ring <= last_page)) return;
    bf16_t* const kept = (turn ? t.kcache : t.vcache) + cache_row_offset(t.page_table, t.table_stride, slot, pos, t.page_size, t.ring,
                                                                         t.nkv, head - t.nh - (turn ? 0 : t.nkv), t.hd);
    *(uint4*)(kept + a) = lo;
    *(uint4*)(kept + b) = hi;
}

struct ShortShape { int tb, splits; };

// Tiles a block and parts of K: the least of what a compute unit's rounds of blocks bring in and of the planes, written and
// read at the rate of all 256.  Both rates are fits: 64 to 256 rows of 12288 x 4096, 6144 x 4096 and 15360 x 5120 take 0.85 to
// 1.27 of what they give, and the choice is within 3 % of the best of a dozen others.  Where two are near each other it changes with
// the rows: 12288 x 4096, us, 6 tiles and 2 parts / 12 and 4: 96 rows 29.0 / 31.5, 112 31.8 / 32.6, 128 32.6 / 33.5, 144 35.5 /
// 35.8, 160 36.0 / 36.9, 161 38.6 / 37.3, 192 40.6 / 40.2, 224 44.8 / 45.3.
static ShortShape short_shape(int M, int tiles, int K) {
    const int mt = (M + 31) / 32, most = min(14, 26 - 2 * mt);
    ShortShape best = {2, 1};
    double least = -1.0;
    for (int s = 1; s <= 4; s *= 2) {
        if (K / 64 < 8 * s) break;
        for (int t = 2; t <= most; ++t) {
            const long long rounds = ((long long)(tiles + t - 1) / t * s + 255) / 256;
            const double cost = (double)rounds * ((K / 64 + s - 1) / s + 3) * (mt * 32 * 128 + t * 2048) / 38.0 +
                                2.0 * s * M * tiles * 64 / 4000.0;
            if (least < 0 || cost < least) { least = cost; best = {t, s}; }
        }
    }
    return best;
}

template <int MT>
static int launch_short(const bf16_t* X, const bf16_t* Wt, float* P, int M, int K, int tiles, ShortShape shape, hipStream_t st) {
    const dim3 grid((tiles + shape.tb - 1) / shape.tb, shape.splits);
#define ILLM_SHORT(NT, WN)                                                                                               \
    if constexpr (2 * MT + NT * WN <= 26) {                                                                              \
        hipLaunchKernelGGL((gemm_short_kernel<MT, NT, WN, 2 * MT + NT * WN <= 20 ? 4 : 3>), grid, dim3(128 * WN), 0, st, X, Wt, P, \
                           M, K, tiles, shape.tb, shape.splits);                                                         \
        return illm_launch_status();                                                                                     \
    }
    if (shape.tb <= 4) ILLM_SHORT(2, 2)
    if (shape.tb <= 6) ILLM_SHORT(3, 2)
    if (shape.tb <= 8) ILLM_SHORT(2, 4)
    if (shape.tb <= 10) ILLM_SHORT(5, 2)
    if (shape.tb <= 12) ILLM_SHORT(3, 4)
    if (shape.tb <= 14) ILLM_SHORT(7, 2)
#undef ILLM_SHORT
    return ILLM_ERR_ARG;
}

static int short_planes(const void* X, const void* Wt, float* P, size_t p_bytes, int M, int K, int tiles, ShortShape* taken,
                        hipStream_t st) {
    const ShortShape shape = short_shape(M, tiles, K);
    if ((size_t)shape.splits * M * tiles * 64 > p_bytes) return ILLM_ERR_ARG;
    *taken = shape;
    const bf16_t *x = (const bf16_t*)X, *w = (const bf16_t*)Wt;
    switch ((M + 31) / 32) {
        case 1: return launch_short<1>(x, w, P, M, K, tiles, shape, st);
        case 2: return launch_short<2>(x, w, P, M, K, tiles, shape, st);
        case 3: return launch_short<3>(x, w, P, M, K, tiles, shape, st);
        case 4: return launch_short<4>(x, w, P, M, K, tiles, shape, st);
        case 5: return launch_short<5>(x, w, P, M, K, tiles, shape, st);
        case 6: return launch_short<6>(x, w, P, M, K, tiles, shape, st);
        case 7: return launch_short<7>(x, w, P, M, K, tiles, shape, st);
        default: return launch_short<8>(x, w, P, M, K, tiles, shape, st);
    }
}

static bool short_args(const void* X, const void* Wt, const void* P, const void* Y, int M, long long rows, int K) {
    return X && Wt && P && Y && M > 0 && M <= 256 && rows > 0 && rows <= 1 << 26 && K > 0 && K % 64 == 0 && rows * K * 2 <= 0xffffffffLL &&
           ((uintptr_t)X | (uintptr_t)Wt | (uintptr_t)P | (uintptr_t)Y) % 16 == 0;
}

extern "C" int illm_gemm_short_splits(int M, int rows, int K) {
    return M <= 0 || M > 256 || rows <= 0 || K <= 0 ? 0 : short_shape(M, (rows + 15) / 16, K).splits;
}

extern "C" int illm_gemm_short_gate_up(const void* X, const void* Wt, void* P, size_t p_bytes, void* Y, int M, int F, int K,
                                       float limit, float alpha, void* stream) {
    if (F <= 0 || F % 8 || !short_args(X, Wt, P, Y, M, 2LL * F, K) || !(limit >= 0.f)) return ILLM_ERR_ARG;
    const int tiles = F / 8;
    ShortShape shape;
    const int rc = short_planes(X, Wt, (float*)P, p_bytes, M, K, tiles, &shape, (hipStream_t)stream);
    if (rc != ILLM_OK) return rc;
    hipLaunchKernelGGL(gate_up_planes_kernel, dim3((tiles + 255) / 256, M), dim3(256), 0, (hipStream_t)stream, (const float*)P,
                       (bf16_t*)Y, shape.splits, M, tiles, limit, alpha);
    return illm_launch_status();
}

extern "C" int illm_gemm_short_qkv(const void* X, const void* Wt, void* P, size_t p_bytes, void* Y, int M, int K,
                                   const float* cos_sin, int max_pos, const int32_t* row_pos, const int32_t* row_slot,
                                   const int32_t* slot_len, void* kcache, void* vcache, const int32_t* page_table,
                                   int table_stride, int page_size, int ring, int nh, int nkv, int hd, void* stream) {
    if (nh <= 0 || nkv <= 0 || hd <= 0 || hd % 16 || (nh + 2LL * nkv) * hd > 1 << 26 || !cos_sin || max_pos <= 0 || !row_pos ||
        !row_slot || !kcache || !vcache || !page_table || table_stride <= 0 || page_size <= 0 || ring < 0)
        return ILLM_ERR_ARG;
    const int N = (nh + 2 * nkv) * hd, tiles = N / 16;
    if (!short_args(X, Wt, P, Y, M, N, K)) return ILLM_ERR_ARG;
    ShortShape shape;
    const int rc = short_planes(X, Wt, (float*)P, p_bytes, M, K, tiles, &shape, (hipStream_t)stream);
    if (rc != ILLM_OK) return rc;
    const GsQkv t = {cos_sin, row_pos, row_slot, slot_len, (bf16_t*)kcache, (bf16_t*)vcache, page_table, table_stride, page_size,
                     ring, nh, nkv, hd};
    hipLaunchKernelGGL(qkv_planes_kernel, dim3((tiles + 255) / 256, M), dim3(256), 0, (hipStream_t)stream, (const float*)P, (bf16_t*)Y,
                       shape.splits, M, tiles, t);
    return illm_launch_status();
}
