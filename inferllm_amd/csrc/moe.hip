// Routed feed-forward (mixture of experts): the router's choice, the grouping of (token, choice)
// pairs by expert, the experts' products over their own rows, and the weighted sum.
//
// A pair p = t * top + k is token t's k-th choice.  Pairs are grouped by expert into tiles of at
// most MOE_TILE rows; a block of the product kernels takes one tile and some output columns, a wave
// one column at a time with the lanes cutting K among them, so a matrix is read once per tile and
// a row's sum depends on nothing but the row (its order over K is fixed by the lane pattern).  The
// order of the pairs inside an expert's group is whatever the grouping's counters gave: it moves
// rows between tiles and changes no value.
#include "api.h"
#include "common.h"
#include "gemm_turns.h"

#define MOE_TILE 8

// ---------------------------------------------------------------- router
// z[t, e] = sum_k x[t, k] w[e, k] with a float32 matrix of few rows (a router): float32 products
// and sums.  Every sum runs over K in the same order whatever its companions and their number, so
// that near-tied experts are the same for a prompt's row and for the same token alone: a wave's lanes
// take four neighbouring k each (one where K % 4), 256 (64) a turn, and the lanes' sums are added
// half by half of the wave, then by quarters, down to neighbours.
__device__ __forceinline__ float4 ld4_f32(const void* p, int dt, size_t i) {
    if (dt == ILLM_BF16) {
        const uint2 u = *(const uint2*)((const bf16_t*)p + i);
        return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                           __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u));
    }
    return *(const float4*)((const float*)p + i);
}

// wave_sum without a trip through LDS, the same additions in the same order: the other half of the wave, the
// row of sixteen lanes beside, then within a row the lane 8, 4, 2 and 1 on (once lanes l and l ^ 8 hold the
// same number, the lane 4 on holds that of l ^ 4, and so on down).
template <int CTRL>
__device__ __forceinline__ float few_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float few_wave_sum(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = __int_as_float(r[0]) + __int_as_float(r[1]);
    r = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = __int_as_float(r[0]) + __int_as_float(r[1]);
    v += few_dpp<0x128>(v);
    v += few_dpp<0x124>(v);
    v += few_dpp<0x122>(v);
    v += few_dpp<0x121>(v);
    return v;
}

// Up to 16 tokens (single tokens of a batch): a wave an output of a token, V neighbouring k a lane, eight
// turns of the lanes asked for before the first is used.  Bound by that trip to memory; with 8 tokens a wave it
// was the chain of its loads and of 8 sums of 6 exchanges each: 64 outputs of K = 2,048 for 8 tokens 14.2 -> 2.2
// us, 160 of 5,120 29.6 -> 4.7 (two tokens a wave 2.8 and 4.8, four 3.6 and 6.8).  grid (T, ceil(NE / 4)).
template <int DT, int V>
__global__ void __launch_bounds__(256)
few_outputs_few_tokens_kernel(const void* __restrict__ x, const float* __restrict__ w, float* __restrict__ z, int NE,
                              int K) {
    constexpr int AHEAD = 8;
    const size_t t = blockIdx.x;
    const int e = blockIdx.y * 4 + wave_index(), lane = threadIdx.x & 63;
    if (e >= NE) return;
    const float* wr = w + (size_t)e * K;
    float acc = 0.f;
    for (int k0 = lane * V; k0 < K; k0 += 64 * V * AHEAD) {
        float wv[AHEAD][V], xv[AHEAD][V];
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {               // (past K: the first turn's again, not used)
            const int k = k0 + 64 * V * a < K ? k0 + 64 * V * a : k0;
            if (V == 4) {
                *(float4*)wv[a] = *(const float4*)(wr + k);
                *(float4*)xv[a] = ld4_f32(x, DT, t * K + k);
            } else {
                wv[a][0] = wr[k];
                xv[a][0] = ld_f(x, DT, t * K + k);
            }
        }
        loads_asked_for();
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            if (k0 + 64 * V * a >= K) continue;
#pragma unroll
            for (int j = 0; j < V; ++j) acc += xv[a][j] * wv[a][j];
        }
    }
    acc = few_wave_sum(acc);
    if (lane == 0) z[t * NE + e] = acc;
}

// More tokens: a wave takes 4 outputs and 8 tokens at a time (a chunk of a row of w serves 8 tokens, a chunk of
// a token's row 4 outputs), V neighbouring k a lane, the next turn's loads on their way beside this turn's products.  Rows past
// the last are the last again: a load behind a branch on the type or the row is waited for before the next is asked
// for, which had been the kernel's time (64 outputs of K = 2,048 for 64 / 2,964 bfloat16 tokens
// 15 / 73 -> 8.5 / 26 us, 160 of 5,120 for 2,964 444 -> 132).  grid (ceil(T / 8), ceil(NE / 16)).
template <int DT, int V>
__global__ void __launch_bounds__(256)
few_outputs_f32_kernel(const void* __restrict__ x, const float* __restrict__ w,
                       float* __restrict__ z, int T, int NE, int K) {
    const int t0 = blockIdx.x * 8;
    const int e0 = (blockIdx.y * 4 + wave_index()) * 4, lane = threadIdx.x & 63;
    if (e0 >= NE) return;
    const int nt = T - t0 < 8 ? T - t0 : 8;
    const float* wr[4];
    size_t xr[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) wr[j] = w + (size_t)(e0 + j < NE ? e0 + j : NE - 1) * K;
#pragma unroll
    for (int i = 0; i < 8; ++i) xr[i] = (size_t)min(t0 + i, T - 1) * K;
    float v[32];                                        // sum 4 i + j: token i, output j
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i] = 0.f;
    // (as they lie in memory: 4, 8 or 16 bytes)
    typedef float w_t __attribute__((ext_vector_type(V)));
    typedef uint32_t h_t __attribute__((ext_vector_type(V == 4 ? 2 : 1)));
    struct Turn { w_t w[4], x[DT == ILLM_F32 ? 8 : 1]; h_t h[DT == ILLM_BF16 ? 8 : 1]; };
    auto ask = [&](Turn& t, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) t.w[j] = *(const w_t*)(wr[j] + k);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (DT == ILLM_F32) t.x[i] = *(const w_t*)((const float*)x + xr[i] + k);
            else if constexpr (V == 4) t.h[i] = *(const h_t*)((const bf16_t*)x + xr[i] + k);
            else t.h[i] = ((const bf16_t*)x)[xr[i] + k];
        }
    };
    auto add = [&](const Turn& t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float xv[V];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if constexpr (DT == ILLM_F32) xv[e] = t.x[i][e];
                else xv[e] = __uint_as_float(V == 1 || !(e & 1) ? t.h[i][e / 2] << 16 : t.h[i][e / 2] & 0xffff0000u);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < V; ++e) v[4 * i + j] += xv[e] * t.w[j][e];
        }
    };
    const int first = lane * V, step = 64 * V;
    if (first < K) {
        Turn t0_, t1_;
        ask(t0_, first);
        for (int k = first; k < K; k += 2 * step) {
            ask(t1_, k + step < K ? k + step : first);  // (past K: the first turn's again, not used)
            __builtin_amdgcn_sched_barrier(0);
            add(t0_);
            if (k + step >= K) break;
            ask(t0_, k + 2 * step < K ? k + 2 * step : first);
            __builtin_amdgcn_sched_barrier(0);
            add(t1_);
        }
    }
    // 32 sums over 64 lanes by halving: at the step that pairs lanes l and l ^ b a lane keeps the sums whose
    // number has that step's bit where l has b, 1 for b = 32 up to 16 for b = 2
#pragma unroll
    for (int b = 32, n = 16; b > 1; b >>= 1, n >>= 1) {
        const bool up = (lane & b) != 0;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const float keep = up ? v[2 * i + 1] : v[2 * i], send = up ? v[2 * i] : v[2 * i + 1];
            v[i] = keep + __shfl_xor(send, b, ILLM_WAVE);
        }
    }
    const float sum = v[0] + __shfl_xor(v[0], 1, ILLM_WAVE);
    const int mine = (int)(__brev((uint32_t)lane) >> 26) & 31;      // lane bit 5 is the sum's bit 0, .., bit 1 its bit 4
    const int i = mine >> 2, j = mine & 3;
    if (!(lane & 1) && i < nt && e0 + j < NE) z[(size_t)(t0 + i) * NE + e0 + j] = sum;
}

extern "C" int illm_few_outputs_f32(const void* x, int x_dt, const float* w, float* z, int T, int NE,
                                    int K, void* stream) {
    if (T < 0 || NE <= 0 || NE > 65535 * 4 || K <= 0 || !illm_dtype_ok(x_dt)) return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    hipStream_t st = (hipStream_t)stream;
    if (T <= 16) {
#define GO(DT_, V_)                                                                                          \
    hipLaunchKernelGGL((few_outputs_few_tokens_kernel<DT_, V_>), dim3(T, (NE + 3) / 4), dim3(256), 0, st, x, w, \
                       z, NE, K)
        if (K % 4) {
            if (x_dt == ILLM_BF16) GO(ILLM_BF16, 1);
            else GO(ILLM_F32, 1);
        } else if (x_dt == ILLM_BF16) GO(ILLM_BF16, 4);
        else GO(ILLM_F32, 4);
#undef GO
        return illm_launch_status();
    }
#define GO(DT_, V_)                                                                                          \
    hipLaunchKernelGGL((few_outputs_f32_kernel<DT_, V_>), dim3((T + 7) / 8, (NE + 15) / 16), dim3(256), 0, st, x, w, z, T, NE, K)
    if (K % 4) {
        if (x_dt == ILLM_BF16) GO(ILLM_BF16, 1);
        else GO(ILLM_F32, 1);
    } else if (x_dt == ILLM_BF16) GO(ILLM_BF16, 4);
    else GO(ILLM_F32, 4);
#undef GO
    return illm_launch_status();
}

// Scores of a router's outputs: their softmax, or every output's sigmoid.
#define MOE_SCORE_SOFTMAX 0
#define MOE_SCORE_SIGMOID 1
// What an expert does with its gate and up products: silu(gate) * up, or with both clamped
// (gate from above, up on both sides, at `limit`) gate * sigmoid(1.702 gate) * (up + 1).
#define MOE_ACT_SILU 0
#define MOE_ACT_CLAMPED 1
// Experts without a gate: the up product alone, act(z) = max(z, 0)^2 (as `act_kind` of a product that
// is not gated; any other kind there leaves the product as it is).
#define MOE_ACT_RELU2 2
__device__ __forceinline__ float moe_act(float gate, float up, int act_kind, float limit) {
    if (act_kind == MOE_ACT_SILU) return (gate / (1.0f + expf(-gate))) * up;
    gate = fminf(gate, limit);
    up = fminf(fmaxf(up, -limit), limit);
    return (gate / (1.0f + expf(-1.702f * gate))) * (up + 1.0f);
}
static inline bool moe_act_ok(int act_kind, int gated) {
    return act_kind == MOE_ACT_SILU || act_kind == (gated ? MOE_ACT_CLAMPED : MOE_ACT_RELU2);
}
// what a product without a gate leaves of a sum (`rounded`: the activations' type is bfloat16, which
// the product takes before the activation, as a product of its own would leave it)
__device__ __forceinline__ float moe_plain_act(float v, int act_kind, bool rounded) {
    if (act_kind != MOE_ACT_RELU2) return v;
    v = fmaxf(rounded ? bf16_to_f32(f32_to_bf16(v)) : v, 0.f);
    return v * v;
}

// One wave per token: s = the scores of all NE outputs (float32), choice score = s + correction,
// the `top` largest choice scores (lowest index on ties) in falling order; weights are scale * s.
// `groups` > 0: the outputs are that many equal groups of neighbours, of which only the `keep` with the
// largest sums of their two largest choice scores (lowest index on ties) can be chosen from.
// EPL: outputs a lane holds, 1 for up to 64 (the exponentials of seven that are not there: 64 outputs, 6 chosen, 8 tokens
// 5.2 -> 4.6 us, 2,964 6.7 -> 5.5), else MOE_EPL.
#define MOE_EPL 8                                   // up to 512 experts
template <int EPL>
__device__ __forceinline__ void
moe_route_row(const float* zr, const void* __restrict__ corr, int corr_dt, int NE, int top,
              int32_t* __restrict__ idx_row, float* __restrict__ wt_row, int32_t* idx_copy,
              int score_kind, float scale, int groups, int keep) {
    __shared__ float choice[64 * EPL], group_score[64 * EPL];
    const int lane = threadIdx.x & 63;
    float s[EPL], c[EPL];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const int e = lane + 64 * i;
        s[i] = e < NE ? zr[e] : -INFINITY;
        mx = fmaxf(mx, s[i]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        s[i] = lane + 64 * i < NE ? expf(s[i] - mx) : 0.f;
        sum += s[i];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const int e = lane + 64 * i;
        // softmax over all outputs, or every output's own sigmoid
        s[i] = score_kind == MOE_SCORE_SIGMOID ? (e < NE ? 1.0f / (1.0f + expf(-zr[e])) : 0.f) : s[i] / sum;
        c[i] = e < NE ? s[i] + (corr ? ld_f(corr, corr_dt, e) : 0.f) : -INFINITY;
    }
    if (groups > 0) {                                  // (the block is this one wave)
        const int size = NE / groups;
#pragma unroll
        for (int i = 0; i < EPL; ++i)
            if (lane + 64 * i < NE) choice[lane + 64 * i] = c[i];
        __syncthreads();
        for (int g = lane; g < groups; g += 64) {
            float a = -INFINITY, b = -INFINITY;        // the two largest
            for (int j = 0; j < size; ++j) {
                const float v = choice[g * size + j];
                if (v > a) { b = a; a = v; }
                else if (v > b) b = v;
            }
            group_score[g] = size > 1 ? a + b : a;
        }
        __syncthreads();
        for (int g = lane; g < groups; g += 64) {
            const float mine = group_score[g];
            int before = 0;
            for (int j = 0; j < groups; ++j)
                if (group_score[j] > mine || (group_score[j] == mine && j < g)) ++before;
            choice[g] = before < keep ? 1.f : 0.f;     // (the choice scores have been read)
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            const int e = lane + 64 * i;
            if (e < NE && choice[e / size] == 0.f) c[i] = -INFINITY;
        }
    }
    // Up to 64 outputs, all choice scores finite: an output's place is the number of outputs ahead of it
    // (a larger score, or the same and a lower index), counted in one pass over the lanes instead of
    // `top` searches of 12 exchanges each (64 outputs, 6 chosen: 9.0 -> 4.6 us).  A search costs as much as
    // counting some 20 outputs: of 64 outputs 1 or 2 chosen take 3.8 and 4.6 us by searches, 5.5 by counting.
    if (NE <= 64 && NE <= 20 * top && groups == 0 && __all(lane >= NE || fabsf(c[0]) < INFINITY)) {
        int place = 0;
        for (int j = 0; j < NE; ++j) {
            const float o = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c[0]), j));
            place += o > c[0] || (o == c[0] && j < lane);
        }
        if (lane < NE && place < top) {
            idx_row[place] = lane;
            wt_row[place] = scale * s[0];
            if (idx_copy) idx_copy[place] = lane;
        }
        return;
    }
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int be = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            const int e = lane + 64 * i;
            if (e < NE && (c[i] > best || (c[i] == best && e < be))) { best = c[i]; be = e; }
        }
        for (int o = 32; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, 64);
            const int oe = __shfl_xor(be, o, 64);
            if (ob > best || (ob == best && oe < be)) { best = ob; be = oe; }
        }
        float w = 0.f;
#pragma unroll
        for (int i = 0; i < EPL; ++i)
            if (lane + 64 * i == be) { w = s[i]; c[i] = -INFINITY; }
        w = wave_sum(w);                               // only the owner's lane holds a value
        if (lane == 0) {
            idx_row[k] = be;
            wt_row[k] = scale * w;
            if (idx_copy) idx_copy[k] = be;
        }
    }
}

template <int EPL>
__global__ void __launch_bounds__(64)
moe_route_kernel(const float* __restrict__ z, const void* __restrict__ corr, int corr_dt, int NE,
                 int top, int32_t* __restrict__ idx, float* __restrict__ wt, int score_kind, float scale,
                 int groups, int keep) {
    const size_t t = blockIdx.x;
    moe_route_row<EPL>(z + t * NE, corr, corr_dt, NE, top, idx + t * top, wt + t * top, nullptr, score_kind, scale, groups,
                       keep);
}

static bool moe_route_args(const void* corr, int corr_dt, int T, int NE, int top, int score_kind, int groups, int keep) {
    return !(groups < 0 || (groups > 0 && (NE % groups || keep <= 0 || keep > groups || top > keep * (NE / groups)))) &&
           (score_kind == MOE_SCORE_SOFTMAX || score_kind == MOE_SCORE_SIGMOID) && T >= 0 && NE > 0 && NE <= 64 * MOE_EPL &&
           top > 0 && top <= NE && (!corr || illm_dtype_ok(corr_dt));
}

extern "C" int illm_moe_route(const float* z, const void* corr, int corr_dt, int T, int NE, int top,
                              int32_t* idx, float* wt, int score_kind, float scale, int groups, int keep,
                              void* stream) {
    if (!moe_route_args(corr, corr_dt, T, NE, top, score_kind, groups, keep)) return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    if (NE <= 64)
        hipLaunchKernelGGL(moe_route_kernel<1>, dim3(T), dim3(64), 0, (hipStream_t)stream, z, corr, corr_dt, NE, top, idx, wt,
                           score_kind, scale, groups, keep);
    else
        hipLaunchKernelGGL(moe_route_kernel<MOE_EPL>, dim3(T), dim3(64), 0, (hipStream_t)stream, z, corr, corr_dt, NE, top, idx,
                           wt, score_kind, scale, groups, keep);
    return illm_launch_status();
}

// ---------------------------------------------------------------- grouping
// One block.  order[NP]: the pairs whose expert is a real one (< NEr), grouped by expert.
// tiles[3 i ..]: (expert, first place in `order`, rows) of tile i; tiles[3 max_tiles] = number of
// tiles.  Counters live in LDS and are cleared here, so nothing needs clearing between calls.
#define MOE_MAX_EXPERTS 512
__device__ __forceinline__ void
moe_group_pairs(const int32_t* idx, int NP, int NEr, int32_t* __restrict__ order,
                int32_t* __restrict__ tiles, int max_tiles, int tile_rows) {
    __shared__ int cnt[MOE_MAX_EXPERTS], offs[MOE_MAX_EXPERTS], tile0[MOE_MAX_EXPERTS + 1];
    for (int e = threadIdx.x; e < NEr; e += blockDim.x) cnt[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < NP; p += blockDim.x) {
        const int e = idx[p];
        if (e >= 0 && e < NEr) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (threadIdx.x < 64) {                            // places and tiles before each expert: one wave, 64 a turn
        int o = 0, tl = 0;
        for (int e0 = 0; e0 < NEr; e0 += 64) {
            const int e = e0 + threadIdx.x, n = e < NEr ? cnt[e] : 0, t = (n + tile_rows - 1) / tile_rows;
            int so = n, st = t;                        // sums up to and with this lane
            for (int d = 1; d < 64; d <<= 1) {
                const int uo = __shfl_up(so, d, 64), ut = __shfl_up(st, d, 64);
                if ((int)threadIdx.x >= d) { so += uo; st += ut; }
            }
            if (e < NEr) { offs[e] = o + so - n; tile0[e] = tl + st - t; }
            o += __shfl(so, 63, 64);
            tl += __shfl(st, 63, 64);
        }
        if (threadIdx.x == 0) {
            tile0[NEr] = tl;
            tiles[3 * (size_t)max_tiles] = tl < max_tiles ? tl : max_tiles;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NEr; e += blockDim.x) {
        const int n = cnt[e];
        for (int s = 0, i = tile0[e]; s < n && i < max_tiles; s += tile_rows, ++i) {
            tiles[3 * (size_t)i] = e;
            tiles[3 * (size_t)i + 1] = offs[e] + s;
            tiles[3 * (size_t)i + 2] = n - s < tile_rows ? n - s : tile_rows;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NEr; e += blockDim.x) cnt[e] = offs[e];     // now the write cursors
    __syncthreads();
    for (int p = threadIdx.x; p < NP; p += blockDim.x) {
        const int e = idx[p];
        if (e >= 0 && e < NEr) order[atomicAdd(&cnt[e], 1)] = p;
    }
}

__global__ void __launch_bounds__(1024)
moe_group_kernel(const int32_t* __restrict__ idx, int NP, int NEr, int32_t* __restrict__ order,
                 int32_t* __restrict__ tiles, int max_tiles, int tile_rows) {
    moe_group_pairs(idx, NP, NEr, order, tiles, max_tiles, tile_rows);
}

// The choice and the grouping of up to 16 tokens in one launch, a wave a token: the pairs go from one to the other through LDS.
// us in a graph, 64 outputs, 6 chosen, two kernels / this: 1 token
// 6.4 / 5.6, 8 tokens 6.9 / 5.8, 16 tokens 7.2 / 7.1.
#define MOE_FEW_TOKENS 16
#define MOE_FEW_TOP 16
__global__ void __launch_bounds__(64 * MOE_FEW_TOKENS)
moe_route_group_kernel(const float* __restrict__ z, const void* __restrict__ corr, int corr_dt, int NE, int top, int32_t* __restrict__ idx,
                       float* __restrict__ wt, int score_kind, float scale, int T, int NEr, int32_t* __restrict__ order,
                       int32_t* __restrict__ tiles, int max_tiles, int tile_rows) {
    __shared__ int32_t chosen[MOE_FEW_TOKENS * MOE_FEW_TOP];
    const int t = wave_index();
    if (t < T)
        moe_route_row<1>(z + (size_t)t * NE, corr, corr_dt, NE, top, idx + t * top, wt + t * top, chosen + t * top, score_kind,
                         scale, 0, 0);
    __syncthreads();
    moe_group_pairs(chosen, T * top, NEr, order, tiles, max_tiles, tile_rows);
}

extern "C" int illm_moe_route_group(const float* z, const void* corr, int corr_dt, int T, int NE, int top, int32_t* idx, float* wt,
                                    int score_kind, float scale, int NEr, int32_t* order, int32_t* tiles, int max_tiles,
                                    int tile_rows, void* stream) {
    if (!moe_route_args(corr, corr_dt, T, NE, top, score_kind, 0, 0) || T < 1 || T > MOE_FEW_TOKENS || NE > 64 || top > MOE_FEW_TOP ||
        NEr < 0 || NEr > MOE_MAX_EXPERTS || max_tiles < 0 || tile_rows <= 0)
        return ILLM_ERR_ARG;
    hipLaunchKernelGGL(moe_route_group_kernel, dim3(1), dim3(64 * T), 0, (hipStream_t)stream, z, corr, corr_dt, NE, top, idx, wt,
                       score_kind, scale, T, NEr, order, tiles, max_tiles, tile_rows);
    return illm_launch_status();
}

extern "C" int illm_moe_tile_rows(void) { return MOE_TILE; }

extern "C" int illm_moe_group(const int32_t* idx, int NP, int NEr, int32_t* order, int32_t* tiles,
                              int max_tiles, int tile_rows, void* stream) {
    if (NP < 0 || NEr < 0 || NEr > MOE_MAX_EXPERTS || max_tiles < 0 || tile_rows <= 0)
        return ILLM_ERR_ARG;
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, idx, NP, NEr,
                       order, tiles, max_tiles, tile_rows);
    return illm_launch_status();
}

// ---------------------------------------------------------------- the experts' products
// grid (tiles, column groups).  X rows: pair p reads row p / x_div of X (x_div = top for the
// tokens' rows, 1 for rows that are per pair already).  GATED: W holds [gate (N) | up (N)] rows per
// expert and Y = silu(X Wg^T) * (X Wu^T); else Y = X W^T.  Y rows are per pair.  A wave takes two
// columns at a time, so that their rows of W are in flight together.
template <int DT, int V, bool GATED>
__global__ void __launch_bounds__(256)
moe_rows_kernel(const void* __restrict__ X, int x_div, const void* __restrict__ W,
                const int32_t* __restrict__ order, const int32_t* __restrict__ tiles, int max_tiles,
                void* __restrict__ Y, int N, int K, int cols_per_block, int act_kind, float limit,
                const float* __restrict__ row_w) {
    const int tile = blockIdx.x;
    if (tile >= tiles[3 * (size_t)max_tiles]) return;
    const int e = tiles[3 * (size_t)tile], first = tiles[3 * (size_t)tile + 1];
    const int n = tiles[3 * (size_t)tile + 2];
    const int w = wave_index(), lane = threadIdx.x & 63;
    int pair[MOE_TILE];
#pragma unroll
    for (int r = 0; r < MOE_TILE; ++r) pair[r] = r < n ? order[first + r] : 0;
    const size_t wrows = GATED ? 2 * (size_t)N : (size_t)N;
    const int c_end = min(N, (int)(blockIdx.y + 1) * cols_per_block);
    for (int col = blockIdx.y * cols_per_block + 2 * w; col < c_end; col += 8) {
        const bool two = col + 1 < c_end;
        const size_t wa0 = ((size_t)e * wrows + col) * K, wa1 = two ? wa0 + K : wa0;
        const size_t up = (size_t)N * K;
        float a[2][MOE_TILE], g[2][MOE_TILE];
#pragma unroll
        for (int r = 0; r < MOE_TILE; ++r) { a[0][r] = a[1][r] = 0.f; g[0][r] = g[1][r] = 0.f; }
#pragma unroll 2
        for (int k = lane * V; k < K; k += 64 * V) {
            float w0[V], w1[V], u0[V], u1[V];
            ldv<DT, V>(W, wa0 + k, w0);
            ldv<DT, V>(W, wa1 + k, w1);
            if (GATED) { ldv<DT, V>(W, wa0 + up + k, u0); ldv<DT, V>(W, wa1 + up + k, u1); }
#pragma unroll
            for (int r = 0; r < MOE_TILE; ++r) {
                if (r < n) {
                    float x[V];
                    ldv<DT, V>(X, (size_t)(pair[r] / x_div) * K + k, x);
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        a[0][r] += x[j] * w0[j];
                        a[1][r] += x[j] * w1[j];
                        if (GATED) { g[0][r] += x[j] * u0[j]; g[1][r] += x[j] * u1[j]; }
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < MOE_TILE; ++r) {
            if (r < n) {
                a[0][r] = wave_sum(a[0][r]); a[1][r] = wave_sum(a[1][r]);
                if (GATED) { g[0][r] = wave_sum(g[0][r]); g[1][r] = wave_sum(g[1][r]); }
            }
        }
        if (lane < 2 && (lane == 0 || two)) {
#pragma unroll
            for (int r = 0; r < MOE_TILE; ++r) {
                if (r < n) {
                    float v = lane ? a[1][r] : a[0][r];
                    if (GATED) {
                        // the products take the activations' type before the activation, as a
                        // product of its own would leave them
                        float gate = v, upv = lane ? g[1][r] : g[0][r];
                        if (row_w) { gate *= row_w[pair[r]]; upv *= row_w[pair[r]]; }   // W (w x) = w (W x)
                        if (DT == ILLM_BF16) { gate = bf16_to_f32(f32_to_bf16(gate)); upv = bf16_to_f32(f32_to_bf16(upv)); }
                        v = moe_act(gate, upv, act_kind, limit);
                    } else
                        v = moe_plain_act(row_w ? v * row_w[pair[r]] : v, act_kind, DT == ILLM_BF16);
                    if (DT == ILLM_BF16) ((bf16_t*)Y)[(size_t)pair[r] * N + col + lane] = f32_to_bf16(v);
                    else ((float*)Y)[(size_t)pair[r] * N + col + lane] = v;
                }
            }
        }
    }
}

extern "C" int illm_moe_rows(const void* X, int x_div, const void* W, int dt, int gated,
                             const int32_t* order, const int32_t* tiles, int max_tiles, void* Y,
                             int N, int K, int act_kind, float limit, const float* row_w,
                             void* stream) {
    if (!moe_act_ok(act_kind, gated) || x_div <= 0 || N <= 0 || K <= 0 || max_tiles < 0 || max_tiles > 2147483647 / 3 ||
        !illm_dtype_ok(dt))
        return ILLM_ERR_ARG;
    if (max_tiles == 0) return ILLM_OK;
    const int cols = 32;
    const dim3 grid(max_tiles, (N + cols - 1) / cols);
    if (grid.y > 65535) return ILLM_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
#define GO(DT_, V_, G_)                                                                          \
    hipLaunchKernelGGL((moe_rows_kernel<DT_, V_, G_>), grid, dim3(256), 0, st, X, x_div, W, order, \
                       tiles, max_tiles, Y, N, K, cols, act_kind, limit, row_w)
    if (dt == ILLM_BF16) {
        if (K % 8 == 0) { if (gated) GO(ILLM_BF16, 8, true); else GO(ILLM_BF16, 8, false); }
        else { if (gated) GO(ILLM_BF16, 1, true); else GO(ILLM_BF16, 1, false); }
    } else {
        if (K % 4 == 0) { if (gated) GO(ILLM_F32, 4, true); else GO(ILLM_F32, 4, false); }
        else { if (gated) GO(ILLM_F32, 1, true); else GO(ILLM_F32, 1, false); }
    }
#undef GO
    return illm_launch_status();
}

// The same products for tiles of up to 16 MT pairs on the matrix cores (bfloat16, K % 32 == 0):
// MFMA 16x16x32 with 16 rows of W as the A operand and 16 of the tile's X rows as the B operand,
// both read in operand order straight from memory (lane (r, q) = (lane % 16, lane / 16) holds 8
// consecutive k of row r at k0 + 8 q; the tile's X rows stay in the caches, W is read once a
// tile).  A wave takes NT groups of 16 output columns at a time and all MT row groups, so an X
// operand serves NT (gated: 2 NT) products; the sum over K runs in one fixed order, so a row's
// result does not depend on its tile.  grid (tiles, column groups of 64 NT).
typedef __bf16 moe_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float moe_f32x4_t __attribute__((ext_vector_type(4)));

template <int MT, int NT, bool GATED, bool AHEAD, int KU>
__global__ void __launch_bounds__(256)
moe_rows_mfma_kernel(const bf16_t* __restrict__ X, int x_div, const bf16_t* __restrict__ W,
                     const int32_t* __restrict__ order, const int32_t* __restrict__ tiles,
                     int max_tiles, bf16_t* __restrict__ Y, int N, int K, int act_kind, float limit,
                     const float* __restrict__ row_w) {
    const int tile = blockIdx.x;
    if (tile >= tiles[3 * (size_t)max_tiles]) return;
    const int e = tiles[3 * (size_t)tile], first = tiles[3 * (size_t)tile + 1];
    const int n = tiles[3 * (size_t)tile + 2];
    const int w = wave_index(), lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    int pair[MT];
    const bf16_t* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int i = mt * 16 + r;
        pair[mt] = order[first + (i < n ? i : n - 1)];          // rows beyond the tile: read, not written
        xp[mt] = X + (size_t)(pair[mt] / x_div) * K + q * 8;
    }
    const size_t wrows = GATED ? 2 * (size_t)N : (size_t)N;
    const int n0 = (blockIdx.y * 4 + w) * 16 * NT;
    if (n0 >= N) return;
    const bf16_t* wa[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int wr = n0 + nt * 16 + r < N ? n0 + nt * 16 + r : N - 1;
        wa[nt] = W + ((size_t)e * wrows + wr) * K + q * 8;
    }
    const size_t up = (size_t)N * K;
    moe_f32x4_t a[NT][MT], g[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            a[nt][mt] = (moe_f32x4_t){0.f, 0.f, 0.f, 0.f};
            g[nt][mt] = a[nt][mt];
        }
    if constexpr (KU > 1) {
        // few accumulators (single tokens): KU / 2 steps of 32 k at a time in two sets of registers, the
        // next set asked for before this one is multiplied
        constexpr int H = KU / 2;
        struct Set { moe_bf16x8_t w0[H][NT], w1[H][NT], x[H][MT]; };
        auto load = [&](Set& s, int k) __attribute__((always_inline)) {
            const int kc = k < K ? k : K - 32 * H;               // (past the end: not used)
#pragma unroll
            for (int u = 0; u < H; ++u) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    s.w0[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + kc + 32 * u);
                    if (GATED) s.w1[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + up + kc + 32 * u);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) s.x[u][mt] = *(const moe_bf16x8_t*)(xp[mt] + kc + 32 * u);
            }
            __builtin_amdgcn_sched_barrier(0);                   // (else a product's loads are put right before it)
        };
        auto multiply = [&](const Set& s) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < H; ++u)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        a[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.w0[u][nt], s.x[u][mt], a[nt][mt], 0, 0, 0);
                        if (GATED)
                            g[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.w1[u][nt], s.x[u][mt], g[nt][mt], 0, 0, 0);
                    }
            __builtin_amdgcn_sched_barrier(0);
        };
        Set s0, s1;
        load(s0, 0);
        for (int k = 0; k < K; k += 32 * KU) {
            load(s1, k + 32 * H);
            multiply(s0);
            load(s0, k + 64 * H);
            multiply(s1);
        }
    } else {
        // the operands of the next 32 k are asked for before this step's products are issued
        moe_bf16x8_t w0[NT], w1[NT], x[MT];
    #pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            w0[nt] = *(const moe_bf16x8_t*)(wa[nt]);
            if (GATED) w1[nt] = *(const moe_bf16x8_t*)(wa[nt] + up);
        }
    #pragma unroll
        for (int mt = 0; mt < MT; ++mt) x[mt] = *(const moe_bf16x8_t*)(xp[mt]);
        for (int k = 0; k < K; k += 32) {
            moe_bf16x8_t w0n[NT], w1n[NT], xn[MT];
            const int kn = k + 32 < K ? k + 32 : k;            // the last step loads its own again
            if (!AHEAD && k > 0) {
                // (many accumulators: no second set of operands; other waves hide the loads)
    #pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    w0[nt] = *(const moe_bf16x8_t*)(wa[nt] + k);
                    if (GATED) w1[nt] = *(const moe_bf16x8_t*)(wa[nt] + up + k);
                }
    #pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[mt] = *(const moe_bf16x8_t*)(xp[mt] + k);
            }
            if (AHEAD) {
    #pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    w0n[nt] = *(const moe_bf16x8_t*)(wa[nt] + kn);
                    if (GATED) w1n[nt] = *(const moe_bf16x8_t*)(wa[nt] + up + kn);
                }
    #pragma unroll
                for (int mt = 0; mt < MT; ++mt) xn[mt] = *(const moe_bf16x8_t*)(xp[mt] + kn);
            }
    #pragma unroll
            for (int nt = 0; nt < NT; ++nt)
    #pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    a[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[nt], x[mt], a[nt][mt], 0, 0, 0);
                    if (GATED)
                        g[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[nt], x[mt], g[nt][mt], 0, 0, 0);
                }
            if (AHEAD) {
    #pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    w0[nt] = w0n[nt];
                    if (GATED) w1[nt] = w1n[nt];
                }
    #pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[mt] = xn[mt];
            }
        }
    }
    // a[nt][mt][i] belongs to the pair of row mt * 16 + r and column n0 + 16 nt + 4 q + i
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        if (mt * 16 + r >= n) continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = n0 + 16 * nt + 4 * q + i;
                if (col >= N) continue;
                float v = a[nt][mt][i];
                if (GATED) {
                    const float rw = row_w ? row_w[pair[mt]] : 1.0f;          // W (w x) = w (W x)
                    const float gate = bf16_to_f32(f32_to_bf16(a[nt][mt][i] * rw));
                    const float upv = bf16_to_f32(f32_to_bf16(g[nt][mt][i] * rw));
                    v = moe_act(gate, upv, act_kind, limit);
                } else
                    v = moe_plain_act(row_w ? v * row_w[pair[mt]] : v, act_kind, true);
                Y[(size_t)pair[mt] * N + col] = f32_to_bf16(v);
            }
    }
}

// The value of the lane 8 further within 16.
__device__ __forceinline__ moe_bf16x8_t moe_turn8(illm_u32x4_t v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)v[i], 0x128, 0xf, 0xf, true);   // row_ror:8
    return *(const moe_bf16x8_t*)&v;
}

// The same for tiles of up to 16 pairs of few tokens, K % 64 == 0, W read in whole 128-byte lines: a load brings 64 k of 8
// rows (lanes r < 8 hold the first 32 k of row r, the others the second 32 of row r - 8), and a product of the lines as
// they are is followed by one of the lines turned by 8 lanes, so that rows 0 .. 7 of the sums take the steps of 32 k one
// after the other, as above: the same bits.  (Rows 8 .. 15 of the sums are never read.)  Bound by reading the chosen
// experts once.  A block is one (tile, group of columns), the groups of a tile one after the other: with the tile as the
// faster index its blocks all went to one of the eight XCDs wherever the number of tiles is a multiple of 8, and 30 experts
// make 3 tiles for some XCDs and 4 for others.  2,048 x 1,408, 64 experts, 6 a token, gate|up and down in us, matrices cold,
// before / now: 4 tokens 68 + 24.2 / 47.9 + 24.8, 8 tokens 75.7 + 34.2 / 69.1 + 34.1, 16 tokens 121 + 96 / 102 + 53, 24
// tokens 134 + 74 / 111 + 59 (2.8 to 5.8 TB/s).  NH: groups of 8 columns a wave takes; S: steps of 64 k a set of registers
// holds, two sets in turn.
template <int NH, bool GATED, int S>
__global__ void __launch_bounds__(256)
moe_lines_kernel(const bf16_t* __restrict__ X, int x_div, const bf16_t* __restrict__ W,
                 const int32_t* __restrict__ order, const int32_t* __restrict__ tiles, int max_tiles,
                 bf16_t* __restrict__ Y, int N, int K, int act_kind, float limit, const float* __restrict__ row_w,
                 int groups) {
    const int tile = blockIdx.x / groups, group = blockIdx.x - tile * groups;
    if (tile >= tiles[3 * (size_t)max_tiles]) return;
    const int e = tiles[3 * (size_t)tile], first = tiles[3 * (size_t)tile + 1], n = tiles[3 * (size_t)tile + 2];
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int n0 = (group * 4 + wave_index()) * 8 * NH;
    if (n0 >= N) return;
    constexpr int NW = GATED ? 2 * NH : NH;                           // (gate rows, then up rows)
    const size_t wrows = GATED ? 2 * (size_t)N : (size_t)N;
    const illm_u32x4_t* wp[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int row = min(n0 + (i % NH) * 8 + (r & 7), N - 1) + (i / NH) * N;
        wp[i] = (const illm_u32x4_t*)(W + ((size_t)e * wrows + row) * K + (q + 4 * (r >> 3)) * 8);
    }
    const int pair = order[first + min(r, n - 1)];                    // rows beyond the tile: read, not written
    const illm_u32x4_t* xp = (const illm_u32x4_t*)(X + (size_t)(pair / x_div) * K + q * 8);
    moe_f32x4_t acc[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) acc[i] = (moe_f32x4_t){0.f, 0.f, 0.f, 0.f};
    struct Set { illm_u32x4_t w[S][NW], x[S][2]; };
    const int steps = K / 64;
    auto load = [&](Set& s, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int at = min(k + u, steps - 1) * 8;                 // (past the end: not used)
#pragma unroll
            for (int i = 0; i < NW; ++i) s.w[u][i] = __builtin_nontemporal_load(wp[i] + at);
            s.x[u][0] = xp[at];
            s.x[u][1] = xp[at + 4];
        }
        __builtin_amdgcn_sched_barrier(0);                            // (else a product's loads are put right before it)
    };
    auto multiply = [&](const Set& s, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            if (k + u >= steps) continue;
#pragma unroll
            for (int i = 0; i < NW; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const moe_bf16x8_t*)&s.w[u][i], *(const moe_bf16x8_t*)&s.x[u][0],
                                                                 acc[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NW; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(moe_turn8(s.w[u][i]), *(const moe_bf16x8_t*)&s.x[u][1], acc[i], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    Set s0, s1;
    load(s0, 0);
    for (int k = 0; k < steps; k += 2 * S) {
        load(s1, k + S);
        multiply(s0, k);
        load(s0, k + 2 * S);
        multiply(s1, k + S);
    }
    // acc[h][i] belongs to the pair of row r and column n0 + 8 h + 4 q + i
    if (r >= n || q >= 2) return;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = n0 + 8 * h + 4 * q + i;
            if (col >= N) continue;
            float v = acc[h][i];
            if (GATED) {
                const float rw = row_w ? row_w[pair] : 1.0f;          // W (w x) = w (W x)
                const float gate = bf16_to_f32(f32_to_bf16(v * rw));
                const float upv = bf16_to_f32(f32_to_bf16(acc[(GATED ? NH : 0) + h][i] * rw));
                v = moe_act(gate, upv, act_kind, limit);
            } else
                v = moe_plain_act(row_w ? v * row_w[pair] : v, act_kind, true);
            Y[(size_t)pair * N + col] = f32_to_bf16(v);
        }
}

// Tiles of 64 pairs (prompts), K % 64 == 0: as above with the tile's X rows shared by the block's
// four waves through LDS, 64 k at a time in two buffers (a thread brings 32 bytes of one row; the
// 16-byte pieces of a row are placed at piece ^ (row % 8), so that the 16 rows a product's operand
// reads lie in different banks); one barrier a slab.  W stays a stream of each wave's own rows,
// asked for one slab ahead.
template <int NT, bool GATED>
__global__ void __launch_bounds__(256)
moe_rows_mfma_lds_kernel(const bf16_t* __restrict__ X, int x_div, const bf16_t* __restrict__ W,
                         const int32_t* __restrict__ order, const int32_t* __restrict__ tiles,
                         int max_tiles, bf16_t* __restrict__ Y, int N, int K, int act_kind,
                         float limit, const float* __restrict__ row_w) {
    constexpr int MT = 4;
    __shared__ uint4 xs[2][64 * 8];
    const int tile = blockIdx.x;
    if (tile >= tiles[3 * (size_t)max_tiles]) return;          // the whole block leaves together
    const int e = tiles[3 * (size_t)tile], first = tiles[3 * (size_t)tile + 1];
    const int n = tiles[3 * (size_t)tile + 2];
    const int w = wave_index(), lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int lr = threadIdx.x >> 2, lc = (threadIdx.x & 3) * 2;       // the row and pieces this thread brings
    const bf16_t* lx = X + (size_t)(order[first + (lr < n ? lr : n - 1)] / x_div) * K + lc * 8;
    const int s0 = lr * 8 + (lc ^ (lr & 7)), s1 = lr * 8 + ((lc + 1) ^ (lr & 7));
    int pair[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int i = mt * 16 + r;
        pair[mt] = order[first + (i < n ? i : n - 1)];
    }
    const size_t wrows = GATED ? 2 * (size_t)N : (size_t)N;
    const int n0 = (blockIdx.y * 4 + w) * 16 * NT;             // (a wave beyond N works on row N - 1 and writes nothing)
    const bf16_t* wa[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int wr = n0 + nt * 16 + r < N ? n0 + nt * 16 + r : N - 1;
        wa[nt] = W + ((size_t)e * wrows + wr) * K + q * 8;
    }
    const size_t up = (size_t)N * K;
    moe_f32x4_t a[NT][MT], g[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            a[nt][mt] = (moe_f32x4_t){0.f, 0.f, 0.f, 0.f};
            g[nt][mt] = a[nt][mt];
        }
    moe_bf16x8_t w0[2][NT], w1[2][NT];
    uint4 xa = *(const uint4*)lx, xb = *(const uint4*)(lx + 8);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            w0[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + 32 * u);
            if (GATED) w1[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + up + 32 * u);
        }
    xs[0][s0] = xa;
    xs[0][s1] = xb;
    __syncthreads();
    for (int k = 0; k < K; k += 64) {
        const int buf = (k >> 6) & 1;
        const int kn = k + 64 < K ? k + 64 : k;                  // the last slab asks for itself again
        moe_bf16x8_t w0n[2][NT], w1n[2][NT];
        xa = *(const uint4*)(lx + kn);
        xb = *(const uint4*)(lx + kn + 8);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                w0n[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + kn + 32 * u);
                if (GATED) w1n[u][nt] = *(const moe_bf16x8_t*)(wa[nt] + up + kn + 32 * u);
            }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            moe_bf16x8_t x[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const uint4 v = xs[buf][(mt * 16 + r) * 8 + ((u * 4 + q) ^ (r & 7))];
                x[mt] = *(const moe_bf16x8_t*)&v;
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    a[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[u][nt], x[mt], a[nt][mt], 0, 0, 0);
                    if (GATED)
                        g[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[u][nt], x[mt], g[nt][mt], 0, 0, 0);
                }
        }
        xs[buf ^ 1][s0] = xa;
        xs[buf ^ 1][s1] = xb;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                w0[u][nt] = w0n[u][nt];
                if (GATED) w1[u][nt] = w1n[u][nt];
            }
        __syncthreads();
    }
    if (n0 >= N) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        if (mt * 16 + r >= n) continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = n0 + 16 * nt + 4 * q + i;
                if (col >= N) continue;
                float v = a[nt][mt][i];
                if (GATED) {
                    const float rw = row_w ? row_w[pair[mt]] : 1.0f;          // W (w x) = w (W x)
                    const float gate = bf16_to_f32(f32_to_bf16(a[nt][mt][i] * rw));
                    const float upv = bf16_to_f32(f32_to_bf16(g[nt][mt][i] * rw));
                    v = moe_act(gate, upv, act_kind, limit);
                } else
                    v = moe_plain_act(row_w ? v * row_w[pair[mt]] : v, act_kind, true);
                Y[(size_t)pair[mt] * N + col] = f32_to_bf16(v);
            }
    }
}

// Tiles of up to 128 or 192 pairs (from 3 to 24 pairs an expert on), K % 64 == 0, N % 4 == 0 (192: N % 8): the loop of
// gemm_turns.h over a tile's pairs, X's rows gathered by the loads, and 64 NT rows of W (gated: half of them gate rows, half
// the up rows of the same columns).  X and an expert's W each within the 4 GiB that a load's 32-bit offset reaches; X, W
// and Y on 16-byte addresses.  Block ids go round the 8 XCDs: an XCD takes a stretch of the (tile, columns) there are, the
// columns of a tile one after the other, so that a tile's rows of X and, through an expert's tiles, its rows of W are read
// into that L2 once.
// A loop of two stages with one barrier each, both drained (four waves, tiles of 128 pairs by 128 rows of W, two blocks a
// compute unit) -> this one; 64 experts of 1408 x 2048, 6 chosen, gate|up + down in us: 2,964 tokens 406 + 208 -> 289 + 149
// (of the rows of 192 a third are padding), 1,000 tokens 199 + 97 -> 167 + 95, 64 tokens 174 + 73 -> 139 + 70
// (bound by reading the experts); 8 experts of 8192 x 4096, 1,024 tokens, 2 chosen 478 + 285 -> 425 + 174.  A group of waves without
// pairs in an expert's last tile leaves its products out: 2,964 tokens, both products 456 -> 434, 8 of 8192 x 4096 1,421 -> 1,282.
template <int MT0, int MT1, int NTH, bool GATED>
__global__ void __launch_bounds__(512, 2)
moe_turns_kernel(const bf16_t* __restrict__ X, int x_div, const bf16_t* __restrict__ W,
                 const int32_t* __restrict__ order, const int32_t* __restrict__ tiles, int max_tiles,
                 bf16_t* __restrict__ Y, int N, int K, int act_kind, float limit, const float* __restrict__ row_w) {
    using T = Turns<MT0, MT1, NTH, NTH>;
    constexpr int COLS = GATED ? T::BN / 2 : T::BN;
    __shared__ illm_u32x4_t x0a[T::UX0], x1a[T::UX1], w0a[T::UW0], w1a[T::UW1];
    __shared__ illm_u32x4_t x0b[T::UX0], x1b[T::UX1], w0b[T::UW0], w1b[T::UW1];
    const int cols = (N + COLS - 1) / COLS, total = tiles[3 * (size_t)max_tiles] * cols;
    if ((int)blockIdx.x >= total) return;                      // the whole block leaves together
    const int xcd = blockIdx.x & 7, at = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
    const int tile = at / cols, n0 = (at - tile * cols) * COLS;
    const int e = tiles[3 * (size_t)tile], first = tiles[3 * (size_t)tile + 1], n = tiles[3 * (size_t)tile + 2];
    T t;
    t.begin();
    const uint32_t K2 = (uint32_t)K * 2u;
    const size_t wrows = GATED ? 2 * (size_t)N : (size_t)N;
    struct Loads {
        const T& t;
        __amdgpu_buffer_rsrc_t rx, rw;
        uint32_t ox0[T::CX0], ox1[T::CX1], ow0[T::CW0], ow1[T::CW1], at, last;     // at: byte offset of stage s + 2
        __device__ __forceinline__ void x1(illm_u32x4_t* to) const { t.load(to, rx, ox1, min(at - 128, last)); }
        __device__ __forceinline__ void w0(illm_u32x4_t* to) const { t.load(to, rw, ow0, min(at, last)); }
        __device__ __forceinline__ void x0(illm_u32x4_t* to) const { t.load(to, rx, ox0, min(at, last)); }
        __device__ __forceinline__ void w1(illm_u32x4_t* to) { t.load(to, rw, ow1, min(at, last)); at += 128; }
    } ld = {t, illm_buffer(X, 0xffffffffu), illm_buffer(W + (size_t)e * wrows * K, wrows * K * 2), {}, {}, {}, {}, 0, K2 - 128};
    auto x_at = [&](int row) { return (uint32_t)(order[first + min(row, n - 1)] / x_div) * K2 + t.lc; };
    auto w_at = [&](typename T::WAt w, int half) {
        const int c = turns_column<NTH>(w.tile, w.row);
        return (uint32_t)(n0 + (GATED ? w.wave * NTH * 16 + c + half * N : (2 * w.wave + half) * NTH * 16 + c)) * K2 + t.lc;
    };
#pragma unroll
    for (int i = 0; i < T::CX0; ++i) ld.ox0[i] = x_at(t.template x_row<MT0>(i, 0));
#pragma unroll
    for (int i = 0; i < T::CX1; ++i) ld.ox1[i] = x_at(t.template x_row<MT1>(i, MT0 * 16));
#pragma unroll
    for (int i = 0; i < NTH; ++i) {
        ld.ow0[i] = w_at(t.template w_row<NTH>(i), 0);
        ld.ow1[i] = w_at(t.template w_row<NTH>(i), 1);
    }
    t.clear();
    ld.w0(w0a); ld.x0(x0a); ld.w1(w1a);                        // (stages past the end: the last one again, not used)
    ld.x1(x1a);
    ld.w0(w0b); ld.x0(x0b); ld.w1(w1b);
    t.start(w0a);
    const int stages = K / 64, there = n - t.wm * T::MT * 16;        // (an expert's last tile may hold few pairs)
    const bool on0 = there > 0, on1 = there > MT0 * 16;
    for (int s = 0; s < stages; s += 2) {
        t.template stage<0>(x0a, x1a, w0a, w1a, x1b, w0b, ld, on0, on1);
        if (s + 1 < stages) t.template stage<1>(x0b, x1b, w0b, w1b, x1a, w0a, ld, on0, on1);
    }
    t.end();
    // acc[i][j][v]: pair wm MT 16 + 16 j + r, the i-th tile's column turns_column(i, 4 q + v)
#pragma unroll
    for (int j = 0; j < T::MT; ++j) {
        const int row = t.wm * T::MT * 16 + 16 * j + t.r;
        if (row >= n) continue;
        const int pair = order[first + row];
        const float rw = row_w ? row_w[pair] : 1.0f;           // W (w x) = w (W x)
#pragma unroll
        for (int h = 0; h < (GATED ? 1 : 2); ++h) {
            const int col = n0 + (GATED ? t.wn : 2 * t.wn + h) * NTH * 16 + t.q * 4 * NTH;
            if (col >= N) continue;
            uint32_t o[2 * NTH];
#pragma unroll
            for (int i = 0; i < NTH; ++i) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if constexpr (GATED) {
                        const float gate = bf16_to_f32(f32_to_bf16(t.acc[i][j][u] * rw));
                        const float upv = bf16_to_f32(f32_to_bf16(t.acc[NTH + i][j][u] * rw));
                        v[u] = moe_act(gate, upv, act_kind, limit);
                    } else {
                        const float a = t.acc[h * NTH + i][j][u];
                        v[u] = moe_plain_act(row_w ? a * rw : a, act_kind, true);
                    }
                }
                o[2 * i] = pack_bf16x2(v[0], v[1]);
                o[2 * i + 1] = pack_bf16x2(v[2], v[3]);
            }
            bf16_t* const to = Y + (size_t)pair * N + col;
            if constexpr (NTH == 2) *(uint4*)to = make_uint4(o[0], o[1], o[2], o[3]);
            else *(uint2*)to = make_uint2(o[0], o[1]);
        }
    }
}

extern "C" int illm_moe_rows_mfma(const void* X, int x_div, const void* W, int gated, int tile_rows,
                                  const int32_t* order, const int32_t* tiles, int max_tiles,
                                  void* Y, int N, int K, int act_kind, float limit,
                                  const float* row_w, void* stream) {
    if (!moe_act_ok(act_kind, gated) || x_div <= 0 || N <= 0 || K <= 0 || K % 32 || max_tiles < 0 || max_tiles > 2147483647 / 3 ||
        (tile_rows != 16 && tile_rows != 32 && tile_rows != 64 && tile_rows != 128 && tile_rows != 192))
        return ILLM_ERR_ARG;
    if (max_tiles == 0) return ILLM_OK;
    hipStream_t st = (hipStream_t)stream;
    if (tile_rows == 128 || tile_rows == 192) {
        // 192 pairs by 256 rows of W, one block a compute unit; 128 by 128, two (which one: `_moe_tiling`)
        const int beyond = tile_rows == 192 ? 256 : 128;       // rows of W that a block's loads may go past the end
        if (K % 64 || N % (tile_rows == 192 ? 8 : 4) || (long long)(gated ? 2 : 1) * (N + beyond) * K * 2 >= 0xffffffffLL ||
            ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16)
            return ILLM_ERR_ARG;
        const int width = beyond / (gated ? 2 : 1);
        const long long blocks = (long long)max_tiles * ((N + width - 1) / width);
        if (blocks > 0x7fffffLL) return ILLM_ERR_ARG;
#define GO_TURNS(MT0_, MT1_, NTH_, G_)                                                             \
    hipLaunchKernelGGL((moe_turns_kernel<MT0_, MT1_, NTH_, G_>), dim3((unsigned)blocks), dim3(512), 0, st, (const bf16_t*)X, \
                       x_div, (const bf16_t*)W, order, tiles, max_tiles, (bf16_t*)Y, N, K, act_kind, limit, row_w)
        if (tile_rows == 192) { if (gated) GO_TURNS(4, 2, 2, true); else GO_TURNS(4, 2, 2, false); }
        else { if (gated) GO_TURNS(2, 2, 1, true); else GO_TURNS(2, 2, 1, false); }
#undef GO_TURNS
        return illm_launch_status();
    }
    if (tile_rows == 64 && K % 64 == 0) {
        const int nt = gated ? 2 : 4;
        const dim3 grid(max_tiles, (N + 64 * nt - 1) / (64 * nt));
        if (grid.y > 65535) return ILLM_ERR_ARG;
        if (gated)
            hipLaunchKernelGGL((moe_rows_mfma_lds_kernel<2, true>), grid, dim3(256), 0, st, (const bf16_t*)X,
                               x_div, (const bf16_t*)W, order, tiles, max_tiles, (bf16_t*)Y, N, K, act_kind, limit, row_w);
        else
            hipLaunchKernelGGL((moe_rows_mfma_lds_kernel<4, false>), grid, dim3(256), 0, st, (const bf16_t*)X,
                               x_div, (const bf16_t*)W, order, tiles, max_tiles, (bf16_t*)Y, N, K, act_kind, limit, row_w);
        return illm_launch_status();
    }
#define GO(MT_, NT_, G_, KU_)                                                                      \
    do {                                                                                           \
        const dim3 grid(max_tiles, (N + 64 * NT_ - 1) / (64 * NT_));                               \
        if (grid.y > 65535) return ILLM_ERR_ARG;                                                   \
        hipLaunchKernelGGL((moe_rows_mfma_kernel<MT_, NT_, G_, (MT_ * NT_ <= 16), KU_>), grid, dim3(256), 0, st, \
                           (const bf16_t*)X, x_div, (const bf16_t*)W, order, tiles, max_tiles,     \
                           (bf16_t*)Y, N, K, act_kind, limit, row_w);                              \
    } while (0)
    if (tile_rows == 16) {
        // W by whole lines from 8 tiles on, and where the columns alone make blocks enough (1 token with 6 of 64 experts,
        // 2,048 x 1,408: 21.5 + 10.2 us below, 25.0 + 12.5 by lines; 2 tokens 39.7 + 17.1 / 35.7 + 17.3).  The down
        // products take 16 columns a wave while that leaves waves enough (2,048 x 1,408, us with 8 / 16 columns: 8 tokens
        // 40.1 / 34.1, 16 tokens 65.5 / 53.1; 1,024 x 2,816 of 8 experts, 4 tokens 13.5 / 21.4).
        const bool wide = !gated && (long long)max_tiles * N >= 32768;
        const int groups = (N + (wide ? 63 : 31)) / (wide ? 64 : 32);
        const long long blocks = (long long)max_tiles * groups;
        if (K % 64 == 0 && (max_tiles >= 8 || (long)max_tiles * ((N + 255) / 256) >= 512) && blocks < (1 << 23)) {
#define GO_LINES(NH_, G_, S_)                                                                      \
    hipLaunchKernelGGL((moe_lines_kernel<NH_, G_, S_>), dim3((unsigned)blocks), dim3(256), 0, st, (const bf16_t*)X, x_div, \
                       (const bf16_t*)W, order, tiles, max_tiles, (bf16_t*)Y, N, K, act_kind, limit, row_w, groups)
            if (gated) GO_LINES(1, true, 2);
            else if (wide) GO_LINES(2, false, 1);
            else GO_LINES(1, false, 2);
#undef GO_LINES
        } else if ((long)max_tiles * ((N + 255) / 256) < 512) {
            // few tiles: 16 columns a wave, so that more waves share the reading
            if (K % 256 == 0) { if (gated) GO(1, 1, true, 8); else GO(1, 1, false, 8); }
            else if (K % 128 == 0) { if (gated) GO(1, 1, true, 4); else GO(1, 1, false, 4); }
            else if (K % 64 == 0) { if (gated) GO(1, 1, true, 2); else GO(1, 1, false, 2); }
            else { if (gated) GO(1, 1, true, 1); else GO(1, 1, false, 1); }
        } else { if (gated) GO(1, 4, true, 1); else GO(1, 4, false, 1); }
    }
    else if (tile_rows == 32) { if (gated) GO(2, 4, true, 1); else GO(2, 4, false, 1); }
    else { if (gated) GO(4, 2, true, 1); else GO(4, 4, false, 1); }    // wider column blocks measured slower
#undef GO
    return illm_launch_status();
}

// ---------------------------------------------------------------- weighted sum
// grid (tokens, chunks of 256 columns): out[t] = sum_k wt[t, k] * (idx[t, k] < NEr ? Y[t top + k] : h[t])
//                                         (+ sigmoid(h[t] . sg) * shared[t]), float32.
#define MOE_COMBINE_TOP 16                          // choices held in registers (more: read again)
__global__ void __launch_bounds__(256)
moe_combine_kernel(const void* __restrict__ h, int dt, const int32_t* __restrict__ idx,
                   const float* __restrict__ wt, const void* __restrict__ Y,
                   const void* __restrict__ shared, const void* __restrict__ sg, int sg_dt,
                   float* __restrict__ out, int E, int top, int NEr) {
    __shared__ float red[16];
    const size_t t = blockIdx.x;
    int ce[MOE_COMBINE_TOP];
    float cw[MOE_COMBINE_TOP];
#pragma unroll
    for (int k = 0; k < MOE_COMBINE_TOP; ++k) {
        ce[k] = k < top ? idx[t * top + k] : 0;
        cw[k] = k < top ? (wt ? wt[t * top + k] : 1.f) : 0.f;
    }
    float gate = 0.f;
    if (shared) {
        gate = 1.f;
        if (sg) {
            float d = 0.f;
            for (int i = threadIdx.x; i < E; i += blockDim.x) d += ld_f(h, dt, t * E + i) * ld_f(sg, sg_dt, i);
            d = block_sum(d, red);
            gate = 1.0f / (1.0f + expf(-d));
        }
    }
    const int i_end = min(E, (int)(blockIdx.y + 1) * 256);
    for (int i = blockIdx.y * 256 + threadIdx.x; i < i_end; i += 256) {
        const float hv = ld_f(h, dt, t * E + i);
        float acc = 0.f;
        if (top <= MOE_COMBINE_TOP) {
            float v[MOE_COMBINE_TOP];
#pragma unroll
            for (int k = 0; k < MOE_COMBINE_TOP; ++k)
                v[k] = k < top && ce[k] < NEr ? ld_f(Y, dt, (t * top + k) * E + i) : hv;
#pragma unroll
            for (int k = 0; k < MOE_COMBINE_TOP; ++k)
                if (k < top) acc += cw[k] * v[k];
        } else {
            for (int k = 0; k < top; ++k) {
                const int e = idx[t * top + k];
                acc += (wt ? wt[t * top + k] : 1.f) * (e < NEr ? ld_f(Y, dt, (t * top + k) * E + i) : hv);
            }
        }
        if (shared) acc += gate * ld_f(shared, dt, t * E + i);
        out[t * E + i] = acc;
    }
}

// The same with V neighbouring columns a thread (16-byte loads from 16-byte addresses; E % V == 0, top <= MOE_COMBINE_TOP) and a
// block a token: the gate's dot product is formed once a token, and all of a thread's rows are asked for
// together (2,964 tokens of 2,048, 6 chosen: 157 -> 25 us; 8 tokens 7.0 -> 5.0; in a graph, with the choice's test ahead of each
// load 19.0 and 3.6, without 17.3 and 2.7; of one or two choices no more are asked for than two: 2,964 tokens, one chosen, with eight
// 11.0, with two 9.1).  Up to MOE_COMBINE_FEW tokens a
// block 256 V columns of a token, each with the gate's product for itself: tokens of 7,168, 8 chosen, one block
// against several, by column first: 8 tokens 12.7, 14.4, 7.9 us; 128 tokens 37, 14.7, 9.4; 256 tokens in float32
// 49, 17.8, 22.4.
#define MOE_COMBINE_FEW 128
template <int DT, int V, int TOP>
__global__ void __launch_bounds__(256)
moe_combine_vec_kernel(const void* __restrict__ h, const int32_t* __restrict__ idx, const float* __restrict__ wt,
                       const void* __restrict__ Y, const void* __restrict__ shared, const void* __restrict__ sg,
                       int sg_dt, float* __restrict__ out, int E, int top, int NEr) {
    __shared__ float red[16];
    const size_t t = blockIdx.x;
    float gate = shared ? 1.f : 0.f;
    if (shared && sg) {
        float d = 0.f;
        for (int i = threadIdx.x * V; i < E; i += 256 * V) {
            float hv[V];
            ldv<DT, V>(h, t * E + i, hv);
#pragma unroll
            for (int j = 0; j < V; ++j) d += hv[j] * ld_f(sg, sg_dt, i + j);
        }
        d = block_sum(d, red);
        gate = 1.0f / (1.0f + expf(-d));
    }
    for (int i = (blockIdx.y * 256 + threadIdx.x) * V; i < E; i += gridDim.y * 256 * V) {
        float acc[V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = 0.f;
        // (no load behind a branch: every choice's row, or h's for one that is no expert, is on its way before the first is used)
        float r[TOP][V], w[TOP];
#pragma unroll
        for (int k = 0; k < TOP; ++k) {
            const size_t p = t * top + min(k, top - 1);
            const bool real = idx[p] < NEr;                    // the same in all lanes
            w[k] = wt ? wt[p] : 1.f;
            ldv<DT, V>(real ? Y : h, (real ? p : t) * E + i, r[k]);
        }
        float sv[V];
        if (shared) ldv<DT, V>(shared, t * E + i, sv);
#pragma unroll
        for (int k = 0; k < TOP; ++k)
            if (k < top)
#pragma unroll
                for (int j = 0; j < V; ++j) acc[j] += w[k] * r[k][j];
        if (shared) {
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += gate * sv[j];
        }
#pragma unroll
        for (int j = 0; j < V; j += 4)
            *(float4*)(out + t * E + i + j) = make_float4(acc[j], acc[j + 1], acc[j + 2], acc[j + 3]);
    }
}

extern "C" int illm_moe_combine(const void* h, int dt, const int32_t* idx, const float* wt,
                                const void* Y, const void* shared, const void* sg, int sg_dt,
                                float* out, int T, int E, int top, int NEr, void* stream) {
    if (T < 0 || E <= 0 || top <= 0 || !illm_dtype_ok(dt) || (sg && !illm_dtype_ok(sg_dt)) ||
        (E + 255) / 256 > 65535)
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    const uintptr_t at = (uintptr_t)h | (uintptr_t)Y | (uintptr_t)shared | (uintptr_t)out;
    if (top <= MOE_COMBINE_TOP && E % (dt == ILLM_BF16 ? 8 : 4) == 0 && at % 16 == 0) {
        const int V = dt == ILLM_BF16 ? 8 : 4, parts = T <= MOE_COMBINE_FEW ? (E + 256 * V - 1) / (256 * V) : 1;
#define ILLM_COMBINE(DT, V, TOP)                                                                                          \
    hipLaunchKernelGGL((moe_combine_vec_kernel<DT, V, TOP>), dim3(T, parts), dim3(256), 0, (hipStream_t)stream, h, idx, wt, Y, \
                       shared, sg, sg_dt, out, E, top, NEr)
        if (dt == ILLM_BF16) {
            if (top <= 2) ILLM_COMBINE(ILLM_BF16, 8, 2);
            else if (top <= 8) ILLM_COMBINE(ILLM_BF16, 8, 8);
            else ILLM_COMBINE(ILLM_BF16, 8, 16);
        } else if (top <= 2) ILLM_COMBINE(ILLM_F32, 4, 2);
        else if (top <= 8) ILLM_COMBINE(ILLM_F32, 4, 8);
        else ILLM_COMBINE(ILLM_F32, 4, 16);
#undef ILLM_COMBINE
        return illm_launch_status();
    }
    hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (E + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                       h, dt, idx, wt, Y, shared, sg, sg_dt, out, E, top, NEr);
    return illm_launch_status();
}
