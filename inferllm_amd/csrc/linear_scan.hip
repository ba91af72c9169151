// What stands around the plain gated recurrence (illm_gated_scan with `correct` 0,
//     S <- g S + k (beta v)^T;   o = S^T q,   S [key dim, value dim] float32 per head)
// for two mixers that keep such a state.
//
// A state-space mixer with a scalar decay a head (state-space duality):
//   ssm_prepare   short causal convolution with bias over time of the x | B | C columns of the input
//                 projection (the taps before a step's first row from the kept tail), SiLU;
//                 dt = softplus(dt + dt_bias), g = exp(-exp(A_log) dt), beta = dt; k = B, q = C of the
//                 head's group, v = x
//   ssm_finish    y = (o + D x) silu(z), RMS norm in `norm_groups` equal parts of the row, weight
//
// A matrix memory with exponential gates held in range by a running maximum m (from 0):
//   memory_rows   q dim^-1/2, k, and v with a column of ones behind it as float32 (the state's
//                 last column is then the normaliser n = sum of the weighted keys)
//   memory_gates  i = cap tanh((i + b_i) / cap), f = logsigmoid(cap tanh((f + b_f) / cap)),
//                 m_t = max(f + m_(t-1), i), g = exp(f + m_(t-1) - m_t), beta = exp(i - m_t), token
//                 after token per sequence and head, m kept per sequence
//   memory_finish o / (max(|n . q|, exp(-m)) + 1e-6), RMS norm per head, weight, sigmoid gate
//
// Everything but the stored projections is float32.  A sequence's rows in a step are consecutive.
#include <math.h>

#include "api.h"
#include "common.h"

#define SCAN_MAX_TAPS 8

__device__ __forceinline__ float ls_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float ls_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float ls_log_sigmoid(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

// ---------------------------------------------------------------- state-space mixer
// grid (rows, NB); 256 threads over the convolution's channels.  U [T, u_stride]: columns
// [x_off, x_off + C) = x (H dv) | B (G N) | C (G N) before the convolution, dt_off: H columns.
// `update_tail`: every sequence brings one row, and the thread that has read a channel's taps also
// writes its tail for the next step.
__global__ void __launch_bounds__(256)
ssm_prepare_kernel(const void* __restrict__ U, int dt, int u_stride, int x_off, int dt_off,
                   const float* __restrict__ conv_w, const float* __restrict__ conv_b, int taps,
                   void* __restrict__ tail, const int32_t* __restrict__ row_slot,
                   const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                   float* __restrict__ qn, float* __restrict__ kn, float* __restrict__ vv,
                   float* __restrict__ beta, float* __restrict__ dec, int G, int H, int N, int dv,
                   int update_tail) {
    const int r = blockIdx.x, NB = gridDim.y;
    const int inner = H * dv, GN = G * N, C = inner + 2 * GN, K = taps - 1;
    const int slot = row_slot[r];
    int before = 0;                                     // rows of this sequence ahead of r in the step, up to K
    while (before < K && r - before - 1 >= 0 && row_slot[r - before - 1] == slot) ++before;
    for (int c = blockIdx.y * 256 + threadIdx.x; c < C; c += 256 * NB) {
        float x[SCAN_MAX_TAPS], cw[SCAN_MAX_TAPS];
#pragma unroll
        for (int j = 0; j < SCAN_MAX_TAPS; ++j) {
            x[j] = cw[j] = 0.f;
            if (j < taps) {
                const int d = K - j;                    // tap j looks d tokens back
                x[j] = d <= before ? ld_f(U, dt, (size_t)(r - d) * u_stride + x_off + c)
                                   : ld_f(tail, dt, ((size_t)slot * K + (K - (d - before))) * C + c);
                cw[j] = conv_w[(size_t)c * taps + j];
            }
        }
        float a = conv_b[c];
#pragma unroll
        for (int j = 0; j < SCAN_MAX_TAPS; ++j) {
            if (j < taps) {
                a = fmaf(cw[j], x[j], a);
                if (update_tail && j > 0) st_f(tail, dt, ((size_t)slot * K + (j - 1)) * C + c, x[j]);
            }
        }
        const float y = a * ls_sigmoid(a);
        if (c < inner) vv[(size_t)r * inner + c] = y;
        else if (c < inner + GN) kn[(size_t)r * GN + (c - inner)] = y;
        else qn[(size_t)r * GN + (c - inner - GN)] = y;
    }
    for (int i = blockIdx.y * 256 + threadIdx.x; i < H; i += 256 * NB) {
        const float step = ls_softplus(ld_f(U, dt, (size_t)r * u_stride + dt_off + i) + dt_bias[i]);
        beta[(size_t)r * H + i] = step;
        dec[(size_t)r * H + i] = expf(-expf(a_log[i]) * step);
    }
}

// The same of prompts (no tails written) where four channels lie together: a thread takes four channels of `rows` rows
// one after the other, its weights in registers, every input read once (a thread a channel and row read the weights
// and the rows before again for each: 2,964 rows of 6,144 channels 209 us).  grid (ceil(T / rows), ceil(C / 1024)).  The
// taps are added in the same order: the same bits.
template <int DT, int TAPS>
__global__ void __launch_bounds__(256)
ssm_prepare_rows_kernel(const void* __restrict__ U, int u_stride, int x_off, int dt_off, const float* __restrict__ conv_w,
                        const float* __restrict__ conv_b, const void* __restrict__ tail,
                        const int32_t* __restrict__ row_slot, const float* __restrict__ a_log,
                        const float* __restrict__ dt_bias, float* __restrict__ qn, float* __restrict__ kn,
                        float* __restrict__ vv, float* __restrict__ beta, float* __restrict__ dec, int T, int G, int H,
                        int N, int dv, int rows) {
    constexpr int K = TAPS - 1;
    const int inner = H * dv, GN = G * N, C = inner + 2 * GN;
    const int r0 = blockIdx.x * rows, r1 = min(r0 + rows, T);
    const int c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (blockIdx.y == 0) {
        for (int i = threadIdx.x; i < (r1 - r0) * H; i += 256) {
            const int h = i % H;
            const size_t r = r0 + i / H;
            const float step = ls_softplus(ld_f(U, DT, r * u_stride + dt_off + h) + dt_bias[h]);
            beta[r * H + h] = step;
            dec[r * H + h] = expf(-expf(a_log[h]) * step);
        }
    }
    if (c >= C) return;
    float w[4 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) *(float4*)(w + 4 * j) = ((const float4*)(conv_w + (size_t)c * TAPS))[j];
    const float4 bias = *(const float4*)(conv_b + c);
    auto input = [&](int r) { return ld_f4(U, DT, ((size_t)r * u_stride + x_off + c) / 4); };
    float4 x[TAPS], next = input(r0);
    int had = -1;
    float* to = c < inner ? vv + c : c < inner + GN ? kn + (c - inner) : qn + (c - inner - GN);
    const size_t to_row = c < inner ? inner : GN;
    for (int r = r0; r < r1; ++r) {
        const int slot = row_slot[r];
        if (slot != had) {                              // the inputs ahead of the sequence's first row here
            int before = 0;
            while (before < K && r - before - 1 >= 0 && row_slot[r - before - 1] == slot) ++before;
#pragma unroll
            for (int j = 0; j < K; ++j) {
                const int d = K - j;                    // tap j looks d tokens back
                x[j] = d <= before ? input(r - d) : ld_f4(tail, DT, (((size_t)slot * K + (K - (d - before))) * C + c) / 4);
            }
            had = slot;
        }
        x[K] = next;
        if (r + 1 < r1) next = input(r + 1);
        float4 a = bias;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            a.x = fmaf(w[j], x[j].x, a.x);
            a.y = fmaf(w[TAPS + j], x[j].y, a.y);
            a.z = fmaf(w[2 * TAPS + j], x[j].z, a.z);
            a.w = fmaf(w[3 * TAPS + j], x[j].w, a.w);
        }
        *(float4*)(to + r * to_row) = make_float4(a.x * ls_sigmoid(a.x), a.y * ls_sigmoid(a.y), a.z * ls_sigmoid(a.z),
                                                  a.w * ls_sigmoid(a.w));
#pragma unroll
        for (int j = 0; j < K; ++j) x[j] = x[j + 1];
    }
}

extern "C" int illm_ssm_prepare(const void* U, int dt, int u_stride, int x_off, int dt_off,
                                const float* conv_w, const float* conv_b, int taps, void* tail,
                                const int32_t* row_slot, const float* a_log, const float* dt_bias,
                                float* qn, float* kn, float* vv, float* beta, float* dec, int T, int G,
                                int H, int N, int dv, int update_tail, void* stream) {
    if (T < 0 || G <= 0 || H <= 0 || H % G || N <= 0 || dv <= 0 || taps < 1 || taps > SCAN_MAX_TAPS ||
        !illm_dtype_ok(dt) || x_off < 0 || dt_off < 0 || x_off + H * dv + 2 * G * N > u_stride ||
        dt_off + H > u_stride)
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    const int C = H * dv + 2 * G * N, most = (C + 255) / 256;
    const size_t unit = dt == ILLM_BF16 ? 8 : 16;
    if (!update_tail && taps >= 2 && taps <= 4 && T > 16 && (H * dv) % 4 == 0 && (G * N) % 4 == 0 && u_stride % 4 == 0 &&
        x_off % 4 == 0 && ((uintptr_t)U | (uintptr_t)tail) % unit == 0 &&
        ((uintptr_t)conv_w | (uintptr_t)conv_b | (uintptr_t)qn | (uintptr_t)kn | (uintptr_t)vv) % 16 == 0) {
        // as many rows a thread, up to 8, as leave about 1,024 blocks
        const int by = (C + 1023) / 1024, rows = max(1, min(8, (int)((long long)T * by / 1024)));
        const dim3 grid((T + rows - 1) / rows, by);
#define ROWS(DT_, TAPS_)                                                                                              \
    hipLaunchKernelGGL((ssm_prepare_rows_kernel<DT_, TAPS_>), grid, dim3(256), 0, (hipStream_t)stream, U, u_stride, x_off, \
                       dt_off, conv_w, conv_b, tail, row_slot, a_log, dt_bias, qn, kn, vv, beta, dec, T, G, H, N, dv, rows)
        if (dt == ILLM_BF16) {
            if (taps == 4) ROWS(ILLM_BF16, 4); else if (taps == 3) ROWS(ILLM_BF16, 3); else ROWS(ILLM_BF16, 2);
        } else {
            if (taps == 4) ROWS(ILLM_F32, 4); else if (taps == 3) ROWS(ILLM_F32, 3); else ROWS(ILLM_F32, 2);
        }
#undef ROWS
        return illm_launch_status();
    }
    int nb = T >= 2048 ? 1 : (2048 + T - 1) / T;        // enough blocks to fill the chip when the rows are few
    nb = nb > most ? most : nb;
    hipLaunchKernelGGL(ssm_prepare_kernel, dim3(T, nb), dim3(256), 0, (hipStream_t)stream, U, dt, u_stride,
                       x_off, dt_off, conv_w, conv_b, taps, tail, row_slot, a_log, dt_bias, qn, kn, vv,
                       beta, dec, G, H, N, dv, update_tail);
    return illm_launch_status();
}

// grid (rows, norm groups); 256 threads.  y_j = (o_j + D[head of j] x_j) silu(z_j) over the part's
// columns, out = y / sqrt(mean over the part of y^2 + eps) * w.  Z [T, z_stride] + z_off.
__global__ void __launch_bounds__(256)
ssm_finish_kernel(const float* __restrict__ o, const float* __restrict__ x,
                  const float* __restrict__ D, const void* __restrict__ Z, int z_dt, int z_stride,
                  int z_off, const void* __restrict__ w, int w_dt, void* __restrict__ out, int out_dt,
                  int inner, int dv, int part, float eps) {
    __shared__ float red[16];
    const size_t r = blockIdx.x;
    const int j0 = blockIdx.y * part;
    float ss = 0.f;
    for (int j = j0 + threadIdx.x; j < j0 + part; j += 256) {
        const float z = ld_f(Z, z_dt, r * z_stride + z_off + j);
        const float y = fmaf(D[j / dv], x[r * inner + j], o[r * inner + j]) * (z * ls_sigmoid(z));
        ss += y * y;
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)part + eps);
    for (int j = j0 + threadIdx.x; j < j0 + part; j += 256) {
        const float z = ld_f(Z, z_dt, r * z_stride + z_off + j);
        const float y = fmaf(D[j / dv], x[r * inner + j], o[r * inner + j]) * (z * ls_sigmoid(z));
        st_f(out, out_dt, r * inner + j, (y * inv) * ld_f(w, w_dt, j));
    }
}

// The same in one pass where four columns lie together: a thread holds up to four groups of four columns, o, x, z and w asked for
// together.  Bound by memory's bytes: 2,964 rows of 4,096 columns in 8 parts, a column at a time and everything read twice, 59 us,
// this 23.
template <int E>
__global__ void __launch_bounds__(256)
ssm_finish_vec4_kernel(const float* __restrict__ o, const float* __restrict__ x, const float* __restrict__ D,
                       const void* __restrict__ Z, int z_dt, int z_stride, int z_off, const void* __restrict__ w, int w_dt,
                       void* __restrict__ out, int out_dt, int inner, int dv, int part, float eps) {
    __shared__ float red[16];
    const size_t r = blockIdx.x;
    const int j0 = blockIdx.y * part;
    float4 ov[E], xv[E], wv[E];
    AnyRaw4 zr[E];
    float d[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int j = j0 + min(4 * (int)(threadIdx.x + blockDim.x * e), part - 4);         // (past the part: its last, not used)
        ov[e] = ((const float4*)o)[(r * inner + j) / 4];
        xv[e] = ((const float4*)x)[(r * inner + j) / 4];
        zr[e] = ld_raw4(Z, z_dt, (r * z_stride + z_off + j) / 4);
        wv[e] = ld_f4_any(w, w_dt, j / 4);
        d[e] = D[j / dv];
    }
    loads_asked_for();
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const float4 z = raw4_f(zr[e], z_dt);
        ov[e] = make_float4(fmaf(d[e], xv[e].x, ov[e].x) * (z.x * ls_sigmoid(z.x)), fmaf(d[e], xv[e].y, ov[e].y) * (z.y * ls_sigmoid(z.y)),
                            fmaf(d[e], xv[e].z, ov[e].z) * (z.z * ls_sigmoid(z.z)), fmaf(d[e], xv[e].w, ov[e].w) * (z.w * ls_sigmoid(z.w)));
        if (4 * (int)(threadIdx.x + blockDim.x * e) < part) ss += sum_sq(ov[e]);
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)part + eps);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int j = 4 * (int)(threadIdx.x + blockDim.x * e);
        if (j < part)
            st_f4(out, out_dt, (r * inner + j0 + j) / 4, make_float4((ov[e].x * inv) * wv[e].x, (ov[e].y * inv) * wv[e].y,
                                                                     (ov[e].z * inv) * wv[e].z, (ov[e].w * inv) * wv[e].w));
    }
}

extern "C" int illm_ssm_finish(const float* o, const float* x, const float* D, const void* Z, int z_dt,
                               int z_stride, int z_off, const void* w, int w_dt, void* out, int out_dt,
                               int T, int H, int dv, int norm_groups, float eps, void* stream) {
    if (T < 0 || H <= 0 || dv <= 0 || norm_groups <= 0 || norm_groups > 65535 ||
        (H * dv) % norm_groups || !illm_dtype_ok(z_dt) || !illm_dtype_ok(w_dt) || !illm_dtype_ok(out_dt) ||
        z_off < 0 || z_off + H * dv > z_stride)
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    const int part = (H * dv) / norm_groups;
    auto four = [](int dt) { return (uintptr_t)(dt == ILLM_BF16 ? 8 : 16); };
    if (part % 4 == 0 && part <= 4096 && dv % 4 == 0 && z_off % 4 == 0 && z_stride % 4 == 0 &&
        ((uintptr_t)o | (uintptr_t)x) % 16 == 0 && (uintptr_t)Z % four(z_dt) == 0 && (uintptr_t)w % four(w_dt) == 0 &&
        (uintptr_t)out % four(out_dt) == 0) {
        const int units = part / 4, threads = units >= 256 ? 256 : (units + 63) / 64 * 64, each = (units + threads - 1) / threads;
#define GO(E)                                                                                                          \
    hipLaunchKernelGGL(ssm_finish_vec4_kernel<E>, dim3(T, norm_groups), dim3(threads), 0, (hipStream_t)stream, o, x, D, Z, z_dt, \
                       z_stride, z_off, w, w_dt, out, out_dt, H * dv, dv, part, eps)
        if (each <= 1) GO(1);
        else if (each <= 2) GO(2);
        else GO(4);
#undef GO
        return illm_launch_status();
    }
    hipLaunchKernelGGL(ssm_finish_kernel, dim3(T, norm_groups), dim3(256), 0, (hipStream_t)stream, o, x, D,
                       Z, z_dt, z_stride, z_off, w, w_dt, out, out_dt, H * dv, dv, (H * dv) / norm_groups, eps);
    return illm_launch_status();
}

// ---------------------------------------------------------------- matrix memory
// The gates of sequence b and head h, one wave, 64 tokens at a time, the next ones' pre-activations on their way.  A token turns
// the maximum m into max(f + m, i); two such steps, (f, i) and then (f', i'), are the one step (f + f', max(i + f', i')), so the
// maxima of 64 tokens are a scan of six exchanges (one token after the other as scalars: 2,048 tokens of 16 heads of 128 129 us with the
// rows' conversion beside it, now 42; 8 sequences of 61 to 1,024 68 -> 27).
template <int DT>
static __device__ __forceinline__ void
memory_gates(int b, int h, const void* __restrict__ U, int u_stride, int i_off, int f_off,
                    const float* __restrict__ i_bias, const float* __restrict__ f_bias, float cap,
                    float* __restrict__ m_state, const int32_t* __restrict__ cu,
                    const int32_t* __restrict__ seq_slot, float* __restrict__ beta,
                    float* __restrict__ dec, float* __restrict__ em, int H) {
    const int lane = threadIdx.x & 63;
    const int r0 = cu[b], n = cu[b + 1] - r0;
    if (n <= 0) return;
    const int slot = seq_slot[b];
    const float bi = i_bias[h], bf = f_bias[h], inv_cap = 1.0f / cap;
    float m = m_state[(size_t)slot * H + h];
    auto row_of = [&](int t0) { return (size_t)(r0 + min(t0 + lane, n - 1)); };
    float iu = ld_f(U, DT, row_of(0) * u_stride + i_off + h), fu = ld_f(U, DT, row_of(0) * u_stride + f_off + h);
    for (int t0 = 0; t0 < n; t0 += 64) {
        const bool ok = t0 + lane < n;
        const float ig = ok ? cap * tanhf((iu + bi) * inv_cap) : -INFINITY;
        const float fg = ok ? ls_log_sigmoid(cap * tanhf((fu + bf) * inv_cap)) : 0.f;
        if (t0 + 64 < n) {
            iu = ld_f(U, DT, row_of(t0 + 64) * u_stride + i_off + h);
            fu = ld_f(U, DT, row_of(t0 + 64) * u_stride + f_off + h);
        }
        float F = fg, I = ig;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const float fp = __shfl_up(F, d, ILLM_WAVE), ip = __shfl_up(I, d, ILLM_WAVE);
            if (lane >= d) {
                I = fmaxf(ip + F, I);
                F = fp + F;
            }
        }
        const float m_mine = fmaxf(F + m, I), left = __shfl_up(m_mine, 1, ILLM_WAVE), m_before = lane ? left : m;
        m = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m_mine), 63));      // (past the last token: its maximum)
        if (ok) {
            const size_t row = row_of(t0);
            dec[row * H + h] = expf(fg + m_before - m_mine);
            beta[row * H + h] = expf(ig - m_mine);
            em[row * H + h] = expf(-m_mine);
        }
    }
    if (lane == 0) m_state[(size_t)slot * H + h] = m;
}

// grid (gate blocks + rows, ceil(max(H dk, H (dv + 1)) / 256)); 256 threads, an entry of q, k and v each (a block a row, which
// went through them one after another, took 9.3 us for 8 rows of 2,048, this 4.7).  The first blocks of the grid's first row
// take four (sequence, head) pairs' gates each, which need nothing of the rest: as a kernel behind the
// rows -> beside them, 16 heads of 128 x 128, 1 / 8 / 64 single tokens 5.0 / 4.6 / 5.1 -> 3.7 / 4.0 / 3.6 us.
// U [T, u_stride] = [q (H dk) | k (H dk) | v (H dv) | ...].
template <int DT>
__global__ void __launch_bounds__(256)
memory_prepare_kernel(const void* __restrict__ U, int u_stride, float* __restrict__ qn,
                      float* __restrict__ kn, float* __restrict__ vv, int H, int dk, int dv, float qscale, int gate_blocks,
                      int n_seqs, int i_off, int f_off, const float* __restrict__ i_bias, const float* __restrict__ f_bias,
                      float cap, float* __restrict__ m_state, const int32_t* __restrict__ cu,
                      const int32_t* __restrict__ seq_slot, float* __restrict__ beta, float* __restrict__ dec,
                      float* __restrict__ em) {
    if ((int)blockIdx.x < gate_blocks) {
        const int unit = blockIdx.x * 4 + wave_index();
        if (blockIdx.y == 0 && unit < n_seqs * H)
            memory_gates<DT>(unit / H, unit % H, U, u_stride, i_off, f_off, i_bias, f_bias, cap, m_state, cu, seq_slot, beta,
                             dec, em, H);
        return;
    }
    const size_t r = blockIdx.x - gate_blocks;
    const int nq = H * dk, nv = H * (dv + 1), i = blockIdx.y * 256 + threadIdx.x;
    const int h = i / (dv + 1), j = i - h * (dv + 1);
    float q = 0.f, k = 0.f, v = 1.0f;
    if (i < nq) {
        q = ld_f(U, DT, r * u_stride + i);
        k = ld_f(U, DT, r * u_stride + nq + i);
    }
    if (i < nv && j < dv) v = ld_f(U, DT, r * u_stride + 2 * nq + h * dv + j);
    if (i < nq) {
        qn[r * nq + i] = q * qscale;
        kn[r * nq + i] = k;
    }
    if (i < nv) vv[r * nv + i] = v;
}

extern "C" int illm_memory_prepare(const void* U, int dt, int u_stride, int i_off, int f_off,
                                   const float* i_bias, const float* f_bias, float cap, float* m_state,
                                   const int32_t* cu, const int32_t* seq_slot, float* qn, float* kn,
                                   float* vv, float* beta, float* dec, float* em, int T, int n_seqs,
                                   int H, int dk, int dv, void* stream) {
    if (T < 0 || n_seqs < 0 || n_seqs > 65535 || H <= 0 || H > 65535 || dk <= 0 || dv <= 0 ||
        !illm_dtype_ok(dt) || !(cap > 0.f) || 2 * H * dk + H * dv > u_stride || i_off < 0 || f_off < 0 ||
        i_off + H > u_stride || f_off + H > u_stride)
        return ILLM_ERR_ARG;
    if (T == 0 || n_seqs == 0) return ILLM_OK;
    const int widest = H * dk > H * (dv + 1) ? H * dk : H * (dv + 1);
    if ((widest + 255) / 256 > 65535) return ILLM_ERR_ARG;
    const long long gate_blocks = ((long long)n_seqs * H + 3) / 4;
    if (gate_blocks * 4 > 0x7fffffff || gate_blocks + T > 0x7fffffff) return ILLM_ERR_ARG;
    const dim3 grid((unsigned)(gate_blocks + T), (widest + 255) / 256);
#define ILLM_MEMORY_PREPARE(DT)                                                                                     \
    hipLaunchKernelGGL(memory_prepare_kernel<DT>, grid, dim3(256), 0, (hipStream_t)stream, U, u_stride, qn, kn, vv, H, dk, dv, \
                       1.0f / sqrtf((float)dk), (int)gate_blocks, n_seqs, i_off, f_off, i_bias, f_bias, cap, m_state, cu, \
                       seq_slot, beta, dec, em)
    if (dt == ILLM_BF16) ILLM_MEMORY_PREPARE(ILLM_BF16);
    else ILLM_MEMORY_PREPARE(ILLM_F32);
#undef ILLM_MEMORY_PREPARE
    return illm_launch_status();
}

// grid (rows, ceil(H / 4)); a wave a head.  o [T, H, dv + 1]: the last column is n . q.
//   y_j = o_j / (max(|n . q|, exp(-m)) + 1e-6);  out = y / sqrt(mean_j y^2 + eps) * w[h dv + j] * sigmoid(z)
// Heads of up to 64 CS columns (CS 0: any) in one pass, a lane's columns, z and w asked for together: 2,964 rows of 16 heads of
// 128, a block a head and everything read when it is needed 25 us, this 21.
template <int CS>
__global__ void __launch_bounds__(256)
memory_finish_kernel(const float* __restrict__ o, const float* __restrict__ em,
                     const void* __restrict__ w, int w_dt, const void* __restrict__ Z, int z_dt,
                     int z_stride, int z_off, void* __restrict__ out, int out_dt, int H, int dv, float eps) {
    const size_t r = blockIdx.x;
    const int h = blockIdx.y * 4 + wave_index(), lane = threadIdx.x & 63;
    if (h >= H) return;
    const float* op = o + (r * H + h) * (dv + 1);
    const size_t z0 = r * z_stride + z_off + (size_t)h * dv;
    const float nq = op[dv], e0 = em[r * H + h];
    if constexpr (CS > 0) {
        float y[CS], z[CS], wt[CS];
#pragma unroll
        for (int c = 0; c < CS; ++c) {
            const int j = min(lane + 64 * c, dv - 1);
            y[c] = op[j];
            z[c] = ld_f(Z, z_dt, z0 + j);
            wt[c] = ld_f(w, w_dt, (size_t)h * dv + j);
        }
        const float den = fmaxf(fabsf(nq), e0) + 1e-6f;
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < CS; ++c) {
            y[c] /= den;
            if (lane + 64 * c < dv) ss += y[c] * y[c];
        }
        const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
        for (int c = 0; c < CS; ++c)
            if (lane + 64 * c < dv)
                st_f(out, out_dt, (r * H + h) * dv + lane + 64 * c, (y[c] * inv) * wt[c] * ls_sigmoid(z[c]));
        return;
    }
    const float den = fmaxf(fabsf(nq), e0) + 1e-6f;
    float ss = 0.f;
    for (int j = lane; j < dv; j += 64) {
        const float y = op[j] / den;
        ss += y * y;
    }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)dv + eps);
    for (int j = lane; j < dv; j += 64)
        st_f(out, out_dt, (r * H + h) * dv + j,
             ((op[j] / den) * inv) * ld_f(w, w_dt, (size_t)h * dv + j) * ls_sigmoid(ld_f(Z, z_dt, z0 + j)));
}

extern "C" int illm_memory_finish(const float* o, const float* em, const void* w, int w_dt, const void* Z,
                                  int z_dt, int z_stride, int z_off, void* out, int out_dt, int T, int H,
                                  int dv, float eps, void* stream) {
    if (T < 0 || H <= 0 || H > 65535 || dv <= 0 || !illm_dtype_ok(w_dt) || !illm_dtype_ok(z_dt) ||
        !illm_dtype_ok(out_dt) || z_off < 0 || z_off + H * dv > z_stride)
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
#define GO(CS)                                                                                                         \
    hipLaunchKernelGGL(memory_finish_kernel<CS>, dim3(T, (H + 3) / 4), dim3(256), 0, (hipStream_t)stream, o, em, w, w_dt, Z, \
                       z_dt, z_stride, z_off, out, out_dt, H, dv, eps)
    if (dv <= 64) GO(1);
    else if (dv <= 128) GO(2);
    else if (dv <= 256) GO(4);
    else GO(0);
#undef GO
    return illm_launch_status();
}

// ---------------------------------------------------------------- gated linear attention
// The plain gated rule with a decay per key channel: from the projections U [T, u_stride] (q at
// q_off, k at k_off, both H dk wide, v at v_off, H dv wide) and the decays' pre-activations
// Z [T, z_stride] (H dk wide) with their bias zb:
//   q dk^-1/2, k, v as float32; decay = sigmoid(Z + zb)^(1 / tau) = exp(logsigmoid(Z + zb) / tau);
//   the token's weight is 1.
// grid (rows); 256 threads.
__global__ void __launch_bounds__(256)
gla_prepare_kernel(const void* __restrict__ U, int dt, int u_stride, int q_off, int k_off, int v_off,
                   const void* __restrict__ Z, int z_dt, int z_stride, const float* __restrict__ zb,
                   float inv_tau, float* __restrict__ qn, float* __restrict__ kn,
                   float* __restrict__ vv, float* __restrict__ beta, float* __restrict__ dec, int H,
                   int dk, int dv) {
    const size_t t = blockIdx.x;
    const float qs = 1.0f / sqrtf((float)dk);
    for (int e = threadIdx.x; e < H * dk; e += 256) {
        qn[t * H * dk + e] = ld_f(U, dt, t * u_stride + q_off + e) * qs;
        kn[t * H * dk + e] = ld_f(U, dt, t * u_stride + k_off + e);
        dec[t * H * dk + e] = expf(ls_log_sigmoid(ld_f(Z, z_dt, t * z_stride + e) + zb[e]) * inv_tau);
    }
    for (int e = threadIdx.x; e < H * dv; e += 256) vv[t * H * dv + e] = ld_f(U, dt, t * u_stride + v_off + e);
    for (int e = threadIdx.x; e < H; e += 256) beta[t * H + e] = 1.0f;
}

// The same four columns a thread where offsets, strides and widths are multiples of 4: grid
// (rows, ceil(max(H dk, H dv) / 1024)).  A block a row, a column at a time, took 11.2 us for 8 rows of
// 2,048, this 4.8; 2,964 rows 26 and 18.
__global__ void __launch_bounds__(256)
gla_prepare_vec4_kernel(const void* __restrict__ U, int dt, int u_stride, int q_off, int k_off, int v_off,
                        const void* __restrict__ Z, int z_dt, int z_stride, const float* __restrict__ zb,
                        float inv_tau, float* __restrict__ qn, float* __restrict__ kn, float* __restrict__ vv,
                        float* __restrict__ beta, float* __restrict__ dec, int H, int dk, int dv) {
    const size_t t = blockIdx.x;
    const int g = blockIdx.y * 256 + threadIdx.x, nk4 = H * dk / 4, nv4 = H * dv / 4;
    const float qs = 1.0f / sqrtf((float)dk);
    const int gk = g < nk4 ? g : 0, gv = g < nv4 ? g : 0;
    const float4 q = ld_f4_any(U, dt, (t * u_stride + q_off) / 4 + gk), k = ld_f4_any(U, dt, (t * u_stride + k_off) / 4 + gk);
    const float4 z = ld_f4_any(Z, z_dt, t * z_stride / 4 + gk), b = ((const float4*)zb)[gk];
    const float4 v = ld_f4_any(U, dt, (t * u_stride + v_off) / 4 + gv);
    loads_asked_for();
    if (g < nk4) {
        ((float4*)qn)[t * nk4 + g] = make_float4(q.x * qs, q.y * qs, q.z * qs, q.w * qs);
        ((float4*)kn)[t * nk4 + g] = k;
        ((float4*)dec)[t * nk4 + g] = make_float4(
            expf(ls_log_sigmoid(z.x + b.x) * inv_tau), expf(ls_log_sigmoid(z.y + b.y) * inv_tau),
            expf(ls_log_sigmoid(z.z + b.z) * inv_tau), expf(ls_log_sigmoid(z.w + b.w) * inv_tau));
    }
    if (g < nv4) ((float4*)vv)[t * nv4 + g] = v;
    if (g < H) beta[t * H + g] = 1.0f;
}

extern "C" int illm_gla_prepare(const void* U, int dt, int u_stride, int q_off, int k_off, int v_off,
                                const void* Z, int z_dt, int z_stride, const float* zb, float tau,
                                float* qn, float* kn, float* vv, float* beta, float* dec, int T, int H,
                                int dk, int dv, void* stream) {
    if (T < 0 || H <= 0 || dk <= 0 || dv <= 0 || !illm_dtype_ok(dt) || !illm_dtype_ok(z_dt) || !(tau > 0.f) ||
        q_off < 0 || k_off < 0 || v_off < 0 || q_off + H * dk > u_stride || k_off + H * dk > u_stride ||
        v_off + H * dv > u_stride || H * dk > z_stride)
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    const int widest = H * dk > H * dv ? H * dk : H * dv;
    // Rows of at most 256 columns are one turn of a block's threads a column each: 4 heads of 64 take 3.0 us that way
    // and 3.4 by groups of four.  (dv >= 4: a row's H weights are within its groups of four.)
    if (widest > 256 && ((H * dk) | (H * dv) | q_off | k_off | v_off | u_stride | z_stride) % 4 == 0 && widest / 4 >= H &&
        (widest / 4 + 255) / 256 <= 65535 &&
        ((uintptr_t)U | (uintptr_t)Z | (uintptr_t)zb | (uintptr_t)qn | (uintptr_t)kn | (uintptr_t)vv | (uintptr_t)dec) % 16 == 0) {
        hipLaunchKernelGGL(gla_prepare_vec4_kernel, dim3(T, (widest / 4 + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           U, dt, u_stride, q_off, k_off, v_off, Z, z_dt, z_stride, zb, 1.0f / tau, qn, kn, vv, beta,
                           dec, H, dk, dv);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(gla_prepare_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, U, dt, u_stride,
                       q_off, k_off, v_off, Z, z_dt, z_stride, zb, 1.0f / tau, qn, kn, vv, beta, dec, H, dk, dv);
    return illm_launch_status();
}

// ---------------------------------------------------------------- a gated linear recurrent unit
// Per channel c of `C`, in `nb` equal blocks of cb channels: with u the recurrence's input,
//   r = sigmoid(Wr[b] u_b + br),  i = sigmoid(Wi[b] u_b + bi)        (square maps within a block)
//   a = exp(-rate r softplus(lam)),  x = sqrt(1 - a^2) i u
//   S <- a S + x,   out = S gelu_tanh(Y + yb)
// lru_gates gives a and x; lru_scan runs the recurrence from the kept state [slots][C] and back
// into it and multiplies by the other branch.  All float32 but the stored Y and the output.
//
// grid (ceil(T / ROWS), nb); 256 threads over a block's outputs; the rows' inputs go through LDS, laid
// out [input][row] so that a thread reads one input of all its rows in 16-byte pieces.  Steps of few
// rows take tiles of 4 rows (more blocks), longer ones tiles of 16.  Wt [2][nb][cb in][cb out] float32:
// the two maps transposed, so that the threads of a wave read neighbouring outputs of one input.
template <int ROWS>
__global__ void __launch_bounds__(256)
lru_gates_kernel(const float* __restrict__ u, const float* __restrict__ Wt, const float* __restrict__ br,
                 const float* __restrict__ bi, const float* __restrict__ lam, float rate,
                 float* __restrict__ a_out, float* __restrict__ x_out, int T, int C, int cb) {
    extern __shared__ __attribute__((aligned(16))) float us[];                   // [cb][ROWS], then the slices' partial sums
    const int t0 = blockIdx.x * ROWS, b = blockIdx.y, nb = C / cb;
    const int rows = min(ROWS, T - t0);
    for (int e = threadIdx.x; e < ROWS * cb; e += 256) {
        const int r = e / cb, i = e - r * cb;
        us[i * ROWS + r] = r < rows ? u[(size_t)(t0 + r) * C + (size_t)b * cb + i] : 0.f;
    }
    __syncthreads();
    const float* wr = Wt + (size_t)b * cb * cb;
    const float* wi = Wt + ((size_t)nb + b) * cb * cb;
    // a block narrower than the thread block cuts its inputs into S slices, one a group of cb
    // threads, whose sums are added in slice order
    const int S = cb < 256 ? 256 / cb : 1;
    const int per = (cb + S - 1) / S;
    float* part = us + (size_t)cb * ROWS;           // [S][cb][2 ROWS]
    for (int o0 = 0; o0 < cb; o0 += 256) {
        const int o = S > 1 ? (int)threadIdx.x % cb : o0 + (int)threadIdx.x;
        const int sl = S > 1 ? (int)threadIdx.x / cb : 0;
        const bool live = o < cb && sl < S;
        float ar[ROWS], ai[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) ar[r] = ai[r] = 0.f;
        if (live) {
            const int i_lo = sl * per, i_hi = min(cb, i_lo + per);
#pragma unroll 8
            for (int i = i_lo; i < i_hi; ++i) {
                const float w1 = wr[(size_t)i * cb + o], w2 = wi[(size_t)i * cb + o];
                const float4* xr = (const float4*)(us + i * ROWS);
#pragma unroll
                for (int r4 = 0; r4 < ROWS / 4; ++r4) {
                    const float4 x = xr[r4];
                    ar[4 * r4 + 0] = fmaf(w1, x.x, ar[4 * r4 + 0]); ai[4 * r4 + 0] = fmaf(w2, x.x, ai[4 * r4 + 0]);
                    ar[4 * r4 + 1] = fmaf(w1, x.y, ar[4 * r4 + 1]); ai[4 * r4 + 1] = fmaf(w2, x.y, ai[4 * r4 + 1]);
                    ar[4 * r4 + 2] = fmaf(w1, x.z, ar[4 * r4 + 2]); ai[4 * r4 + 2] = fmaf(w2, x.z, ai[4 * r4 + 2]);
                    ar[4 * r4 + 3] = fmaf(w1, x.w, ar[4 * r4 + 3]); ai[4 * r4 + 3] = fmaf(w2, x.w, ai[4 * r4 + 3]);
                }
            }
        }
        if (S > 1) {
            if (live) {
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    part[((size_t)sl * cb + o) * 2 * ROWS + r] = ar[r];
                    part[((size_t)sl * cb + o) * 2 * ROWS + ROWS + r] = ai[r];
                }
            }
            __syncthreads();
            if (live && sl == 0) {
                for (int s2 = 1; s2 < S; ++s2) {
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) {
                        ar[r] += part[((size_t)s2 * cb + o) * 2 * ROWS + r];
                        ai[r] += part[((size_t)s2 * cb + o) * 2 * ROWS + ROWS + r];
                    }
                }
            }
        }
        if (!live || sl != 0) continue;
        const int c = b * cb + o;
        const float sp = ls_softplus(lam[c]), b1 = br[c], b2 = bi[c];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (r >= rows) continue;
            const float rg = ls_sigmoid(ar[r] + b1), ig = ls_sigmoid(ai[r] + b2);
            const float log_a = -rate * rg * sp;
            a_out[(size_t)(t0 + r) * C + c] = expf(log_a);
            // 1 - a^2 as -expm1(2 log a): a decay close to 1 keeps its digits
            x_out[(size_t)(t0 + r) * C + c] = sqrtf(fmaxf(-expm1f(2.0f * log_a), 0.f)) * ig * us[o * ROWS + r];
        }
    }
}

// The same for steps of few rows and maps of 64 channels or more, sum for sum in the same order (a row's gates are
// the same bits alone and among many): 32 outputs and 4 rows a block, grid (ceil(T / 4), nb, ceil(cb / 32)); a
// wave has both gates of the outputs and one of the slices that a map's inputs are cut into, S waves.
// Bound by the trips to memory of a thread's inputs, AHEAD of which are under way twice over; a block with all
// outputs of a map had 8 of each gate and left compute units idle: 16 maps of 128 x 128, 8 rows 14.3 -> 5.5 us,
// 128 rows 15.3 -> 8.9; 8 of 256 x 256, 8 rows 38.6 -> 11.3; 16 of 64 x 64, 1 row 5.9 -> 3.9.  (Below 64 the tiles of many
// rows: 16 of 32 x 32, 1 row 4.1 us against 5.2.)
#define LRU_FEW_ROWS 4
template <int AHEAD>
__global__ void __launch_bounds__(256)
lru_gates_few_kernel(const float* __restrict__ u, const float* __restrict__ Wt, const float* __restrict__ br,
                     const float* __restrict__ bi, const float* __restrict__ lam, float rate,
                     float* __restrict__ a_out, float* __restrict__ x_out, int T, int C, int cb, int S) {
    extern __shared__ __attribute__((aligned(16))) float us[];        // [cb][4 rows]
    __shared__ float part[4][LRU_FEW_ROWS][64];                       // the slices' sums
    const int t0 = blockIdx.x * LRU_FEW_ROWS, b = blockIdx.y, nb = C / cb, rows = min(LRU_FEW_ROWS, T - t0);
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
    const int o = blockIdx.z * 32 + (lane & 31);
    const float* const wp = Wt + ((size_t)(lane >= 32 ? nb : 0) + b) * cb * cb + min(o, cb - 1);
    const float* const up = u + (size_t)t0 * C + (size_t)b * cb;
    const int per = (cb + S - 1) / S, lo = wave * per, hi = min(cb, lo + per);
    float w0[AHEAD], w1[AHEAD];
    auto ask = [&](float* w, int i0) __attribute__((always_inline)) {           // (past the range: its last, not used)
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) w[k] = wp[(size_t)min(i0 + k, cb - 1) * cb];
        __builtin_amdgcn_sched_barrier(0);
    };
    ask(w0, lo);
    for (int i = tid; i < cb; i += blockDim.x) {
        float4 x;
        x.x = up[i];
        x.y = rows > 1 ? up[(size_t)C + i] : 0.f;
        x.z = rows > 2 ? up[2 * (size_t)C + i] : 0.f;
        x.w = rows > 3 ? up[3 * (size_t)C + i] : 0.f;
        ((float4*)us)[i] = x;
    }
    __syncthreads();
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    auto take = [&](float w, int i) __attribute__((always_inline)) {
        const float4 x = ((const float4*)us)[i];
        acc.x = fmaf(w, x.x, acc.x); acc.y = fmaf(w, x.y, acc.y);
        acc.z = fmaf(w, x.z, acc.z); acc.w = fmaf(w, x.w, acc.w);
    };
    auto multiply = [&](const float* w, int i0) __attribute__((always_inline)) {
        if (i0 + AHEAD <= hi) {
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) take(w[k], i0 + k);
        } else {
#pragma unroll
            for (int k = 0; k < AHEAD; ++k)
                if (i0 + k < hi) take(w[k], i0 + k);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int i0 = lo; i0 < hi; i0 += 2 * AHEAD) {
        ask(w1, i0 + AHEAD);
        multiply(w0, i0);
        ask(w0, i0 + 2 * AHEAD);
        multiply(w1, i0 + AHEAD);
    }
    if (S > 1) {
#pragma unroll
        for (int r = 0; r < LRU_FEW_ROWS; ++r) part[wave][r][lane] = ((const float*)&acc)[r];
        __syncthreads();
        if (wave > 0) return;
        for (int s = 1; s < S; ++s) {
            acc.x += part[s][0][lane]; acc.y += part[s][1][lane];
            acc.z += part[s][2][lane]; acc.w += part[s][3][lane];
        }
    }
    // lanes below 32 hold their output's first gate, those above its second: rows 0 and 1 to the ones, 2 and 3 to the others
    const bool high = lane >= 32;
    const float4 oth = make_float4(__shfl_xor(acc.x, 32, ILLM_WAVE), __shfl_xor(acc.y, 32, ILLM_WAVE),
                                   __shfl_xor(acc.z, 32, ILLM_WAVE), __shfl_xor(acc.w, 32, ILLM_WAVE));
    if (o >= cb) return;
    const int c = b * cb + o;
    const float sp = ls_softplus(lam[c]), b1 = br[c], b2 = bi[c];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = (high ? 2 : 0) + k;
        if (r >= rows) continue;
        const float ar = high ? (k ? oth.w : oth.z) : (k ? acc.y : acc.x), ai = high ? (k ? acc.w : acc.z) : (k ? oth.y : oth.x);
        const float rg = ls_sigmoid(ar + b1), ig = ls_sigmoid(ai + b2);
        const float log_a = -rate * rg * sp;
        a_out[(size_t)(t0 + r) * C + c] = expf(log_a);
        // 1 - a^2 as -expm1(2 log a): a decay close to 1 keeps its digits
        x_out[(size_t)(t0 + r) * C + c] = sqrtf(fmaxf(-expm1f(2.0f * log_a), 0.f)) * ig * us[o * LRU_FEW_ROWS + r];
    }
}

// Steps of many rows and maps of whole waves of outputs (cb % 64 == 0), again the same sums: 16 rows and up to 256 outputs a
// block, grid (ceil(T / 16), nb, ceil(cb / 256)); a wave has 64 outputs' gates of one slice of the inputs.  The rows' inputs
// are the same for a wave's lanes and come through the scalar cache, so that the loop is the weights' loads and multiply-adds
// with a scalar operand (by way of LDS its reads took as long as they).  us, that kernel -> this: 200 / 2,964 rows of 16 maps of
// 128 x 128 28 / 126 -> 19 / 86, 2,964 of 8 of 256 x 256 247 -> 137, of 16 of 256 x 256 334 -> 247.  (The next turn's weights ahead, or
// 4 or 16 inputs a turn: no faster.)
__global__ void __launch_bounds__(256)
lru_gates_rows_kernel(const float* __restrict__ u, const float* __restrict__ Wt, const float* __restrict__ br,
                      const float* __restrict__ bi, const float* __restrict__ lam, float rate,
                      float* __restrict__ a_out, float* __restrict__ x_out, int T, int C, int cb, int S) {
    constexpr int ROWS = 16, IN = 8;                     // IN: inputs a turn
    extern __shared__ __attribute__((aligned(16))) float part[];      // [S - 1][cb][2 ROWS] sums of the slices after the first
    const int t0 = blockIdx.x * ROWS, b = blockIdx.y, nb = C / cb, rows = min(ROWS, T - t0);
    const int lane = threadIdx.x & 63, wave = wave_index(), chunks = S > 1 ? cb / 64 : 4;
    const int sl = wave / chunks, o = (blockIdx.z * 4 + wave % chunks) * 64 + lane;
    const bool live = sl < S && o < cb;                  // (a wave's lanes alike)
    const int per = cb / S;
    float ar[ROWS], ai[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) ar[r] = ai[r] = 0.f;
    if (live) {
        const float* const wr = Wt + (size_t)b * cb * cb + o;
        const float* const wi = Wt + ((size_t)nb + b) * cb * cb + o;
        const float* const up = u + (size_t)t0 * C + (size_t)b * cb;
        for (int i0 = sl * per; i0 < (sl + 1) * per; i0 += IN) {
            float w1[IN], w2[IN];
#pragma unroll
            for (int k = 0; k < IN; ++k) {
                w1[k] = wr[(size_t)(i0 + k) * cb];
                w2[k] = wi[(size_t)(i0 + k) * cb];
            }
#pragma unroll
            for (int k4 = 0; k4 < IN; k4 += 4)
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    const float4 x = *(const float4*)(up + (size_t)min(r, rows - 1) * C + i0 + k4);
                    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        ar[r] = fmaf(w1[k4 + k], xs[k], ar[r]);
                        ai[r] = fmaf(w2[k4 + k], xs[k], ai[r]);
                    }
                }
        }
    }
    if (S > 1) {
        if (live && sl > 0) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                part[(((size_t)(sl - 1) * 2 * ROWS) + r) * cb + o] = ar[r];
                part[(((size_t)(sl - 1) * 2 * ROWS) + ROWS + r) * cb + o] = ai[r];
            }
        }
        __syncthreads();
        if (sl == 0)
            for (int s = 1; s < S; ++s)
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    ar[r] += part[((size_t)(s - 1) * 2 * ROWS + r) * cb + o];
                    ai[r] += part[((size_t)(s - 1) * 2 * ROWS + ROWS + r) * cb + o];
                }
    }
    if (!live || sl > 0) return;
    const int c = b * cb + o;
    const float sp = ls_softplus(lam[c]), b1 = br[c], b2 = bi[c];
    float x[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) x[r] = u[(size_t)min(t0 + r, T - 1) * C + c];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if (r >= rows) continue;
        const float rg = ls_sigmoid(ar[r] + b1), ig = ls_sigmoid(ai[r] + b2);
        const float log_a = -rate * rg * sp;
        a_out[(size_t)(t0 + r) * C + c] = expf(log_a);
        // 1 - a^2 as -expm1(2 log a): a decay close to 1 keeps its digits
        x_out[(size_t)(t0 + r) * C + c] = sqrtf(fmaxf(-expm1f(2.0f * log_a), 0.f)) * ig * x[r];
    }
}

template <int ROWS>
static int lru_gates_launch(const float* u, const float* Wt, const float* br, const float* bi,
                            const float* lam, float rate, float* a_out, float* x_out, int T, int C,
                            int nb, hipStream_t st) {
    const int cb = C / nb;
    const int slices = cb < 256 ? 256 / cb : 1;
    const size_t lds = ((size_t)ROWS * cb + (slices > 1 ? (size_t)slices * cb * 2 * ROWS : 0)) * sizeof(float);
    if (lds > 64 * 1024) return ILLM_ERR_ARG;
    if (lds > 48 * 1024 &&
        hipFuncSetAttribute((const void*)lru_gates_kernel<ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
        return ILLM_ERR_LAUNCH;
    hipLaunchKernelGGL(lru_gates_kernel<ROWS>, dim3((T + ROWS - 1) / ROWS, nb), dim3(256), lds, st, u, Wt, br,
                       bi, lam, rate, a_out, x_out, T, C, cb);
    return illm_launch_status();
}

extern "C" int illm_lru_gates(const float* u, const float* Wt, const float* br, const float* bi,
                              const float* lam, float rate, float* a_out, float* x_out, int T, int C,
                              int nb, void* stream) {
    if (T < 0 || C <= 0 || nb <= 0 || C % nb || nb > 65535) return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    const int cb = C / nb;
    if (T <= 128 && cb >= 64 && cb <= 4096) {
        const int S = cb < 256 ? 256 / cb : 1;
        const size_t lds = (size_t)cb * LRU_FEW_ROWS * sizeof(float);
#define GO(AHEAD_)                                                                                                 \
    do {                                                                                                           \
        if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)lru_gates_few_kernel<AHEAD_>,                        \
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) \
            return ILLM_ERR_LAUNCH;                                                                                \
        hipLaunchKernelGGL(lru_gates_few_kernel<AHEAD_>, dim3((T + LRU_FEW_ROWS - 1) / LRU_FEW_ROWS, nb, (cb + 31) / 32), \
                           dim3(64 * S), lds, (hipStream_t)stream, u, Wt, br, bi, lam, rate, a_out, x_out, \
                           T, C, cb, S);                                                                           \
    } while (0)
        if ((cb + S - 1) / S <= 32) GO(16);
        else GO(32);
#undef GO
        return illm_launch_status();
    }
    if (T > 128 && cb % 64 == 0 && cb <= 4096 && (uintptr_t)u % 16 == 0) {
        const int S = cb < 256 ? 256 / cb : 1;
        const size_t lds = (size_t)(S - 1) * cb * 32 * sizeof(float);
        hipLaunchKernelGGL(lru_gates_rows_kernel, dim3((T + 15) / 16, nb, (cb + 255) / 256), dim3(256), lds, (hipStream_t)stream, u,
                           Wt, br, bi, lam, rate, a_out, x_out, T, C, cb, S);
        return illm_launch_status();
    }
    // tiles of 16 rows where a block's inputs of 16 rows fit LDS (blocks of up to 1,024 channels)
    if (T <= 128 || C / nb > 1024)
        return lru_gates_launch<4>(u, Wt, br, bi, lam, rate, a_out, x_out, T, C, nb, (hipStream_t)stream);
    return lru_gates_launch<16>(u, Wt, br, bi, lam, rate, a_out, x_out, T, C, nb, (hipStream_t)stream);
}

__device__ __forceinline__ float ls_gelu_tanh(float z) {
    return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// grid (sequences, ceil(C / 256)); a thread walks its channel through the sequence's rows.
__global__ void __launch_bounds__(256)
lru_scan_kernel(const float* __restrict__ a, const float* __restrict__ x, float* __restrict__ state,
                const void* __restrict__ Y, int y_dt, int y_stride, int y_off,
                const float* __restrict__ yb, void* __restrict__ out, int out_dt,
                const int32_t* __restrict__ cu, const int32_t* __restrict__ seq_slot, int C) {
    const int b = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= C) return;
    const int r0 = cu[b], n = cu[b + 1] - r0;
    if (n <= 0) return;
    const int slot = seq_slot[b];
    float S = state[(size_t)slot * C + c];
    const float bias = yb ? yb[c] : 0.f;
    for (int t = 0; t < n; ++t) {
        const size_t at = (size_t)(r0 + t) * C + c;
        S = fmaf(a[at], S, x[at]);
        const float y = ls_gelu_tanh(ld_f(Y, y_dt, (size_t)(r0 + t) * y_stride + y_off + c) + bias);
        st_f(out, out_dt, at, S * y);
    }
    state[(size_t)slot * C + c] = S;
}

// The same recurrence for long steps, in three launches over chunks of LRU_CHUNK rows:
//   lru_chunk_sums   per (sequence, chunk, channel): the chunk's product of decays P and its sum B
//                    from a state of zero (S_end = P S_start + B)
//   lru_chunk_carry  per (sequence, channel): the state at every chunk's start, chunk after chunk
//                    (and the sequence's last state back into the slot)
//   lru_chunk_apply  per (sequence, chunk, channel): the recurrence again from the chunk's start
//                    state, with the other branch multiplied in
// A row's state is then summed in another order than token by token: it differs in rounding only.
#define LRU_CHUNK 32
__global__ void __launch_bounds__(256)
lru_chunk_sums_kernel(const float* __restrict__ a, const float* __restrict__ x, float* __restrict__ P,
                      float* __restrict__ B, const int32_t* __restrict__ cu, int C, int max_chunks) {
    const int b = blockIdx.z, ch = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int r0 = cu[b], n = cu[b + 1] - r0;
    const int t0 = ch * LRU_CHUNK;
    if (t0 >= n) return;
    const int t1 = min(n, t0 + LRU_CHUNK);
    float p = 1.f, s = 0.f;
    for (int t = t0; t < t1; ++t) {
        const size_t at = (size_t)(r0 + t) * C + c;
        const float av = a[at];
        s = fmaf(av, s, x[at]);
        p *= av;
    }
    const size_t o = ((size_t)b * max_chunks + ch) * C + c;
    P[o] = p;
    B[o] = s;
}

__global__ void __launch_bounds__(256)
lru_chunk_carry_kernel(const float* __restrict__ P, float* __restrict__ B, float* __restrict__ state,
                       const int32_t* __restrict__ cu, const int32_t* __restrict__ seq_slot, int C,
                       int max_chunks) {
    const int b = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int n = cu[b + 1] - cu[b];
    if (n <= 0) return;
    const int chunks = (n + LRU_CHUNK - 1) / LRU_CHUNK, slot = seq_slot[b];
    float S = state[(size_t)slot * C + c];
    for (int ch = 0; ch < chunks; ++ch) {
        const size_t o = ((size_t)b * max_chunks + ch) * C + c;
        const float next = fmaf(P[o], S, B[o]);
        B[o] = S;                                   // the chunk's start state, for lru_chunk_apply
        S = next;
    }
    state[(size_t)slot * C + c] = S;
}

__global__ void __launch_bounds__(256)
lru_chunk_apply_kernel(const float* __restrict__ a, const float* __restrict__ x,
                       const float* __restrict__ S0, const void* __restrict__ Y, int y_dt, int y_stride,
                       int y_off, const float* __restrict__ yb, void* __restrict__ out, int out_dt,
                       const int32_t* __restrict__ cu, int C, int max_chunks) {
    const int b = blockIdx.z, ch = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int r0 = cu[b], n = cu[b + 1] - r0;
    const int t0 = ch * LRU_CHUNK;
    if (t0 >= n) return;
    const int t1 = min(n, t0 + LRU_CHUNK);
    float S = S0[((size_t)b * max_chunks + ch) * C + c];
    const float bias = yb ? yb[c] : 0.f;
    for (int t = t0; t < t1; ++t) {
        const size_t at = (size_t)(r0 + t) * C + c;
        S = fmaf(a[at], S, x[at]);
        const float y = ls_gelu_tanh(ld_f(Y, y_dt, (size_t)(r0 + t) * y_stride + y_off + c) + bias);
        st_f(out, out_dt, at, S * y);
    }
}

// `scratch`: 2 * n_seqs * ceil(max_rows / 32) * C floats for steps of 64 rows a sequence or more
// (null, or fewer rows: a thread walks its channel through the whole sequence).
extern "C" int illm_lru_scan(const float* a, const float* x, float* state, const void* Y, int y_dt,
                             int y_stride, int y_off, const float* yb, void* out, int out_dt,
                             const int32_t* cu, const int32_t* seq_slot, int n_seqs, int max_rows, int C,
                             float* scratch, void* stream) {
    if (n_seqs < 0 || C <= 0 || !illm_dtype_ok(y_dt) || !illm_dtype_ok(out_dt) || y_off < 0 ||
        y_off + C > y_stride || n_seqs > 65535 || max_rows < 0)
        return ILLM_ERR_ARG;
    if (n_seqs == 0) return ILLM_OK;
    hipStream_t st = (hipStream_t)stream;
    const int cblocks = (C + 255) / 256;
    if (scratch && max_rows >= 2 * LRU_CHUNK) {
        const int chunks = (max_rows + LRU_CHUNK - 1) / LRU_CHUNK;
        if (chunks > 65535) return ILLM_ERR_ARG;
        float* P = scratch;
        float* B = scratch + (size_t)n_seqs * chunks * C;
        hipLaunchKernelGGL(lru_chunk_sums_kernel, dim3(cblocks, chunks, n_seqs), dim3(256), 0, st, a, x, P, B, cu,
                           C, chunks);
        hipLaunchKernelGGL(lru_chunk_carry_kernel, dim3(cblocks, n_seqs), dim3(256), 0, st, P, B, state, cu,
                           seq_slot, C, chunks);
        hipLaunchKernelGGL(lru_chunk_apply_kernel, dim3(cblocks, chunks, n_seqs), dim3(256), 0, st, a, x, B, Y,
                           y_dt, y_stride, y_off, yb, out, out_dt, cu, C, chunks);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(lru_scan_kernel, dim3(n_seqs, cblocks), dim3(256), 0, st, a, x, state, Y, y_dt,
                       y_stride, y_off, yb, out, out_dt, cu, seq_slot, C);
    return illm_launch_status();
}
