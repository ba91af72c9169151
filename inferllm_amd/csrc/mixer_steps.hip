// Single tokens (one row a sequence) through mixers whose state per head is a matrix S [dk, dv], float32: what stands around the
// plain gated rule S <- diag(g) S + k (beta v)^T, o = S^T q (delta_rule.hip, linear_scan.hip) in the recurrence's own kernel.
//
// A block takes a head of a sequence: 16 waves, wave w rows [w NR, w NR + NR) of S, a lane the columns lane, lane + 64, ...; a
// row's k, q and decay are one lane's and are read off it.  The partial sums meet in LDS in wave order; wave 0 forms the output.
// A kernel of a decode step costs 4 to 5 us whatever it does, and these are bound by their trips to memory: the numbers of the
// projection and the state are asked for together.  us in a graph, inputs, recurrence and output as kernels of their own -> here:
//                                                          1 sequence       8             16            64
//   matrix memory, 16 heads of 128 x 129                  14.5 -> 6.0   20.0 -> 7.1   23.8 -> 8.8   52.1 -> 30.7
//   gated linear attention, 16 heads of 64 x 128, with
//   the decays' product and the copy of its rows          12.5 -> 4.7   14.7 -> 5.3   17.2 -> 6.4   29.5 -> 17.0
//   state-space mixer, 64 heads of 128 x 64 (two kernels) 15.4 -> 9.0   21.4 -> 14.2  27.3 -> 21.0  71.4 -> 70.5
// (64 sequences of the last: 268 MB of state at 3.9 TB/s.)
#include <math.h>

#include "api.h"
#include "common.h"

#define STEP_WAVES 16
#define STEP_MAX_TAPS 8

__device__ __forceinline__ float ms_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float ms_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float ms_log_sigmoid(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

template <int DT>
__device__ __forceinline__ float ms_ld(const void* p, size_t i) {
    return DT == ILLM_BF16 ? bf16_to_f32(((const bf16_t*)p)[i]) : ((const float*)p)[i];
}

// A wave's rows of a head's state: columns past dv and rows past dk read ones that are there and are not written back.
template <int NR, int CS>
struct StepState {
    float s[NR][CS];
    __device__ __forceinline__ void ask(const float* sp, int i0, int dk, int dv, int stride) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int ii = 0; ii < NR; ++ii)
#pragma unroll
            for (int c = 0; c < CS; ++c) s[ii][c] = sp[(size_t)min(i0 + ii, dk - 1) * stride + min(lane + 64 * c, dv - 1)];
    }
    // S <- g S + k u^T and the wave's part of S^T q; lane ii holds row i0 + ii's g, k and q (k = q = 0 past dk)
    __device__ __forceinline__ void turn(float g_l, float k_l, float q_l, const float (&u)[CS], float (&o)[CS]) {
#pragma unroll
        for (int c = 0; c < CS; ++c) o[c] = 0.f;
#pragma unroll
        for (int ii = 0; ii < NR; ++ii) {
            const float g = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_l), ii));
            const float k = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(k_l), ii));
            const float q = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q_l), ii));
#pragma unroll
            for (int c = 0; c < CS; ++c) {
                s[ii][c] = fmaf(k, u[c], s[ii][c] * g);
                o[c] = fmaf(s[ii][c], q, o[c]);
            }
        }
    }
    __device__ __forceinline__ void keep(float* sp, int i0, int dk, int dv, int stride) const {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int ii = 0; ii < NR; ++ii)
#pragma unroll
            for (int c = 0; c < CS; ++c)
                if (i0 + ii < dk && lane + 64 * c < dv) sp[(size_t)(i0 + ii) * stride + lane + 64 * c] = s[ii][c];
    }
};

template <int N>
__device__ __forceinline__ float step_sum(const float (*red)[N], int c) {
    float t[4] = {red[0][c], red[1][c], red[2][c], red[3][c]};
#pragma unroll
    for (int w = 4; w < STEP_WAVES; ++w) t[w & 3] += red[w][c];
    return (t[0] + t[1]) + (t[2] + t[3]);
}

// A matrix memory (see linear_scan.hip): grid (H, rows).  U [rows, u_stride] = [q (H dk) | k (H dk) | v (H dv) | ..], the gates'
// columns at i_off and f_off, the output gate's at z_off; state [slots][H][dk][dv + 1], its last column the normaliser.
template <int DT, int NR, int CS>
__global__ void __launch_bounds__(64 * STEP_WAVES)
memory_step_kernel(const void* __restrict__ U, int u_stride, int i_off, int f_off, int z_off, const float* __restrict__ i_bias,
                   const float* __restrict__ f_bias, float cap, float* __restrict__ m_state, float* __restrict__ state,
                   const int32_t* __restrict__ row_slot, const void* __restrict__ w, int w_dt, void* __restrict__ out, int H,
                   int dk, int dv, float qscale, float eps) {
    __shared__ float red[STEP_WAVES][64 * CS + 1];
    const int h = blockIdx.x, r = blockIdx.y, lane = threadIdx.x & 63, wave = wave_index(), i0 = wave * NR;
    const int slot = row_slot[r], mine = min(i0 + lane, dk - 1);
    const size_t u0 = (size_t)r * u_stride;
    float* const sp = state + ((size_t)slot * H + h) * dk * (dv + 1);
    float q = ms_ld<DT>(U, u0 + (size_t)h * dk + mine) * qscale, k = ms_ld<DT>(U, u0 + (size_t)(H + h) * dk + mine);
    const float iu = ms_ld<DT>(U, u0 + i_off + h), fu = ms_ld<DT>(U, u0 + f_off + h), bi = i_bias[h], bf = f_bias[h];
    const float m_before = m_state[(size_t)slot * H + h];
    float v[CS], z[CS], wt[CS];
#pragma unroll
    for (int c = 0; c < CS; ++c) {
        const size_t col = (size_t)h * dv + min(lane + 64 * c, dv - 1);
        v[c] = ms_ld<DT>(U, u0 + 2 * (size_t)H * dk + col);
        z[c] = ms_ld<DT>(U, u0 + z_off + col);
        wt[c] = ld_f(w, w_dt, col);
    }
    StepState<NR, CS> S;
    S.ask(sp, i0, dk, dv, dv + 1);
    float norm = sp[(size_t)mine * (dv + 1) + dv];
    loads_asked_for();
    const bool live = lane < NR && i0 + lane < dk;
    if (!live) q = k = 0.f;
    const float inv_cap = 1.0f / cap;
    const float ig = cap * tanhf((iu + bi) * inv_cap), fg = ms_log_sigmoid(cap * tanhf((fu + bf) * inv_cap));
    const float m = fmaxf(fg + m_before, ig), g = expf(fg + m_before - m), beta = expf(ig - m);
#pragma unroll
    for (int c = 0; c < CS; ++c) v[c] *= beta;
    float o[CS];
    S.turn(g, k, q, v, o);
    norm = fmaf(k, beta, norm * g);
    S.keep(sp, i0, dk, dv, dv + 1);
    if (live) sp[(size_t)(i0 + lane) * (dv + 1) + dv] = norm;
#pragma unroll
    for (int c = 0; c < CS; ++c) red[wave][lane + 64 * c] = o[c];
    const float nq = wave_sum(live ? norm * q : 0.f);
    if (lane == 0) red[wave][64 * CS] = nq;
    __syncthreads();
    if (wave != 0) return;
    if (lane == 0) m_state[(size_t)slot * H + h] = m;
    const float den = fmaxf(fabsf(step_sum(red, 64 * CS)), expf(-m)) + 1e-6f;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CS; ++c) {
        o[c] = step_sum(red, lane + 64 * c) / den;
        if (lane + 64 * c < dv) ss += o[c] * o[c];
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
    for (int c = 0; c < CS; ++c)
        if (lane + 64 * c < dv)
            st_f(out, DT, ((size_t)r * H + h) * dv + lane + 64 * c, (o[c] * inv) * wt[c] * ms_sigmoid(z[c]));
}

// Gated linear attention: grid (H, rows).  U's columns q, k (H dk), v and the gate's z (H dv) at their offsets and the decays'
// `ra` inner numbers at a_off; decay = sigmoid(W_a2 a + bias)^(1 / tau), W_a2 [H dk, ra] of U's type, its product in float32.
template <int DT, int NR, int CS>
__global__ void __launch_bounds__(64 * STEP_WAVES)
gla_step_kernel(const void* __restrict__ U, int u_stride, int q_off, int k_off, int v_off, int z_off, int a_off, int ra,
                const void* __restrict__ w_a2, const float* __restrict__ a2_bias, float inv_tau, float* __restrict__ state,
                const int32_t* __restrict__ row_slot, const void* __restrict__ w, int w_dt, void* __restrict__ out, int H, int dk,
                int dv, float qscale, float eps) {
    __shared__ float red[STEP_WAVES][64 * CS];
    const int h = blockIdx.x, r = blockIdx.y, lane = threadIdx.x & 63, wave = wave_index(), i0 = wave * NR;
    const int slot = row_slot[r], mine = min(i0 + lane, dk - 1);
    const size_t u0 = (size_t)r * u_stride, row = (size_t)h * dk + mine;
    float* const sp = state + ((size_t)slot * H + h) * dk * dv;
    float q = ms_ld<DT>(U, u0 + q_off + row) * qscale, k = ms_ld<DT>(U, u0 + k_off + row);
    const float zb = a2_bias[row];
    float v[CS], z[CS], wt[CS];
#pragma unroll
    for (int c = 0; c < CS; ++c) {
        const int in = min(lane + 64 * c, dv - 1);
        v[c] = ms_ld<DT>(U, u0 + v_off + (size_t)h * dv + in);
        z[c] = ms_ld<DT>(U, u0 + z_off + (size_t)h * dv + in);
        wt[c] = ld_f(w, w_dt, in);
    }
    float4 a[4], b[4];                                  // the first 16 of the inner numbers ahead of the state
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a[j] = ld_f4(U, DT, (u0 + a_off) / 4 + min(j, ra / 4 - 1));
        b[j] = ld_f4(w_a2, DT, row * (ra / 4) + min(j, ra / 4 - 1));
    }
    StepState<NR, CS> S;
    S.ask(sp, i0, dk, dv, dv);
    loads_asked_for();
    float za = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (4 * j < ra) za = fmaf(a[j].w, b[j].w, fmaf(a[j].z, b[j].z, fmaf(a[j].y, b[j].y, fmaf(a[j].x, b[j].x, za))));
    for (int j = 4; j < ra / 4; ++j) {
        const float4 c = ld_f4(U, DT, (u0 + a_off) / 4 + j), d = ld_f4(w_a2, DT, row * (ra / 4) + j);
        za = fmaf(c.w, d.w, fmaf(c.z, d.z, fmaf(c.y, d.y, fmaf(c.x, d.x, za))));
    }
    const float g = expf(ms_log_sigmoid(za + zb) * inv_tau);
    if (!(lane < NR && i0 + lane < dk)) q = k = 0.f;
    float o[CS];
    S.turn(g, k, q, v, o);
    S.keep(sp, i0, dk, dv, dv);
#pragma unroll
    for (int c = 0; c < CS; ++c) red[wave][lane + 64 * c] = o[c];
    __syncthreads();
    if (wave != 0) return;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CS; ++c) {
        o[c] = step_sum(red, lane + 64 * c);
        if (lane + 64 * c < dv) ss += o[c] * o[c];
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
    for (int c = 0; c < CS; ++c)
        if (lane + 64 * c < dv)
            st_f(out, DT, ((size_t)r * H + h) * dv + lane + 64 * c, o[c] * inv * wt[c] * (z[c] * ms_sigmoid(z[c])));
}

// A state-space mixer (see linear_scan.hip): grid (H, rows).  The short convolution of the head's x and of its group's B and C,
// the recurrence, y = (o + D x) silu(z), left to the norm over groups of heads in ssm_step_norm_kernel, which also moves the
// kept inputs of B and C on: a group's heads read them here.
template <int DT, int NR, int CS>
__global__ void __launch_bounds__(64 * STEP_WAVES)
ssm_step_kernel(const void* __restrict__ U, int u_stride, int x_off, int dt_off, int z_off, const float* __restrict__ conv_w,
                const float* __restrict__ conv_b, int taps, void* __restrict__ tail, float* __restrict__ state,
                const int32_t* __restrict__ row_slot, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                const float* __restrict__ D, float* __restrict__ y, int G, int H, int N, int dv) {
    __shared__ float red[STEP_WAVES][64 * CS], xs[768];
    const int h = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = wave_index(), i0 = wave * NR;
    const int slot = row_slot[r], mine = min(i0 + lane, N - 1), gh = h / (H / G);
    const int inner = H * dv, GN = G * N, C = inner + 2 * GN, K = taps - 1;
    const size_t u0 = (size_t)r * u_stride;
    float* const sp = state + ((size_t)slot * H + h) * N * dv;
    const float du = ms_ld<DT>(U, u0 + dt_off + h), db = dt_bias[h], al = a_log[h], Dh = D[h];
    float z[CS];
#pragma unroll
    for (int c = 0; c < CS; ++c) z[c] = ms_ld<DT>(U, u0 + z_off + (size_t)h * dv + min(lane + 64 * c, dv - 1));
    const bool turned = tid < dv + 2 * N;
    const int in = tid - dv, c = tid < dv ? h * dv + tid : in < N ? inner + gh * N + in : inner + GN + gh * N + (in - N);
    float x[STEP_MAX_TAPS], cw[STEP_MAX_TAPS], bias = 0.f;
#pragma unroll
    for (int j = 0; j < STEP_MAX_TAPS; ++j) {
        x[j] = cw[j] = 0.f;
        if (turned && j < taps) {
            x[j] = j < K ? ms_ld<DT>(tail, ((size_t)slot * K + j) * C + c) : ms_ld<DT>(U, u0 + x_off + c);
            cw[j] = conv_w[(size_t)c * taps + j];
        }
    }
    if (turned) bias = conv_b[c];
    StepState<NR, CS> S;
    S.ask(sp, i0, N, dv, dv);
    loads_asked_for();
    if (turned) {
        float a = bias;
#pragma unroll
        for (int j = 0; j < STEP_MAX_TAPS; ++j)
            if (j < taps) {
                a = fmaf(cw[j], x[j], a);
                if (j > 0 && tid < dv) st_f(tail, DT, ((size_t)slot * K + (j - 1)) * C + c, x[j]);
            }
        xs[tid] = a * ms_sigmoid(a);
    }
    const float step = ms_softplus(du + db), g = expf(-expf(al) * step);
    __syncthreads();
    float k = xs[dv + mine], q = xs[dv + N + mine], u[CS], o[CS];
    if (!(lane < NR && i0 + lane < N)) q = k = 0.f;
#pragma unroll
    for (int i = 0; i < CS; ++i) u[i] = step * xs[min(lane + 64 * i, dv - 1)];
    S.turn(g, k, q, u, o);
    S.keep(sp, i0, N, dv, dv);
#pragma unroll
    for (int i = 0; i < CS; ++i) red[wave][lane + 64 * i] = o[i];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int i = 0; i < CS; ++i) {
        const int j = lane + 64 * i;
        if (j < dv) y[(size_t)r * inner + (size_t)h * dv + j] = fmaf(Dh, xs[j], step_sum(red, j)) * (z[i] * ms_sigmoid(z[i]));
    }
}

// grid (rows, norm groups); 256 threads.  out = y / sqrt(mean over the part of y^2 + eps) * w, and the group's share of the kept
// inputs' columns [first, C).
template <int DT>
__global__ void __launch_bounds__(256)
ssm_step_norm_kernel(const float* __restrict__ y, const void* __restrict__ w, int w_dt, void* __restrict__ out, int inner, int part,
                     float eps, const void* __restrict__ U, int u_stride, int x_off, int taps, void* __restrict__ tail,
                     const int32_t* __restrict__ row_slot, int C) {
    __shared__ float red[16];
    const size_t r = blockIdx.x;
    const int j0 = blockIdx.y * part, K = taps - 1, share = (C - inner + gridDim.y - 1) / gridDim.y;
    float v[8], wt[8];
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int j = threadIdx.x + 256 * e;
        v[e] = j < part ? y[r * inner + j0 + j] : 0.f;
        wt[e] = j < part ? ld_f(w, w_dt, j0 + j) : 0.f;
    }
    const int slot = row_slot[r], c1 = min(C, inner + (int)(blockIdx.y + 1) * share);
    for (int c = inner + blockIdx.y * share + threadIdx.x; c < c1; c += 256) {
        float x[STEP_MAX_TAPS];
#pragma unroll
        for (int j = 1; j < STEP_MAX_TAPS; ++j)
            if (j <= K) x[j] = j < K ? ms_ld<DT>(tail, ((size_t)slot * K + j) * C + c) : ms_ld<DT>(U, r * u_stride + x_off + c);
#pragma unroll
        for (int j = 1; j < STEP_MAX_TAPS; ++j)
            if (j <= K) st_f(tail, DT, ((size_t)slot * K + (j - 1)) * C + c, x[j]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
    ss = block_sum<4>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)part + eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int j = threadIdx.x + 256 * e;
        if (j < part) st_f(out, DT, r * inner + j0 + j, (v[e] * inv) * wt[e]);
    }
}

// The head sizes that these kernels take: dk to 256 rows, dv to 256 columns.
static bool step_sizes(int dt, int B, int H, int dk, int dv) {
    return illm_dtype_ok(dt) && B >= 0 && B <= 65535 && H > 0 && dk > 0 && dk <= 256 && dv > 0 && dv <= 256;
}

#define STEP_ROWS(DT_, CS_)                     \
    if (dk <= 64) GO(DT_, 4, CS_);              \
    else if (dk <= 128) GO(DT_, 8, CS_);        \
    else GO(DT_, 16, CS_)
#define STEP_COLS(DT_)                          \
    if (dv <= 64) { STEP_ROWS(DT_, 1); }        \
    else if (dv <= 128) { STEP_ROWS(DT_, 2); }  \
    else { STEP_ROWS(DT_, 4); }
#define STEP_TYPES()                            \
    if (dt == ILLM_BF16) { STEP_COLS(ILLM_BF16) } else { STEP_COLS(ILLM_F32) }

extern "C" int illm_memory_step(const void* U, int dt, int u_stride, int i_off, int f_off, int z_off, const float* i_bias,
                                const float* f_bias, float cap, float* m_state, float* state, const int32_t* row_slot,
                                const void* w, int w_dt, void* out, int B, int H, int dk, int dv, float eps, void* stream) {
    if (!step_sizes(dt, B, H, dk, dv) || !illm_dtype_ok(w_dt) || !(cap > 0.f) || i_off < 0 || f_off < 0 || z_off < 0 ||
        2LL * H * dk + (long long)H * dv > u_stride || i_off + H > u_stride || f_off + H > u_stride ||
        z_off + (long long)H * dv > u_stride)
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
#define GO(DT_, NR_, CS_)                                                                                                \
    hipLaunchKernelGGL((memory_step_kernel<DT_, NR_, CS_>), dim3(H, B), dim3(64 * STEP_WAVES), 0, (hipStream_t)stream, U, \
                       u_stride, i_off, f_off, z_off, i_bias, f_bias, cap, m_state, state, row_slot, w, w_dt, out, H, dk, dv, \
                       1.0f / sqrtf((float)dk), eps)
    STEP_TYPES()
#undef GO
    return illm_launch_status();
}

extern "C" int illm_gla_step(const void* U, int dt, int u_stride, int q_off, int k_off, int v_off, int z_off, int a_off, int ra,
                             const void* w_a2, const float* a2_bias, float tau, float* state, const int32_t* row_slot,
                             const void* w, int w_dt, void* out, int B, int H, int dk, int dv, float eps, void* stream) {
    if (!step_sizes(dt, B, H, dk, dv) || !illm_dtype_ok(w_dt) || !(tau > 0.f) || ra <= 0 || ra % 4 || a_off < 0 || a_off % 4 ||
        u_stride % 4 || q_off < 0 || k_off < 0 || v_off < 0 || z_off < 0 || a_off + (long long)ra > u_stride ||
        q_off + (long long)H * dk > u_stride || k_off + (long long)H * dk > u_stride || v_off + (long long)H * dv > u_stride ||
        z_off + (long long)H * dv > u_stride || ((uintptr_t)U | (uintptr_t)w_a2) % (dt == ILLM_BF16 ? 8 : 16))
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
#define GO(DT_, NR_, CS_)                                                                                                \
    hipLaunchKernelGGL((gla_step_kernel<DT_, NR_, CS_>), dim3(H, B), dim3(64 * STEP_WAVES), 0, (hipStream_t)stream, U, u_stride, \
                       q_off, k_off, v_off, z_off, a_off, ra, w_a2, a2_bias, 1.0f / tau, state, row_slot, w, w_dt, out, H, dk, dv, \
                       1.0f / sqrtf((float)dk), eps)
    STEP_TYPES()
#undef GO
    return illm_launch_status();
}

extern "C" int illm_ssm_step(const void* U, int dt, int u_stride, int x_off, int dt_off, int z_off, const float* conv_w,
                             const float* conv_b, int taps, void* tail, float* state, const int32_t* row_slot, const float* a_log,
                             const float* dt_bias, const float* D, float* y, const void* w, int w_dt, int norm_groups, float eps,
                             void* out, int B, int G, int H, int N, int dv, void* stream) {
    const int dk = N;
    if (!step_sizes(dt, B, H, N, dv) || !illm_dtype_ok(w_dt) || G <= 0 || H % G || taps < 1 || taps > STEP_MAX_TAPS || x_off < 0 ||
        dt_off < 0 || z_off < 0 || x_off + (long long)H * dv + 2LL * G * N > u_stride || dt_off + H > u_stride ||
        z_off + (long long)H * dv > u_stride || norm_groups <= 0 || norm_groups > 65535 || ((long long)H * dv) % norm_groups ||
        (long long)H * dv / norm_groups > 2048)
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
#define GO(DT_, NR_, CS_)                                                                                                \
    hipLaunchKernelGGL((ssm_step_kernel<DT_, NR_, CS_>), dim3(H, B), dim3(64 * STEP_WAVES), 0, (hipStream_t)stream, U, u_stride, \
                       x_off, dt_off, z_off, conv_w, conv_b, taps, tail, state, row_slot, a_log, dt_bias, D, y, G, H, N, dv)
    STEP_TYPES()
#undef GO
    const int inner = H * dv, C = inner + 2 * G * N;
#define NORM(DT_)                                                                                                        \
    hipLaunchKernelGGL(ssm_step_norm_kernel<DT_>, dim3(B, norm_groups), dim3(256), 0, (hipStream_t)stream, y, w, w_dt, out, inner, \
                       inner / norm_groups, eps, U, u_stride, x_off, taps, tail, row_slot, C)
    if (dt == ILLM_BF16) NORM(ILLM_BF16);
    else NORM(ILLM_F32);
#undef NORM
    return illm_launch_status();
}
