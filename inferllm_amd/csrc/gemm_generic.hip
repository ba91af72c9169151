// Y[M, N] = X[M, K] . W[N, K]^T for any sizes and any mix of float32 / bfloat16
// storage, accumulated in float32 with plain multiply-adds (no matrix cores, no
// reduced-precision mode).  Each output element is summed over k in ascending
// order, whatever its row's place in the batch, so a row gives the same bits
// whether it comes alone or among others.  This is the matrix product of the
// 32-bit path and the fallback for shapes the MFMA kernels do not take.  Two more
// kernels below serve the 32-bit path's common cases faster, both in float32
// throughout: few rows (W read once) and many rows (the matrix cores' float32
// instruction).
//
// The reference's float product is the same sum (src/kern/naive/naive.cpp:363-379);
// its GPU path calls cublasSgemm (src/kern/gpu/kernel_gpu.cu:420-435).
#include <mutex>

#include "api.h"
#include "api_test.h"
#include "common.h"

#define GT 64   // tile of outputs per block (GT x GT)
#define GK 16   // depth of a k step

__global__ void __launch_bounds__(256)
gemm_generic_kernel(const void* __restrict__ X, int x_dt, const void* __restrict__ W, int w_dt,
                    void* __restrict__ Y, int y_dt, int M, int N, int K) {
    __shared__ float xs[GK][GT + 1];
    __shared__ float ws[GK][GT + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += GK) {
        // 64 rows x 16 k per operand, 1024 elements, 4 per thread
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = threadIdx.x + e * 256;
            const int r = idx >> 4, kk = idx & 15;
            const int k = k0 + kk;
            const int m = m0 + r, n = n0 + r;
            xs[kk][r] = (m < M && k < K) ? ld_f(X, x_dt, (size_t)m * K + k) : 0.f;
            ws[kk][r] = (n < N && k < K) ? ld_f(W, w_dt, (size_t)n * K + k) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n < N) st_f(Y, y_dt, (size_t)m * N + n, acc[i][j]);
        }
    }
}

extern "C" int illm_gemm_generic(const void* X, int x_dt, const void* W, int w_dt, void* Y,
                                 int y_dt, int M, int N, int K, void* stream) {
    if (M < 0 || N <= 0 || K <= 0 || !illm_dtype_ok(x_dt) || !illm_dtype_ok(w_dt) ||
        !illm_dtype_ok(y_dt))
        return ILLM_ERR_ARG;
    if (M == 0) return ILLM_OK;
    const int gy = (M + GT - 1) / GT;
    if (gy > 65535) return ILLM_ERR_ARG;
    hipLaunchKernelGGL(gemm_generic_kernel, dim3((N + GT - 1) / GT, gy), dim3(256), 0,
                       (hipStream_t)stream, X, x_dt, W, w_dt, Y, y_dt, M, N, K);
    return illm_launch_status();
}


// ---------------------------------------------------------------- many rows, float32
// The same product for float32 X and W with K a multiple of 16, on the matrix cores' float32
// instruction (MFMA 32x32x2: float32 operands, float32 products and sums; nothing is rounded to
// a shorter type).  A block of four waves takes T x T outputs, a wave T/2 x T/2.  Both operands go
// through LDS as rows of 32 k (two buffers, the next two stages' loads in flight in two register
// sets while this one is multiplied), a chunk of 8 k as its even ones, then its odd ones, read 16
// bytes a lane: half-wave 0 takes the even ones, so that one LDS read is the operand of four
// MFMAs, each of two neighbouring k.  The MFMA's rows are W's (n) and its columns X's (m), so a
// lane holds 4 consecutive n of one m: 16-byte stores.  An output element is summed over k in
// ascending pairs whatever its row's place, the number of rows or T.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4v_t __attribute__((ext_vector_type(4)));
typedef float f32x2v_t __attribute__((ext_vector_type(2)));

#define FM_K 32      // k a stage
#define FM_LD 36     // LDS row stride in floats: the 16-byte reads of 8 rows fall into 32 different banks

template <int T>
__global__ void __launch_bounds__(256, 2)
gemm_f32_mfma_kernel(const float* __restrict__ X, const float* __restrict__ W, void* __restrict__ Y,
                     int y_dt, int M, int N, int K, int m_tiles) {
    constexpr int NT = T / 64;                 // MFMA tiles of a wave along each side
    constexpr int NL = T / 32;                 // 16-byte pieces a thread brings of each operand a stage
    extern __shared__ __attribute__((aligned(16))) float lds[];         // [buffer][X rows, W rows][FM_LD]
    constexpr int BUF = 2 * T * FM_LD;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
    const int r = lane & 31, kh = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    // the blocks that share rows of W run next to each other on one XCD (block ids go round the 8)
    const int xcd = blockIdx.x & 7, j8 = blockIdx.x >> 3;
    const int m0 = (j8 % m_tiles) * T, n0 = ((j8 / m_tiles) * 8 + xcd) * T;
    if (n0 >= N) return;

    // staging: thread t brings 4 k (quad t % 8) of rows t / 8 + 32 e of both operands, the stage's k as
    // a scalar offset (address and mask instructions a stage cost a tenth of the time); rows beyond the matrix read its last row (their
    // outputs are not stored).  K = 32 n + 16: the last stage's loads start 16 k earlier and count
    // from the 17th k on; stages past the end are zeros.
    const int s_row = tid >> 3, s_k = (tid & 7) * 4;
    uint32_t xo[NL], wo[NL];                   // bytes from the block's first row
#pragma unroll
    for (int e = 0; e < NL; ++e) {
        xo[e] = (uint32_t)(min(s_row + 32 * e, M - 1 - m0) * K + min(s_k, K - 4)) * 4u;
        wo[e] = (uint32_t)(min(s_row + 32 * e, N - 1 - n0) * K + min(s_k, K - 4)) * 4u;
    }
    const char* const xbase = (const char*)(X + (size_t)m0 * K);
    const char* const wbase = (const char*)(W + (size_t)n0 * K);
    const bool in_part = K >= FM_K ? s_k >= FM_K / 2 : s_k < K;
    struct Set { f32x4v_t x[NL], w[NL]; };
    const int full = K / FM_K, stages = (K + FM_K - 1) / FM_K;
    auto fetch = [&](Set& g, int st) __attribute__((always_inline)) {
        const size_t at = (size_t)max(0, min(st * FM_K, K - FM_K)) * 4;
#pragma unroll
        for (int e = 0; e < NL; ++e) {
            g.x[e] = *(const f32x4v_t*)(xbase + at + xo[e]);
            g.w[e] = *(const f32x4v_t*)(wbase + at + wo[e]);
        }
    };
    auto stage = [&](Set& g, int st) __attribute__((always_inline)) {
        float* xs = lds + (st & 1) * BUF + s_row * FM_LD + (s_k & ~7) + (s_k & 4) / 2;
        if (st >= full) {
            const bool in = st < stages && in_part;
#pragma unroll
            for (int e = 0; e < NL; ++e) {
                const f32x4v_t zero = {0.f, 0.f, 0.f, 0.f};
                g.x[e] = in ? g.x[e] : zero;
                g.w[e] = in ? g.w[e] : zero;
            }
        }
#pragma unroll
        for (int e = 0; e < NL; ++e) {
            float* ws = xs + T * FM_LD;
            *(f32x2v_t*)(xs + 32 * e * FM_LD) = (f32x2v_t){g.x[e][0], g.x[e][2]};
            *(f32x2v_t*)(xs + 32 * e * FM_LD + 4) = (f32x2v_t){g.x[e][1], g.x[e][3]};
            *(f32x2v_t*)(ws + 32 * e * FM_LD) = (f32x2v_t){g.w[e][0], g.w[e][2]};
            *(f32x2v_t*)(ws + 32 * e * FM_LD + 4) = (f32x2v_t){g.w[e][1], g.w[e][3]};
        }
    };
    f32x16_t acc[NT][NT];                    // [n tile][m tile]
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    struct Ops { f32x4v_t a[NT], b[NT]; };     // a wave's operands of 8 k
    auto operands = [&](Ops& o, int st, int c) __attribute__((always_inline)) {
        const float* xb = lds + (st & 1) * BUF + (wm * (T / 2) + r) * FM_LD + 4 * kh + 8 * c;
        const float* wb = lds + (st & 1) * BUF + (T + wn * (T / 2) + r) * FM_LD + 4 * kh + 8 * c;
#pragma unroll
        for (int i = 0; i < NT; ++i) o.a[i] = *(const f32x4v_t*)(wb + 32 * i * FM_LD);
#pragma unroll
        for (int j = 0; j < NT; ++j) o.b[j] = *(const f32x4v_t*)(xb + 32 * j * FM_LD);
    };
    auto multiply = [&](const Ops& o) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[i][s], o.b[j][s], acc[i][j], 0, 0, 0);
        if constexpr (T == 64) __builtin_amdgcn_sched_barrier(0);
    };

    Set g0, g1;
    Ops o0, o1;
    fetch(g0, 0);
    fetch(g1, 1);
    stage(g0, 0);
    __syncthreads();
    // Stage st is multiplied while st + 1 waits in one register set and st + 2 is asked for into the
    // other (stages past the end are zeros).  T = 64: a chunk's operands are read while the chunk
    // before it is multiplied, the next stage's first ones too: its writes and the barrier stand
    // before this stage's last products, so that a block alone on its compute unit goes on (256 rows,
    // 12288 x 4096: 260 -> 249 us, 4096 x 11008: 227 -> 217).  T = 128: the other block of the compute unit
    // fills the gap, and the order by stages is as fast (2,048 rows of 4096 x 11008: 1,422 us, 1,431 so).
    auto turn = [&](Set& next, Set& after, int st) __attribute__((always_inline)) {
        fetch(after, st + 2);
        if constexpr (T == 64) {
            operands(o1, st, 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(o0);
            operands(o0, st, 2);
            __builtin_amdgcn_sched_barrier(0);
            multiply(o1);
            operands(o1, st, 3);
            __builtin_amdgcn_sched_barrier(0);
            multiply(o0);
            stage(next, st + 1);
            __syncthreads();
            operands(o0, st + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            multiply(o1);
        } else {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < FM_K / 8; ++c) {
                Ops o;
                operands(o, st, c);
                multiply(o);
            }
            __builtin_amdgcn_sched_barrier(0);
            stage(next, st + 1);
            __syncthreads();
        }
    };
    if constexpr (T == 64) operands(o0, 0, 0);
    for (int st = 0; st + 1 < stages; st += 2) {
        turn(g1, g0, st);
        turn(g0, g1, st + 1);
    }
    if (stages & 1) turn(g1, g0, stages - 1);
    // acc[i][j][v]: n = n0 + wn * T/2 + 32 i + 8 (v / 4) + 4 kh + v % 4, m = m0 + wm * T/2 + 32 j + r
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int m = m0 + wm * (T / 2) + 32 * j + r;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + wn * (T / 2) + 32 * i + 8 * g + 4 * kh;
                const size_t at = (size_t)m * N + n;
                if (n + 3 < N && (N & 3) == 0 && y_dt == ILLM_F32) {
                    *(float4*)((float*)Y + at) = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1],
                                                             acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) st_f(Y, y_dt, at + v, acc[i][j][4 * g + v]);
                }
            }
    }
}

// The same for short K, where the kernel above has more stages in flight than there are: blocks of 128 x 128,
// stages of 16 k, one ahead, operands k-major in LDS (33 KB, so that four blocks share a compute unit and
// their stores of Y, which is what counts here, overlap).  4,096 rows of 4096 x 16 19 us, and 46 (35 in blocks of 64 x 64)
// above; 2,048 rows of 2048 x 16 9.2 and 13.5.  The same pairs of k in the same order: the same bits.
#define FS_T 128     // outputs of a block along m and along n
#define FS_K 16      // k a stage
#define FS_LD 130    // LDS row stride in floats (4 * FS_LD = 8 mod 32: the stores of a half-wave,
                     // 8 rows x 4 k-quads, fall into 32 different banks)

__global__ void __launch_bounds__(256)
gemm_f32_short_kernel(const float* __restrict__ X, const float* __restrict__ W, void* __restrict__ Y,
                     int y_dt, int M, int N, int K) {
    __shared__ float xs[2][FS_K][FS_LD];
    __shared__ float ws[2][FS_K][FS_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
    const int r = lane & 31, kh = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    const int m0 = blockIdx.y * FS_T, n0 = blockIdx.x * FS_T;

    // staging: thread t brings 4 k (quad t % 4) of rows t / 4 and t / 4 + 64 of both operands;
    // rows beyond the matrix read its last row (their outputs are not stored)
    const int s_row = tid >> 2, s_kq = tid & 3;
    const float* xsrc[2];
    const float* wsrc[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        xsrc[e] = X + (size_t)min(m0 + s_row + 64 * e, M - 1) * K + s_kq * 4;
        wsrc[e] = W + (size_t)min(n0 + s_row + 64 * e, N - 1) * K + s_kq * 4;
    }
    float4 xg[2], wg[2];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            xg[e] = *(const float4*)(xsrc[e] + k0);
            wg[e] = *(const float4*)(wsrc[e] + k0);
        }
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int row = s_row + 64 * e;
            xs[buf][s_kq * 4 + 0][row] = xg[e].x; xs[buf][s_kq * 4 + 1][row] = xg[e].y;
            xs[buf][s_kq * 4 + 2][row] = xg[e].z; xs[buf][s_kq * 4 + 3][row] = xg[e].w;
            ws[buf][s_kq * 4 + 0][row] = wg[e].x; ws[buf][s_kq * 4 + 1][row] = wg[e].y;
            ws[buf][s_kq * 4 + 2][row] = wg[e].z; ws[buf][s_kq * 4 + 3][row] = wg[e].w;
        }
    };
    f32x16_t acc[2][2];                    // [n tile][m tile]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    fetch(0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += FS_K, buf ^= 1) {
        const bool more = k0 + FS_K < K;
        if (more) fetch(k0 + FS_K);
#pragma unroll
        for (int s = 0; s < FS_K / 2; ++s) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = ws[buf][2 * s + kh][wn * 64 + 32 * i + r];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = xs[buf][2 * s + kh][wm * 64 + 32 * j + r];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (more) stage(buf ^ 1);          // (last read before the barrier that ended the stage before)
        __syncthreads();
    }
    // acc[i][j][v]: n = n0 + wn * 64 + 32 i + 8 (v / 4) + 4 kh + v % 4, m = m0 + wm * 64 + 32 j + r
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + wm * 64 + 32 * j + r;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + wn * 64 + 32 * i + 8 * g + 4 * kh;
                const size_t at = (size_t)m * N + n;
                if (n + 3 < N && (N & 3) == 0 && y_dt == ILLM_F32) {
                    *(float4*)((float*)Y + at) = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1],
                                                             acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < N) st_f(Y, y_dt, at + v, acc[i][j][4 * g + v]);
                }
            }
    }
}

static int g_f32_tile = 0;
extern "C" void illm_set_f32_tile(int t) { g_f32_tile = t == 16 || t == 64 || t == 128 ? t : 0; }

// A kernel that needs more dynamic LDS than it may have without asking: asked for once per device.
template <int T>
static int f32_lds_ready(size_t bytes) {
    static bool ready[64] = {};
    static std::mutex lock;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return ILLM_ERR_LAUNCH;
    std::lock_guard<std::mutex> hold(lock);
    if (!ready[dev]) {
        if (hipFuncSetAttribute((const void*)gemm_f32_mfma_kernel<T>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
            return ILLM_ERR_LAUNCH;
        ready[dev] = true;
    }
    return ILLM_OK;
}

template <int T>
static int launch_f32_mfma(const float* X, const float* W, void* Y, int y_dt, int M, int N, int K, hipStream_t st) {
    const long long mt = (M + T - 1) / T, nt = (N + T - 1) / T, blocks = (nt + 7) / 8 * 8 * mt;
    if (blocks > 0x7fffffffLL) return ILLM_ERR_ARG;
    const size_t lds = (size_t)4 * T * FM_LD * sizeof(float);
    const int rc = f32_lds_ready<T>(lds);
    if (rc != ILLM_OK) return rc;
    hipLaunchKernelGGL(gemm_f32_mfma_kernel<T>, dim3((unsigned)blocks), dim3(256), lds, st, X, W, Y, y_dt, M, N, K, (int)mt);
    return illm_launch_status();
}

// float32 X [M, K] and W [N, K], K % 16 == 0; Y float32 or bfloat16.  Else ILLM_ERR_ARG.
extern "C" int illm_gemm_f32_mfma(const float* X, const float* W, void* Y, int y_dt, int M, int N,
                                  int K, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || (K % 16) || !illm_dtype_ok(y_dt) || !X || !W || !Y)
        return ILLM_ERR_ARG;
    const long long m128 = (M + 127) / 128, b128 = m128 * ((N + 127) / 128);
    const long long b64 = (long long)((M + 63) / 64) * ((N + 63) / 64);
    if (m128 > 65535) return ILLM_ERR_ARG;
    if (K >= 1 << 22)                      // a block's rows would pass 2 GiB
        return illm_gemm_generic(X, ILLM_F32, W, ILLM_F32, Y, y_dt, M, N, K, stream);
    // Short K: writing Y is what counts.  The kernel for it from 512 of its blocks on, unless they are rows and columns
    // beyond the matrix for more than a tenth (then up to K = 112), else blocks of 64 x 64.  us in that kernel / in blocks of
    // 64 x 64 / of 128 x 128: 4,096 rows of 4096 x 16 19 / 32 / 49, x 96 41 / 46 / 47, x 320 108 / 122 / 109;
    // 4,096 of 2048 x 48 18 / 20 / 22; 300 of 32000 x 48 20 / 24 / 32, x 160 46 / 41 / 49; 2,048 of 2048 x 32 11 / 9 / 11,
    // x 128 19 / 17 / 19, x 320 35 / 33 / 34 (x 512 - / 51 / 48).
    const bool few_k = K <= 320;
    const bool is_short = g_f32_tile ? g_f32_tile == 16 : few_k && b128 >= 512 && (K <= 112 || 10 * b64 >= 36 * b128);
    if (is_short) {
        hipLaunchKernelGGL(gemm_f32_short_kernel, dim3((N + FS_T - 1) / FS_T, (unsigned)m128), dim3(256), 0, (hipStream_t)stream,
                           X, W, Y, y_dt, M, N, K);
        return illm_launch_status();
    }
    // Blocks of 128 x 128 finish in rounds of one a compute unit (256 blocks of K = 4,096: 280 us, 512
    // 535, 768 800), those of 64 x 64 in rounds of a quarter of that at 0.9 of the rate (256 91 us, 512
    // 157, 1,024 300): the larger ones where their rounds are nearly full.  Measured at 129 to 2,048
    // rows of the 7B shapes; with 128 x 128 alone, stages of 16 k and one stage ahead, 256 rows took
    // 314 us (4096 x 4096), 318 (12288 x 4096), 829 (4096 x 11008) and 545 (22016 x 4096), now 91, 236,
    // 249 and 438; 2,048 rows 562, 1,584, 1,447 and 2,973, now 540, 1,585, 1,428 and 2,894.
    const bool big = g_f32_tile ? g_f32_tile == 128 : !few_k && 10 * 1024 * ((b128 + 255) / 256) <= 11 * b64;
    return big ? launch_f32_mfma<128>(X, W, Y, y_dt, M, N, K, (hipStream_t)stream)
               : launch_f32_mfma<64>(X, W, Y, y_dt, M, N, K, (hipStream_t)stream);
}


// ---------------------------------------------------------------- up to 128 rows, float32
// The same product for up to 128 float32 rows and K a multiple of 32, bound by reading W once:
// MFMA 16x16x4 float32 with operands straight from memory.  A block of 8 waves takes 16 rows of
// W; the waves take pieces of 32 k in turn (wave w pieces w, w + 8, ...: eight neighbouring
// 128-byte segments of a row at a time).  Lane l reads 16 bytes at k = 4 (l / 16) + 16 q of row
// l % 16, of W and of every 16 rows of X alike: element j of that load is the operand of an
// MFMA whose four k are 4 g + j + 16 q, the same four for both operands, so nothing is
// permuted.  The waves' sums are added through LDS in wave order: the order of a sum depends on
// K only, not on the row's place or on the number of rows.

template <int RT, int CT>                      // tiles of 16 rows of X, tiles of 16 rows of W
__global__ void __launch_bounds__(512)
gemm_rows_f32_mfma_kernel(const float* __restrict__ X, const float* __restrict__ W, void* __restrict__ Y,
                          int y_dt, int M, int N, int K) {
    __shared__ f32x4v_t part[8][RT * CT][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16 * CT;
    const float* wsrc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) wsrc[c] = W + (size_t)min(n0 + 16 * c + r16, N - 1) * K + 4 * g;
    const float* xsrc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) xsrc[t] = X + (size_t)min(16 * t + r16, M - 1) * K + 4 * g;
    f32x4v_t acc[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[t][c] = (f32x4v_t){0.f, 0.f, 0.f, 0.f};
    constexpr int U = RT * CT <= 2 ? 4 : (RT <= 4 ? 2 : 1);   // pieces asked for together
    const int pieces = K / 32;
    for (int p = wave; p < pieces; p += 8 * U) {
        f32x4v_t wr[U][CT][2], xr[U][RT][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k0 = 32 * min(p + 8 * u, pieces - 1);      // (past the end: a piece read again, not used)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    wr[u][c][q] = __builtin_nontemporal_load((const f32x4v_t*)(wsrc[c] + k0 + 16 * q));
#pragma unroll
                for (int t = 0; t < RT; ++t) xr[u][t][q] = *(const f32x4v_t*)(xsrc[t] + k0 + 16 * q);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (p + 8 * u < pieces) {
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int t = 0; t < RT; ++t)
#pragma unroll
                            for (int c = 0; c < CT; ++c)
                                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[u][c][q][j], xr[u][t][q][j],
                                                                                 acc[t][c], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) part[wave][t * CT + c][lane] = acc[t][c];
    __syncthreads();
    // acc[t][c][v]: n = n0 + 16 c + 4 g + v, m = 16 t + r16; a thread adds the eight waves' sums
    for (int e = tid; e < RT * CT * 64; e += 512) {
        const int tc = e >> 6, l = e & 63;
        f32x4v_t sum = part[0][tc][l];
#pragma unroll
        for (int w = 1; w < 8; ++w) sum += part[w][tc][l];
        const int m = 16 * (tc / CT) + (l & 15), n = n0 + 16 * (tc % CT) + 4 * (l >> 4);
        if (m >= M) continue;
        const size_t at = (size_t)m * N + n;
        if (n + 3 < N && (N & 3) == 0 && y_dt == ILLM_F32) {
            *(f32x4v_t*)((float*)Y + at) = sum;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < N) st_f(Y, y_dt, at + v, sum[v]);
        }
    }
}

static int g_rows_f32_tiles = 0;     // tests: W tiles a block (1 or 2); 0: the library's choice
extern "C" void illm_set_rows_f32_tiles(int tiles) { g_rows_f32_tiles = tiles == 1 || tiles == 2 ? tiles : 0; }

// float32 X [M <= 128, K] and W [N, K], K % 32 == 0; Y float32 or bfloat16.  Else ILLM_ERR_ARG.
extern "C" int illm_gemm_rows_f32_mfma(const float* X, const float* W, void* Y, int y_dt, int M, int N,
                                       int K, void* stream) {
    if (M <= 0 || M > 128 || N <= 0 || K <= 0 || (K % 32) || !illm_dtype_ok(y_dt) || !X || !W || !Y)
        return ILLM_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    // two tiles of W a block halve what the blocks read of X together: from 17 rows on, where
    // that is most of the traffic, if there are still two blocks for every compute unit
    // (measured at 64 rows: 22016 x 4096 263 -> 204 us, 12288 x 4096 the same, 4096 x 4096 49 -> 65)
    const int rt = (M + 15) / 16;
    const int ct = g_rows_f32_tiles ? g_rows_f32_tiles : (rt >= 2 && N >= 32 * 512 ? 2 : 1);
    const dim3 grid((N + 16 * ct - 1) / (16 * ct)), block(512);
#define ILLM_ROWS_F32(RT)                                                                             \
    case RT:                                                                                          \
        if (ct == 2)                                                                                  \
            hipLaunchKernelGGL((gemm_rows_f32_mfma_kernel<RT, 2>), grid, block, 0, st, X, W, Y, y_dt, M, N, K); \
        else                                                                                          \
            hipLaunchKernelGGL((gemm_rows_f32_mfma_kernel<RT, 1>), grid, block, 0, st, X, W, Y, y_dt, M, N, K); \
        break;
    switch (rt) {
        ILLM_ROWS_F32(1) ILLM_ROWS_F32(2) ILLM_ROWS_F32(3) ILLM_ROWS_F32(4)
        ILLM_ROWS_F32(5) ILLM_ROWS_F32(6) ILLM_ROWS_F32(7) ILLM_ROWS_F32(8)
    }
#undef ILLM_ROWS_F32
    return illm_launch_status();
}


// ---------------------------------------------------------------- few rows, float32
// The same product for M <= 16 rows of float32 X and float32 W (decoding on the 32-bit path),
// bound by reading W once: a block of 4 waves takes R rows of W for MR rows of X (M rounded up to
// 1, 2, 4, 8 or 16), the waves split K in interleaved pieces of 256, a lane multiplies 4 consecutive k
// of every W row with every X row (plain multiply-adds, float32), and the R * MR sums of a wave
// are added over its lanes by a halving exchange that leaves sum number l in lane l (modulo their number; what is left of
// the lanes' bits is added plainly, in the same tree).  The waves' sums are added in wave order.  The order of a sum
// depends on K only, not on the row's place nor on MR.
// AHEAD: a wave's next piece is asked for before this one is multiplied (few blocks).  Whole pieces are asked for without a
// test.  us, matrices cold, 8 rows of sums for up to 8 of X, one piece at a time -> now, 1 and 4 rows: 4096 x 4096 15.4 / 15.2 ->
// 12.7 / 14.3, 12288 x 4096 35.2 / 36.0 -> 31.9 / 33.9, 22016 x 4096 58.3 / 59.5 -> 55.0 / 56.6 (6.4 TB/s), 4096 x 11008 34.2 /
// 34.5 -> 30.2 / 32.1, 512 x 96 3.7 / 3.8 -> 2.4 / 3.0.  The same bits.
// What stood around the products of a decode step of few rows was launches (5.5 us each between the products of a 7B layer,
// 2 to 3 for a tiny model's), so they are taken into them.  us of norm, product and what follows, as kernels -> in one, 1 / 4
// rows: q|k|v 192 x 96 7.1 / 8.0 -> 3.4 / 4.0, 3072 x 1024 9.7 / 10.6 -> 5.6 / 6.8, 6144 x 2048 16.4 / 18.1 -> 12.2 / 13.4;
// gate and up 2 x 256 x 96 6.2 / 7.3 -> 3.1 / 3.8, 2 x 8192 x 2048 26.2 / 27.5 -> 22.2 / 23.9, 2 x 11008 x 4096 60.5 / 62.2 -> 55.1
// / 56.5; the add costs 0.4.
// NORM: X holds rows whose RMS norm (weight `nw`, `eps`) is to be multiplied: x nw is multiplied, the block, which reads the
// whole rows anyway, sums their squares, and the sums are scaled by 1 / sqrt(mean + eps) at the end.
// EPI GEMV_ADD: float32 Y += the product.  GEMV_ACT: W = [gate | up] of N rows each, a block takes R / 2 of either; Y = the
// activation of the two sums (silu(gate) up, or the clamped one with limit > 0).  GEMV_QKV: the rows of W are the q, k and
// v heads, a block takes four pairs (i, i + hd / 2) of one; q rotated into Y, k rotated and v into the cache.
enum { GEMV_PLAIN = 0, GEMV_ADD = 1, GEMV_ACT = 2, GEMV_QKV = 3 };
struct GemvQkv {
    const float* cos_sin;                  // [positions, hd / 2, 2]
    const int32_t *row_pos, *row_slot, *page_table;
    float *kcache, *vcache;
    int table_stride, page_size, ring, nh, nkv, hd;
};

// v[i] of all lanes summed, sum i (modulo S) in v[0] of lane i: at the step that pairs lanes l and l ^ b a lane keeps the sums
// whose number has l's bit b
template <int S>
static __device__ __forceinline__ void lanes_sums(float (&v)[S], int lane) {
#pragma unroll
    for (int b = 1, n2 = S / 2; b < 64; b <<= 1, n2 >>= 1) {
        const bool up = (lane & b) != 0;
        if (b < S) {
#pragma unroll
            for (int i = 0; i < n2; ++i) {
                const float keep = up ? v[2 * i + 1] : v[2 * i];
                const float send = up ? v[2 * i] : v[2 * i + 1];
                v[i] = keep + __shfl_xor(send, b, ILLM_WAVE);
            }
        } else {
            v[0] += __shfl_xor(v[0], b, ILLM_WAVE);
        }
    }
}

template <int MR, int R, bool AHEAD, bool NORM = false, int EPI = GEMV_PLAIN>
__global__ void __launch_bounds__(256, MR == 4 && !AHEAD ? 4 : 1)
gemv_rows_f32_kernel(const float* __restrict__ X, const float* __restrict__ W, void* __restrict__ Y,
                     int y_dt, int M, int N, int K, const float* __restrict__ nw, float eps, float limit, float alpha, GemvQkv a) {
    constexpr bool HALVES = EPI == GEMV_ACT || EPI == GEMV_QKV;      // the second R / 2 rows of W belong to the first
    constexpr int S = R * MR, RN = HALVES ? R / 2 : R;               // sums; columns (pairs) a block makes
    static_assert(S <= 64 && (S & (S - 1)) == 0, "");
    __shared__ float part[4][S];
    __shared__ float part_ss[4][MR];
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int n0 = blockIdx.x * RN;
    const int head = EPI == GEMV_QKV ? n0 / (a.hd / 2) : 0, pair0 = EPI == GEMV_QKV ? n0 - head * (a.hd / 2) : 0;
    const float *wrow[R], *xrow[MR];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        size_t at = (r < RN ? (size_t)0 : (size_t)N) + min(n0 + r % RN, N - 1);
        if (EPI == GEMV_QKV) at = (size_t)head * a.hd + pair0 + r % RN + (r < RN ? 0 : a.hd / 2);
        wrow[r] = W + at * K + wave * 256;
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) xrow[m] = X + (size_t)min(m, M - 1) * K + wave * 256;
    // (what the lanes that finish q, k and v need is a chain of three loads: its first before W, the next before the lanes'
    // sums, the wait for either behind other work.  All of it at the end took a tiny model's step 2 us a layer longer)
    const bool finishes = EPI == GEMV_QKV && wave == 0 && lane % MR < M && lane < S / 2;
    int pos = 0, slot = 0;
    if (finishes) {
        pos = a.row_pos[lane % MR];
        slot = a.row_slot[lane % MR];
    }
    float acc[R][MR];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;
    float ss[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) ss[m] = 0.f;

    struct Piece { f32x4v_t w[R]; };                         // (W is used once: loads that do not stay in the caches)
    auto load = [&](Piece& p, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r) p.w[r] = __builtin_nontemporal_load((const f32x4v_t*)(wrow[r] + k + lane * 4));
        if (AHEAD) __builtin_amdgcn_sched_barrier(0);        // (else they are put right before their use)
    };
    auto multiply = [&](const Piece& p, int k) __attribute__((always_inline)) {
        const float4 g = NORM ? *(const float4*)(nw + wave * 256 + k + lane * 4) : make_float4(1.f, 1.f, 1.f, 1.f);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float4 x = *(const float4*)(xrow[m] + k + lane * 4);
            if (NORM) {
                ss[m] += (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w);
                x.x *= g.x; x.y *= g.y; x.z *= g.z; x.w *= g.w;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float a = acc[r][m];
                a = fmaf(p.w[r].x, x.x, a);
                a = fmaf(p.w[r].y, x.y, a);
                a = fmaf(p.w[r].z, x.z, a);
                a = fmaf(p.w[r].w, x.w, a);
                acc[r][m] = a;
            }
        }
    };
    const int whole = (K - wave * 256) / 256, n = (whole + 3) / 4;         // this wave's whole pieces: 0, 1024, ...
    if (MR == 8) {                                         // (whole pieces by themselves: 61 -> 63 us for 22016 x 4096)
        for (int k = 0; k + wave * 256 + lane * 4 < K; k += 1024) {
            Piece p;
            load(p, k);
            multiply(p, k);
        }
    } else if (!AHEAD) {
        for (int i = 0; i < n; ++i) {
            Piece p;
            load(p, i * 1024);
            multiply(p, i * 1024);
        }
    } else if (whole > 0) {
        Piece p0, p1;
        load(p0, 0);
        for (int i = 0; i < n; i += 2) {
            load(p1, min(i + 1, n - 1) * 1024);
            multiply(p0, i * 1024);
            if (i + 1 >= n) break;
            load(p0, min(i + 2, n - 1) * 1024);
            multiply(p1, (i + 1) * 1024);
        }
    }
    if (MR != 8 && K % 256 && K / 256 % 4 == wave && lane * 4 < K % 256) {            // the last piece, K is a multiple of 4
        const int k = K / 1024 * 1024;
        Piece p;
        load(p, k);
        multiply(p, k);
    }
    float2 cs = make_float2(1.f, 0.f);
    int page = 0;
    if (finishes) {
        if (head < a.nh + a.nkv) cs = *(const float2*)(a.cos_sin + ((size_t)pos * (a.hd / 2) + pair0 + lane / MR) * 2);
        const int lp = pos / a.page_size;                                  // (`cache_row_offset` in two steps)
        if (head >= a.nh) page = a.page_table[(size_t)slot * a.table_stride + (a.ring > 0 ? lp % a.ring : lp)];
    }
    float v[S];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) v[r * MR + m] = acc[r][m];
    lanes_sums(v, lane);
    if (lane < S) part[wave][lane] = v[0];
    if (NORM) {
        lanes_sums(ss, lane);
        if (lane < MR) part_ss[wave][lane] = ss[0];
    }
    __syncthreads();
    if (wave == 0 && lane < S) {
        float t = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
        const int r = lane / MR, m = lane % MR;
        if (NORM) {
            const float sum = ((part_ss[0][m] + part_ss[1][m]) + part_ss[2][m]) + part_ss[3][m];
            t *= 1.0f / sqrtf(sum / (float)K + eps);
        }
        if (EPI == GEMV_ACT) {
            const float u = __shfl(t, (lane + S / 2) & 63, ILLM_WAVE);     // (of the gates' lanes: the up sum)
            if (limit > 0.f) {
                const float g = fminf(t, limit);
                t = g / (1.0f + expf(-alpha * g)) * (fminf(fmaxf(u, -limit), limit) + 1.0f);
            } else {
                t = (t / (1.0f + expf(-t))) * u;
            }
        }
        if (EPI == GEMV_QKV) {
            const float u = __shfl(t, (lane + S / 2) & 63, ILLM_WAVE);     // (of the first rows' lanes: the partner's sum)
            if (m < M && r < RN) {
                const bool turned = head < a.nh + a.nkv;
                const int kvh = turned ? head - a.nh : head - a.nh - a.nkv;
                float* to = (float*)Y + ((size_t)m * (a.nh + 2 * a.nkv) + head) * a.hd + pair0 + r;
                if (head >= a.nh)
                    to = (turned ? a.kcache : a.vcache) +
                         (((size_t)page * a.nkv + kvh) * a.page_size + pos % a.page_size) * a.hd + pair0 + r;
                to[0] = turned ? t * cs.x - u * cs.y : t;
                to[a.hd / 2] = turned ? t * cs.y + u * cs.x : u;
            }
            return;
        }
        if (m < M && r < RN && n0 + r < N) {
            const size_t at = (size_t)m * N + n0 + r;
            if (EPI == GEMV_ADD) ((float*)Y)[at] += t;
            else st_f(Y, y_dt, at, t);
        }
    }
}

// float32 X [M <= 16, K] and W [N, K], K % 4 == 0; Y float32 or bfloat16.  Else ILLM_ERR_ARG.
extern "C" int illm_gemv_rows_f32(const float* X, const float* W, void* Y, int y_dt, int M, int N,
                                  int K, void* stream) {
    if (M <= 0 || M > 16 || N <= 0 || K <= 0 || (K % 4) || !illm_dtype_ok(y_dt)) return ILLM_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    // (blocks of 16 rows of W were slower than these of 8: 72 against 60 us for 22016 x 4096)
#define ILLM_GEMV(MR, R, AHEAD)                                                                                      \
    hipLaunchKernelGGL((gemv_rows_f32_kernel<MR, R, AHEAD>), dim3((N + R - 1) / R), dim3(256), 0, st, X, W, Y, y_dt, M, N, K, \
                       (const float*)nullptr, 0.f, 0.f, 0.f, GemvQkv{})
    const bool ahead = N <= 8192;                  // (blocks enough hide the loads: 22016 x 4096 of 8 rows 61 -> 70 us)
    if (M > 8) ILLM_GEMV(16, 4, true);
    else if (M > 4) ILLM_GEMV(8, 8, false);
    else if (M > 2) { if (ahead) ILLM_GEMV(4, 8, true); else ILLM_GEMV(4, 8, false); }
    else if (M > 1) { if (ahead) ILLM_GEMV(2, 8, true); else ILLM_GEMV(2, 8, false); }
    else { if (ahead) ILLM_GEMV(1, 8, true); else ILLM_GEMV(1, 8, false); }
#undef ILLM_GEMV
    return illm_launch_status();
}

// The same for M <= 8 rows with what surrounds the product taken in: norm_w [K] (and eps) the RMS norm of X's rows, or null;
// epi 0: Y [M, N] float32 = the product, 1: Y += the product (without a norm), 2: W [2 N, K] = [gate | up], Y = their
// activation (limit 0: silu(gate) up; else the clamped one of `alpha`).
#define ILLM_GEMV_F(MR, AHEAD, NORM, EPI)                                                                             \
    hipLaunchKernelGGL((gemv_rows_f32_kernel<MR, 8, AHEAD, NORM, EPI>), dim3(blocks), dim3(256), 0, (hipStream_t)stream, \
                       X, W, Y, (int)ILLM_F32, M, N, K, norm_w, eps, limit, alpha, qkv)
#define ILLM_GEMV_M(NORM, EPI)                                                                                        \
    do {                                                                                                              \
        if (M > 4) ILLM_GEMV_F(8, false, NORM, EPI);                                                                  \
        else if (M > 2) { if (ahead) ILLM_GEMV_F(4, true, NORM, EPI); else ILLM_GEMV_F(4, false, NORM, EPI); }        \
        else if (M > 1) { if (ahead) ILLM_GEMV_F(2, true, NORM, EPI); else ILLM_GEMV_F((NORM ? 4 : 2), false, NORM, EPI); } \
        else { if (ahead) ILLM_GEMV_F(1, true, NORM, EPI); else ILLM_GEMV_F(1, false, NORM, EPI); }                   \
    } while (0)
// (2 rows with a norm, the next piece not ahead: sums for 4 rows, whose code is the better one: 2 x 8192 x 2048 25.8 -> 23.4 us,
// 2 x 13824 x 5120 93.6 -> 86.1)
extern "C" int illm_gemv_rows_f32_fused(const float* X, const float* W, float* Y, int M, int N, int K, const float* norm_w,
                                        float eps, int epi, float limit, float alpha, void* stream) {
    if (!X || !W || !Y || M <= 0 || M > 8 || N <= 0 || K <= 0 || (K % 4) || epi < GEMV_PLAIN || epi > GEMV_ACT ||
        (norm_w && epi == GEMV_ADD))
        return ILLM_ERR_ARG;
    const bool ahead = N <= 8192 / (epi == GEMV_ACT ? 2 : 1);        // (as above, by rows of W)
    const int cols = epi == GEMV_ACT ? 4 : 8, blocks = (N + cols - 1) / cols;
    const GemvQkv qkv{};
    if (norm_w) {
        if (epi == GEMV_ACT) ILLM_GEMV_M(true, GEMV_ACT);
        else ILLM_GEMV_M(true, GEMV_PLAIN);
    } else {
        if (epi == GEMV_ACT) ILLM_GEMV_M(false, GEMV_ACT);
        else if (epi == GEMV_ADD) ILLM_GEMV_M(false, GEMV_ADD);
        else return illm_gemv_rows_f32(X, W, Y, ILLM_F32, M, N, K, stream);
    }
    return illm_launch_status();
}

// The q|k|v product of M <= 8 single tokens with the rotation of q and k (pairs (i, i + hd / 2) of a head, hd % 8 == 0) and
// the store of k and v: row m at position row_pos[m] of slot row_slot[m].  Y [M, (nh + 2 nkv) hd]: only q is written.
extern "C" int illm_gemv_qkv_f32(const float* X, const float* W, float* Y, int M, int K, const float* norm_w, float eps,
                                 const float* cos_sin, int max_pos, const int32_t* row_pos, const int32_t* row_slot,
                                 float* kcache, float* vcache, const int32_t* page_table, int table_stride, int page_size,
                                 int ring, int nh, int nkv, int hd, void* stream) {
    if (!X || !W || !Y || M <= 0 || M > 8 || K <= 0 || (K % 4) || nh <= 0 || nkv <= 0 || hd <= 0 || (hd % 8) || !cos_sin ||
        max_pos <= 0 || !row_pos || !row_slot || !kcache || !vcache || !page_table || page_size <= 0 || table_stride <= 0 ||
        (nh + 2LL * nkv) * hd > 0x7fffffff)
        return ILLM_ERR_ARG;
    const GemvQkv qkv = {cos_sin, row_pos, row_slot, page_table, kcache, vcache, table_stride, page_size, ring, nh, nkv, hd};
    const int N = (nh + 2 * nkv) * hd, blocks = N / 8;
    const float limit = 0.f, alpha = 0.f;
#define ILLM_GEMV_QKV(NORM)                                                                                           \
    do {                                                                                                              \
        if (M > 4) ILLM_GEMV_F(8, false, NORM, GEMV_QKV);                                                             \
        else if (M > 2) ILLM_GEMV_F(4, true, NORM, GEMV_QKV);                                                         \
        else if (M > 1) ILLM_GEMV_F(2, true, NORM, GEMV_QKV);                                                         \
        else ILLM_GEMV_F(1, true, NORM, GEMV_QKV);                                                                    \
    } while (0)
    if (norm_w) ILLM_GEMV_QKV(true);
    else ILLM_GEMV_QKV(false);
#undef ILLM_GEMV_QKV
    return illm_launch_status();
}
#undef ILLM_GEMV_M
#undef ILLM_GEMV_F
