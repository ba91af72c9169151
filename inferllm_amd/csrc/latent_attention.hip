// Latent attention: every token keeps one low-rank latent row c [R] (RMS-normed) and one rotated
// key part kr [dr] that all heads share; a head's key is [W_uk c | kr] and its value W_uv c.
//
// Rows of several tokens (whole prompts) build every head's keys and values from the step's own
// latent rows (`illm_latent_pack`) and go through the library's prompt attention.  Single tokens
// never build them: with qa_h = [W_uk,h^T q_h | q_h,rot] the score of key j is qa_h . [c_j | kr_j],
// and the weighted sum of values is W_uv,h (sum_j p_j c_j), so one token's attention is a walk over
// the cached latent rows that all heads of a block share (`illm_latent_attn_decode`), followed by
// the small product with W_uv and the output gate (`illm_latent_merge_up`).
//
// Scores, softmax statistics, the norm of the latent, rotation and the running sums are float32.
#include "api.h"
#include "common.h"

// ---------------------------------------------------------------- norm, rotation, cache store
// One block per row of y = [q: H (dn + dr) | down: R + dr | gate: H] (row stride ncols).
// The latent is normed (float32 statistics), the shared key part and every head's rotated query
// part are rotated in pairs (2i, 2i+1), i < rot/2, by the float32 table [max_pos][rot/2][2];
// latent and key part go to the paged cache [page][row][R + dr] and to c_out / kr_out.
__device__ __forceinline__ void
latent_store_row(const int t, void* __restrict__ y, int dt, int ncols, int H, int dn, int dr, int R,
                 int rot, const float* __restrict__ cos_sin, int max_pos,
                 const void* __restrict__ nw, int nw_dt, float eps,
                 const int32_t* __restrict__ row_pos, const int32_t* __restrict__ row_slot,
                 const int32_t* __restrict__ slot_len, void* __restrict__ cache,
                 const int32_t* __restrict__ page_table, int table_stride, int page_size,
                 int ring, void* __restrict__ c_out, void* __restrict__ kr_out,
                 void* __restrict__ cache_t, const bool rotate_q) {
    __shared__ float red[16];
    int pos = row_pos[t];
    const size_t row = (size_t)t * ncols;
    const size_t down = row + (size_t)H * (dn + dr);
    float ss = 0.f;
    for (int i = threadIdx.x; i < R; i += blockDim.x) {
        const float v = ld_f(y, dt, down + i);
        ss += v * v;
    }
    ss = block_sum(ss, red);
    const float scale = 1.0f / sqrtf(ss / (float)R + eps);
    bool store = cache != nullptr;
    size_t dst = 0, dst_t = 0;
    if (store) {
        const int slot = row_slot[t];
        if (ring > 0 && slot_len) {
            // a later row of this step lands on the same ring page: this one is already outside
            const int last_page = (slot_len[slot] - 1) / page_size;
            if (pos / page_size + ring <= last_page) store = false;
        }
        if (store) {
            int lp = pos / page_size;
            if (ring > 0) lp %= ring;
            const int phys = page_table[(size_t)slot * table_stride + lp];
            dst = ((size_t)phys * page_size + (pos % page_size)) * (size_t)(R + dr);
            dst_t = (size_t)phys * R * page_size + (pos % page_size);
        }
    }
    for (int i = threadIdx.x; i < R; i += blockDim.x) {
        const float v = (ld_f(y, dt, down + i) * scale) * ld_f(nw, nw_dt, i);
        if (c_out) st_f(c_out, dt, (size_t)t * R + i, v);
        if (store) st_f(cache, dt, dst + i, v);
        if (store && cache_t) st_f(cache_t, dt, dst_t + (size_t)i * page_size, v);   // [page][dim][row]
    }
    if (pos >= max_pos) pos = max_pos - 1;
    const float* cs = cos_sin ? cos_sin + (size_t)pos * rot : nullptr;   // [rot/2][2]
    const int half = cs ? rot / 2 : 0;
    const size_t ksrc = down + R;
    for (int i = threadIdx.x; i < half; i += blockDim.x) {
        const float c = cs[2 * i], s = cs[2 * i + 1];
        const float u = ld_f(y, dt, ksrc + 2 * i), v = ld_f(y, dt, ksrc + 2 * i + 1);
        const float a = u * c - v * s, b = v * c + u * s;
        if (kr_out) { st_f(kr_out, dt, (size_t)t * dr + 2 * i, a); st_f(kr_out, dt, (size_t)t * dr + 2 * i + 1, b); }
        if (store) { st_f(cache, dt, dst + R + 2 * i, a); st_f(cache, dt, dst + R + 2 * i + 1, b); }
    }
    for (int e = 2 * half + threadIdx.x; e < dr; e += blockDim.x) {       // dims beyond the rotated ones
        const float v = ld_f(y, dt, ksrc + e);
        if (kr_out) st_f(kr_out, dt, (size_t)t * dr + e, v);
        if (store) st_f(cache, dt, dst + R + e, v);
    }
    for (int u = threadIdx.x; rotate_q && u < H * half; u += blockDim.x) {
        const int h = u / half, i = u - h * half;
        const size_t base = row + (size_t)h * (dn + dr) + dn;
        const float c = cs[2 * i], s = cs[2 * i + 1];
        const float a = ld_f(y, dt, base + 2 * i), b = ld_f(y, dt, base + 2 * i + 1);
        st_f(y, dt, base + 2 * i, a * c - b * s);
        st_f(y, dt, base + 2 * i + 1, b * c + a * s);
    }
}

__global__ void __launch_bounds__(256)
latent_rope_store_kernel(void* __restrict__ y, int dt, int ncols, int H, int dn, int dr, int R,
                         int rot, const float* __restrict__ cos_sin, int max_pos,
                         const void* __restrict__ nw, int nw_dt, float eps,
                         const int32_t* __restrict__ row_pos, const int32_t* __restrict__ row_slot,
                         const int32_t* __restrict__ slot_len, void* __restrict__ cache,
                         const int32_t* __restrict__ page_table, int table_stride, int page_size,
                         int ring, void* __restrict__ c_out, void* __restrict__ kr_out,
                         void* __restrict__ cache_t) {
    latent_store_row(blockIdx.x, y, dt, ncols, H, dn, dr, R, rot, cos_sin, max_pos, nw, nw_dt, eps,
                     row_pos, row_slot, slot_len, cache, page_table, table_stride, page_size, ring,
                     c_out, kr_out, cache_t, true);
}

extern "C" int illm_latent_rope_store(void* y, int dt, int ncols, int T, int H, int dn, int dr,
                                      int R, int rot, const float* cos_sin, int max_pos,
                                      const void* norm_w, int norm_dt, float eps,
                                      const int32_t* row_pos, const int32_t* row_slot,
                                      const int32_t* slot_len, void* cache,
                                      const int32_t* page_table, int table_stride, int page_size,
                                      int ring, void* c_out, void* kr_out, void* cache_t,
                                      void* stream) {
    if (T < 0 || H <= 0 || dn < 0 || dr < 0 || R <= 0 || !illm_dtype_ok(dt) || !illm_dtype_ok(norm_dt) ||
        ncols < H * (dn + dr) + R + dr)
        return ILLM_ERR_ARG;
    if (cos_sin && (rot <= 0 || rot > dr || (rot & 1) || max_pos <= 0)) return ILLM_ERR_ARG;
    if (cache && (!page_table || !row_slot || page_size <= 0 || table_stride <= 0)) return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    hipLaunchKernelGGL(latent_rope_store_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, y, dt,
                       ncols, H, dn, dr, R, rot, cos_sin, max_pos, norm_w, norm_dt, eps, row_pos,
                       row_slot, slot_len, cache, page_table, table_stride, page_size, ring, c_out,
                       kr_out, cache_t);
    return illm_launch_status();
}

// ---------------------------------------------------------------- packed rows for prompt attention
// out[t] = [q heads | k heads | v heads], every head P wide: q_h = [y's q_h (dn + dr) | 0],
// k_h = [kvu's key part h (dn) | kr (dr) | 0], v_h = [kvu's value part h (dv) | 0].
// kvu [T, H dn + H dv] is the product of the latent rows with [W_uk ; W_uv].
__global__ void __launch_bounds__(256)
latent_pack_kernel(const void* __restrict__ y, int dt, int ncols, const void* __restrict__ kvu,
                   const void* __restrict__ kr, void* __restrict__ out, int H, int dn, int dr,
                   int dv, int P) {
    const size_t t = blockIdx.x;
    const int HP = H * P, dq = dn + dr;
    const size_t kvrow = t * (size_t)(H * (dn + dv));
    for (int e = threadIdx.x; e < 3 * HP; e += blockDim.x) {
        const int which = e / HP, rem = e - which * HP;
        const int h = rem / P, d = rem - h * P;
        float v = 0.f;
        if (which == 0) {
            if (d < dq) v = ld_f(y, dt, t * ncols + (size_t)h * dq + d);
        } else if (which == 1) {
            if (d < dn) v = ld_f(kvu, dt, kvrow + (size_t)h * dn + d);
            else if (d < dq) v = ld_f(kr, dt, t * dr + (d - dn));
        } else if (d < dv) {
            v = ld_f(kvu, dt, kvrow + (size_t)H * dn + (size_t)h * dv + d);
        }
        st_f(out, dt, t * (size_t)(3 * HP) + e, v);
    }
}

// bfloat16, every width a multiple of 8: 16 bytes a thread and turn (2,964 rows of 16 heads of 192: 57 us an element).
__global__ void __launch_bounds__(256)
latent_pack_vec8_kernel(const bf16_t* __restrict__ y, int ncols, const bf16_t* __restrict__ kvu,
                        const bf16_t* __restrict__ kr, bf16_t* __restrict__ out, int H, int dn, int dr, int dv, int P) {
    const size_t t = blockIdx.x;
    const int HP = H * P, dq = dn + dr;
    const bf16_t* const kv = kvu + t * (size_t)(H * (dn + dv));
    for (int e = threadIdx.x * 8; e < 3 * HP; e += 256 * 8) {
        const int which = e / HP, rem = e - which * HP;
        const int h = rem / P, d = rem - h * P;
        const bf16_t* from = nullptr;
        if (which == 0) {
            if (d < dq) from = y + t * ncols + (size_t)h * dq + d;
        } else if (which == 1) {
            if (d < dn) from = kv + (size_t)h * dn + d;
            else if (d < dq) from = kr + t * dr + (d - dn);
        } else if (d < dv) {
            from = kv + (size_t)H * dn + (size_t)h * dv + d;
        }
        *(uint4*)(out + t * (size_t)(3 * HP) + e) = from ? *(const uint4*)from : make_uint4(0, 0, 0, 0);
    }
}

extern "C" int illm_latent_pack(const void* y, int dt, int ncols, const void* kvu, const void* kr,
                                void* out, int T, int H, int dn, int dr, int dv, int P,
                                void* stream) {
    if (T < 0 || H <= 0 || dn < 0 || dr < 0 || dv <= 0 || P < dn + dr || P < dv || !illm_dtype_ok(dt))
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    if (dt == ILLM_BF16 && (ncols | dn | dr | dv | P) % 8 == 0 &&
        ((uintptr_t)y | (uintptr_t)kvu | (uintptr_t)kr | (uintptr_t)out) % 16 == 0) {
        hipLaunchKernelGGL(latent_pack_vec8_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)y, ncols,
                           (const bf16_t*)kvu, (const bf16_t*)kr, (bf16_t*)out, H, dn, dr, dv, P);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(latent_pack_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, y, dt, ncols,
                       kvu, kr, out, H, dn, dr, dv, P);
    return illm_launch_status();
}

// out[t, h dv + v] = attn[t, h P + v] * sigmoid(y[t, gate_off + h]): the output gate per head.
__global__ void __launch_bounds__(256)
latent_gate_kernel(const void* __restrict__ attn, const void* __restrict__ y, int dt, int ncols,
                   int gate_off, void* __restrict__ out, int H, int dv, int P) {
    const size_t t = blockIdx.x;
    for (int e = threadIdx.x; e < H * dv; e += blockDim.x) {
        const int h = e / dv, v = e - h * dv;
        const float g = ld_f(y, dt, t * ncols + gate_off + h);
        const float a = ld_f(attn, dt, t * (size_t)(H * P) + (size_t)h * P + v);
        st_f(out, dt, t * (size_t)(H * dv) + e, a * (1.0f / (1.0f + expf(-g))));
    }
}

// bfloat16, dv and P multiples of 8: 16 bytes a thread and turn (2,964 rows of 2,048: 17 us an element).
__global__ void __launch_bounds__(256)
latent_gate_vec8_kernel(const bf16_t* __restrict__ attn, const bf16_t* __restrict__ y, int ncols, int gate_off,
                        bf16_t* __restrict__ out, int H, int dv, int P) {
    const size_t t = blockIdx.x;
    for (int e = threadIdx.x * 8; e < H * dv; e += 256 * 8) {
        const int h = e / dv, v = e - h * dv;
        const float g = bf16_to_f32(y[t * ncols + gate_off + h]);
        const uint4 a = *(const uint4*)(attn + t * (size_t)(H * P) + (size_t)h * P + v);
        const float s = 1.0f / (1.0f + expf(-g));
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            o[k] = pack_bf16x2(__uint_as_float(w[k] << 16) * s, __uint_as_float(w[k] & 0xffff0000u) * s);
        *(uint4*)(out + t * (size_t)(H * dv) + e) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

extern "C" int illm_latent_gate(const void* attn, const void* y, int dt, int ncols, int gate_off,
                                void* out, int T, int H, int dv, int P, void* stream) {
    if (T < 0 || H <= 0 || dv <= 0 || P < dv || gate_off < 0 || gate_off + H > ncols || !illm_dtype_ok(dt))
        return ILLM_ERR_ARG;
    if (T == 0) return ILLM_OK;
    if (dt == ILLM_BF16 && (dv | P) % 8 == 0 && ((uintptr_t)attn | (uintptr_t)out) % 16 == 0) {
        hipLaunchKernelGGL(latent_gate_vec8_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)attn,
                           (const bf16_t*)y, ncols, gate_off, (bf16_t*)out, H, dv, P);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(latent_gate_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream, attn, y, dt,
                       ncols, gate_off, out, H, dv, P);
    return illm_launch_status();
}

// ---------------------------------------------------------------- queries against latent rows
struct LatentStore {              // what the store of a row needs (see illm_latent_rope_store)
    int rot, max_pos, nw_dt, table_stride, page_size, ring;
    float eps;
    const float* cos_sin;
    const void* nw;
    const int32_t* row_pos;
    const int32_t* row_slot;
    void* cache;
    void* cache_t;
    const int32_t* page_table;
};

// The rot part of a head's query in LDS (qs[dn ..]) rotated at the row's position.
__device__ __forceinline__ void rotate_in_lds(float* qs, int dn, const LatentStore& st, int b) {
    if (!st.cos_sin) return;
    int pos = st.row_pos[b];
    if (pos >= st.max_pos) pos = st.max_pos - 1;
    const float* cs = st.cos_sin + (size_t)pos * st.rot;
    for (int i = threadIdx.x; i < st.rot / 2; i += blockDim.x) {
        const float c = cs[2 * i], s = cs[2 * i + 1];
        const float a = qs[dn + 2 * i], v = qs[dn + 2 * i + 1];
        qs[dn + 2 * i] = a * c - v * s;
        qs[dn + 2 * i + 1] = v * c + a * s;
    }
    __syncthreads();
}

// qa[b, h] = [sum_d q[b, h, d] W_uk[h dn + d, :] (R) | q[b, h, dn:] (dr)], float32.  grid (B, H).
// FUSED (grid (B, H + 1)): the query's rot part is rotated here, on its way (y keeps the
// unrotated one), and block (b, H) norms, rotates and stores row b's latent and key part.
template <bool FUSED>
__global__ void __launch_bounds__(256)
latent_absorb_q_kernel(void* __restrict__ y, int dt, int ncols, const void* __restrict__ wuk,
                       int w_dt, void* __restrict__ qa, int qa_dt, int H, int dn, int dr, int R,
                       LatentStore st) {
    extern __shared__ __attribute__((aligned(16))) float qs[];
    const int b = blockIdx.x, h = blockIdx.y;
    if (FUSED && h == H) {
        latent_store_row(b, y, dt, ncols, H, dn, dr, R, st.rot, st.cos_sin, st.max_pos, st.nw, st.nw_dt,
                         st.eps, st.row_pos, st.row_slot, nullptr, st.cache, st.page_table,
                         st.table_stride, st.page_size, st.ring, nullptr, nullptr, st.cache_t, false);
        return;
    }
    const size_t src = (size_t)b * ncols + (size_t)h * (dn + dr);
    for (int d = threadIdx.x; d < dn + dr; d += blockDim.x) qs[d] = ld_f(y, dt, src + d);
    __syncthreads();
    if (FUSED) rotate_in_lds(qs, dn, st, b);
    const size_t dst = ((size_t)b * H + h) * (size_t)(R + dr);
    for (int r = threadIdx.x; r < R; r += blockDim.x) {
        float acc = 0.f;
#pragma unroll 8
        for (int d = 0; d < dn; ++d) acc += qs[d] * ld_f(wuk, w_dt, ((size_t)h * dn + d) * R + r);
        st_f(qa, qa_dt, dst + r, acc);
    }
    for (int e = threadIdx.x; e < dr; e += blockDim.x) st_f(qa, qa_dt, dst + R + e, qs[dn + e]);
}

// The same for bfloat16 W_uk with R % 8 == 0 and R <= 512: a thread holds 8 neighbouring latent
// dims (one 16-byte load a row of W_uk) and takes every (256 / (R / 8))-th plain dim; the groups'
// sums are added through LDS in group order.  Taken where the kernel after this would have more blocks than the chip takes at once.
template <bool FUSED>
__global__ void __launch_bounds__(256)
latent_absorb_q_bf16_kernel(void* __restrict__ y, int dt, int ncols,
                            const bf16_t* __restrict__ wuk, void* __restrict__ qa, int qa_dt, int H,
                            int dn, int dr, int R, LatentStore st) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* qs = sm;                       // [dn + dr]
    float* part = sm + dn + dr;           // [groups][R]
    const int b = blockIdx.x, h = blockIdx.y;
    if (FUSED && h == H) {
        latent_store_row(b, y, dt, ncols, H, dn, dr, R, st.rot, st.cos_sin, st.max_pos, st.nw, st.nw_dt,
                         st.eps, st.row_pos, st.row_slot, nullptr, st.cache, st.page_table,
                         st.table_stride, st.page_size, st.ring, nullptr, nullptr, st.cache_t, false);
        return;
    }
    const size_t src = (size_t)b * ncols + (size_t)h * (dn + dr);
    for (int d = threadIdx.x; d < dn + dr; d += 256) qs[d] = ld_f(y, dt, src + d);
    __syncthreads();
    if (FUSED) rotate_in_lds(qs, dn, st, b);
    const int per_row = R / 8, groups = 256 / per_row;
    const int c = threadIdx.x % per_row, g = threadIdx.x / per_row;
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    if (g < groups) {
        const bf16_t* wp = wuk + (size_t)h * dn * R + c * 8;
#pragma unroll 4
        for (int d = g; d < dn; d += groups) {
            const uint4 u = *(const uint4*)(wp + (size_t)d * R);
            const float q = qs[d];
            const uint32_t uw[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i] += q * __uint_as_float(uw[i] << 16);
                acc[2 * i + 1] += q * __uint_as_float(uw[i] & 0xffff0000u);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) part[(size_t)g * R + c * 8 + i] = acc[i];
    }
    __syncthreads();
    const size_t dst = ((size_t)b * H + h) * (size_t)(R + dr);
    for (int r = threadIdx.x; r < R; r += 256) {
        float a = 0.f;
        for (int gg = 0; gg < groups; ++gg) a += part[(size_t)gg * R + r];
        st_f(qa, qa_dt, dst + r, a);
    }
    for (int e = threadIdx.x; e < dr; e += 256) st_f(qa, qa_dt, dst + R + e, qs[dn + e]);
}

// Up to 512 heads of rows: grid (B, H or H + 1, chunks of 128 latent dims), a thread's 8 dims of every 16th plain dim, 8 rows of
// W_uk asked for ahead of the query's way through LDS.  Bound by trips to memory one after another.  With the store, 16
// heads of 128 + 64, us, the kernel above / this: 8 rows of 192 dims 5.1 / 4.4, 320 6.6 / 5.7, 512 7.3 / 6.3; 33 rows
// 5.4 / 5.5, 6.9 / 6.3, 7.8 / 7.6; 64 rows 6.0 / 7.2, 7.8 / 8.9, 9.6 / 10.4.
template <bool FUSED>
__global__ void __launch_bounds__(256)
latent_absorb_q_few_kernel(void* __restrict__ y, int dt, int ncols,
                            const bf16_t* __restrict__ wuk, void* __restrict__ qa, int qa_dt, int H,
                            int dn, int dr, int R, LatentStore st) {
    constexpr int COLS = 128, LANES = COLS / 8, GROUPS = 256 / LANES, AHEAD = 8;
    extern __shared__ __attribute__((aligned(16))) float qs[];           // [dn + dr]
    __shared__ __attribute__((aligned(16))) float part[GROUPS][COLS];
    const int b = blockIdx.x, h = blockIdx.y, r0 = blockIdx.z * COLS;
    if (FUSED && h == H) {
        if (blockIdx.z == 0)
            latent_store_row(b, y, dt, ncols, H, dn, dr, R, st.rot, st.cos_sin, st.max_pos, st.nw, st.nw_dt,
                             st.eps, st.row_pos, st.row_slot, nullptr, st.cache, st.page_table,
                             st.table_stride, st.page_size, st.ring, nullptr, nullptr, st.cache_t, false);
        return;
    }
    const int c = threadIdx.x % LANES, g = threadIdx.x / LANES;
    const bool live = r0 + 8 * c < R;
    const bf16_t* const wp = wuk + (size_t)h * dn * R + (live ? r0 + 8 * c : 0);
    uint4 u[AHEAD];
    auto ask = [&](int d0) __attribute__((always_inline)) {              // (past the last row: the last, times nothing)
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) u[k] = *(const uint4*)(wp + (size_t)min(d0 + g + GROUPS * k, dn - 1) * R);
    };
    if (dn > 0) ask(0);
    loads_asked_for();
    const size_t src = (size_t)b * ncols + (size_t)h * (dn + dr);
    for (int d = threadIdx.x; d < dn + dr; d += 256) qs[d] = ld_f(y, dt, src + d);
    __syncthreads();
    if (FUSED) rotate_in_lds(qs, dn, st, b);
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    for (int d0 = 0; d0 < dn; d0 += GROUPS * AHEAD) {
        if (d0) ask(d0);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const int d = d0 + g + GROUPS * k;
            if (d >= dn) continue;
            const float q = qs[d];
            const uint32_t uw[4] = {u[k].x, u[k].y, u[k].z, u[k].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i] += q * __uint_as_float(uw[i] << 16);
                acc[2 * i + 1] += q * __uint_as_float(uw[i] & 0xffff0000u);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i += 4) *(float4*)&part[g][c * 8 + i] = make_float4(acc[i], acc[i + 1], acc[i + 2], acc[i + 3]);
    __syncthreads();
    const size_t dst = ((size_t)b * H + h) * (size_t)(R + dr);
    for (int r = threadIdx.x; r < min(COLS, R - r0); r += 256) {
        float a = 0.f;
#pragma unroll
        for (int gg = 0; gg < GROUPS; ++gg) a += part[gg][r];
        st_f(qa, qa_dt, dst + r0 + r, a);
    }
    if (blockIdx.z == 0)
        for (int e = threadIdx.x; e < dr; e += 256) st_f(qa, qa_dt, dst + R + e, qs[dn + e]);
}

template <bool FUSED>
static int launch_absorb_q(void* y, int dt, int ncols, const void* wuk, int w_dt, void* qa, int qa_dt,
                           int B, int H, int dn, int dr, int R, const LatentStore& st,
                           hipStream_t stream) {
    const dim3 grid(B, FUSED ? H + 1 : H);
    if (w_dt == ILLM_BF16 && R % 8 == 0 && R <= 512 && R >= 8 && (dn + dr) * sizeof(float) <= 40 * 1024 && (uintptr_t)wuk % 16 == 0) {
        if ((long long)B * H <= 512)
            hipLaunchKernelGGL(latent_absorb_q_few_kernel<FUSED>, dim3(grid.x, grid.y, (R + 127) / 128), dim3(256),
                               (dn + dr) * sizeof(float), stream, y, dt, ncols, (const bf16_t*)wuk, qa, qa_dt, H, dn, dr, R, st);
        else
            hipLaunchKernelGGL(latent_absorb_q_bf16_kernel<FUSED>, grid, dim3(256), ((dn + dr) + (256 / (R / 8)) * R) * sizeof(float),
                               stream, y, dt, ncols, (const bf16_t*)wuk, qa, qa_dt, H, dn, dr, R, st);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(latent_absorb_q_kernel<FUSED>, grid, dim3(256), (size_t)(dn + dr) * sizeof(float),
                       stream, y, dt, ncols, wuk, w_dt, qa, qa_dt, H, dn, dr, R, st);
    return illm_launch_status();
}

extern "C" int illm_latent_absorb_q(const void* y, int dt, int ncols, const void* wuk, int w_dt,
                                    void* qa, int qa_dt, int B, int H, int dn, int dr, int R,
                                    void* stream) {
    if (B < 0 || H <= 0 || H > 65534 || dn < 0 || dr < 0 || R <= 0 || !illm_dtype_ok(dt) ||
        !illm_dtype_ok(w_dt) || !illm_dtype_ok(qa_dt) || ncols < H * (dn + dr))
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
    LatentStore st = {};
    return launch_absorb_q<false>((void*)y, dt, ncols, wuk, w_dt, qa, qa_dt, B, H, dn, dr, R, st,
                                  (hipStream_t)stream);
}

extern "C" int illm_latent_store_absorb(void* y, int dt, int ncols, int B, int H, int dn, int dr,
                                        int R, int rot, const float* cos_sin, int max_pos,
                                        const void* norm_w, int norm_dt, float eps,
                                        const int32_t* row_pos, const int32_t* row_slot, void* cache,
                                        const int32_t* page_table, int table_stride, int page_size,
                                        int ring, void* cache_t, const void* wuk, int w_dt, void* qa,
                                        int qa_dt, void* stream) {
    if (B < 0 || H <= 0 || H > 65534 || dn < 0 || dr < 0 || R <= 0 || !illm_dtype_ok(dt) ||
        !illm_dtype_ok(w_dt) || !illm_dtype_ok(qa_dt) || !illm_dtype_ok(norm_dt) ||
        ncols < H * (dn + dr) + R + dr || !row_pos)
        return ILLM_ERR_ARG;
    if (cos_sin && (rot <= 0 || rot > dr || (rot & 1) || max_pos <= 0)) return ILLM_ERR_ARG;
    if (cache && (!page_table || !row_slot || page_size <= 0 || table_stride <= 0)) return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
    LatentStore st;
    st.rot = rot; st.max_pos = max_pos; st.nw_dt = norm_dt; st.table_stride = table_stride;
    st.page_size = page_size; st.ring = ring; st.eps = eps; st.cos_sin = cos_sin; st.nw = norm_w;
    st.row_pos = row_pos; st.row_slot = row_slot; st.cache = cache; st.cache_t = cache_t;
    st.page_table = page_table;
    return launch_absorb_q<true>(y, dt, ncols, wuk, w_dt, qa, qa_dt, B, H, dn, dr, R, st,
                                 (hipStream_t)stream);
}

// ---------------------------------------------------------------- one token over the latent cache
// grid (sequences, splits, groups of HG = 4 HGW heads); 256 threads.  A split takes whole tiles of
// TK keys aligned at absolute positions; a tile of latent rows goes through LDS once for all heads
// of the block.  Wave w owns heads 4-wise: HGW heads, whose scores, softmax statistics and sums it
// keeps to itself; lane = (key of the tile, part of the row), lanes of one key share the row's
// dims in turn and add their partial scores.  For the sums a lane holds latent dims lane + 64 c.
// Each block leaves (sums [R], max, weight) per head in `partial`.
template <int DT>
__device__ __forceinline__ float lds_elem(const char* ks, size_t i) {
    return DT == ILLM_BF16 ? bf16_to_f32(((const bf16_t*)ks)[i]) : ((const float*)ks)[i];
}

template <int DT, int HGW, int RC>
__global__ void __launch_bounds__(256)
latent_decode_kernel(const float* __restrict__ qa, const void* __restrict__ cache,
                     const int32_t* __restrict__ page_table, int table_stride, int page_size,
                     int ring, const int32_t* __restrict__ seq_slot,
                     const int32_t* __restrict__ seq_len, int len_more,
                     float* __restrict__ partial, int nsplit, int H, int R, int dr, float scale,
                     int window, int TK, int kstride) {
    extern __shared__ __attribute__((aligned(16))) size_t smem_raw[];
    const int D = R + dr, HG = 4 * HGW;
    size_t* rowoff = smem_raw;                         // [TK]
    float* qs = (float*)(rowoff + TK);                 // [HG][D]
    float* ps = qs + (size_t)HG * D;                   // [HG][TK]
    char* ks = (char*)(ps + (size_t)HG * TK);          // [TK][kstride] in storage type
    const int b = blockIdx.x, split = blockIdx.y, h0 = blockIdx.z * HG;
    const int len = seq_len[b] + len_more, slot = seq_slot[b];
    const int lo = window > 0 ? (len - window > 0 ? len - window : 0) : 0;
    const int tile0 = lo / TK, tile1 = (len - 1) / TK + 1;
    const int per = (tile1 - tile0 + nsplit - 1) / nsplit;
    const int ta = tile0 + split * per;
    const int tb = ta + per < tile1 ? ta + per : tile1;
    for (int e = threadIdx.x; e < HG * D; e += 256) {
        const int hh = e / D, d = e - hh * D;
        qs[e] = h0 + hh < H ? qa[((size_t)b * H + h0 + hh) * D + d] : 0.f;
    }
    const int w = wave_index(), lane = threadIdx.x & 63;
    const int NP = 64 / TK, j = lane % TK, part = lane / TK;
    float m[HGW], l[HGW], acc[HGW][RC];
#pragma unroll
    for (int i = 0; i < HGW; ++i) {
        m[i] = -INFINITY; l[i] = 0.f;
#pragma unroll
        for (int c = 0; c < RC; ++c) acc[i][c] = 0.f;
    }
    for (int tile = ta; tile < tb; ++tile) {
        const int k0 = tile * TK;
        __syncthreads();                               // the tile before has been used up
        if (threadIdx.x < TK) {
            const int p = k0 + threadIdx.x;
            int lp = p / page_size;
            if (ring > 0) lp %= ring;
            const int phys = page_table[(size_t)slot * table_stride + lp];
            rowoff[threadIdx.x] = ((size_t)phys * page_size + (p % page_size)) * (size_t)D;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < TK * D; e += 256) {
            const int jj = e / D, d = e - jj * D;
            const int p = k0 + jj;
            const bool ok = p >= lo && p < len;
            if (DT == ILLM_BF16)
                ((bf16_t*)ks)[(size_t)jj * kstride + d] = ok ? ((const bf16_t*)cache)[rowoff[jj] + d] : (bf16_t)0;
            else
                ((float*)ks)[(size_t)jj * kstride + d] = ok ? ((const float*)cache)[rowoff[jj] + d] : 0.f;
        }
        __syncthreads();
        float s[HGW];
#pragma unroll
        for (int i = 0; i < HGW; ++i) s[i] = 0.f;
        for (int d = part; d < D; d += NP) {
            const float kv = lds_elem<DT>(ks, (size_t)j * kstride + d);
#pragma unroll
            for (int i = 0; i < HGW; ++i) s[i] += qs[(size_t)(w * HGW + i) * D + d] * kv;
        }
        for (int off = TK; off < 64; off <<= 1) {
#pragma unroll
            for (int i = 0; i < HGW; ++i) s[i] += __shfl_xor(s[i], off, 64);
        }
        const int p = k0 + j;
        const bool ok = p >= lo && p < len;
#pragma unroll
        for (int i = 0; i < HGW; ++i) {
            const float sc = ok ? s[i] * scale : -INFINITY;
            const float mn = fmaxf(m[i], wave_max(sc));
            const float alpha = m[i] == -INFINITY ? 0.f : expf(m[i] - mn);
            const float pj = ok ? expf(sc - mn) : 0.f;
            l[i] = l[i] * alpha + wave_sum(part == 0 ? pj : 0.f);
            m[i] = mn;
            if (part == 0) ps[(size_t)(w * HGW + i) * TK + j] = pj;
#pragma unroll
            for (int c = 0; c < RC; ++c) acc[i][c] *= alpha;
        }
        __syncthreads();
        const int j_lo = lo - k0 > 0 ? lo - k0 : 0;
        const int j_hi = len - k0 < TK ? len - k0 : TK;
        for (int jj = j_lo; jj < j_hi; ++jj) {
            float pw[HGW];
#pragma unroll
            for (int i = 0; i < HGW; ++i) pw[i] = ps[(size_t)(w * HGW + i) * TK + jj];
#pragma unroll
            for (int c = 0; c < RC; ++c) {
                const int r = lane + 64 * c;
                const float kv = r < R ? lds_elem<DT>(ks, (size_t)jj * kstride + r) : 0.f;
#pragma unroll
                for (int i = 0; i < HGW; ++i) acc[i][c] += pw[i] * kv;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < HGW; ++i) {
        const int h = h0 + w * HGW + i;
        if (h >= H) continue;
        float* dst = partial + (((size_t)b * H + h) * nsplit + split) * (size_t)(R + 4);
#pragma unroll
        for (int c = 0; c < RC; ++c) {
            const int r = lane + 64 * c;
            if (r < R) dst[r] = acc[i][c];
        }
        if (lane == 0) { dst[R] = m[i]; dst[R + 1] = l[i]; }
    }
}

template <int DT, int HGW>
static int launch_latent_decode(int RC, dim3 grid, size_t smem, hipStream_t st, const float* qa,
                                const void* cache, const int32_t* page_table, int table_stride,
                                int page_size, int ring, const int32_t* seq_slot,
                                const int32_t* seq_len, int len_more, float* partial, int nsplit,
                                int H, int R, int dr, float scale, int window, int TK, int kstride) {
#define GO(RC_)                                                                                   \
    do {                                                                                          \
        if (smem > 48 * 1024 &&                                                                   \
            hipFuncSetAttribute((const void*)latent_decode_kernel<DT, HGW, RC_>,                  \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) { \
            (void)hipGetLastError();                                                              \
            return ILLM_ERR_ARG;                                                                  \
        }                                                                                         \
        hipLaunchKernelGGL((latent_decode_kernel<DT, HGW, RC_>), grid, dim3(256), smem, st, qa,   \
                           cache, page_table, table_stride, page_size, ring, seq_slot, seq_len,   \
                           len_more, partial, nsplit, H, R, dr, scale, window, TK, kstride);      \
        return illm_launch_status();                                                              \
    } while (0)
    switch (RC) {
        case 1: GO(1);
        case 2: GO(2);
        case 4: GO(4);
        case 8: GO(8);
        default: GO(16);
    }
#undef GO
}

extern "C" int illm_latent_attn_decode(const float* qa, const void* cache, int dt,
                                       const int32_t* page_table, int table_stride, int page_size,
                                       int ring, const int32_t* seq_slot, const int32_t* seq_len,
                                       int len_more, float* partial, int nsplit, int B, int H,
                                       int R, int dr, float scale, int window, void* stream) {
    if (B < 0 || H <= 0 || R <= 0 || R > 1024 || dr < 0 || nsplit < 1 || nsplit > 65535 ||
        page_size <= 0 || page_size % 8 || table_stride <= 0 || !illm_dtype_ok(dt) || !partial)
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
    const int D = R + dr;
    const int HGW = H >= 16 ? 4 : (H >= 8 ? 2 : 1), HG = 4 * HGW;
    const int groups = (H + HG - 1) / HG;
    if (groups > 65535) return ILLM_ERR_ARG;
    const int rc = (R + 63) / 64;
    const int RC = rc <= 1 ? 1 : (rc <= 2 ? 2 : (rc <= 4 ? 4 : (rc <= 8 ? 8 : 16)));
    // row stride of a tile in LDS: lanes that read the same dim of different keys hit different banks
    int kstride;
    if (dt == ILLM_BF16) {
        kstride = (D + 1) & ~1;
        if ((kstride / 2) % 2 == 0) kstride += 2;
    } else {
        kstride = D | 1;
    }
    const size_t esz = dt == ILLM_BF16 ? 2 : 4;
    int TK = 64;
    size_t smem = 0;
    for (; TK >= 8; TK >>= 1) {
        smem = (size_t)TK * 8 + (size_t)HG * D * 4 + (size_t)HG * TK * 4 + (size_t)TK * kstride * esz;
        if (page_size % TK == 0 && smem <= 128 * 1024) break;
    }
    if (TK < 8) return ILLM_ERR_ARG;
    const dim3 grid(B, nsplit, groups);
    hipStream_t st = (hipStream_t)stream;
#define CALL(DT_, HGW_)                                                                            \
    return launch_latent_decode<DT_, HGW_>(RC, grid, smem, st, qa, cache, page_table, table_stride, \
                                           page_size, ring, seq_slot, seq_len, len_more, partial,   \
                                           nsplit, H, R, dr, scale, window, TK, kstride)
    if (dt == ILLM_BF16) {
        if (HGW == 4) CALL(ILLM_BF16, 4);
        if (HGW == 2) CALL(ILLM_BF16, 2);
        CALL(ILLM_BF16, 1);
    }
    if (HGW == 4) CALL(ILLM_F32, 4);
    if (HGW == 2) CALL(ILLM_F32, 2);
    CALL(ILLM_F32, 1);
#undef CALL
}

// The same walk on the matrix cores for a bfloat16 cache (R % 16 == 0, (R + dr) % 8 == 0, pages of
// a multiple of 32 rows), with a second copy of the latent rows laid out [page][dim][row]
// (`cache_t`).  A block is one wave: a group of 16 heads, one range of keys, 32 keys at a time.
// Scores: MFMA 16x16x32 with 16 keys as the A operand (8 neighbouring dims of a cache row, read in
// operand order straight from memory) and the 16 heads' queries as the B operand (bfloat16, read
// the same way; they stay in the cache): lane (r, q) = (lane % 16, lane / 16) is left with head r's scores of keys 4 q .. 4 q + 3 of
// either half of the 32.  Those 8 weights are the B operand of the second product as they stand:
// its contraction takes the keys in that order, and the A operand, 16 latent dims by these 8 keys,
// is two 8-byte loads from the transposed copy.  Keys that are not seen get weight 0 and their
// loaded values are masked (a freed page may hold anything).  The sums stay in registers
// (R / 16 accumulators of 4); statistics in float32.
// Bound by trips to memory one after another; keys and values are asked for in turn (with the values early 192 + 64 dims took
// 10.3 and 35.8 us for 1 sequence of 3,000 and 32 of 1,000 to 2,000, so 9.4 and 31.2).  Wider latents: the kernel after this.
typedef __bf16 la_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float la_f32x4_t __attribute__((ext_vector_type(4)));

template <int RT>
__global__ void __launch_bounds__(64)
latent_decode_mfma_kernel(const bf16_t* __restrict__ qa, const bf16_t* __restrict__ cache,
                          const bf16_t* __restrict__ cache_t,
                          const int32_t* __restrict__ page_table, int table_stride, int page_size,
                          int ring, const int32_t* __restrict__ seq_slot,
                          const int32_t* __restrict__ seq_len, int len_more,
                          float* __restrict__ partial, int nsplit, int H, int R, int dr, float scale,
                          int window) {
    const int D = R + dr;
    const int b = blockIdx.x, split = blockIdx.y, h0 = blockIdx.z * 16;
    const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
    const int len = seq_len[b] + len_more, slot = seq_slot[b];
    const int lo = window > 0 ? (len - window > 0 ? len - window : 0) : 0;
    const int tile0 = lo / 32, tile1 = (len - 1) / 32 + 1;
    const int per = (tile1 - tile0 + nsplit - 1) / nsplit;
    const int ta = tile0 + split * per;
    const int tb = ta + per < tile1 ? ta + per : tile1;
    asm volatile("" ::"s"(slot));                    // (asked for with the length, not behind the branch)
    if (ta >= tb) {                                  // a range without keys: its sums are not read
        if (q == 0 && h0 + r < H) {
            float* dst = partial + (((size_t)b * H + h0 + r) * nsplit + split) * (size_t)(R + 4);
            dst[R] = -INFINITY;
            dst[R + 1] = 0.f;
        }
        return;
    }
    // the lane's query row (heads beyond the last read the last one's; their results are dropped)
    const bf16_t* qp = qa + ((size_t)b * H + (h0 + r < H ? h0 + r : H - 1)) * D + 8 * q;
    la_f32x4_t o[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) o[rt] = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const la_bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int tile = ta; tile < tb; ++tile) {
        const int k0 = tile * 32;
        int lp = k0 / page_size;
        if (ring > 0) lp %= ring;
        const int phys = page_table[(size_t)slot * table_stride + lp];
        const int rowb = k0 % page_size;
        const bf16_t* kp0 = cache + ((size_t)phys * page_size + rowb + r) * D + 8 * q;
        const bf16_t* kp1 = kp0 + (size_t)16 * D;
        la_f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
        const bf16_t* tp = cache_t + ((size_t)phys * R + r) * page_size + rowb + 4 * q;
        constexpr int CH = RT < 8 ? RT : 8, U = 6;          // row groups whose loads are in flight together, steps of the scores
        uint2 c0[CH], c1[CH];
        // U steps of 32 dims at a time: all their loads are asked for before the first product
        int d0 = 0;
        for (; d0 + 32 * U <= D; d0 += 32 * U) {
            la_bf16x8_t qv[U], ka[U], kb[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                qv[u] = *(const la_bf16x8_t*)(qp + d0 + 32 * u);
                ka[u] = *(const la_bf16x8_t*)(kp0 + d0 + 32 * u);
                kb[u] = *(const la_bf16x8_t*)(kp1 + d0 + 32 * u);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[u], qv[u], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[u], qv[u], s1, 0, 0, 0);
            }
        }
        for (; d0 < D; d0 += 32) {                   // what is left, the last step maybe in part
            la_bf16x8_t qv = zero8, ka = zero8, kb = zero8;
            if (d0 + 8 * q < D) {
                qv = *(const la_bf16x8_t*)(qp + d0);
                ka = *(const la_bf16x8_t*)(kp0 + d0);
                kb = *(const la_bf16x8_t*)(kp1 + d0);
            }
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qv, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, qv, s1, 0, 0, 0);
        }
        float sc[8];
        bool ok[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p0 = k0 + 4 * q + i, p1 = p0 + 16;
            ok[i] = p0 >= lo && p0 < len;
            ok[4 + i] = p1 >= lo && p1 < len;
            sc[i] = ok[i] ? s0[i] * scale : -INFINITY;
            sc[4 + i] = ok[4 + i] ? s1[i] * scale : -INFINITY;
        }
        float mt = sc[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mt = fmaxf(mt, sc[i]);
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float mn = fmaxf(m, mt);
        const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
        float pw[8], ls = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            pw[i] = ok[i] ? expf(sc[i] - mn) : 0.f;
            ls += pw[i];
        }
        ls += __shfl_xor(ls, 16, 64);
        ls += __shfl_xor(ls, 32, 64);
        l = l * alpha + ls;
        m = mn;
        uint4 pu;
        pu.x = pack_bf16x2(pw[0], pw[1]); pu.y = pack_bf16x2(pw[2], pw[3]);
        pu.z = pack_bf16x2(pw[4], pw[5]); pu.w = pack_bf16x2(pw[6], pw[7]);
        const la_bf16x8_t pv = *(const la_bf16x8_t*)&pu;
        const uint32_t k01 = (ok[0] ? 0xffffu : 0u) | (ok[1] ? 0xffff0000u : 0u);
        const uint32_t k23 = (ok[2] ? 0xffffu : 0u) | (ok[3] ? 0xffff0000u : 0u);
        const uint32_t k45 = (ok[4] ? 0xffffu : 0u) | (ok[5] ? 0xffff0000u : 0u);
        const uint32_t k67 = (ok[6] ? 0xffffu : 0u) | (ok[7] ? 0xffff0000u : 0u);
#pragma unroll
        for (int r0 = 0; r0 < RT; r0 += CH) {
#pragma unroll
            for (int u = 0; u < CH; ++u) {
                const int rt = (r0 + u) * 16 < R ? r0 + u : 0;      // beyond R: loaded, not used
                c0[u] = *(const uint2*)(tp + (size_t)rt * 16 * page_size);
                c1[u] = *(const uint2*)(tp + (size_t)rt * 16 * page_size + 16);
            }
#pragma unroll
            for (int u = 0; u < CH; ++u) {
                const int rt = r0 + u;
                if (rt * 16 < R) {
                    uint4 cu;
                    cu.x = c0[u].x & k01; cu.y = c0[u].y & k23; cu.z = c1[u].x & k45; cu.w = c1[u].y & k67;
                    o[rt][0] *= alpha; o[rt][1] *= alpha; o[rt][2] *= alpha; o[rt][3] *= alpha;
                    o[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const la_bf16x8_t*)&cu, pv, o[rt], 0, 0, 0);
                }
            }
        }
    }
    // o[rt][i] = sum of head h0 + r over latent dim 16 rt + 4 q + i
    const int h = h0 + r;
    if (h < H) {
        float* dst = partial + (((size_t)b * H + h) * nsplit + split) * (size_t)(R + 4);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (rt * 16 < R) {
                *(la_f32x4_t*)(dst + rt * 16 + 4 * q) = o[rt];       // rows of R + 4 floats: 16-byte aligned
            }
        }
        if (q == 0) { dst[R] = m; dst[R + 1] = l; }
    }
}

// The same by four waves a block where R > 256: a wave takes every fourth step of 32 dims of the scores, whose parts
// meet in LDS, then the softmax (each wave for itself) and a quarter of the latent dims of the sums: a tile's keys and values, 90 KB
// that a single wave asks for in five turns, are one trip of four waves.  U: steps a wave, 4 U >= D / 32.
// One wave a block -> this, us, 16 heads of 512 + 64 dims: 1 sequence of 600 / 3,000 keys 8.9 / 15.4 -> 5.9 / 9.7, 8 of 400 9.7 ->
// 6.5, 8 of 62 to 1,040 12.6 -> 10.7, 16 of 1,000 16.2 -> 13.2, 32 of 1,500 34.6 -> 33.7, 64 of 2,000 79.7 -> 78.1.
template <int U>
__global__ void __launch_bounds__(256)
latent_decode_mfma_wide_kernel(const bf16_t* __restrict__ qa, const bf16_t* __restrict__ cache, const bf16_t* __restrict__ cache_t,
                               const int32_t* __restrict__ page_table, int table_stride, int page_size, int ring,
                               const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_len, int len_more,
                               float* __restrict__ partial, int nsplit, int H, int R, int dr, float scale, int window) {
    constexpr int NV = 8;                                  // row groups of 16 latent dims a wave: R <= 512
    __shared__ la_f32x4_t part[2][4][2][64];
    const int D = R + dr;
    const int b = blockIdx.x, split = blockIdx.y, h0 = blockIdx.z * 16;
    const int lane = threadIdx.x & 63, w = wave_index(), r = lane & 15, q = lane >> 4;
    const int len = seq_len[b] + len_more, slot = seq_slot[b];
    const int lo = window > 0 ? (len - window > 0 ? len - window : 0) : 0;
    const int tile0 = lo / 32, tile1 = (len - 1) / 32 + 1;
    const int per = (tile1 - tile0 + nsplit - 1) / nsplit;
    const int ta = tile0 + split * per;
    const int tb = ta + per < tile1 ? ta + per : tile1;
    asm volatile("" ::"s"(slot));                    // (asked for with the length, not behind the branch)
    const int h = h0 + r;
    float* const dst = partial + (((size_t)b * H + min(h, H - 1)) * nsplit + split) * (size_t)(R + 4);
    if (ta >= tb) {                                  // a range without keys: its sums are not read
        if (w == 0 && q == 0 && h < H) {
            dst[R] = -INFINITY;
            dst[R + 1] = 0.f;
        }
        return;
    }
    // the wave's dims of the lane's query row (heads beyond the last read the last one's; steps past the end are zeros)
    const bf16_t* qp = qa + ((size_t)b * H + min(h, H - 1)) * D;
    const la_bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    int at[U];
    bool there[U];
    la_bf16x8_t qv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int d = 32 * (w + 4 * u) + 8 * q;
        there[u] = d < D;
        at[u] = there[u] ? d : 0;
        qv[u] = *(const la_bf16x8_t*)(qp + at[u]);
    }
    la_f32x4_t o[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) o[v] = (la_f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    for (int tile = ta; tile < tb; ++tile) {
        const int k0 = tile * 32;
        int lp = k0 / page_size;
        if (ring > 0) lp %= ring;
        const int phys = page_table[(size_t)slot * table_stride + lp];
        const int rowb = k0 % page_size;
        const bf16_t* kp0 = cache + ((size_t)phys * page_size + rowb + r) * D;
        const bf16_t* kp1 = kp0 + (size_t)16 * D;
        const bf16_t* tp = cache_t + ((size_t)phys * R + r) * page_size + rowb + 4 * q;
        la_bf16x8_t ka[U], kb[U];
        uint2 c0[NV], c1[NV];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ka[u] = *(const la_bf16x8_t*)(kp0 + at[u]);
            kb[u] = *(const la_bf16x8_t*)(kp1 + at[u]);
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const size_t row = (size_t)min((w * NV + v) * 16, R - 16) * page_size;      // beyond R: loaded, not used
            c0[v] = *(const uint2*)(tp + row);
            c1[v] = *(const uint2*)(tp + row + 16);
        }
        __builtin_amdgcn_sched_barrier(0);           // (else every product's loads are put right before it)
        la_f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const la_bf16x8_t x = there[u] ? qv[u] : zero8;
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(there[u] ? ka[u] : zero8, x, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(there[u] ? kb[u] : zero8, x, s1, 0, 0, 0);
        }
        la_f32x4_t (*sums)[2][64] = part[tile & 1];
        sums[w][0][lane] = s0;
        sums[w][1][lane] = s1;
        __syncthreads();
        s0 = (sums[0][0][lane] + sums[1][0][lane]) + (sums[2][0][lane] + sums[3][0][lane]);
        s1 = (sums[0][1][lane] + sums[1][1][lane]) + (sums[2][1][lane] + sums[3][1][lane]);
        float sc[8];
        bool ok[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p0 = k0 + 4 * q + i, p1 = p0 + 16;
            ok[i] = p0 >= lo && p0 < len;
            ok[4 + i] = p1 >= lo && p1 < len;
            sc[i] = ok[i] ? s0[i] * scale : -INFINITY;
            sc[4 + i] = ok[4 + i] ? s1[i] * scale : -INFINITY;
        }
        float mt = sc[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mt = fmaxf(mt, sc[i]);
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float mn = fmaxf(m, mt);
        const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
        float pw[8], ls = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            pw[i] = ok[i] ? expf(sc[i] - mn) : 0.f;
            ls += pw[i];
        }
        ls += __shfl_xor(ls, 16, 64);
        ls += __shfl_xor(ls, 32, 64);
        l = l * alpha + ls;
        m = mn;
        uint4 pu;
        pu.x = pack_bf16x2(pw[0], pw[1]); pu.y = pack_bf16x2(pw[2], pw[3]);
        pu.z = pack_bf16x2(pw[4], pw[5]); pu.w = pack_bf16x2(pw[6], pw[7]);
        const la_bf16x8_t pv = *(const la_bf16x8_t*)&pu;
        const uint32_t k01 = (ok[0] ? 0xffffu : 0u) | (ok[1] ? 0xffff0000u : 0u);
        const uint32_t k23 = (ok[2] ? 0xffffu : 0u) | (ok[3] ? 0xffff0000u : 0u);
        const uint32_t k45 = (ok[4] ? 0xffffu : 0u) | (ok[5] ? 0xffff0000u : 0u);
        const uint32_t k67 = (ok[6] ? 0xffffu : 0u) | (ok[7] ? 0xffff0000u : 0u);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            uint4 cu;
            cu.x = c0[v].x & k01; cu.y = c0[v].y & k23; cu.z = c1[v].x & k45; cu.w = c1[v].y & k67;
            o[v][0] *= alpha; o[v][1] *= alpha; o[v][2] *= alpha; o[v][3] *= alpha;
            o[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const la_bf16x8_t*)&cu, pv, o[v], 0, 0, 0);
        }
    }
    // o[v][i] = sum of head h over latent dim 16 (8 w + v) + 4 q + i
    if (h < H) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int d = (w * NV + v) * 16;
            if (d < R) *(la_f32x4_t*)(dst + d + 4 * q) = o[v];               // rows of R + 4 floats: 16-byte aligned
        }
        if (w == 0 && q == 0) { dst[R] = m; dst[R + 1] = l; }
    }
}

extern "C" int illm_latent_attn_decode_mfma(const void* qa, const void* cache, const void* cache_t,
                                            const int32_t* page_table, int table_stride,
                                            int page_size, int ring, const int32_t* seq_slot,
                                            const int32_t* seq_len, int len_more, float* partial,
                                            int nsplit, int B, int H, int R, int dr, float scale,
                                            int window, void* stream) {
    if (B < 0 || H <= 0 || R <= 0 || R > 512 || R % 16 || dr < 0 || (R + dr) % 8 || nsplit < 1 ||
        nsplit > 65535 || page_size <= 0 || page_size % 32 || table_stride <= 0 || !partial ||
        !cache || !cache_t)
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
    const int groups = (H + 15) / 16;
    if (groups > 65535) return ILLM_ERR_ARG;
    const dim3 grid(B, nsplit, groups);
    hipStream_t st = (hipStream_t)stream;
#define GO(KERNEL, THREADS)                                                                        \
    hipLaunchKernelGGL(KERNEL, grid, dim3(THREADS), 0, st, (const bf16_t*)qa, (const bf16_t*)cache, (const bf16_t*)cache_t, \
                       page_table, table_stride, page_size, ring, seq_slot, seq_len, len_more, partial, nsplit, H, R, dr, scale, \
                       window)
    if (R <= 64) GO(latent_decode_mfma_kernel<4>, 64);
    else if (R <= 128) GO(latent_decode_mfma_kernel<8>, 64);
    else if (R <= 256) GO(latent_decode_mfma_kernel<16>, 64);
    else if (R + dr <= 512) GO(latent_decode_mfma_wide_kernel<4>, 256);
    else if (R + dr <= 640) GO(latent_decode_mfma_wide_kernel<5>, 256);
    else if (R + dr <= 1024) GO(latent_decode_mfma_wide_kernel<8>, 256);
    else GO(latent_decode_mfma_kernel<32>, 64);
#undef GO
    return illm_launch_status();
}

// grid (B, H, chunks of 32 value dims): combine the splits, multiply the combined latent sum by
// W_uv's rows of the head (a wave a value dim, lanes over the latent dims) and by the head's
// output gate.  Every chunk's block combines the splits for itself, those up to the last that holds keys (the
// ranges are cut for the longest sequence): a few by a thread a dim, more in 16-byte loads by all threads, eight
// loads in flight either way, in an order that their number and R fix (512 dims: 63 ranges 10.5 -> 7.7 us with a
// thread a dim walking all of them one by one, 16 of 64 sequences 28.4 -> 22.3; 128 dims: 64 ranges 7.5 -> 6.5, 4 ranges 5.9
// -> 6.0, and 7.2 with the second pass through LDS).
__global__ void __launch_bounds__(256)
latent_merge_up_kernel(const float* __restrict__ partial, int nsplit, const void* __restrict__ wuv,
                       int w_dt, const void* __restrict__ y, int dt, int ncols, int gate_off,
                       void* __restrict__ out, int H, int R, int dv) {
    // [R] combined sums, [nsplit] weights, then, on 16 bytes, [1024] where R % 4 == 0
    extern __shared__ __attribute__((aligned(16))) float ol[];
    float* ws = ol + R;
    __shared__ int filled;                             // ranges up to the last that holds keys
    const int b = blockIdx.x, h = blockIdx.y;
    const float* base = partial + ((size_t)b * H + h) * nsplit * (size_t)(R + 4);
    const int w = wave_index(), lane = threadIdx.x & 63;
    if (w == 0) {
        // the ranges' (max, sum), asked for together: lane s holds range s, s + 64, ...; weights exp(m_s - M) / total
        auto at = [&](int s, int i, float none) __attribute__((always_inline)) {
            return s < nsplit ? base[(size_t)s * (R + 4) + R + i] : none;
        };
        const float m0 = at(lane, 0, -INFINITY), l0 = at(lane, 1, 0.f);
        float M = m0;
        for (int s = lane + 64; s < nsplit; s += 64) M = fmaxf(M, at(s, 0, -INFINITY));
        M = wave_max(M);
        float tot = 0.f, e0 = 0.f;
        int last = 0;
        for (int s0 = 0; s0 < nsplit; s0 += 64) {
            const float ms = s0 ? at(s0 + lane, 0, -INFINITY) : m0, ls = s0 ? at(s0 + lane, 1, 0.f) : l0;
            const float e = ms == -INFINITY ? 0.f : expf(ms - M);
            tot += ls * e;
            if (s0) { if (s0 + lane < nsplit) ws[s0 + lane] = e; }
            else e0 = e;
            const unsigned long long some = __ballot(ms != -INFINITY);
            if (some) last = s0 + 64 - __clzll(some);
        }
        tot = wave_sum(tot);
        if (lane == 0) filled = last;
        if (lane < nsplit) ws[lane] = e0 / tot;
        for (int s = lane + 64; s < nsplit; s += 64) ws[s] = ws[s] / tot;
    }
    __syncthreads();
    // (few ranges, narrow latents: walking them costs less than the second pass through LDS)
    const bool few = filled <= (R <= 256 ? 24 : 8);
    if (!few && R % 4 == 0 && R <= 1024 && (uintptr_t)partial % 16 == 0) {
        // a thread takes four neighbouring dims of every `turns`-th range, eight loads in flight
        const int r4 = R / 4, turns = 256 / r4, at = threadIdx.x % r4, mine = threadIdx.x / r4;
        float* sums = ol + ((R + nsplit + 3) & ~3);    // [turns][R]
        if (mine < turns) {
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int s0 = mine; s0 < filled; s0 += 8 * turns) {
                float4 v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int s = s0 + u * turns;
                    v[u] = *(const float4*)(base + (size_t)(s < filled ? s : s0) * (R + 4) + 4 * at);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int s = s0 + u * turns;
                    const float g = s < filled ? ws[s] : 0.f;
                    a.x += v[u].x * g; a.y += v[u].y * g; a.z += v[u].z * g; a.w += v[u].w * g;
                }
            }
            *(float4*)(sums + (size_t)mine * R + 4 * at) = a;
        }
        __syncthreads();
        for (int r = threadIdx.x; r < R; r += 256) {
            float a = sums[r];
            for (int t = 1; t < turns; ++t) a += sums[(size_t)t * R + r];
            ol[r] = a;
        }
    } else {
        // a thread a dim, range after range, eight loads in flight
        for (int r = threadIdx.x; r < R; r += 256) {
            float a = 0.f;
            for (int s0 = 0; s0 < filled; s0 += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = base[(size_t)min(s0 + u, filled - 1) * (R + 4) + r];
#pragma unroll
                for (int u = 0; u < 8; ++u) a += s0 + u < filled ? v[u] * ws[s0 + u] : 0.f;
            }
            ol[r] = a;
        }
    }
    __syncthreads();
    const float g = ld_f(y, dt, (size_t)b * ncols + gate_off + h);
    const float gate = 1.0f / (1.0f + expf(-g));
    if (w_dt == ILLM_BF16 && R % 8 == 0) {
        // 16-byte loads: a lane takes 8 neighbouring latent dims of a row of W_uv
        const bf16_t* wp = (const bf16_t*)wuv;
        const int v_end = min(dv, (int)(blockIdx.z + 1) * 32);
        for (int v0 = blockIdx.z * 32 + 4 * w; v0 < v_end; v0 += 16) {   // four rows of W_uv in flight a wave
            float dot[4] = {0.f, 0.f, 0.f, 0.f};
            for (int r = lane * 8; r < R; r += 512) {
                uint4 u[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int v = v0 + j < v_end ? v0 + j : v_end - 1;
                    u[j] = *(const uint4*)(wp + ((size_t)h * dv + v) * R + r);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t uw[4] = {u[j].x, u[j].y, u[j].z, u[j].w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        dot[j] += __uint_as_float(uw[i] << 16) * ol[r + 2 * i];
                        dot[j] += __uint_as_float(uw[i] & 0xffff0000u) * ol[r + 2 * i + 1];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = wave_sum(dot[j]);
                if (lane == 0 && v0 + j < v_end)
                    st_f(out, dt, (size_t)b * H * dv + (size_t)h * dv + v0 + j, d * gate);
            }
        }
        return;
    }
    const int v_hi = min(dv, (int)(blockIdx.z + 1) * 32);
    for (int v = blockIdx.z * 32 + w; v < v_hi; v += 4) {
        const size_t wr = ((size_t)h * dv + v) * R;
        float dot = 0.f;
        for (int r = lane; r < R; r += 64) dot += ld_f(wuv, w_dt, wr + r) * ol[r];
        dot = wave_sum(dot);
        if (lane == 0) st_f(out, dt, (size_t)b * H * dv + (size_t)h * dv + v, dot * gate);
    }
}

// The same for 256 < R <= 512 and bfloat16 W_uv: everything is asked for at once, the block's 32 rows of W_uv (eight a wave),
// the ranges' statistics and the first 16 ranges' sums, whether they hold keys or not (what a range without keys holds is
// dropped).  us, 128 value dims, one trip after another -> this: one row and 19 ranges 6.6 -> 5.4,
// 8 rows of 13 ranges 8.0 -> 6.1, of up to 33 8.4 -> 7.2; 16 of 32 10.0 both, 32 rows and more, whose blocks are more than the
// chip takes at once and hide each other's trips, 15.3 -> 19.2.  Blocks of one head follow each other 8 apart where heads are a
// multiple of 8: its rows of W_uv stay in one XCD's L2.
__global__ void __launch_bounds__(256)
latent_merge_up_wide_kernel(const float* __restrict__ partial, int nsplit, const bf16_t* __restrict__ wuv,
                            const void* __restrict__ y, int dt, int ncols, int gate_off, void* __restrict__ out, int H, int R,
                            int dv) {
    extern __shared__ __attribute__((aligned(16))) float ws[];      // [nsplit] weights
    __shared__ __attribute__((aligned(16))) float sums[2][512];
    __shared__ int filled;                                // ranges up to the last that holds keys
    const int h = blockIdx.x, b = blockIdx.y, lane = threadIdx.x & 63, w = wave_index();
    const float* const base = partial + ((size_t)b * H + h) * nsplit * (size_t)(R + 4);
    auto stat = [&](int s, int i, float none) __attribute__((always_inline)) {
        return s < nsplit ? base[(size_t)s * (R + 4) + R + i] : none;
    };
    float m0 = -INFINITY, l0 = 0.f;
    if (w == 0) { m0 = stat(lane, 0, -INFINITY); l0 = stat(lane, 1, 0.f); }
    // a thread takes four neighbouring dims of every other range
    const int dim = (threadIdx.x & 127) * 4, mine = threadIdx.x >> 7;
    float4 v[8];
    auto ask = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            v[u] = *(const float4*)(base + (size_t)min(s0 + 2 * u + mine, nsplit - 1) * (R + 4) + min(dim, R - 4));
    };
    ask(0);
    const float gv = ld_f(y, dt, (size_t)b * ncols + gate_off + h);
    const int at = min(lane * 8, R - 8), v0 = blockIdx.z * 32 + 8 * w;
    uint4 up[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) up[j] = *(const uint4*)(wuv + ((size_t)h * dv + min(v0 + j, dv - 1)) * R + at);
    loads_asked_for();
    if (w == 0) {
        // lane s holds range s, s + 64, ...; weights exp(m_s - M) / total
        float M = m0;
        for (int s = lane + 64; s < nsplit; s += 64) M = fmaxf(M, stat(s, 0, -INFINITY));
        M = wave_max(M);
        float tot = 0.f;
        int last = 0;
        for (int s0 = 0; s0 < nsplit; s0 += 64) {
            const float ms = s0 ? stat(s0 + lane, 0, -INFINITY) : m0, ls = s0 ? stat(s0 + lane, 1, 0.f) : l0;
            const float e = ms == -INFINITY ? 0.f : expf(ms - M);
            tot += ls * e;
            if (s0 + lane < nsplit) ws[s0 + lane] = e;
            const unsigned long long some = __ballot(ms != -INFINITY);
            if (some) last = s0 + 64 - __clzll(some);
        }
        tot = wave_sum(tot);
        if (lane == 0) filled = last;
        for (int s = lane; s < nsplit; s += 64) ws[s] = ws[s] / tot;
    }
    __syncthreads();
    const int ranges = filled;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < ranges; s0 += 16) {
        if (s0) ask(s0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int s = s0 + 2 * u + mine;
            if (s >= ranges) continue;
            const float g = ws[s];
            a.x += v[u].x * g; a.y += v[u].y * g; a.z += v[u].z * g; a.w += v[u].w * g;
        }
    }
    *(float4*)&sums[mine][dim] = a;
    __syncthreads();
    const float gate = 1.0f / (1.0f + expf(-gv));
    float c[8], dot[8];
    const bool live = lane * 8 < R;
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = live ? sums[0][at + i] + sums[1][at + i] : 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t uw[4] = {up[j].x, up[j].y, up[j].z, up[j].w};
        dot[j] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            dot[j] += __uint_as_float(uw[i] << 16) * c[2 * i];
            dot[j] += __uint_as_float(uw[i] & 0xffff0000u) * c[2 * i + 1];
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int j = 0; j < 8; ++j) dot[j] += __shfl_xor(dot[j], o, 64);
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (lane == j && v0 + j < dv) st_f(out, dt, (size_t)b * H * dv + (size_t)h * dv + v0 + j, dot[j] * gate);
}

extern "C" int illm_latent_merge_up(const float* partial, int nsplit, const void* wuv, int w_dt,
                                    const void* y, int dt, int ncols, int gate_off, void* out,
                                    int B, int H, int R, int dv, void* stream) {
    if (B < 0 || H <= 0 || H > 65535 || R <= 0 || dv <= 0 || nsplit < 1 || !illm_dtype_ok(dt) ||
        !illm_dtype_ok(w_dt) || gate_off < 0 || gate_off + H > ncols)
        return ILLM_ERR_ARG;
    if (B == 0) return ILLM_OK;
    if ((dv + 31) / 32 > 65535) return ILLM_ERR_ARG;
    if ((long long)B * H <= 128 && R > 256 && R <= 512 && R % 8 == 0 && w_dt == ILLM_BF16 && nsplit <= 8192 &&
        ((uintptr_t)partial | (uintptr_t)wuv) % 16 == 0) {
        hipLaunchKernelGGL(latent_merge_up_wide_kernel, dim3(H, B, (dv + 31) / 32), dim3(256), (size_t)nsplit * sizeof(float),
                           (hipStream_t)stream, partial, nsplit, (const bf16_t*)wuv, y, dt, ncols, gate_off, out, H, R, dv);
        return illm_launch_status();
    }
    hipLaunchKernelGGL(latent_merge_up_kernel, dim3(B, H, (dv + 31) / 32), dim3(256), (size_t)(R + nsplit + 4 + (R % 4 == 0 && R <= 1024 ? 1024 : 0)) * sizeof(float),
                       (hipStream_t)stream, partial, nsplit, wuv, w_dt, y, dt, ncols, gate_off, out,
                       H, R, dv);
    return illm_launch_status();
}
