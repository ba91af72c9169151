// The inner loop of products of many bfloat16 rows, sums in float32 (MFMA 16x16x32): a block of eight waves in two groups
// of four, one wave of each on every SIMD.  The groups take turns: while one multiplies, the other reads its next operands
// from LDS and asks memory for later stages, and a barrier after each turn changes them over, so that the matrix cores of
// a SIMD always have one wave's products and its LDS and load instructions are the other wave's.
//
// A block's tile is 2 (groups) x MT tiles of 16 rows of X by 4 (waves of a group) x NT tiles of 16 rows of W.  A wave's MT
// tiles are MT0 and MT1, its NT tiles NT0 and NT1; a stage is 64 k and has four turns a group, one for each pair of those
// parts: X0 W0, X0 W1, X1 W1, X1 W0.  Stages stand in two sets of LDS arrays, each part in an array of its own: X0, X1, W0
// and W1 of stage s are read in turns 0, 2, 3 (of the stage before) and 1.  Two turns after its last reads a part is
// overwritten by the loads of the stage two further on, which so have six turns to arrive: no turn waits for the newest
// five, and every wait is a count (MID below).  Every sum takes the steps of 32 k one after the other.
//
// What bounds it: LDS.  256 x 256 outputs read 196 KB and write 64 KB of LDS a stage, 2,080 of its cycles, beside 2,048 of
// the matrix cores; with real numbers instead of zeros the chip's power does (8,192^3: 1.78 PFLOP/s of zeros, 1.52 of
// normal deviates).  Four waves of 128 x 128 (131 KB a stage, one wave a SIMD): 0.93 to 1.08.
#pragma once
#include "common.h"

typedef __bf16 turns_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float turns_f32x4_t __attribute__((ext_vector_type(4)));

template <int VM>
__device__ __forceinline__ void turns_wait_loads() {
    static_assert(VM < 64, "the wait count");
    __builtin_amdgcn_s_waitcnt(0x0f70 | (VM & 15) | ((VM >> 4) << 14));
}

// The column, within a wave's columns of one part, of row rr of the part's tile i: with two tiles a lane's sums are 8
// neighbouring columns of a row of X, with one 4.
template <int NTH>
__device__ __forceinline__ int turns_column(int i, int rr) {
    return NTH == 2 ? (rr >> 2) * 8 + i * 4 + (rr & 3) : rr;
}

template <int MT0, int MT1, int NT0, int NT1>
struct Turns {
    static constexpr int MT = MT0 + MT1, NT = NT0 + NT1, BM = 32 * MT, BN = 64 * NT;
    // 16-byte units of the LDS arrays; loads a wave (8 rows of 128 bytes each)
    static constexpr int UX0 = MT0 * 256, UX1 = MT1 * 256, UW0 = NT0 * 512, UW1 = NT1 * 512;
    static constexpr int CX0 = MT0 / 2, CX1 = MT1 / 2, CW0 = NT0, CW1 = NT1, ALL = CX0 + CX1 + CW0 + CW1;
    static_assert(MT0 % 2 == 0 && MT1 % 2 == 0 && NT0 <= 2 && NT1 <= 2, "whole loads");

    turns_f32x4_t acc[NT][MT];
    illm_u32x4_t xf[MT0 > MT1 ? MT0 : MT1][2], w0[2][NT0][2], w1[NT1][2];
    int wave, wm, wn, r, q, c0, c1, lr, lc;

    __device__ __forceinline__ void begin() {
        const int lane = threadIdx.x & 63;
        wave = wave_index(); wm = wave >> 2; wn = wave & 3;
        r = lane & 15; q = lane >> 4;
        c0 = q ^ (r & 7); c1 = (4 + q) ^ (r & 7);              // 16-byte piece c of row t stands at place c ^ (t % 8)
        lr = lane >> 3; lc = ((lane & 7) ^ lr) * 16;
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) acc[i][j] = (turns_f32x4_t){0.f, 0.f, 0.f, 0.f};
    }
    // The tile's row that this lane's i-th load of a part of X brings, and of W: the wave (of four) whose columns
    // they are, the tile of the part and the row in it.
    template <int MTH>
    __device__ __forceinline__ int x_row(int i, int base) const {
        const int rho = (i * 8 + wave) * 8 + lr, g = rho / (MTH * 16);
        return g * (MT * 16) + base + (rho - g * MTH * 16);
    }
    struct WAt { int wave, tile, row; };
    template <int NTH>
    __device__ __forceinline__ WAt w_row(int i) const {
        const int rho = (i * 8 + wave) * 8 + lr, w = rho / (NTH * 16), in = rho - w * NTH * 16;
        return {w, in >> 4, in & 15};
    }
    template <int C>
    __device__ __forceinline__ void load(illm_u32x4_t* to, __amdgpu_buffer_rsrc_t rs, const uint32_t (&from)[C], uint32_t at) const {
#pragma unroll
        for (int i = 0; i < C; ++i) ld16_lds(rs, to + (i * 8 + wave) * 64, from[i], at);
    }
    template <int MTH>
    __device__ __forceinline__ void read_x(const illm_u32x4_t* a) {
#pragma unroll
        for (int j = 0; j < MTH; ++j) {
            xf[j][0] = a[(wm * MTH * 16 + j * 16 + r) * 8 + c0];
            xf[j][1] = a[(wm * MTH * 16 + j * 16 + r) * 8 + c1];
        }
    }
    template <int NTH>
    __device__ __forceinline__ void read_w(illm_u32x4_t (&to)[NTH][2], const illm_u32x4_t* a) const {
#pragma unroll
        for (int i = 0; i < NTH; ++i) {
            to[i][0] = a[(wn * NTH * 16 + i * 16 + r) * 8 + c0];
            to[i][1] = a[(wn * NTH * 16 + i * 16 + r) * 8 + c1];
        }
    }
    // The turn's products, once every wave's loads for the other group's and this group's next reads have arrived (all but
    // the newest VM of this wave's) and the other group's products are on their way.  on: a group whose rows of X are not there
    // leaves the products out (the same in all lanes).
    template <int VM, int NTH, int NB, int MTH, int MB>
    __device__ __forceinline__ void multiply(const illm_u32x4_t (&w)[NTH][2], bool on) {
        __builtin_amdgcn_sched_barrier(0);
        turns_wait_loads<VM>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        if (on) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int i = 0; i < NTH; ++i)
#pragma unroll
                    for (int j = 0; j < MTH; ++j)
                        acc[NB + i][MB + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            *(const turns_bf16x8_t*)&w[i][kk], *(const turns_bf16x8_t*)&xf[j][kk], acc[NB + i][MB + j], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    // Stage s of set A (P = s % 2).  ld.x1(to) asks for part X1 of stage s + 1, ld.w0, ld.x0 and ld.w1 for parts of s + 2.
    // on0, on1: whether any of the group's rows of X0 and of X1 are there.
    template <int P, class Loads>
    __device__ __forceinline__ void stage(illm_u32x4_t* x0a, illm_u32x4_t* x1a, illm_u32x4_t* w0a, illm_u32x4_t* w1a,
                                          illm_u32x4_t* x1b, illm_u32x4_t* w0b, Loads& ld, bool on0 = true, bool on1 = true) {
        read_x<MT0>(x0a); ld.x1(x1b);
        multiply<ALL + CX1, NT0, 0, MT0, 0>(w0[P], on0);
        read_w(w1, w1a); ld.w0(w0a);
        multiply<ALL + CW0, NT1, NT0, MT0, 0>(w1, on0);
        read_x<MT1>(x1a); ld.x0(x0a);
        multiply<ALL + CX0, NT1, NT0, MT1, MT0>(w1, on1);
        read_w(w0[1 - P], w0b); ld.w1(w1a);
        multiply<ALL + CW1, NT0, 0, MT1, MT0>(w0[P], on1);
    }
    // Before the first stage, with W0 X0 W1 X1 of stage 0 and W0 X0 W1 of stage 1 asked for in this order; the second
    // group starts a turn later.  end: every wave's barriers are then as many.
    __device__ __forceinline__ void start(const illm_u32x4_t* w0a) {
        __builtin_amdgcn_sched_barrier(0);
        turns_wait_loads<ALL + CX0 + CW1>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_w(w0[0], w0a);
        __builtin_amdgcn_sched_barrier(0);
        turns_wait_loads<ALL + CW1>();
        __builtin_amdgcn_s_barrier();
        if (wm == 1) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void end() const {
        __builtin_amdgcn_sched_barrier(0);
        if (wm == 0) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_waitcnt(0x0f70);                    // no load into LDS outlives the block
    }
};
