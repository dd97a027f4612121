// vrt_gemm.hpp -- the row-batch projections of the prefill and the batched decode on MFMA
// (vrt_gemm.hip): operand layouts and launches.
//
// Operand order. Both operands of v_mfma_f32_16x16x32_f16 hold 16 rows x 32 consecutive k: lane l
// gives row l % 16, k = 8 (l / 16) + j, j < 8. Activations and weights are kept in memory as
// such units, 512 halves each, in lane order, so a wave's operand load is one contiguous 1 KB, from
// memory straight to registers or to LDS, and an LDS read of it is conflict-free without padding.
//   activations [row tile of 16][K / 32][hi, lo][512]   (f16 high and low parts, A = hi + lo)
//   weights     [row tile of 16][K / 32][512]           (the Q8_0 quants as f16, exact)
//   scales      [K / 32][npad]                          (fp32), npad = N rounded up to 128
// One unit of K is one Q8_0 block, so a block's scale multiplies whole MFMA results.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vrt {

constexpr uint32_t kGmRowPad = 128;   // rows of an activation buffer and of a weight matrix: whole tiles

// Offset (halves) of element (row, k) of an activation buffer with nkb = K / 32: its high part;
// the low part is kGmLo further.
constexpr uint32_t kGmLo = 512;
__host__ __device__ __forceinline__ uint64_t gm_off(uint32_t row, uint32_t k, uint32_t nkb) {
    return (static_cast<uint64_t>(row >> 4) * nkb + (k >> 5)) * 1024u + ((k >> 3) & 3u) * 128u + (row & 15u) * 8u + (k & 7u);
}
// Halves of an activation buffer of `rows` rows (padded to whole tiles) and K columns.
__host__ __device__ __forceinline__ uint64_t gm_size(uint64_t rows, uint32_t K) {
    return (rows + kGmRowPad - 1u) / kGmRowPad * kGmRowPad * K * 2u;
}

// x = hi + lo. The product that x often is must be rounded to fp32 before it is rounded to f16: left to
// itself the compiler rounds it to f16 in one step (v_fma_mixlo_f16) for the subtraction and in two
// for the stored hi, and where the two differ (about one value in 2^13) the pair is one f16 ulp off.
__device__ __forceinline__ void gm_split(float x, _Float16& hi, _Float16& lo) {
    asm("" : "+v"(x));
    hi = static_cast<_Float16>(x);
    lo = static_cast<_Float16>(x - static_cast<float>(hi));
}

// gelu_tanh(gate) * up (shaders/gelu_mul.comp:23-31) with 0.5 x (1 + tanh u) = x / (1 + e^(-2u)), which has no
// cancellation where tanh u is close to -1. The hardware's exponential and reciprocal are approximate to 1 ulp: the
// exponential's error counts by 1 - s of the quotient's share s, and the quotient is corrected once with the
// rounding error of 1 + e carried along. Error against 64 bits over gates N(0, 1), 2-norm: 3.7e-8; with tanhf in the
// reference's order of operations 4.5e-8; without the correction 5.3e-8. Time of the function alone: 0.73 of
// tanhf's, 1.8 times that without the correction. Past the exponential's range the quotient is 0.
__device__ __forceinline__ float gm_gelu_mul(float x, float up) {
#pragma clang fp contract(off)
    const float t = x * __builtin_fmaf(-0.1029432397f, x * x, -2.302208198f);   // -2 u log2 e
    const float e = __builtin_amdgcn_exp2f(fminf(t, 126.0f)), d = 1.0f + e;
    const float lo = e <= 1.0f ? e - (d - 1.0f) : 1.0f - (d - e);   // 1 + e = d + lo
    const float r = __builtin_amdgcn_rcpf(d), q = x * r;
    const float y = __builtin_fmaf(__builtin_fmaf(-q, lo, __builtin_fmaf(-d, q, x)), r, q);
    return (t > 126.0f ? x * 0.0f : y) * up;
}

// 64 lanes x 16 (or 4) bytes from base + voff straight into LDS at lds + lane * 16 (or 4). In
// assembly so that the waits are placed by hand: the compiler would wait for every such load in
// flight before any LDS read.
__device__ __forceinline__ void gm_lds16(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void gm_lds4(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :: "v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}

struct GmArgs {
    const _Float16* a;     // activations, M rows
    const _Float16* w;     // weights, N rows
    const float* ws;       // their block scales [nkb][npad]
    float* c;              // C [M][N] fp32 (row stride ldc), split z at c + z * c_bs; or, gate/up:
    _Float16* o;           // gelu_tanh(gate) * up as an activation buffer of N / 2 columns
    uint64_t c_bs;
    uint32_t ldc;
    uint32_t M, N, nkb, npad;
};

// C = A x W^T, or with glu (w: gate and up rows interleaved in groups of 16, 16 gate rows first)
// gelu_tanh(gate) * up. gm_splits: the K splits that suit this shape (1: none);
// the consumer adds the partials in split order.
constexpr uint32_t kGmSplitWgs = 160;   // K is split up to this many 64 x 64 tiles, in four at most:
constexpr uint64_t kGmSplitFloats = 4ull * kGmSplitWgs * 64u * 64u;   //   so many partial sums
uint32_t gm_splits(uint32_t M, uint32_t N, uint32_t nkb);
int gm_run(const GmArgs& G, uint32_t splits, bool glu, hipStream_t s);
// The same with the residual fold and norm that come before it (G.a unused; at most 16 rows):
// h_out = f * (scale(f) * w_post) + h (f nullptr: no fold, nothing written), and the projection of
// (h_out * scale(h_out)) * w_next. h_out is another buffer than h. A non-finite h_out lowers *nonfinite to code.
struct GmNorm {
    const float* h;
    const float* f;
    float* h_out;
    const float* w_post;
    const float* w_next;
    uint32_t* nonfinite;
    uint32_t code;
    float eps;
};
bool gm_norm_fits(uint32_t M, uint32_t nkb);
int gm_run_norm(const GmArgs& G, const GmNorm& R, bool glu, hipStream_t s);
int gm_setup();   // once per device before gm_lm: its LDS limit
// One-time expansion of Q8_0 rows into a weight matrix: up to three matrices concatenated
// (rows0, rows1, the rest), or with glu the gate (w0) and up (w1) rows interleaved. Rows N..npad-1
// are zero with scale 0.
int gm_expand(const uint8_t* w0, const uint8_t* w1, const uint8_t* w2, uint32_t rows0, uint32_t rows1, uint32_t N,
              uint32_t nkb, bool glu, _Float16* wh, float* ws, hipStream_t s);
// logits [M][V] = x W^T over V Q8_0 rows of nkb blocks in their file layout, x an activation buffer, and the best
// logit (am_better) of each row in each of gm_lm_chunks runs of the V rows: best [M][chunks]. gm_lm_fits: the table is
// 16-byte aligned and readable in whole 16-byte units, and a tile of it fits LDS.
constexpr uint32_t kGmLdsMax = 160u * 1024u;
constexpr uint32_t kGmLmMaxChunks = 512;
struct GmBest {
    float value;
    uint32_t index;
};
bool gm_lm_fits(const uint8_t* table, uint64_t readable, uint32_t V, uint32_t nkb);
uint32_t gm_lm_chunks(uint32_t M, uint32_t nkb);
int gm_lm(const uint8_t* table, uint32_t V, uint32_t nkb, const _Float16* x, uint32_t M, float* logits, GmBest* best,
          hipStream_t s);

}  // namespace vrt
