// vrt_prefill.hip -- batched prompt prefill of the Gemma 3 executor: every prompt position of
// a block at once. The projections are Q8_0 x activation GEMMs on MFMA, attention is causal
// with the local/global pattern, and the last position runs the fused LM head + argmax of the
// decode step. Afterwards the KV cache holds positions 0..T-1 exactly as T serial decode
// steps would have left it (src/gemma3.cpp:2099-2111), so decoding continues at T.
//
// GEMM numerics. C[m][n] = sum_b s[n][b] * sum_{k in b} A[m][k] * q[n][k] with s the block's
// f16 scale and q its int8 quants (exact in f16). A (fp32 activations) is split as
// A = hi + lo with hi = f16(A) and lo = f16(A - hi), so the two f16 MFMA products carry ~22
// bits of A; every f16 x f16 product is exact in fp32 and the MFMA accumulates in fp32. The
// per-block partial is scaled by s in fp32 and added to the fp32 accumulator.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <initializer_list>
#include <utility>
#include <vector>

#include "vrt_g3_errors.hpp"
#include "vrt_g3_internal.hpp"
#include "vrt_gemm.hpp"
#include "vrt_q8_device.hpp"

namespace vrt {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr uint32_t kPfThreads = 256;
constexpr uint32_t kPfMaxSplits = 4;   // K splits of a projection, at most (gm_splits, pf_splits_q8)
constexpr uint64_t kPfExpandBudget = 16ull << 30;   // device bytes for the prefill's expanded weights
constexpr uint32_t kPfTile = 64;     // attention score rows are padded to a multiple of this

// ---- row kernels ---------------------------------------------------------------------------

__device__ __forceinline__ void pf_split(float x, _Float16* hi, _Float16* lo) {
    _Float16 h, l;
    gm_split(x, h, l);
    *hi = h;
    *lo = l;
}

// pf_split of four consecutive values (8-byte aligned destinations).
__device__ __forceinline__ void pf_split4(f4 x, _Float16* hi, _Float16* lo) {
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    half4 h, l;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        _Float16 a, b;
        gm_split(x[k], a, b);
        h[k] = a;
        l[k] = b;
    }
    *reinterpret_cast<half4*>(hi) = h;
    *reinterpret_cast<half4*>(lo) = l;
}

// 1.0f / std::sqrt(float(sum_sq / n) + eps) (src/gemma3.cpp:967-983).
__device__ __forceinline__ float pf_rms_scale(double ss, uint32_t n, float eps) {
#pragma clang fp contract(off)
    return 1.0f / sqrtf(static_cast<float>(ss / static_cast<double>(n)) + eps);
}

// h[t] = dequantised embedding row of tokens[t] * emb_scale (src/gemma3.cpp:1106-1136).
__global__ void __launch_bounds__(kPfThreads) k_pf_embed(const uint8_t* tok_embd, const uint32_t* tokens, uint32_t d,
                                                         float emb_scale, float* h) {
#pragma clang fp contract(off)
    const uint32_t t = blockIdx.x;
    const uint8_t* row = tok_embd + static_cast<uint64_t>(tokens[t]) * (d / 32u) * 34u;
    for (uint32_t i = threadIdx.x; i < d; i += kPfThreads) {
        const uint8_t* b = row + (i >> 5) * 34u;
        const float sc = half_bits_to_float(static_cast<uint32_t>(b[0]) | (static_cast<uint32_t>(b[1]) << 8));
        h[static_cast<uint64_t>(t) * d + i] = (sc * static_cast<float>(static_cast<int8_t>(b[2 + (i & 31u)]))) * emb_scale;
    }
}

// One wave per row t (four rows per workgroup, `rows` rows in all; n <= 256 NQ elements, a multiple
// of 32; lane l owns the runs of four from 4 l + 256 k; the sums are wave reductions, with no
// barrier). With f (the previous sublayer's output, the sum of nsplit partial rows f + s * sstride
// added in order s = 0, 1, ...): h = f * (scale(f) * w_post) + h (rms_norm_inplace then
// add_inplace, src/gemma3.cpp:1036-1042, :1703-1711, :1849-1855). Then, with w_next: the GEMM
// input (h * scale(h)) * w_next into the activation buffer x (rms_norm_into, :991-996), or with
// `into` 0 h * (scale(h) * w_next) (rms_norm_inplace, the output norm :1866-1868). nonfinite:
// lowest block whose residual went non-finite (:1857-1863), reported through st->nonfinite.
template <uint32_t NQ>
__global__ void __launch_bounds__(kPfThreads) k_pf_norm_w(float* h, const float* f, uint32_t nsplit, uint64_t sstride,
                                                          const float* w_post, const float* w_next, uint32_t n, float eps,
                                                          _Float16* x, G3State* st, uint32_t block, uint32_t rows,
                                                          uint32_t into) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t t = blockIdx.x * (kPfThreads / 64u) + (threadIdx.x >> 6);
    if (t >= rows) return;   // whole wave
    float* hr = h + static_cast<uint64_t>(t) * n;
    // Every load is issued at a clamped, in-bounds index and masked afterwards, so the loads of
    // a row are in flight together (no branch, hence no wait, between them).
    uint32_t ic[NQ];
    bool live[NQ];
#pragma unroll
    for (uint32_t k = 0; k < NQ; ++k) {
        live[k] = 4u * lane + 256u * k < n;
        ic[k] = min(4u * lane + 256u * k, n - 4u);
    }
    f4 hv[NQ], wp[NQ], wn[NQ];
#pragma unroll
    for (uint32_t k = 0; k < NQ; ++k) {
        hv[k] = *reinterpret_cast<const f4*>(hr + ic[k]);
        wp[k] = w_post ? *reinterpret_cast<const f4*>(w_post + ic[k]) : f4{0.0f, 0.0f, 0.0f, 0.0f};
        wn[k] = w_next ? *reinterpret_cast<const f4*>(w_next + ic[k]) : f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (f) {
        const float* fr = f + static_cast<uint64_t>(t) * n;
        f4 fv[NQ];
        if (nsplit == 1u) {
#pragma unroll
            for (uint32_t k = 0; k < NQ; ++k) fv[k] = *reinterpret_cast<const f4*>(fr + ic[k]);
        } else {   // every partial is loaded before the first add, then the partials are added in split order
            f4 fp[NQ][kPfMaxSplits];
#pragma unroll
            for (uint32_t q = 0; q < kPfMaxSplits; ++q) {
                const float* fq = fr + min(q, nsplit - 1u) * sstride;
#pragma unroll
                for (uint32_t k = 0; k < NQ; ++k) fp[k][q] = *reinterpret_cast<const f4*>(fq + ic[k]);
            }
#pragma unroll
            for (uint32_t k = 0; k < NQ; ++k) {
                fv[k] = fp[k][0];
#pragma unroll
                for (uint32_t q = 1; q < kPfMaxSplits; ++q)
                    if (q < nsplit)
#pragma unroll
                        for (int e = 0; e < 4; ++e) fv[k][e] += fp[k][q][e];
            }
        }
        double ss = 0.0;
#pragma unroll
        for (uint32_t k = 0; k < NQ; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (!live[k]) fv[k][e] = 0.0f;
                ss += static_cast<double>(fv[k][e]) * static_cast<double>(fv[k][e]);
            }
        const float sc = pf_rms_scale(wave_red_sum_d(ss), n, eps);
        int bad = 0;
#pragma unroll
        for (uint32_t k = 0; k < NQ; ++k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) hv[k][e] = fv[k][e] * (sc * wp[k][e]) + hv[k][e];
            if (live[k]) {
                *reinterpret_cast<f4*>(hr + ic[k]) = hv[k];
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= !__builtin_isfinite(hv[k][e]);
            }
        }
        if (bad) atomicMin(&st->nonfinite, g3_code_nonfinite(block));
    }
    if (!w_next) return;
    double ss = 0.0;
#pragma unroll
    for (uint32_t k = 0; k < NQ; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = live[k] ? hv[k][e] : 0.0f;
            ss += static_cast<double>(v) * static_cast<double>(v);
        }
    const float sc = pf_rms_scale(wave_red_sum_d(ss), n, eps);
#pragma unroll
    for (uint32_t k = 0; k < NQ; ++k) {
        f4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = into ? (hv[k][e] * sc) * wn[k][e] : hv[k][e] * (sc * wn[k][e]);
        if (live[k]) {
            const uint64_t o = gm_off(t, ic[k], n / 32u);
            pf_split4(y, x + o, x + o + kGmLo);
        }
    }
}

// out[i] = sum over s < nsplit, in order, of the split partials x[s * n + i] of one row.
__global__ void __launch_bounds__(kPfThreads) k_pf_sum(const float* x, uint32_t nsplit, uint32_t n, float* out) {
#pragma clang fp contract(off)
    for (uint32_t i = threadIdx.x; i < n; i += kPfThreads) {
        float v = 0.0f;
        for (uint32_t q = 0; q < nsplit; ++q) v += x[static_cast<uint64_t>(q) * n + i];
        out[i] = v;
    }
}

// gelu_tanh(gate) * up (shaders/gelu_mul.comp:23-31), every operation rounded to fp32.
__device__ __forceinline__ float pf_gelu_mul(float x, float up) {
#pragma clang fp contract(off)
    const float cubic = x * x * x;
    const float g = 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * cubic)));
    return g * up;
}


// ---- GEMM on MFMA: Q8_0 weights ---------------------------------------------------------------

struct PfGemm {
    const _Float16* a;       // A [M][K], an activation buffer (vrt_gemm.hpp)
    const uint8_t* w[3];     // W as Q8_0 matrices concatenated along N (rows[i] rows each)
    uint32_t rows[3];
    uint32_t nseg;
    float* c;                // C [M][N] fp32 (row stride N; split z at c + z * c_bs), or with glu
    _Float16* o;             //   gelu_tanh(gate) * up as an activation buffer of N / 2 columns
    uint64_t c_bs;
    uint32_t M, N, K;
    uint32_t glu;            // w[0] = gate, w[1] = up (N = 2F)
};

// C[M][N] = A[M][K] (f16 hi/lo) x W^T with W the Q8_0 rows (segments concatenated along N).
// Workgroup tile: 64 rows of A x 64 * WN rows of W; wave w computes rows 32 (w / 2) and the
// WN 32-column MFMA tiles from 32 WN (w % 2). K advances 64 (two Q8_0 blocks) per step through
// two LDS stages: A as f16 hi and lo [64][64], W as its exact int8 quants in f16 [64 WN][64]
// plus the fp32 block scales; one barrier per step hands a stage over. Per Q8_0 block and tile the
// two f16 MFMA chains (A hi, A lo) accumulate the exact products in fp32 and the block's partial
// is scaled by the column's scale into the fp32 accumulator. MFMA operands
// (v_mfma_f32_32x32x16_f16): lane l gives A[m = l % 32][k = 8 (l / 32) + j] and B[k][n = l % 32]
// for j < 8 of each 16-wide k step; result r of lane l is C[8 (r / 4) + 4 (l / 32) + r % 4]
// [l % 32]. blockIdx.z splits K: split z covers K blocks [z nkb / S, (z + 1) nkb / S) and writes
// C + z * c_bs; the consumer adds the S partial tiles in split order.
constexpr uint32_t kQgBM = 64;
constexpr uint32_t kQgBK = 64;
constexpr uint32_t kQgPitch = kQgBK * 2u + 16u;   // LDS row pitch in bytes (f16 rows, padded)

constexpr uint32_t kQgAhead = 4;   // K steps whose loads are in flight ahead of the one computed
constexpr uint32_t kQgChunk = 12;  // K steps per straight-line chunk of the main loop

// Epilogue of the Q8_0 GEMMs: with G.glu the wave holding a 64-column group's up columns hands
// them to the wave holding its gate columns through `xch` (LDS of at least NWN / 2 x 16 x 64
// floats per 32-row band, free once the K loop is done), which writes gelu_tanh(gate) * up as
// f16 hi/lo; otherwise the fp32 tile goes to split z's slice of C.
template <int WN, int NWN>
__device__ __forceinline__ void pf_gemm_epilogue(const PfGemm& G, const float16v (&acc)[WN], uint32_t z, uint32_t m0,
                                                 uint32_t n0, uint32_t wm, uint32_t wn, uint32_t kh, uint32_t l32,
                                                 uint32_t lane, float* xch) {
    if (G.glu) {
        // the wave holding a group's up columns hands them to the wave holding its gate columns
        // (gelu_tanh(gate) * up, shaders/gelu_mul.comp:23-31)
        static_assert(WN == 1, "one 32-column MFMA tile per wave");
        __syncthreads();   // every wave is done reading the LDS stages
        const uint32_t pair = wm * (NWN / 2u) + (wn >> 1);
        if (wn & 1u) {
#pragma unroll
            for (int r = 0; r < 16; ++r) xch[(pair * 16u + r) * 64u + lane] = acc[0][r];
        }
        __syncthreads();
        if (wn & 1u) return;
        const uint32_t F = G.N / 2u;
        const uint32_t col = n0 / 2u + 32u * (wn >> 1) + l32;
        if (col >= F) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t row = m0 + 32u * wm + 8u * (r / 4) + 4u * kh + (r % 4);
            if (row < G.M) {
                const uint64_t o = gm_off(row, col, F / 32u);
                pf_split(pf_gelu_mul(acc[0][r], xch[(pair * 16u + r) * 64u + lane]), G.o + o, G.o + o + kGmLo);
            }
        }
        return;
    }
    float* c = G.c + static_cast<uint64_t>(z) * G.c_bs;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const uint32_t col = n0 + 32u * (WN * wn + j) + l32;
        if (col >= G.N) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t row = m0 + 32u * wm + 8u * (r / 4) + 4u * kh + (r % 4);
            if (row < G.M) c[static_cast<uint64_t>(row) * G.N + col] = acc[j][r];
        }
    }
}

template <int WN, int NWN>
__global__ void __launch_bounds__(128 * NWN) k_pf_gemm_q8(PfGemm G) {
    constexpr uint32_t NT = 128u * NWN;          // threads: 2 x NWN waves
    constexpr uint32_t BN = 32u * WN * NWN;      // W rows per tile
    constexpr uint32_t AU = 2u * kQgBM * 8u / NT / 2u;   // A 16-byte units per thread and array
    __shared__ __align__(16) unsigned char s_a[2][2][kQgBM * kQgPitch];   // [stage][hi, lo]
    __shared__ __align__(16) unsigned char s_w[2][BN * kQgPitch];          // [stage] quants
    __shared__ float s_sc[2][BN][2];                                       // [stage][row][block]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t kh = lane >> 5, l32 = lane & 31u;
    const uint32_t m0 = blockIdx.y * kQgBM, n0 = blockIdx.x * BN;
    const uint32_t nkb = G.K >> 5;                                         // Q8_0 blocks along K
    const uint32_t S = gridDim.z, z = blockIdx.z;
    const uint32_t kb_lo = nkb * z / S, kb_hi = nkb * (z + 1u) / S;
    const uint32_t nsteps = (kb_hi - kb_lo + 1u) / 2u;
    const uint64_t row_bytes = static_cast<uint64_t>(nkb) * 34u;

    // One K step in registers: A units u = t + NT j of hi and of lo, in the order of the activation buffer (16-row
    // tile u / 128, block u / 64 % 2, k octet u / 16 % 4, row u % 16), so that a wave's load is one contiguous
    // 1 KB, and the 34-byte W block of thread t < 2 BN (row t / 2, block t % 2). (Units along a row touch 16
    // lines per load of eight rows: a step of 8 sequences at head_dim 40, six blocks, 360 us against 313.)
    struct Stage {
        v4u a[2][AU];  // [hi, lo][unit]
        uint32_t d[8]; // dwords at the block start rounded down to 4 bytes
        uint32_t u0;   // 16 bits at that start + 32, 16 bits at the block start + 32
        uint32_t u1;
        uint32_t sh;   // block start & 3 (0 or 2)
        bool wl;       // W block live
    };
    typedef const __attribute__((address_space(1))) v4u* gv4;
    const uint32_t wr = tid >> 1, wb = tid & 1u;
    static_assert(2u * BN <= NT, "one W block per thread");
    const bool wlive_t = tid < 2u * BN && n0 + wr < G.N;
    const uint8_t* wrow = G.w[0];
    if (G.glu) {   // 64-column groups: 32 gate rows, then the same 32 up rows
        const uint32_t n = wlive_t ? n0 + wr : 0u;
        wrow = ((n & 63u) < 32u ? G.w[0] : G.w[1]) + static_cast<uint64_t>(32u * (n >> 6) + (n & 31u)) * row_bytes;
    } else {
        uint32_t r = wlive_t ? n0 + wr : 0u;
        if (G.nseg > 1u && r >= G.rows[0]) {
            r -= G.rows[0];
            wrow = G.w[1];
            if (G.nseg > 2u && r >= G.rows[1]) {
                r -= G.rows[1];
                wrow = G.w[2];
            }
        }
        wrow += static_cast<uint64_t>(r) * row_bytes;
    }
    // Every load is issued unconditionally at a clamped, in-bounds address (dead data is zeroed
    // when it is stored): with no branch around a load the compiler counts the loads in flight
    // exactly, so the wait for step j's data does not also wait for the later steps of the ring.
    typedef const __attribute__((address_space(1))) uint32_t* gu32;
    typedef const __attribute__((address_space(1))) uint16_t* gu16;
    auto load = [&](uint32_t step, Stage& R) {
        const uint32_t kb = kb_lo + 2u * step;
#pragma unroll
        for (uint32_t j = 0; j < AU; ++j) {
            const uint32_t u = tid + NT * j, r = 16u * (u >> 7) + (u & 15u), c = (u >> 4) & 7u;
            const uint32_t k = 32u * kb + 8u * c;
            const uint32_t rr = min(m0 + r, G.M - 1u), kk = min(k, 32u * kb_hi - 8u);
            const uintptr_t o = reinterpret_cast<uintptr_t>(G.a + gm_off(rr, kk, nkb));
            R.a[0][j] = *reinterpret_cast<gv4>(o);
            R.a[1][j] = *reinterpret_cast<gv4>(o + 2u * kGmLo);
        }
        const uint32_t b = kb + wb;
        R.wl = wlive_t && b < kb_hi;
        // the block's 34 bytes: 8 dwords from its start rounded down (2 bytes before it when the
        // start is 2 mod 4), then the 16 bits at that start + 32 and at the block start + 32; no
        // byte past the block is read
        const uintptr_t base = reinterpret_cast<uintptr_t>(wrow) + 34u * min(b, kb_hi - 1u);
        const uintptr_t lb = base & ~uintptr_t(3);
        R.sh = static_cast<uint32_t>(base & 3u);
#pragma unroll
        for (int j = 0; j < 8; ++j) R.d[j] = reinterpret_cast<gu32>(lb)[j];
        R.u0 = *reinterpret_cast<gu16>(lb + 32u);
        R.u1 = *reinterpret_cast<gu16>(base + 32u);
    };
    auto store = [&](const Stage& R, uint32_t st, uint32_t step) {
        const uint32_t kb = kb_lo + 2u * step;
#pragma unroll
        for (uint32_t j = 0; j < AU; ++j) {
            const uint32_t u = tid + NT * j, r = 16u * (u >> 7) + (u & 15u), c = (u >> 4) & 7u;
            const bool live = m0 + r < G.M && 32u * kb + 8u * c < 32u * kb_hi;
#pragma unroll
            for (uint32_t p = 0; p < 2; ++p)
                *reinterpret_cast<v4u*>(&s_a[st][p][r * kQgPitch + c * 16u]) = live ? R.a[p][j] : v4u{0u, 0u, 0u, 0u};
        }
        if (tid >= 2u * BN) return;
        // quants at window offset sh + 2: shift 2 (sh == 0) or whole dwords from d[1] (sh == 2)
        const uint32_t d8 = R.sh ? (R.u0 | (R.u1 << 16)) : R.u0;
        uint32_t q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t hi = j < 7 ? R.d[j + 1] : d8;
            q[j] = R.wl ? (R.sh ? hi : __builtin_amdgcn_alignbyte(hi, R.d[j], 2u)) : 0u;
        }
        unsigned char* dst = &s_w[st][wr * kQgPitch + wb * 64u];
#pragma unroll
        for (int j = 0; j < 4; ++j) {   // 8 quants (two dwords) -> 8 f16 per 16-byte store
            half8 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(q[2 * j] >> (8 * i))));
                v[4 + i] = static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(q[2 * j + 1] >> (8 * i))));
            }
            *reinterpret_cast<half8*>(dst + 16u * j) = v;
        }
        s_sc[st][wr][wb] = R.wl ? half_bits_to_float(R.sh ? (R.d[0] >> 16) : (R.d[0] & 0xffffu)) : 0.0f;
    };

    const uint32_t wm = wave / NWN, wn = wave % NWN;
    float16v acc[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = float16v{};
    auto compute = [&](uint32_t st) {
        const unsigned char* pa_hi = &s_a[st][0][(32u * wm + l32) * kQgPitch + 16u * kh];
        const unsigned char* pa_lo = &s_a[st][1][(32u * wm + l32) * kQgPitch + 16u * kh];
#pragma unroll
        for (uint32_t b = 0; b < 2; ++b) {   // the step's two Q8_0 blocks
            half8 ah[2], al[2];
#pragma unroll
            for (uint32_t ks = 0; ks < 2; ++ks) {
                ah[ks] = *reinterpret_cast<const half8*>(pa_hi + 64u * b + 32u * ks);
                al[ks] = *reinterpret_cast<const half8*>(pa_lo + 64u * b + 32u * ks);
            }
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint32_t nl = 32u * (WN * wn + j) + l32;   // the lane's column in the tile
                const unsigned char* pw = &s_w[st][nl * kQgPitch + 64u * b + 16u * kh];
                const half8 w0 = *reinterpret_cast<const half8*>(pw), w1 = *reinterpret_cast<const half8*>(pw + 32u);
                float16v p = {};
                p = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[0], w0, p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[0], w0, p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[1], w1, p, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[1], w1, p, 0, 0, 0);
                const float sc = s_sc[st][nl][b];
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][r] += sc * p[r];
            }
        }
    };

    // The K loop runs in straight-line chunks of kQgChunk steps with a ring of kQgAhead register
    // stages: step j's loads are issued kQgAhead steps before it is stored to LDS, so they
    // overlap the MFMAs of the steps in between. Every load is issued unconditionally (clamped,
    // in-bounds addresses; steps past the end re-load the last one and are never stored), and
    // no loaded value crosses a chunk boundary: with no branch around a load and no value live
    // across a back edge, the compiler waits for exactly the step it stores.
    static_assert(kQgAhead <= kQgChunk, "ring inside a chunk");
    for (uint32_t i = 0; i < nsteps; i += kQgChunk) {
        Stage R[kQgAhead];
        auto clamp = [&](uint32_t j) { return min(i + j, nsteps - 1u); };
#pragma unroll
        for (uint32_t u = 0; u < kQgAhead; ++u) load(clamp(u), R[u]);
#pragma unroll
        for (uint32_t u = 0; u < kQgChunk; ++u) {
            const uint32_t j = i + u;
            if (j < nsteps) {
                // stage j & 1 was last read by step j - 2, which every wave finished before the
                // barrier of step j - 1
                store(R[u % kQgAhead], j & 1u, j);
                __syncthreads();
            }
            if (u + kQgAhead < kQgChunk) load(clamp(u + kQgAhead), R[u % kQgAhead]);
            if (j < nsteps) compute(j & 1u);
        }
    }
    pf_gemm_epilogue<WN, NWN>(G, acc, z, m0, n0, wm, wn, kh, l32, lane, reinterpret_cast<float*>(&s_a[0][0][0]));
}

// Operand layouts of the attention keys and values (per 32-key tile, so that every MFMA operand
// load of a wave is one contiguous 1 KB): the key rows of a tile are stored in the order pkey
// (bits 2 and 3 of the index swapped, an involution), and for S^T = K Q^T the k step s, lane
// half f and row m of the A operand hold K[32 tile + pkey(m)][16 s + 8 f + j], j < 8; for
// O^T += V^T E^T the d tile dt, k step sk, lane half f and row m hold V[32 tile + 16 sk + 8 f + j]
// [32 dt + m]. With the pkey order, S^T's result r of lane half f is key 16 (r / 8) + 8 f +
// r % 8 of the tile, which is the key of O^T's k slot 8 f + j of k step sk = r / 8, j = r % 8.
__device__ __forceinline__ uint32_t pf_pkey(uint32_t w) {
    return (w & ~12u) | ((w & 4u) << 1) | ((w & 8u) >> 1);
}
__device__ __forceinline__ uint64_t pf_kswz(uint32_t t, uint32_t d, uint32_t hd) {
    const uint32_t tile = t >> 5, m = pf_pkey(t & 31u);
    return ((static_cast<uint64_t>(tile) * (hd / 16u) + (d >> 4)) * 2u + ((d >> 3) & 1u)) * 256u + m * 8u + (d & 7u);
}
__device__ __forceinline__ uint64_t pf_vswz(uint32_t t, uint32_t d, uint32_t hd) {
    const uint32_t tile = t >> 5, w = t & 31u;
    return ((static_cast<uint64_t>(tile) * (hd / 32u) + (d >> 5)) * 2u + (w >> 4)) * 512u + ((w >> 3) & 1u) * 256u +
           (d & 31u) * 8u + (w & 7u);
}

// Queries in operand order: per (32-row tile, head) and k step s, lane half f and row m of the B operand of
// S^T hold Q[32 tile + m][16 s + 8 f + j], j < 8 (1 KB per step).
__device__ __forceinline__ uint64_t pf_qswz(uint32_t t, uint32_t h, uint32_t d, uint32_t H, uint32_t hd) {
    return ((static_cast<uint64_t>(t >> 5) * H + h) * (hd / 16u) + (d >> 4)) * 512u + ((d >> 3) & 1u) * 256u + (t & 31u) * 8u + (d & 7u);
}

// ---- QK-norm, RoPE, KV cache ------------------------------------------------------------

// Four consecutive cache entries from entry i on (fp32, or 16-bit in the first half of the buffer).
__device__ __forceinline__ void kv_store4(float* c, uint64_t i, f4 x, uint32_t kv16) {
    if (!kv16) {
        *reinterpret_cast<f4*>(c + i) = x;
        return;
    }
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    u16x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = kv16_bits(x[e], kv16);
    *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(c) + i) = b;
}

// Row t of qkv = [q (H heads x hd) | k (hd) | v (hd)], the sum of nsplit partials: QK-norm per head
// (src/gemma3.cpp:1045-1104), NeoX RoPE at position p0 + t (:1371-1424), q as f16 hi/lo in
// pf_qswz order; then k and v go to the KV cache slot of the position when it is still in the window
// after the segment (the serial loop's eviction leaves exactly those, :1590-1600); with kv16 (1 fp16,
// 2 bf16) the cache holds 16-bit entries and k and v are rounded to them first (the attention below
// then sees the cached values, as the serial loop does). The attention operands as f16 hi/lo: k and
// v in the pf_kswz / pf_vswz tile layouts. Rows t >= T write the zero padding keys and values
// (keys past the prompt are masked, and zero values keep the masked products zero).
// One workgroup per eight rows, one wave per row. Lane l holds the dims 4 l .. 4 l + 3 of every head
// (hd <= 256), so loads, cache stores and operand stores are 8 to 16 bytes per lane, the sums of
// squares are wave reductions and a RoPE partner sits hd / 8 lanes away. The values of the eight
// rows, consecutive in the value operand, meet in LDS and leave as 16-byte stores (one row per
// workgroup and two-byte stores: 14.4 us at 2048 rows).
constexpr uint32_t kPfQkRows = 8;
constexpr uint32_t kPfQkHeads = 5;   // heads in flight per wave (four query heads and the key: one round)
__global__ void __launch_bounds__(64 * kPfQkRows) k_pf_qk(const float* qkv, uint32_t nsplit, uint64_t sstride, uint32_t T,
                                                          uint32_t H, uint32_t hd, const float* q_norm,
                                                          const float* k_norm, const float* cos_t, const float* sin_t,
                                                          float eps, float* kc, float* vc, uint32_t slots, _Float16* qhi,
                                                          _Float16* qlo, _Float16* khi, _Float16* klo, _Float16* vhi,
                                                          _Float16* vlo, uint32_t kv16, uint32_t p0, uint32_t qo) {
#pragma clang fp contract(off)
    __shared__ __align__(16) float s_v[kPfQkRows][256];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t t = blockIdx.x * kPfQkRows + wave, kt = qo + t, pos = p0 + t;
    const uint32_t nqkv = (H + 2u) * hd, half = hd >> 1;
    const uint32_t i = min(4u * lane, hd - 4u);   // this lane's dims (clamped: lanes past hd store nothing)
    const bool live = 4u * lane < hd;
    f4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (t < T) {   // whole wave
        const float* row = qkv + static_cast<uint64_t>(t) * nqkv + i;
        // four elements of the row, the split partials added in order
        auto at = [&](uint32_t o) {
            f4 x = *reinterpret_cast<const f4*>(row + o);
            for (uint32_t z = 1; z < nsplit; ++z) {
                const f4 y = *reinterpret_cast<const f4*>(row + z * sstride + o);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] += y[e];
            }
            return x;
        };
        const bool keep = t + slots >= T;   // the last `slots` positions of the segment reach the ring
        const uint64_t slot = static_cast<uint64_t>(pos % slots) * hd + i;
        const bool lower = i < half;
        const uint32_t ri = lower ? i : i - half;
        const f4 cs = *reinterpret_cast<const f4*>(cos_t + static_cast<uint64_t>(pos) * half + ri);
        const f4 sn = *reinterpret_cast<const f4*>(sin_t + static_cast<uint64_t>(pos) * half + ri);
        const f4 wq = *reinterpret_cast<const f4*>(q_norm + i), wk = *reinterpret_cast<const f4*>(k_norm + i);
        v = at((H + 1u) * hd);
        const uint32_t partner = lower ? lane + (hd >> 3) : lane - (hd >> 3);
        for (uint32_t h0 = 0; h0 <= H; h0 += kPfQkHeads) {   // H query heads, then the key head
            f4 x[kPfQkHeads];
#pragma unroll
            for (uint32_t k = 0; k < kPfQkHeads; ++k) x[k] = at(min(h0 + k, H) * hd);
#pragma unroll
            for (uint32_t k = 0; k < kPfQkHeads; ++k) {
                const uint32_t hh = h0 + k;
                if (hh > H) break;
                double sq = 0.0;
#pragma unroll
                for (int e = 0; e < 4; ++e) sq += live ? static_cast<double>(x[k][e]) * static_cast<double>(x[k][e]) : 0.0;
                const float sc = pf_rms_scale(wave_red_sum_d(sq), hd, eps);
                f4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) {   // values *= scale * weights (src/gemma3.cpp:1097-1102)
                    const float a = x[k][e] * (sc * (hh < H ? wq[e] : wk[e]));
                    const float b = __shfl(a, static_cast<int>(partner & 63u));
                    y[e] = lower ? a * cs[e] - b * sn[e] : a * cs[e] + b * sn[e];
                }
                if (hh < H) {
                    const uint64_t o = pf_qswz(t, hh, i, H, hd);
                    if (live) pf_split4(y, qhi + o, qlo + o);
                } else {   // 16-bit KV: the key as the cache holds it, for the cache and the attention
                    if (kv16) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] = kv16_float(kv16_bits(y[e], kv16), kv16);
                    }
                    const uint64_t o = pf_kswz(kt, i, hd);
                    if (live) {
                        pf_split4(y, khi + o, klo + o);
                        if (keep) kv_store4(kc, slot, y, kv16);
                    }
                }
            }
        }
        if (kv16) {   // v is not normed
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = kv16_float(kv16_bits(v[e], kv16), kv16);
        }
        if (live && keep) kv_store4(vc, slot, v, kv16);
    } else if (live) {
        const uint64_t o = pf_kswz(kt, i, hd);
        pf_split4(v, khi + o, klo + o);
    }
    if (live) *reinterpret_cast<f4*>(&s_v[wave][i]) = v;
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < hd; d += 64u * kPfQkRows) {   // qo is a multiple of 32: eight keys of one run
        half8 hi, lo;
#pragma unroll
        for (uint32_t r = 0; r < kPfQkRows; ++r) {
            _Float16 a, b;
            gm_split(s_v[r][d], a, b);
            hi[r] = a;
            lo[r] = b;
        }
        const uint64_t o = pf_vswz(kt - wave, d, hd);
        *reinterpret_cast<half8*>(vhi + o) = hi;
        *reinterpret_cast<half8*>(vlo + o) = lo;
    }
}

// A segment's history for the attention: key coordinates j < nh hold positions kb + j, read
// from the block's KV cache (ring slot (kb + j) % slots, fp32 or 16-bit entries as the cache
// holds them) and written in the pf_kswz / pf_vswz layouts as f16 hi/lo, as k_pf_qk writes a
// segment's own rows. One workgroup per key coordinate.
__global__ void __launch_bounds__(kPfThreads) k_pf_kv_hist(const float* kc, const float* vc, uint32_t slots, uint32_t kv16,
                                                          uint32_t kb, uint32_t nh, uint32_t hd, _Float16* khi,
                                                          _Float16* klo, _Float16* vhi, _Float16* vlo) {
    const uint32_t j = blockIdx.x;
    if (j >= nh) return;
    const uint64_t slot = static_cast<uint64_t>((kb + j) % slots) * hd;
    for (uint32_t i = threadIdx.x; i < hd; i += kPfThreads) {
        const float k = kv16 ? kv16_float(reinterpret_cast<const uint16_t*>(kc)[slot + i], kv16) : kc[slot + i];
        const float v = kv16 ? kv16_float(reinterpret_cast<const uint16_t*>(vc)[slot + i], kv16) : vc[slot + i];
        const uint64_t ko = pf_kswz(j, i, hd), vo = pf_vswz(j, i, hd);
        pf_split(k, khi + ko, klo + ko);
        pf_split(v, vhi + vo, vlo + vo);
    }
}

// ---- causal attention ----------------------------------------------------------------------

// The pairs (query tile i of 32 rows, head h), numbered i H + h, are dealt in groups of four to
// workgroups, one pair per wave; a group's key range [ks, ke) is the union of its tiles' (one tile's
// when H is a multiple of four), cut into chunks of A.kc keys, one workgroup each. In key
// coordinates (a segment's history first, its rows from A.qo) tile i's first query sits at
// qk0 = A.qo + 32 i; it sees the keys from the window's start for qk0, rounded down to 32, up to
// min(A.qo + T, qk0 + 32).
// All four waves read the same keys and values, loaded straight to LDS one tile ahead (128 KB in two
// stages at hd 256 with low parts), one barrier per tile. A wave keeps its queries and its O^T in
// registers, which leaves one wave per SIMD: what overlaps has to be in one instruction stream. Tile
// n's softmax runs between the products S^T = K Q^T of tile n + 1, and the scores of tile n + 1 are
// read out between the products O^T += V^T E^T of tile n (three f16 products each of the hi/lo parts; lane l on
// query l % 32). One after the other (and with the operand reads left to the scheduler, behind a full
// wait each) a tile took 9000 cycles, 3072 of them products.
// The softmax is in base 2 (the scale times log2 e, v_exp_f32). The running maximum m moves, and O^T
// is rescaled, only when a tile's scores exceed it by more than kPfAttSlack for some query: e_j =
// 2^(v_j - m) then stays below 2^kPfAttSlack, in the same relative precision. Each tile's sum of e_j
// in fp32 is added to a running sum in double.
// LO false: a 16-bit KV cache, whose entries are exact in f16, so the low parts of K and V are zero
// and their products are left out.
// A group whose range is one chunk is finished here (out = O / sum into the activation buffer);
// otherwise the pairs' partials go to opart/mpart/lpart, in register order, and k_pf_attn_merge
// combines them in the next launch. Same result as the masked softmax of src/gemma3.cpp:1602-1696
// over the full row up to rounding; a softmax sum that is not > 0 and finite flags the block.
// MFMA operand layouts (v_mfma_f32_32x32x16_f16): lane l gives A[m = l % 32][k = 8 (l / 32) + j]
// and B[k = 8 (l / 32) + j][n = l % 32], j < 8; result r of lane l is C[8 (r / 4) + 4 (l / 32) +
// r % 4][l % 32].
constexpr uint32_t kPfAttPairs = 4;        // pairs per workgroup (waves)
constexpr uint32_t kPfAttParts = 8192;     // partials kept, at most, if that is one per pair
constexpr uint32_t kPfAttMaxChunks = 64;   // chunks of a range, at most (of two key tiles, at least)
constexpr uint32_t kPfAttFew = 32;         // pairs of a k_pf_attn_few launch, at most
constexpr float kPfAttSlack = 8.0f;
struct PfAttn {
    const _Float16* qhi;   // queries, normed and rotated, in pf_qswz order
    const _Float16* qlo;
    const _Float16* khi;   // keys in pf_kswz order, by key coordinate (32-key tiles)
    const _Float16* klo;
    const _Float16* vhi;   // values in pf_vswz order
    const _Float16* vlo;
    _Float16* o;           // output, an activation buffer of H * hd columns: row q - o_row of query row q
    uint32_t o_row;        //   (earlier query rows of the first tile are not written)
    float* opart;          // [pairs][nch][32 hd] chunk partials sum_j e_j v_j (pairs of the launch)
    float* mpart;          // [pairs][nch][32] their maxima (base 2)
    double* lpart;         // [pairs][nch][32] their sums of e_j
    G3State* st;
    uint32_t T, H, window, block;
    uint32_t kc, nch;      // keys per chunk (a multiple of 32), chunks of the longest range
    uint32_t pair0, pairs;   // first pair of the launch, pairs from it
    uint32_t per, groups;    // pairs per group (kPfAttPairs; k_pf_attn_few: 1), groups
    uint32_t qo;           // key coordinate of query row 0 (keys before it: an earlier segment's history)
    float scale2;          // attention scale times log2(e): the scores in base 2
};

// Key range [ks, ke) of the query tiles i0..i1 (key coordinates, 32 rows each).
__host__ __device__ __forceinline__ void pf_att_range(uint32_t qo, uint32_t T, uint32_t window, uint32_t i0, uint32_t i1,
                                                      uint32_t& ks, uint32_t& ke) {
    const uint32_t q0 = qo + 32u * i0, q1 = qo + 32u * i1 + 32u;
    ke = q1 < qo + T ? q1 : qo + T;
    ks = window != 0u && q0 + 1u > window ? (q0 + 1u - window) & ~31u : 0u;
}
// ... of group g (pairs pair0 + per g and on).
__host__ __device__ __forceinline__ void pf_att_group(const PfAttn& A, uint32_t g, uint32_t& ks, uint32_t& ke) {
    const uint32_t a = A.pair0 + A.per * g, last = A.pair0 + A.pairs - 1u;
    const uint32_t b = a + A.per - 1u < last ? a + A.per - 1u : last;
    pf_att_range(A.qo, A.T, A.window, a / A.H, b / A.H, ks, ke);
}

// O^T tiles times alpha, in the accumulation registers they live in: as plain code the multiplication
// would move all of them to VGPRs and back in every tile, taken or not. The compiler does not see the
// accesses inside the assembly, so the waits are here: the leading ones cover an MFMA's last write, the trailing
// one the next MFMA's read. The empty statements on every tile tie them down: volatile statements keep
// their order, no product that writes a tile can follow the first row of them, and none that reads one can
// precede the last.
template <uint32_t DT>
__device__ __forceinline__ void att_rescale(float16v (&o)[DT], float alpha) {
#pragma unroll
    for (uint32_t j = 0; j < DT; ++j) asm volatile("" : "+a"(o[j]));
    asm volatile("s_nop 15\n\ts_nop 7");
#pragma unroll
    for (uint32_t j = 0; j < DT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float x = o[j][r], t;
            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                         : "+a"(x), "=&v"(t)
                         : "v"(alpha));
            o[j][r] = x;
        }
    asm volatile("s_nop 7");
#pragma unroll
    for (uint32_t j = 0; j < DT; ++j) asm volatile("" : "+a"(o[j]));
}

template <uint32_t HD, bool LO>
__global__ void __launch_bounds__(256, 1) k_pf_attn(PfAttn A) {
#pragma clang fp contract(off)
    constexpr uint32_t KS = HD / 16u;               // k steps of S^T
    constexpr uint32_t DT = HD / 32u;               // d tiles of O^T
    constexpr uint32_t NP = LO ? 2u : 1u;           // parts of K and V
    constexpr uint32_t UK = NP * KS, UV = NP * 2u * DT;   // 1 KB operand units of a key tile: K, V
    constexpr uint32_t kAhead = 3u;                 // operand reads ahead of their products
    __shared__ __align__(1024) unsigned char s_k[2][UK * 1024u];
    __shared__ __align__(1024) unsigned char s_v[2][UV * 1024u];
    // Windowed ranges: workgroup b runs on XCD b % 8 and each XCD takes a contiguous eighth of the
    // (group, chunk) units, so neighbouring groups share their keys in one L2. Full ranges: chunk by
    // chunk, the groups in falling order of length, so every XCD works on the same chunk.
    uint32_t c, g;
    {
        const uint32_t N = gridDim.x;
        uint32_t b = blockIdx.x;
        if (A.window != 0u) {
            if ((N & 7u) == 0u) b = (b & 7u) * (N >> 3) + (b >> 3);
            g = b / A.nch;
            c = b - g * A.nch;
        } else {
            c = b / A.groups;
            g = A.groups - 1u - (b - c * A.groups);
        }
    }
    uint32_t ks, ke;
    pf_att_group(A, g, ks, ke);
    const uint32_t nch = (ke - ks + A.kc - 1u) / A.kc;
    if (c >= nch) return;   // whole workgroup
    const uint32_t k0 = ks + c * A.kc, k1 = min(ke, k0 + A.kc);
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t l32 = lane & 31u, hf = lane >> 5;
    const uint32_t rel = kPfAttPairs * g + wave;            // pair of the launch (its partials' index)
    const bool mine = rel < A.pairs;                        // the last group may be short; every wave loads
    const uint32_t pair = A.pair0 + (mine ? rel : A.pairs - 1u), i = pair / A.H, h = pair - i * A.H;
    const uint32_t T = A.T, qw = A.H * HD;
    const uint32_t q = 32u * i + l32, qk0 = A.qo + 32u * i, qk = qk0 + l32;   // this lane's query: row, key coordinate
    // Loads of key tile n of the chunk: the keys' units, the values' units (unit u by wave u % 4)
    const uint32_t lk = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)&s_k[0][0]));
    const uint32_t lv = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)&s_v[0][0]));
    const uint32_t n_tiles = (k1 - k0 + 31u) >> 5;
    auto load_k = [&](uint32_t n) {
        const uint64_t o = static_cast<uint64_t>((k0 >> 5) + n) * (64u * HD);   // bytes of a tile in each part
#pragma unroll
        for (uint32_t j = 0; j < UK; j += 4u)
            if (const uint32_t u = j + wave; UK % 4u == 0u || u < UK)
                gm_lds16(reinterpret_cast<const char*>(u < KS ? A.khi : A.klo) + o + (u < KS ? u : u - KS) * 1024u, lane * 16u,
                         lk + (n & 1u) * (UK * 1024u) + u * 1024u);
    };
    auto load_v = [&](uint32_t n) {
        const uint64_t o = static_cast<uint64_t>((k0 >> 5) + n) * (64u * HD);
#pragma unroll
        for (uint32_t j = 0; j < UV; j += 4u)
            if (const uint32_t u = j + wave; UV % 4u == 0u || u < UV)
                gm_lds16(reinterpret_cast<const char*>(u < 2u * DT ? A.vhi : A.vlo) + o + (u < 2u * DT ? u : u - 2u * DT) * 1024u,
                         lane * 16u, lv + (n & 1u) * (UV * 1024u) + u * 1024u);
    };
    load_k(0u);
    // the queries (B operand of S^T); rows past T hold stale values, which stay in their own lanes (settle), and
    // their results are never written
    half8 qb[KS][2];
    {
        const uint64_t o = (static_cast<uint64_t>(i) * A.H + h) * (KS * 512u) + 8u * lane;
#pragma unroll
        for (uint32_t k = 0; k < KS; ++k) {
            qb[k][0] = *reinterpret_cast<const half8*>(A.qhi + o + 512u * k);
            qb[k][1] = *reinterpret_cast<const half8*>(A.qlo + o + 512u * k);
        }
        // waited for here: left to the first tile, the wait would be in the loop and drain its loads too
#pragma unroll
        for (uint32_t k = 0; k < KS; ++k)
#pragma unroll
            for (uint32_t e = 0; e < 2u; ++e) asm volatile("" : "+v"(qb[k][e]));
    }
    float m = -INFINITY;   // reference maximum of the scaled scores of query q
    double lsum = 0.0;     // this lane's share of sum_j e_j
    float16v o[DT];        // O^T tiles: d = 32 dt + 8 (r / 4) + 4 hf + r % 4, query q
#pragma unroll
    for (uint32_t j = 0; j < DT; ++j) o[j] = float16v{};
    // S^T of tile n as two chains, sa + sb. Operand reads run kAhead units ahead of their products, in
    // this order; `between(s)`, s < 2 KS, is work for the products around it to cover.
    float16v sa, sb;
    auto scores = [&](uint32_t n, auto between) {
        const unsigned char* pk = &s_k[n & 1u][lane * 16u];
        half8 kf[KS][NP];
        sa = float16v{};
        sb = float16v{};
#pragma unroll
        for (uint32_t k = 0; k < kAhead && k < KS; ++k)
#pragma unroll
            for (uint32_t e = 0; e < NP; ++e) kf[k][e] = *reinterpret_cast<const half8*>(pk + (e * KS + k) * 1024u);
#pragma unroll
        for (uint32_t k = 0; k < KS; ++k) {
            if (k + kAhead < KS)
#pragma unroll
                for (uint32_t e = 0; e < NP; ++e)
                    kf[k + kAhead][e] = *reinterpret_cast<const half8*>(pk + (e * KS + k + kAhead) * 1024u);
            __builtin_amdgcn_sched_barrier(0);
            sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[k][0], qb[k][0], sa, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            between(2u * k);
            __builtin_amdgcn_sched_barrier(0);
            sb = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[k][0], qb[k][1], sb, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            between(2u * k + 1u);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LO) {
                if (k & 1u) sb = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[k][1], qb[k][0], sb, 0, 0, 0);
                else sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[k][1], qb[k][0], sa, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Tile n's scores v in base 2 (scale * log2 e folded in, tmax their maximum): masked where some key of
    // the tile is hidden from some query, then the new reference maximum.
    float v[16], tmax = -INFINITY, alpha = 1.0f;
    bool grown = false;   // O^T is to be rescaled by alpha before the tile's products
    auto settle = [&](uint32_t n) {
        const uint32_t kt = k0 + 32u * n;
        if (!(kt + 31u < k1 && kt + 31u <= qk0 && (A.window == 0u || kt + A.window > qk0 + 31u))) {
            tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t key = kt + 16u * (r / 8) + 8u * hf + (r % 8);
                const bool ok = key < k1 && key <= qk && (A.window == 0u || key + A.window > qk);
                v[r] = ok ? v[r] : -INFINITY;
                tmax = fmaxf(tmax, v[r]);
            }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        // whole wave, but only for its queries: rows past T hold another prompt's, which would decide how this
        // one is rounded. A query with nothing visible yet has m = -inf.
        if (__any(q < T && tmax > m + kPfAttSlack)) {
            const float mn = fmaxf(m, tmax);
            alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            grown = n != 0u;   // O^T is zero before the first tile
            m = mn;
            lsum *= static_cast<double>(alpha);
        }
    };
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");   // queries and the first keys
    load_v(0u);
    if (n_tiles > 1u) load_k(1u);
    scores(0u, [](uint32_t) {});
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        v[r] = (sa[r] + sb[r]) * A.scale2;
        tmax = fmaxf(tmax, v[r]);
    }
    settle(0u);
    float base, es;   // the tile's sum of e_j in fp32, then into the double sum
    float ev[16];
    uint32_t ehu[8], elu[8];   // e as f16 hi and lo, two per register
    // The asm statements keep a value's computation where it stands, between the products (the
    // compiler would sink it to its first use).
    auto soft_exp = [&](uint32_t r) {
        ev[r] = __builtin_amdgcn_exp2f(v[r] - base);   // exp(scale s_j - m ln 2)
        es += ev[r];
        asm volatile("" : "+v"(ev[r]));
    };
    auto soft_split = [&](uint32_t p) {
        typedef _Float16 half2 __attribute__((ext_vector_type(2)));
        half2 h, l;
#pragma unroll
        for (uint32_t e = 0; e < 2u; ++e) {
            h[e] = static_cast<_Float16>(ev[2u * p + e]);
            l[e] = static_cast<_Float16>(ev[2u * p + e] - static_cast<float>(h[e]));
        }
        ehu[p] = __builtin_bit_cast(uint32_t, h);
        elu[p] = __builtin_bit_cast(uint32_t, l);
        asm volatile("" : "+v"(ehu[p]), "+v"(elu[p]));
    };
    // slot t of S: its share of the exponentials, and the splits of the slots before it
    auto soft_slot = [&](uint32_t t, uint32_t S) {
#pragma unroll
        for (uint32_t r = 0; r < 16u; ++r)
            if (r >= 16u * t / S && r < 16u * (t + 1u) / S) soft_exp(r);
        if (t != 0u)
#pragma unroll
            for (uint32_t p = 0; p < 8u; ++p)
                if (p >= 16u * (t - 1u) / S / 2u && p < 16u * t / S / 2u) soft_split(p);
    };
    auto soft_rest = [&](uint32_t S) {
#pragma unroll
        for (uint32_t p = 0; p < 8u; ++p)
            if (p >= 16u * (S - 1u) / S / 2u) soft_split(p);
    };
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    // O^T += V^T E^T of tile n; `between(k)` is work for the products of unit k to cover
    auto values = [&](uint32_t n, auto between) {
        if (grown) {
            att_rescale<DT>(o, alpha);
            grown = false;
        }
        half8 eh[2], el[2];
#pragma unroll
        for (uint32_t e = 0; e < 2u; ++e) {
            eh[e] = __builtin_bit_cast(half8, u4{ehu[4u * e], ehu[4u * e + 1u], ehu[4u * e + 2u], ehu[4u * e + 3u]});
            el[e] = __builtin_bit_cast(half8, u4{elu[4u * e], elu[4u * e + 1u], elu[4u * e + 2u], elu[4u * e + 3u]});
        }
        const unsigned char* pv = &s_v[n & 1u][lane * 16u];
        half8 vf[2u * DT][NP];   // unit 2 j + sk
#pragma unroll
        for (uint32_t k = 0; k < kAhead && k < 2u * DT; ++k)
#pragma unroll
            for (uint32_t e = 0; e < NP; ++e) vf[k][e] = *reinterpret_cast<const half8*>(pv + (e * 2u * DT + k) * 1024u);
#pragma unroll
        for (uint32_t k = 0; k < 2u * DT; ++k) {
            if (k + kAhead < 2u * DT)
#pragma unroll
                for (uint32_t e = 0; e < NP; ++e)
                    vf[k + kAhead][e] = *reinterpret_cast<const half8*>(pv + (e * 2u * DT + k + kAhead) * 1024u);
            __builtin_amdgcn_sched_barrier(0);
            float16v& oj = o[k >> 1];
            oj = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[k][0], eh[k & 1u], oj, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            between(k);
            __builtin_amdgcn_sched_barrier(0);
            oj = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[k][0], el[k & 1u], oj, 0, 0, 0);
            if constexpr (LO) oj = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[k][1], eh[k & 1u], oj, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto begin = [&]() {   // the loads before the last barrier have arrived, and every wave is past them
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    for (uint32_t n = 0; n + 1u < n_tiles; ++n) {
        begin();   // the keys of tile n + 1 and the values of tile n
        if (n + 2u < n_tiles) load_k(n + 2u);
        load_v(n + 1u);
        base = m == -INFINITY ? 0.0f : m;   // nothing visible yet: every e_j is 0
        es = 0.0f;
        scores(n + 1u, [&](uint32_t t) { soft_slot(t, 2u * KS); });
        soft_rest(2u * KS);
        lsum += static_cast<double>(es);
        tmax = -INFINITY;
        values(n, [&](uint32_t k) {         // the next tile's scores
#pragma unroll
            for (uint32_t r = 0; r < 16u; ++r)
                if (r >= 16u * k / (2u * DT) && r < 16u * (k + 1u) / (2u * DT)) {
                    v[r] = (sa[r] + sb[r]) * A.scale2;
                    tmax = fmaxf(tmax, v[r]);
                    asm volatile("" : "+v"(v[r]), "+v"(tmax));
                }
        });
        settle(n + 1u);
    }
    begin();
    base = m == -INFINITY ? 0.0f : m;
    es = 0.0f;
    soft_slot(0u, 1u);
    soft_rest(1u);
    lsum += static_cast<double>(es);
    values(n_tiles - 1u, [](uint32_t) {});
    if (!mine) return;
    lsum += __shfl_xor(lsum, 32);   // both lane halves now hold query q's sum
    if (nch == 1u) {   // the whole key range: normalise and write the output rows
        if (q >= T || q < A.o_row) return;
        const double den = lsum;
        if (hf == 0u && (!(den > 0.0) || !__builtin_isfinite(den)))   // :1666-1670
            atomicMin(&A.st->nonfinite, g3_code_softmax(A.block));
        const float inv = static_cast<float>(1.0 / den);
#pragma unroll
        for (uint32_t j = 0; j < DT; ++j)
#pragma unroll
            for (uint32_t rq = 0; rq < 4u; ++rq) {
                const uint64_t oo = gm_off(q - A.o_row, h * HD + 32u * j + 8u * rq + 4u * hf, qw / 32u);
                pf_split4(f4{o[j][4 * rq] * inv, o[j][4 * rq + 1] * inv, o[j][4 * rq + 2] * inv, o[j][4 * rq + 3] * inv},
                          A.o + oo, A.o + oo + kGmLo);
            }
        return;
    }
    const uint64_t unit = static_cast<uint64_t>(rel) * A.nch + c;
    float* op = A.opart + unit * 32u * HD + lane * 4u;
#pragma unroll
    for (uint32_t j = 0; j < DT; ++j)
#pragma unroll
        for (uint32_t rq = 0; rq < 4u; ++rq)
            *reinterpret_cast<f4*>(op + (4u * j + rq) * 256u) = f4{o[j][4 * rq], o[j][4 * rq + 1], o[j][4 * rq + 2], o[j][4 * rq + 3]};
    if (hf == 0u) {
        A.mpart[unit * 32u + l32] = m;
        A.lpart[unit * 32u + l32] = lsum;
    }
}

// k_pf_attn for launches of few pairs, which four pairs per workgroup would put on a handful of CUs, each with
// a long chain: one pair per workgroup, its four waves splitting the head dimension (wave w: the k steps w,
// w + 4, ... of S^T and the d tiles w, w + 4, ... of O^T). The operands come straight to registers, the
// next tile's during the current one; each wave's partial S^T goes through LDS and every wave adds the
// four in wave order (the same scores in every wave), one barrier per tile. Softmax, results and
// partials as in k_pf_attn. 37 rows: 11.5 -> 8.3 us. Up to kPfAttFew pairs; a prefill
// of six blocks, 4 heads of 256, with this kernel and with k_pf_attn: 8 pairs 318 and 333 us, 16 pairs 361 and 381,
// 24 pairs 409 and 404, 32 pairs 422 and 417 (processes differ by 1%), 64 pairs 497 and 490.
template <uint32_t HD, bool LO>
__global__ void __launch_bounds__(256) k_pf_attn_few(PfAttn A) {
#pragma clang fp contract(off)
    constexpr uint32_t KS = HD / 16u, DT = HD / 32u, NP = LO ? 2u : 1u;
    constexpr uint32_t KW = (KS + 3u) / 4u, DW = (DT + 3u) / 4u;   // k steps and d tiles per wave, at most
    __shared__ __align__(16) float s_s[2][4][16 * 64];
    const uint32_t c = blockIdx.x / A.groups, rel = blockIdx.x - c * A.groups;
    uint32_t ks, ke;
    pf_att_group(A, rel, ks, ke);
    const uint32_t nch = (ke - ks + A.kc - 1u) / A.kc;
    if (c >= nch) return;   // whole workgroup
    const uint32_t k0 = ks + c * A.kc, k1 = min(ke, k0 + A.kc);
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t l32 = lane & 31u, hf = lane >> 5;
    const uint32_t pair = A.pair0 + rel, i = pair / A.H, h = pair - i * A.H, T = A.T, qw = A.H * HD;
    const uint32_t q = 32u * i + l32, qk0 = A.qo + 32u * i, qk = qk0 + l32;
    struct Ops {
        half8 k[KW][NP], v[DW][2][NP];
    };
    auto load = [&](uint32_t kt, Ops& R) {   // steps and tiles past the end: the last one (not used)
        const uint64_t tile = static_cast<uint64_t>(kt >> 5) * (32u * HD) + 8u * lane;
#pragma unroll
        for (uint32_t j = 0; j < KW; ++j) {
            const uint64_t o = tile + min(wave + 4u * j, KS - 1u) * 512u;
            R.k[j][0] = *reinterpret_cast<const half8*>(A.khi + o);
            if constexpr (LO) R.k[j][1] = *reinterpret_cast<const half8*>(A.klo + o);
        }
#pragma unroll
        for (uint32_t j = 0; j < DW; ++j)
#pragma unroll
            for (uint32_t sk = 0; sk < 2u; ++sk) {
                const uint64_t o = tile + (min(wave + 4u * j, DT - 1u) * 2u + sk) * 512u;
                R.v[j][sk][0] = *reinterpret_cast<const half8*>(A.vhi + o);
                if constexpr (LO) R.v[j][sk][1] = *reinterpret_cast<const half8*>(A.vlo + o);
            }
    };
    half8 qb[KW][2];
    {
        const uint64_t o = (static_cast<uint64_t>(i) * A.H + h) * (KS * 512u) + 8u * lane;
#pragma unroll
        for (uint32_t j = 0; j < KW; ++j) {
            qb[j][0] = *reinterpret_cast<const half8*>(A.qhi + o + 512u * min(wave + 4u * j, KS - 1u));
            qb[j][1] = *reinterpret_cast<const half8*>(A.qlo + o + 512u * min(wave + 4u * j, KS - 1u));
        }
    }
    float m = -INFINITY;
    double lsum = 0.0;
    float16v o[DW];
#pragma unroll
    for (uint32_t j = 0; j < DW; ++j) o[j] = float16v{};
    uint32_t buf = 0;
    auto step = [&](uint32_t kt, const Ops& R) {
        float16v sp = {};
#pragma unroll
        for (uint32_t j = 0; j < KW; ++j) {
            if (wave + 4u * j >= KS) continue;
            sp = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.k[j][0], qb[j][0], sp, 0, 0, 0);
            sp = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.k[j][0], qb[j][1], sp, 0, 0, 0);
            if constexpr (LO) sp = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.k[j][1], qb[j][0], sp, 0, 0, 0);
        }
        // (buffer buf was last read two tiles ago, before the barrier of the previous tile)
#pragma unroll
        for (uint32_t rq = 0; rq < 4u; ++rq)
            *reinterpret_cast<f4*>(&s_s[buf][wave][(rq * 64u + lane) * 4u]) = f4{sp[4 * rq], sp[4 * rq + 1], sp[4 * rq + 2], sp[4 * rq + 3]};
        __syncthreads();
        float v[16], tmax = -INFINITY;
#pragma unroll
        for (uint32_t rq = 0; rq < 4u; ++rq) {
            f4 t = *reinterpret_cast<const f4*>(&s_s[buf][0][(rq * 64u + lane) * 4u]);
#pragma unroll
            for (uint32_t w = 1; w < 4u; ++w) {
                const f4 u = *reinterpret_cast<const f4*>(&s_s[buf][w][(rq * 64u + lane) * 4u]);
#pragma unroll
                for (int e = 0; e < 4; ++e) t[e] += u[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * rq + e] = t[e] * A.scale2;
        }
        buf ^= 1u;
        const bool whole = kt + 31u < k1 && kt + 31u <= qk0 && (A.window == 0u || kt + A.window > qk0 + 31u);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t key = kt + 16u * (r / 8) + 8u * hf + (r % 8);
            if (!whole && !(key < k1 && key <= qk && (A.window == 0u || key + A.window > qk))) v[r] = -INFINITY;
            tmax = fmaxf(tmax, v[r]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float mn = fmaxf(m, tmax), base = mn == -INFINITY ? 0.0f : mn;   // nothing visible yet: every e_j is 0
        const float alpha = __builtin_amdgcn_exp2f(m - base);
        m = mn;
        float es = 0.0f;
        half8 eh[2], el[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float e = __builtin_amdgcn_exp2f(v[r] - base);
            es += e;
            eh[r / 8][r % 8] = static_cast<_Float16>(e);
            el[r / 8][r % 8] = static_cast<_Float16>(e - static_cast<float>(eh[r / 8][r % 8]));
        }
        lsum = lsum * static_cast<double>(alpha) + static_cast<double>(es);
#pragma unroll
        for (uint32_t j = 0; j < DW; ++j) {
            if (wave + 4u * j >= DT) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) o[j][r] *= alpha;
#pragma unroll
            for (uint32_t sk = 0; sk < 2u; ++sk) {
                o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.v[j][sk][0], eh[sk], o[j], 0, 0, 0);
                o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.v[j][sk][0], el[sk], o[j], 0, 0, 0);
                if constexpr (LO) o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(R.v[j][sk][1], eh[sk], o[j], 0, 0, 0);
            }
        }
    };
    Ops ra, rb;   // two operand sets in turn
    load(k0, ra);
    for (uint32_t kt = k0; kt < k1; kt += 64u) {
        if (kt + 32u < k1) load(kt + 32u, rb);
        step(kt, ra);
        if (kt + 32u >= k1) break;
        if (kt + 64u < k1) load(kt + 64u, ra);
        step(kt + 32u, rb);
    }
    lsum += __shfl_xor(lsum, 32);
    if (nch == 1u) {
        if (q >= T || q < A.o_row) return;
        const double den = lsum;
        if (wave == 0u && hf == 0u && (!(den > 0.0) || !__builtin_isfinite(den)))   // :1666-1670
            atomicMin(&A.st->nonfinite, g3_code_softmax(A.block));
        const float inv = static_cast<float>(1.0 / den);
#pragma unroll
        for (uint32_t j = 0; j < DW; ++j) {
            if (wave + 4u * j >= DT) continue;
#pragma unroll
            for (uint32_t rq = 0; rq < 4u; ++rq) {
                const uint64_t oo = gm_off(q - A.o_row, h * HD + 32u * (wave + 4u * j) + 8u * rq + 4u * hf, qw / 32u);
                pf_split4(f4{o[j][4 * rq] * inv, o[j][4 * rq + 1] * inv, o[j][4 * rq + 2] * inv, o[j][4 * rq + 3] * inv},
                          A.o + oo, A.o + oo + kGmLo);
            }
        }
        return;
    }
    const uint64_t unit = static_cast<uint64_t>(rel) * A.nch + c;
#pragma unroll
    for (uint32_t j = 0; j < DW; ++j) {
        if (wave + 4u * j >= DT) continue;
#pragma unroll
        for (uint32_t rq = 0; rq < 4u; ++rq)
            *reinterpret_cast<f4*>(A.opart + unit * 32u * HD + (4u * (wave + 4u * j) + rq) * 256u + lane * 4u) =
                f4{o[j][4 * rq], o[j][4 * rq + 1], o[j][4 * rq + 2], o[j][4 * rq + 3]};
    }
    if (wave == 0u && hf == 0u) {
        A.mpart[unit * 32u + l32] = m;
        A.lpart[unit * 32u + l32] = lsum;
    }
}

// Merge of the chunk partials of the groups that k_pf_attn split (one wave per (pair, d tile); pairs
// of one-chunk groups were finished there): lane l on query l % 32, its 16 values of the d tile as
// k_pf_attn held them; in chunk order, with M the running maximum of the chunk maxima m_c, den =
// sum_c 2^(m_c - M) sum_c (double), out = sum_c 2^(m_c - M) O_c / den into the activation buffer.
template <uint32_t HD>
__global__ void __launch_bounds__(256) k_pf_attn_merge(PfAttn A) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, hf = lane >> 5;
    const uint32_t rel = blockIdx.x, j = blockIdx.y * 4u + (threadIdx.x >> 6);
    if (j >= HD / 32u) return;   // whole wave
    uint32_t ks, ke;
    pf_att_group(A, rel / A.per, ks, ke);
    const uint32_t nch = (ke - ks + A.kc - 1u) / A.kc;
    const uint32_t pair = A.pair0 + rel, i = pair / A.H, h = pair - i * A.H, q = 32u * i + l32;
    if (nch == 1u) return;   // whole wave
    const uint64_t unit0 = static_cast<uint64_t>(rel) * A.nch;
    // chunks in groups of kG, every load of a group issued together (indices clamped to the last
    // chunk; the clamped duplicates are not used): one round of loads for up to kG chunks
    constexpr uint32_t kG = 4;
    double den = 0.0;
    f4 acc[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) acc[k] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float M = -INFINITY;
    for (uint32_t c0 = 0; c0 < nch; c0 += kG) {
        float mv[kG];
        double lv[kG];
        f4 x[kG][4];
#pragma unroll
        for (uint32_t k = 0; k < kG; ++k) {
            const uint64_t u = unit0 + min(c0 + k, nch - 1u);
            mv[k] = A.mpart[u * 32u + l32];
            lv[k] = A.lpart[u * 32u + l32];
            const float* src = A.opart + u * 32u * HD + j * 1024u + lane * 4u;
#pragma unroll
            for (uint32_t rq = 0; rq < 4u; ++rq) x[k][rq] = *reinterpret_cast<const f4*>(src + rq * 256u);
        }
        __builtin_amdgcn_sched_barrier(0);   // the group's loads stay ahead of their first use
        // running merge: the group's maximum rescales what is accumulated so far
        float Mg = M;
#pragma unroll
        for (uint32_t k = 0; k < kG; ++k)
            if (c0 + k < nch) Mg = fmaxf(Mg, mv[k]);
        const float fo = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - Mg);
        den *= static_cast<double>(fo);
#pragma unroll
        for (uint32_t rq = 0; rq < 4u; ++rq)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[rq][e] *= fo;
        M = Mg;
#pragma unroll
        for (uint32_t k = 0; k < kG; ++k) {
            if (c0 + k >= nch) break;
            // a chunk with no key that this query sees has m_c = -inf and weight 0
            const float f = mv[k] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mv[k] - M);
            den += lv[k] * static_cast<double>(f);
#pragma unroll
            for (uint32_t rq = 0; rq < 4u; ++rq)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[rq][e] += f * x[k][rq][e];
        }
    }
    if (q >= A.T || q < A.o_row) return;
    if (j == 0u && hf == 0u && (!(den > 0.0) || !__builtin_isfinite(den)))   // :1666-1670
        atomicMin(&A.st->nonfinite, g3_code_softmax(A.block));
    const float inv = static_cast<float>(1.0 / den);
#pragma unroll
    for (uint32_t rq = 0; rq < 4u; ++rq) {
        const uint64_t oo = gm_off(q - A.o_row, h * HD + 32u * j + 8u * rq + 4u * hf, A.H * HD / 32u);
        pf_split4(f4{acc[rq][0] * inv, acc[rq][1] * inv, acc[rq][2] * inv, acc[rq][3] * inv}, A.o + oo, A.o + oo + kGmLo);
    }
}

// ---- host side --------------------------------------------------------------------------

template <int WN, int NWN>
static int pf_launch_q8(const PfGemm& G, uint32_t splits, hipStream_t s) {
    constexpr uint32_t BN = 32u * WN * NWN;
    const dim3 grid((G.N + BN - 1u) / BN, (G.M + kQgBM - 1u) / kQgBM, splits);
    PfGemm arg = G;
    void* args[] = {&arg};
    VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_pf_gemm_q8<WN, NWN>), grid, dim3(128u * NWN), args,
                                  0, s));
    return VRT_OK;
}

// K splits of the GEMMs on the Q8_0 rows: enough workgroups to cover the CUs.
static uint32_t pf_splits_q8(uint32_t M, uint32_t N, uint32_t K) {
    const uint32_t tiles = ((M + kQgBM - 1u) / kQgBM) * ((N + 63u) / 64u);
    const uint32_t s = std::min(kPfMaxSplits, std::max(1u, 256u / std::max(1u, tiles)));
    return std::max(1u, std::min(s, (K / 32u) / 2u));
}

// C[M][N] = A[M][K] (an activation buffer) x W^T, W = Q8_0 matrices concatenated along N, or
// their expansion `ex` where there is one (vrt_gemm.hip). With `used`, the K blocks may be split over
// *used workgroups; C then holds the partial products C + z * M * N, z < *used. With glu (segs: gate, up):
// gelu_tanh(A Wg^T) * (A Wu^T) into the activation buffer o (src/gemma3.cpp:1720-1801 up to the
// down projection).
static int pf_gemm(const _Float16* a, uint32_t M, uint32_t K,
                   std::initializer_list<std::pair<const uint8_t*, uint32_t>> segs, const PfMatrix* ex, float* c,
                   _Float16* o, bool glu, uint32_t* used, hipStream_t s) {
    uint32_t N = 0;
    for (const auto& sg : segs) N += sg.second;
    // any N: rows past N load clamped, in-bounds rows, are zeroed in LDS and never stored
    if (K % 32u != 0u || N == 0u || (glu && N % 64u != 0u))
        return set_error(VRT_ERR_INVALID, "prefill GEMM shape not supported");
    if (ex && ex->h) {
        GmArgs G{};
        G.a = a;
        G.w = static_cast<const _Float16*>(ex->h);
        G.ws = ex->s;
        G.c = c;
        G.o = o;
        G.c_bs = static_cast<uint64_t>(M) * N;
        G.ldc = G.N = N;
        G.M = M;
        G.nkb = K / 32u;
        G.npad = (N + kGmRowPad - 1u) / kGmRowPad * kGmRowPad;
        const uint32_t splits = used ? gm_splits(M, N, G.nkb) : 1u;
        if (used) *used = splits;
        return gm_run(G, splits, glu, s);
    }
    PfGemm G{};
    G.a = a;
    for (const auto& sg : segs) {
        G.w[G.nseg] = sg.first;
        G.rows[G.nseg++] = sg.second;
    }
    G.N = N;
    G.c = c;
    G.o = o;
    G.c_bs = static_cast<uint64_t>(M) * N;
    G.M = M;
    G.K = K;
    G.glu = glu ? 1u : 0u;
    const uint32_t splits = used ? pf_splits_q8(M, N, K) : 1u;
    if (used) *used = splits;
    const uint32_t mt = (M + kQgBM - 1u) / kQgBM;
    return N % 128u == 0u && (N / 128u) * mt >= 128u ? pf_launch_q8<1, 4>(G, splits, s) : pf_launch_q8<1, 2>(G, splits, s);
}

// k_pf_norm_w over `rows` rows of n <= 2048 elements (runs of four per lane: the smallest of 1, 2, 3,
// 4, 6, 8 that covers n).
int pf_norm(float* h, const float* f, uint32_t nsplit, uint64_t sstride, const float* w_post, const float* w_next,
            uint32_t n, float eps, _Float16* x, G3State* st, uint32_t block, uint32_t rows, hipStream_t s, bool into) {
    uint32_t in = into ? 1u : 0u;
    void* args[] = {&h, &f, &nsplit, &sstride, &w_post, &w_next, &n, &eps, &x, &st, &block, &rows, &in};
    const uint32_t nq = (n + 255u) / 256u;
    const void* fn = nq <= 1u   ? reinterpret_cast<const void*>(&k_pf_norm_w<1>)
                     : nq <= 2u ? reinterpret_cast<const void*>(&k_pf_norm_w<2>)
                     : nq <= 3u ? reinterpret_cast<const void*>(&k_pf_norm_w<3>)
                     : nq <= 4u ? reinterpret_cast<const void*>(&k_pf_norm_w<4>)
                     : nq <= 6u ? reinterpret_cast<const void*>(&k_pf_norm_w<6>)
                     : nq <= 8u ? reinterpret_cast<const void*>(&k_pf_norm_w<8>)
                                : nullptr;
    if (!fn || n % 32u != 0u || nsplit > kPfMaxSplits) return set_error(VRT_ERR_INVALID, "prefill norm shape not supported");
    const uint32_t per = kPfThreads / 64u;
    VRT_HIP_CHECK(hipLaunchKernel(fn, dim3((rows + per - 1u) / per), dim3(kPfThreads), args, 0, s));
    return VRT_OK;
}

// Block l's attention norm and q|k|v projection over M rows (glu false: c, *used partials), or its FFN norm and
// gelu_tanh(gate) * up (glu true: the activation buffer o): first h = f * (scale(f) * w_post) + h with f the sum
// of nsplit partials (nullptr: none). Few rows run as one launch, which leaves the new residual in *spare and
// swaps the two pointers; otherwise the norm goes through the activation buffer a.
int pf_norm_project(vrt_g3* g, uint32_t l, bool glu, float** h, float** spare, const float* f, uint32_t nsplit, uint64_t sstride,
                    const float* w_post, uint32_t fold_block, _Float16* a, uint32_t M, float* c, uint32_t* used, _Float16* o,
                    G3State* st, hipStream_t s) {
    const LayerParams& Ly = g->layers[l];
    const uint32_t d = g->cfg.embedding_length, nkb = d / 32u;
    const float* w_next = glu ? Ly.ffn_norm : Ly.attn_norm;
    if (g->pf.lw.empty() || (f && nsplit != 1u) || !gm_norm_fits(M, nkb)) {
        if (int rc = pf_norm(*h, f, nsplit, sstride, w_post, w_next, d, g->P.eps, a, st, fold_block, M, s, true)) return rc;
        return glu ? pf_ffn_glu(g, l, a, M, o, s) : pf_project(g, l, kProjQkv, a, M, c, used, s);
    }
    const PfMatrix& m = glu ? g->pf.lw[l].gu : g->pf.lw[l].qkv;
    GmArgs G{};
    G.w = static_cast<const _Float16*>(m.h);
    G.ws = m.s;
    G.c = c;
    G.o = o;
    G.M = M;
    G.N = glu ? 2u * g->cfg.feed_forward_length : (g->cfg.head_count + 2u) * g->cfg.head_dim;
    G.ldc = G.N;
    G.nkb = nkb;
    G.npad = (G.N + kGmRowPad - 1u) / kGmRowPad * kGmRowPad;
    const GmNorm R{*h, f, *spare, w_post, w_next, &st->nonfinite, g3_code_nonfinite(fold_block), g->P.eps};
    if (used) *used = 1u;
    if (f) std::swap(*h, *spare);
    return gm_run_norm(G, R, glu, s);
}

// Block l's projection `which` over the M rows of the activation buffer a: C = A x W^T, or partial
// z of *used K splits at c + z * M * N.
int pf_project(vrt_g3* g, uint32_t l, uint32_t which, const _Float16* a, uint32_t M, float* c, uint32_t* used, hipStream_t s) {
    const LayerParams& Ly = g->layers[l];
    const PfLayerW* lw = g->pf.lw.empty() ? nullptr : &g->pf.lw[l];
    const uint32_t d = g->cfg.embedding_length, hd = g->cfg.head_dim, qw = g->cfg.head_count * hd;
    const uint32_t F = g->cfg.feed_forward_length;
    switch (which) {
    case kProjQkv: return pf_gemm(a, M, d, {{Ly.wq, qw}, {Ly.wk, hd}, {Ly.wv, hd}}, lw ? &lw->qkv : nullptr, c, nullptr, false, used, s);
    case kProjO: return pf_gemm(a, M, qw, {{Ly.wo, d}}, lw ? &lw->o : nullptr, c, nullptr, false, used, s);
    case kProjDown: return pf_gemm(a, M, F, {{Ly.wd, d}}, lw ? &lw->down : nullptr, c, nullptr, false, used, s);
    default: return set_error(VRT_ERR_INVALID, "unknown projection %u", which);
    }
}

// Block l's gelu_tanh(gate) * up over the M rows of a, into the activation buffer o of F columns.
int pf_ffn_glu(vrt_g3* g, uint32_t l, const _Float16* a, uint32_t M, _Float16* o, hipStream_t s) {
    const LayerParams& Ly = g->layers[l];
    const PfLayerW* lw = g->pf.lw.empty() ? nullptr : &g->pf.lw[l];
    const uint32_t F = g->cfg.feed_forward_length;
    return pf_gemm(a, M, g->cfg.embedding_length, {{Ly.wg, F}, {Ly.wu, F}}, lw ? &lw->gu : nullptr, nullptr, o, true, nullptr, s);
}

// Logits of M rows against the tied Q8_0 embedding table: logits [M][vocab] = x W_embd^T, x an
// activation buffer (MFMA on the Q8_0 rows of the arena, one K split).
int pf_lm_logits(vrt_g3* g, const _Float16* x, uint32_t M, float* logits, hipStream_t s) {
    return pf_gemm(x, M, g->cfg.embedding_length, {{g->P.tok_embd, g->cfg.vocab_size}}, nullptr, logits, nullptr, false, nullptr, s);
}

static uint32_t pf_pad(uint32_t T) { return (T + kPfTile - 1u) / kPfTile * kPfTile; }

int pf_setup(vrt_g3* g, uint32_t max_t) {
    const uint32_t d = g->cfg.embedding_length, H = g->cfg.head_count, hd = g->cfg.head_dim;
    const uint32_t F = g->cfg.feed_forward_length, qw = H * hd, nqkv = qw + 2u * hd;
    PfState& p = g->pf;
    p.max_t = 0;
    if (d > 8u * kPfThreads || hd > 256u || hd % 32u || d % 32u || qw % 32u || F % 32u || nqkv % 32u) return VRT_OK;
    const uint64_t tp = pf_pad(max_t);
    auto take = [&](size_t bytes, void** out) -> int {
        VRT_HIP_CHECK(hipMalloc(out, bytes + 256u));
        g->allocs.push_back(*out);
        return VRT_OK;
    };
    void* q;
    if (int rc = take(static_cast<size_t>(max_t) * d * 4u, &q)) return rc;
    p.h = static_cast<float*>(q);
    if (int rc = take(16u * static_cast<size_t>(d) * 4u, &q)) return rc;   // rows of gm_norm_fits
    p.h2 = static_cast<float*>(q);
    // K splits only while their partials are few (gm_splits, pf_splits_q8)
    if (int rc = take(std::max<size_t>(static_cast<size_t>(max_t) * d, kGmSplitFloats) * 4u, &q)) return rc;
    p.x = static_cast<float*>(q);
    if (int rc = take(gm_size(max_t, std::max(d, qw)) * 2u, &q)) return rc;
    p.a = static_cast<_Float16*>(q);
    if (int rc = take(gm_size(max_t, F) * 2u, &q)) return rc;
    p.g = static_cast<_Float16*>(q);
    if (int rc = take(std::max<size_t>(static_cast<size_t>(max_t) * nqkv, kGmSplitFloats) * 4u, &q)) return rc;
    p.qkv = static_cast<float*>(q);
    if (int rc = take(static_cast<size_t>(tp) * qw * 2u, &q)) return rc;
    p.qhi = static_cast<_Float16*>(q);
    if (int rc = take(static_cast<size_t>(tp) * qw * 2u, &q)) return rc;
    p.qlo = static_cast<_Float16*>(q);
    // keys and values of a segment's history and rows (f16 each): prompts longer than max_t run
    // in segments whose keys reach back to position 0 in a global block
    p.tkv = static_cast<uint32_t>(std::max<uint64_t>(tp, pf_pad(g->cfg.context_length)));
    void** kv[] = {&p.khi, &p.klo, &p.vhi, &p.vlo};
    for (void** b : kv)
        if (int rc = take(static_cast<size_t>(hd) * p.tkv * 2u, b)) return rc;
    // as many partials as any launch of this executor can cut its ranges into (context 512: 512 of 32 KB
    // at 4 heads of 256), up to kPfAttParts
    const uint32_t pairs = H * ((max_t + 31u) / 32u), cut = std::min(kPfAttMaxChunks, (p.tkv + 63u) / 64u);
    p.parts = std::max(pairs, std::min(kPfAttParts, (pairs + kPfAttPairs - 1u) / kPfAttPairs * kPfAttPairs * cut));
    if (int rc = take(static_cast<size_t>(p.parts) * 32u * hd * 4u, &q)) return rc;
    p.opart = static_cast<float*>(q);
    if (int rc = take(static_cast<size_t>(p.parts) * 32u * 4u, &q)) return rc;
    p.mpart = static_cast<float*>(q);
    if (int rc = take(static_cast<size_t>(p.parts) * 32u * 8u, &q)) return rc;
    p.lpart = static_cast<double*>(q);
    // Expanded weights: 2 bytes per quant + 4 per 32 (2.125 bytes per weight, twice the Q8_0
    // matrices' 1.0625), made once here when they fit kPfExpandBudget.
    const uint64_t per_layer = static_cast<uint64_t>(nqkv) * d + static_cast<uint64_t>(d) * qw +
                               2ull * F * d + static_cast<uint64_t>(d) * F;
    const uint64_t total = per_layer * g->layers.size() * 2u + per_layer * g->layers.size() / 8u;
    p.lw.clear();
    if (total <= kPfExpandBudget) {
        p.lw.resize(g->layers.size());
        const hipStream_t s = g->ctx->stream;
        auto expand = [&](const uint8_t* w0, const uint8_t* w1, const uint8_t* w2, uint32_t r0, uint32_t r1, uint32_t N,
                          uint32_t K, bool glu, PfMatrix* m) -> int {
            void* hq;
            void* sq;
            const size_t np = (N + kGmRowPad - 1u) / kGmRowPad * kGmRowPad;
            if (int rc = take(np * K * 2u, &hq)) return rc;
            if (int rc = take(np * (K / 32u) * 4u, &sq)) return rc;
            m->h = hq;
            m->s = static_cast<const float*>(sq);
            return gm_expand(w0, w1, w2, r0, r1, N, K / 32u, glu, static_cast<_Float16*>(hq), static_cast<float*>(sq), s);
        };
        for (size_t l = 0; l < g->layers.size(); ++l) {
            const LayerParams& Ly = g->layers[l];
            PfLayerW& w = p.lw[l];
            if (int rc = expand(Ly.wq, Ly.wk, Ly.wv, qw, hd, nqkv, d, false, &w.qkv)) return rc;
            if (int rc = expand(Ly.wo, Ly.wo, Ly.wo, d, 0u, d, qw, false, &w.o)) return rc;
            if (int rc = expand(Ly.wg, Ly.wu, Ly.wu, F, F, 2u * F, d, true, &w.gu)) return rc;
            if (int rc = expand(Ly.wd, Ly.wd, Ly.wd, d, 0u, d, F, false, &w.down)) return rc;
        }
    }
    p.max_t = max_t;
    return VRT_OK;
}

template <uint32_t HD>
static int pf_attn_launch(const PfAttn& A, bool lo, hipStream_t s) {
    PfAttn arg = A;
    void* args[] = {&arg};
    const void* fn = A.per == 1u ? (lo ? reinterpret_cast<const void*>(&k_pf_attn_few<HD, true>)
                                       : reinterpret_cast<const void*>(&k_pf_attn_few<HD, false>))
                     : lo        ? reinterpret_cast<const void*>(&k_pf_attn<HD, true>)
                                 : reinterpret_cast<const void*>(&k_pf_attn<HD, false>);
    VRT_HIP_CHECK(hipLaunchKernel(fn, dim3(A.groups * A.nch), dim3(256), args, 0, s));
    if (A.nch > 1u)   // some group has several chunks
        VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_pf_attn_merge<HD>), dim3(A.pairs, (HD / 32u + 3u) / 4u),
                                      dim3(256), args, 0, s));
    return VRT_OK;
}

// Keys per chunk of a launch, by a model of its time in key-tile steps of one workgroup (~2 us): a
// workgroup costs its steps and about one more to start and end, 256 CUs hold one each, and a
// chunked launch adds the merge (about two steps, and ~0.03 per workgroup for the partials' traffic).
static void pf_att_chunks(PfAttn& A, uint32_t max_parts) {
    uint32_t longest = 1;   // key tiles of the longest range
    uint64_t total = 0;
    std::vector<uint32_t> len(A.groups);
    for (uint32_t g = 0; g < A.groups; ++g) {
        uint32_t ks, ke;
        pf_att_group(A, g, ks, ke);
        len[g] = (ke - ks + 31u) / 32u;
        longest = std::max(longest, len[g]);
        total += len[g];
    }
    double best = 0.0;
    uint32_t best_kc = 0;
    for (uint32_t n = 1; n <= longest; ++n) {   // n chunks of the longest range
        const uint32_t tiles = (longest + n - 1u) / n;
        if (n > 1u && (tiles < 2u || n > kPfAttMaxChunks || (longest + tiles - 1u) / tiles != n)) continue;
        if (n > 1u && static_cast<uint64_t>(A.groups) * kPfAttPairs * n > max_parts) break;
        uint64_t units = 0;
        for (uint32_t g = 0; g < A.groups; ++g) units += (len[g] + tiles - 1u) / tiles;
        const double avg = static_cast<double>(total + units) / 256.0;
        double t = units <= 256u ? tiles + 1.0 : std::max(tiles + 1.0, avg + 0.5 * tiles);
        if (n > 1u) t += 2.0 + 0.03 * static_cast<double>(units) / 4.0;
        if (best_kc == 0u || t < best) {
            best = t;
            best_kc = 32u * tiles;
        }
    }
    A.kc = best_kc;
    A.nch = (32u * longest + A.kc - 1u) / A.kc;
}

// Causal local/global attention of one block (k_pf_attn) over the queries of p.qhi/p.qlo [T][H hd],
// for the query rows from o_row on; row q goes to row q - o_row of the activation buffer p.a.
static int pf_attention(vrt_g3* g, const LayerParams& Ly, uint32_t T, uint32_t o_row, hipStream_t s, uint32_t qo) {
    const PfState& p = g->pf;
    const uint32_t H = g->cfg.head_count, hd = g->cfg.head_dim;
    PfAttn A{};
    A.qhi = p.qhi;
    A.qlo = p.qlo;
    A.o = p.a;
    A.o_row = o_row;
    A.khi = static_cast<const _Float16*>(p.khi);
    A.klo = static_cast<const _Float16*>(p.klo);
    A.vhi = static_cast<const _Float16*>(p.vhi);
    A.vlo = static_cast<const _Float16*>(p.vlo);
    A.opart = p.opart;
    A.mpart = p.mpart;
    A.lpart = p.lpart;
    A.st = g->P.st;
    A.T = T;
    A.H = H;
    A.window = Ly.slots >= g->cfg.context_length ? 0u : Ly.slots;
    A.block = Ly.index;
    A.scale2 = g->P.attn_scale * 1.4426950408889634f;
    A.qo = qo;
    A.pair0 = o_row / 32u * H;
    A.pairs = (T + 31u) / 32u * H - A.pair0;
    // up to kPfAttFew pairs: one per workgroup, in chunks of four key tiles
    A.per = A.pairs <= kPfAttFew ? 1u : kPfAttPairs;
    A.groups = (A.pairs + A.per - 1u) / A.per;
    if (A.per == 1u) {
        uint32_t longest = 1;
        for (uint32_t i = 0; i < A.groups; ++i) {
            uint32_t ks, ke;
            pf_att_group(A, i, ks, ke);
            longest = std::max(longest, ke - ks);
        }
        const uint32_t most = std::min(32u, p.parts / A.pairs);   // chunks: the merge reads them four at a time
        A.kc = std::max(128u, (longest + 32u * most - 1u) / (32u * most) * 32u);
        A.nch = (longest + A.kc - 1u) / A.kc;
    } else {
        pf_att_chunks(A, p.parts);
    }
    if (A.pairs * static_cast<uint64_t>(A.nch) > p.parts || pf_pad(qo + T) > p.tkv)
        return set_error(VRT_ERR_STATE, "prefill attention workspace too small");
    const bool lo = g->P.kv16 == 0u;   // 16-bit entries have no low parts
    switch (hd) {
    case 32: return pf_attn_launch<32>(A, lo, s);
    case 64: return pf_attn_launch<64>(A, lo, s);
    case 96: return pf_attn_launch<96>(A, lo, s);
    case 128: return pf_attn_launch<128>(A, lo, s);
    case 160: return pf_attn_launch<160>(A, lo, s);
    case 192: return pf_attn_launch<192>(A, lo, s);
    case 224: return pf_attn_launch<224>(A, lo, s);
    case 256: return pf_attn_launch<256>(A, lo, s);
    default: return set_error(VRT_ERR_INVALID, "prefill head_dim not supported");
    }
}

// Prompt positions p0..p0+T-1 on the context's stream (positions before p0 are already in the
// KV cache). With `final`, the last one runs the LM head + argmax (results[p0+T-1], logits when
// want_logits); otherwise the segment ends after the last block's keys and values. The caller
// has reset the step state before the first segment.
int pf_run(vrt_g3* g, uint32_t T, uint32_t p0, bool final) {
    const PfState& p = g->pf;
    hipStream_t s = g->ctx->stream;
    uint32_t d = g->cfg.embedding_length, H = g->cfg.head_count, hd = g->cfg.head_dim;
    const uint32_t nqkv = (H + 2u) * hd, L = g->cfg.block_count;
    const G3Params& P = g->P;
    _Float16* a = p.a;
    float* h = p.h;          // residual stream; from the last block's attention on, its last row
    float* spare = p.h2;
    float* x = p.x;
    float* qkv = p.qkv;
    float eps = P.eps;
    G3State* st = P.st;
    if (T == 0u || T > p.max_t || static_cast<uint64_t>(p0) + T > g->cfg.context_length)
        return set_error(VRT_ERR_STATE, "prefill segment outside the workspace or the context");
    auto launch = [&](const void* fn, dim3 grid, void** args) -> int {
        VRT_HIP_CHECK(hipLaunchKernel(fn, grid, dim3(kPfThreads), args, 0, s));
        return VRT_OK;
    };
    {
        const uint8_t* te = P.tok_embd;
        const uint32_t* tok = P.tokens + p0;
        float es = P.emb_scale;
        void* args[] = {&te, &tok, &d, &es, &h};
        if (int rc = launch(reinterpret_cast<const void*>(&k_pf_embed), dim3(T), args)) return rc;
    }
    uint64_t xs = static_cast<uint64_t>(T) * d;  // one O / down partial [T][d]
    uint32_t s_down = 1;                         // splits of the previous block's down projection
    for (uint32_t l = 0; l < L; ++l) {
        const LayerParams& Ly = g->layers[l];
        // previous block's FFN output into the residual, the attention norm, q|k|v
        uint32_t s_qkv = 1;
        if (int rc = pf_norm_project(g, l, false, &h, &spare, l ? x : nullptr, s_down, xs, l ? g->layers[l - 1].post_ffw : nullptr,
                                     l ? l - 1u : 0u, a, T, qkv, &s_qkv, nullptr, st, s))
            return rc;
        // key coordinates: the history this segment's queries can see (from kb: position 0 in a
        // global block, the window's start rounded down to 32 in a local one), then its rows
        const uint32_t window = Ly.slots >= g->cfg.context_length ? 0u : Ly.slots;
        const uint32_t kb = window != 0u && p0 + 1u > window ? (p0 + 1u - window) & ~31u : 0u;
        uint32_t qo = p0 - kb;
        if (qo != 0u) {
            const float* kc = Ly.kc;
            const float* vc = Ly.vc;
            uint32_t slots = Ly.slots, kvf = P.kv16, kb_ = kb;
            _Float16* khi = static_cast<_Float16*>(p.khi);
            _Float16* klo = static_cast<_Float16*>(p.klo);
            _Float16* vhi = static_cast<_Float16*>(p.vhi);
            _Float16* vlo = static_cast<_Float16*>(p.vlo);
            void* args[] = {&kc, &vc, &slots, &kvf, &kb_, &qo, &hd, &khi, &klo, &vhi, &vlo};
            if (int rc = launch(reinterpret_cast<const void*>(&k_pf_kv_hist), dim3(qo), args)) return rc;
        }
        {
            const float* qn = Ly.q_norm;
            const float* kn = Ly.k_norm;
            const float* ct = Ly.global ? P.cos_g : P.cos_l;
            const float* sn = Ly.global ? P.sin_g : P.sin_l;
            float* kc = Ly.kc;
            float* vc = Ly.vc;
            uint32_t slots = Ly.slots;
            // rows past the segment zero the keys and values up to the next 64 key coordinates
            const uint32_t tp = pf_pad(qo + T) - qo;
            _Float16* khi = static_cast<_Float16*>(p.khi);
            _Float16* klo = static_cast<_Float16*>(p.klo);
            _Float16* vhi = static_cast<_Float16*>(p.vhi);
            _Float16* vlo = static_cast<_Float16*>(p.vlo);
            uint32_t kvf = P.kv16, p0_ = p0, qo_ = qo;
            uint64_t qs = static_cast<uint64_t>(T) * nqkv;
            _Float16 *qhi = p.qhi, *qlo = p.qlo;
            void* args[] = {&qkv, &s_qkv, &qs, &T, &H, &hd, &qn, &kn, &ct, &sn, &eps, &kc, &vc, &slots, &qhi, &qlo, &khi, &klo, &vhi, &vlo,
                            &kvf, &p0_, &qo_};
            VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_pf_qk), dim3(tp / kPfQkRows), dim3(64u * kPfQkRows),
                                          args, 0, s));
        }
        // The last block's output feeds only the LM head, so past its q/k/v (every position's
        // keys and values go to the cache) it runs for the last position alone: attention for
        // that position's query tile, then one row.
        const bool last = l + 1u == L;
        if (last && !final) break;   // an earlier segment: the last block's keys and values are all it leaves
        const uint32_t fr = last ? 1u : T;
        if (last) h += static_cast<uint64_t>(T - 1u) * d;
        if (int rc = pf_attention(g, Ly, T, last ? T - 1u : 0u, s, qo)) return rc;
        uint32_t so = 1;
        if (int rc = pf_project(g, l, kProjO, a, fr, x, &so, s)) return rc;
        // attention output into the residual (the O partials of fr rows), the FFN norm, gate/up
        if (int rc = pf_norm_project(g, l, true, &h, &spare, x, so, static_cast<uint64_t>(fr) * d, Ly.post_attn, Ly.index, a, fr,
                                     nullptr, nullptr, p.g, st, s))
            return rc;
        if (int rc = pf_project(g, l, kProjDown, p.g, fr, x, &s_down, s)) return rc;
    }
    if (!final) return VRT_OK;
    {   // last position: its FFN output (the split partials summed in order) and its residual
        // feed the decode step's final norm + LM head
        float* out = P.f;
        uint32_t nsplit = s_down;
        void* args[] = {&x, &nsplit, &d, &out};
        if (int rc = launch(reinterpret_cast<const void*>(&k_pf_sum), dim3(1), args)) return rc;
    }
    VRT_HIP_CHECK(hipMemcpyAsync(P.hmid, h, d * 4u, hipMemcpyDeviceToDevice, s));
    return g3_enqueue_lm(g, s);
}

}  // namespace vrt
