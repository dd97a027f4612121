// vrt_gemm.hip -- the row-batch projections on MFMA (vrt_gemm.hpp): C = A x W^T over M rows, with A
// fp32 activations as f16 hi + lo and W the expanded Q8_0 quants.
//
// Numerics. C[m][n] = sum_b s[n][b] * sum_{k in b} A[m][k] * q[n][k], s the block's f16 scale and q
// its int8 quants (exact in f16). A = hi + lo with hi = f16(A) and lo = f16(A - hi): the two f16
// products carry ~22 bits of A, every f16 x f16 product is exact in fp32 and the MFMA accumulates
// in fp32. A block's partial is scaled in fp32 and added to the fp32 accumulator.
//
// The weight is the MFMA's first operand: result r of lane l is C[m = l % 16][n = 4 (l / 16) + r],
// four consecutive columns of one row per lane (one 16-byte store, or four consecutive k of the
// next projection's operand).
#include "vrt_gemm.hpp"

#include <algorithm>

#include "vrt_internal.hpp"
#include "vrt_q8_device.hpp"

namespace vrt {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// gelu_tanh(gate) * up (shaders/gelu_mul.comp:23-31) with 0.5 x (1 + tanh u) = x / (1 + e^(-2u)): one
// hardware exponential and one reciprocal (1 ulp each) instead of tanhf, and no cancellation where
// tanh u is close to -1. Below the exponential's overflow the quotient is 0.
__device__ __forceinline__ float gm_gelu_mul(float x, float up) {
    const float t = x * (-2.302208198f - 0.1029432397f * (x * x));   // -2 u log2 e
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t)) * up;
}

// Four consecutive columns c..c+3 of row m into an activation buffer of nkb blocks.
__device__ __forceinline__ void gm_store_split(_Float16* o, uint32_t m, uint32_t c, uint32_t nkb, f4 x) {
    half4 h, l;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        _Float16 a, b;
        gm_split(x[k], a, b);
        h[k] = a;
        l[k] = b;
    }
    const uint64_t off = gm_off(m, c, nkb);
    *reinterpret_cast<half4*>(o + off) = h;
    *reinterpret_cast<half4*>(o + off + kGmLo) = l;
}

// Four consecutive columns n..n+3 of row m into C (row stride ldc); N need not be a multiple of 4.
__device__ __forceinline__ void gm_store_c(float* c, uint32_t ldc, uint32_t N, uint32_t m, uint32_t n, f4 x) {
    float* p = c + static_cast<uint64_t>(m) * ldc + n;
    if ((ldc & 3u) == 0u && n + 4u <= N) {
        *reinterpret_cast<f4*>(p) = x;
        return;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k)
        if (n + k < N) p[k] = x[k];
}

// Tiles of 32 MT rows x 32 NT columns, four waves of 16 MT x 16 NT each (2 x 2). K advances one
// Q8_0 block per step through NS LDS stages filled by direct global-to-LDS loads, NS - 1 steps
// ahead; one barrier per step both hands over the stage that has arrived and frees the one read
// before it.
template <int MT, int NT, int NS, bool GLU>
__global__ void __launch_bounds__(256, 2) k_gm_tile(GmArgs G) {
    static_assert(NT % 2 == 0 && NS >= 3, "whole load slots, stages");
    constexpr uint32_t kA = 4096u * MT, kW = 2048u * NT, kS = 128u * NT;   // stage bytes: A, W, scales
    constexpr uint32_t kStage = kA + kW + kS;
    constexpr uint32_t kLoads = MT + NT / 2u;    // 1 KB loads per wave and stage
    constexpr uint32_t kP = kLoads + 1u;         //   and one of scales
    __shared__ __align__(1024) unsigned char s_buf[NS * kStage];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of column panels with all their
    // row tiles, so the panel's weights are fetched into one L2
    const uint32_t nx = gridDim.x, nm = gridDim.y, total = nx * nm;
    uint32_t b = blockIdx.x + nx * blockIdx.y;
    if ((total & 7u) == 0u) b = (b & 7u) * (total >> 3) + (b >> 3);
    const uint32_t bm = b % nm, bn = b / nm;
    const uint32_t S = gridDim.z, z = blockIdx.z;
    const uint32_t kb_lo = G.nkb * z / S, kb_hi = G.nkb * (z + 1u) / S, nsteps = kb_hi - kb_lo;
    const uint32_t mt0 = bm * 2u * MT, nt0 = bn * 2u * NT;   // first 16-row tile, first 16-column tile
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) unsigned char*)s_buf));
    // this wave's loads of a step: units u = wave kLoads + j of the A units (row tile u / 2, part
    // u % 2), then the W units
    const char* src[kLoads];
    uint32_t inc[kLoads], dst[kLoads];
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
        const uint32_t u = wave * kLoads + j;
        if (u < 4u * MT) {
            src[j] = reinterpret_cast<const char*>(G.a) +
                     ((static_cast<uint64_t>(mt0 + (u >> 1)) * G.nkb + kb_lo) * 2u + (u & 1u)) * 1024u;
            inc[j] = 2048u;
            dst[j] = u * 1024u;
        } else {
            const uint32_t v = u - 4u * MT;
            src[j] = reinterpret_cast<const char*>(G.w) + (static_cast<uint64_t>(nt0 + v) * G.nkb + kb_lo) * 1024u;
            inc[j] = 1024u;
            dst[j] = kA + v * 1024u;
        }
    }
    const uint32_t sq = NT == 2 ? 0u : (wave & (NT / 2u - 1u));   // 256 bytes of scales (waves repeat them)
    const char* ssrc = reinterpret_cast<const char*>(G.ws + static_cast<uint64_t>(kb_lo) * G.npad + 16u * nt0 + 64u * sq);
    auto issue = [&](uint32_t stage) {
        const uint32_t base = lds0 + stage * kStage;
#pragma unroll
        for (uint32_t j = 0; j < kLoads; ++j) {
            gm_lds16(src[j], lane * 16u, base + dst[j]);
            src[j] += inc[j];
        }
        gm_lds4(ssrc, lane * 4u, base + kA + kW + 256u * sq);
        ssrc += static_cast<uint64_t>(G.npad) * 4u;
    };
    const uint32_t wm = wave >> 1, wn = wave & 1u;
    f4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t j = 0; j < NS - 1u; ++j)
        if (j < nsteps) issue(j);
    uint32_t stage = 0;
    for (uint32_t k = 0; k < nsteps; ++k) {
        // step k has arrived when only the loads of the later steps issued so far are in flight
        if (k + NS - 2u < nsteps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(kP * (NS - 2u)) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (k + NS - 1u < nsteps) issue(stage == 0u ? NS - 1u : stage - 1u);
        const unsigned char* pa = s_buf + stage * kStage + wm * MT * 2048u + lane * 16u;
        const unsigned char* pw = s_buf + stage * kStage + kA + wn * NT * 1024u + lane * 16u;
        const unsigned char* ps = s_buf + stage * kStage + kA + kW + wn * NT * 64u + (lane >> 4) * 16u;
        half8 ah[MT], al[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            ah[j] = *reinterpret_cast<const half8*>(pa + 2048 * j);
            al[j] = *reinterpret_cast<const half8*>(pa + 2048 * j + 1024);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const half8 w = *reinterpret_cast<const half8*>(pw + 1024 * i);
            const f4 sc = *reinterpret_cast<const f4*>(ps + 64 * i);
            f4 p[MT];
#pragma unroll
            for (int j = 0; j < MT; ++j) p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, ah[j], f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < MT; ++j) p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, al[j], p[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] += sc[r] * p[j][r];
        }
        stage = stage + 1u == NS ? 0u : stage + 1u;
    }
    const uint32_t ml = lane & 15u, nl = 4u * (lane >> 4);
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const uint32_t m = 16u * (mt0 + wm * MT + j) + ml;
        if (m >= G.M) continue;
        if constexpr (GLU) {
#pragma unroll
            for (int i = 0; i < NT; i += 2) {
                const uint32_t c = 8u * (nt0 + wn * NT + i) + nl;
                if (c >= G.N / 2u) continue;
                f4 y;
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = gm_gelu_mul(acc[i][j][r], acc[i + 1][j][r]);
                gm_store_split(G.o, m, c, G.N / 64u, y);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NT; ++i)
                gm_store_c(G.c + z * G.c_bs, G.ldc, G.N, m, 16u * (nt0 + wn * NT + i) + nl, acc[i][j]);
        }
    }
}

// Few rows: 16 MT rows x 16 NT columns per workgroup, the K blocks shared out over its NW waves
// (wave w takes blocks w, w + NW, ...), U blocks' operands loaded at once from memory to registers.
// Nothing is shared between the waves of the K loop, so there is no LDS stage and no barrier in
// it: at these sizes the time is one memory latency, not bandwidth. The waves' partial tiles are
// added in wave order through LDS.
template <int MT, int NT, int NW, int U, bool GLU>
__global__ void __launch_bounds__(64 * NW) k_gm_rows(GmArgs G) {
    constexpr uint32_t kTiles = MT * NT;
    __shared__ __align__(16) float s_red[NW][kTiles][256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nt0 = blockIdx.x * NT, mt0 = blockIdx.y * MT;
    f4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t k0 = wave; k0 < G.nkb; k0 += NW * U) {
        half8 a[U][MT][2], w[U][NT];
        f4 sc[U][NT];
        // every load is issued at a clamped, in-bounds block; a block past the end counts with scale 0
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t kb = min(k0 + NW * u, G.nkb - 1u);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                w[u][i] = *reinterpret_cast<const half8*>(G.w + (static_cast<uint64_t>(nt0 + i) * G.nkb + kb) * 512u + lane * 8u);
                sc[u][i] = *reinterpret_cast<const f4*>(G.ws + static_cast<uint64_t>(kb) * G.npad + 16u * (nt0 + i) + 4u * (lane >> 4));
            }
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const _Float16* pa = G.a + (static_cast<uint64_t>(mt0 + j) * G.nkb + kb) * 1024u + lane * 8u;
                a[u][j][0] = *reinterpret_cast<const half8*>(pa);
                a[u][j][1] = *reinterpret_cast<const half8*>(pa + kGmLo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // all loads ahead of their first use
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool live = k0 + NW * u < G.nkb;
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    f4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][i], a[u][j][0], f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][i], a[u][j][1], p, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] += (live ? sc[u][i][r] : 0.0f) * p[r];
                }
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) *reinterpret_cast<f4*>(&s_red[wave][i * MT + j][lane * 4u]) = acc[i][j];
    __syncthreads();
    constexpr uint32_t kOut = GLU ? kTiles / 2u : kTiles;   // output tiles: gate/up pairs, or all
    for (uint32_t q = tid; q < kOut * 64u; q += 64u * NW) {
        const uint32_t t = q >> 6, l = q & 63u;
        const uint32_t i = GLU ? 2u * (t / MT) : t / MT, j = t % MT;
        const uint32_t m = 16u * (mt0 + j) + (l & 15u);
        auto total = [&](uint32_t tile) {
            f4 x = *reinterpret_cast<const f4*>(&s_red[0][tile][l * 4u]);
#pragma unroll
            for (uint32_t v = 1; v < NW; ++v) {
                const f4 y = *reinterpret_cast<const f4*>(&s_red[v][tile][l * 4u]);
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] += y[r];
            }
            return x;
        };
        const f4 x = total(i * MT + j);
        if constexpr (GLU) {
            const f4 up = total((i + 1u) * MT + j);
            const uint32_t c = 8u * (nt0 + i) + 4u * (l >> 4);
            if (m >= G.M || c >= G.N / 2u) continue;
            f4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = gm_gelu_mul(x[r], up[r]);
            gm_store_split(G.o, m, c, G.N / 64u, y);
        } else {
            if (m < G.M) gm_store_c(G.c, G.ldc, G.N, m, 16u * (nt0 + i) + 4u * (l >> 4), x);
        }
    }
}

// One thread per (row, block) of the expanded matrix, 16 rows of a tile innermost.
__global__ void __launch_bounds__(256) k_gm_expand(const uint8_t* w0, const uint8_t* w1, const uint8_t* w2, uint32_t rows0,
                                                   uint32_t rows1, uint32_t N, uint32_t npad, uint32_t nkb, uint32_t glu,
                                                   _Float16* wh, float* ws) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;
    if (i >= static_cast<uint64_t>(npad) * nkb) return;
    const uint32_t r = static_cast<uint32_t>(i & 15u), kb = static_cast<uint32_t>((i >> 4) % nkb);
    const uint32_t n = static_cast<uint32_t>((i >> 4) / nkb) * 16u + r;
    _Float16* dst = wh + (i >> 4) * 512u + r * 8u;
    if (n >= N) {
        ws[static_cast<uint64_t>(kb) * npad + n] = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < 32u; ++k) dst[(k >> 3) * 128u + (k & 7u)] = static_cast<_Float16>(0.0f);
        return;
    }
    const uint8_t* src;
    if (glu) src = ((n & 31u) < 16u ? w0 : w1) + static_cast<uint64_t>(16u * (n >> 5) + (n & 15u)) * nkb * 34u;
    else if (n < rows0) src = w0 + static_cast<uint64_t>(n) * nkb * 34u;
    else if (n < rows0 + rows1) src = w1 + static_cast<uint64_t>(n - rows0) * nkb * 34u;
    else src = w2 + static_cast<uint64_t>(n - rows0 - rows1) * nkb * 34u;
    const uint8_t* blk = src + 34u * kb;
    ws[static_cast<uint64_t>(kb) * npad + n] =
        half_bits_to_float(static_cast<uint32_t>(blk[0]) | (static_cast<uint32_t>(blk[1]) << 8));
#pragma unroll
    for (uint32_t o = 0; o < 4u; ++o) {
        half8 v;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) v[k] = static_cast<_Float16>(static_cast<float>(static_cast<int8_t>(blk[2u + 8u * o + k])));
        *reinterpret_cast<half8*>(dst + o * 128u) = v;
    }
}

// ---- launches ----------------------------------------------------------------------------

// Both kernels' rules, from the q|k|v, O, gate/up and down shapes of the 270M model at 1..8192 rows.
// k_gm_rows re-reads an operand per 16 or 32 rows or columns but starts and ends fastest: it is
// the faster one up to M N K = 2^29 (O at 512 rows 6.9 against 9.7 us, down at 256 rows 6.9 against
// 7.1; q|k|v at 1024 rows, 2^30, 14 against 10.6).
static bool gm_use_rows(uint32_t M, uint32_t N, uint32_t nkb) {
    return static_cast<uint64_t>(M) * N * nkb * 32u <= (1ull << 29);
}

// Tile of k_gm_tile: the largest of 128 x 128, 64 x 128 and 64 x 64 that still gives every CU a
// workgroup; K splits for fewer workgroups than half the CUs.
struct GmTile {
    uint32_t mt, nt, splits;
};
static GmTile gm_tile_shape(uint32_t M, uint32_t N, uint32_t nkb, bool glu) {
    auto wgs = [&](uint32_t mt, uint32_t nt) { return ((M + 32u * mt - 1u) / (32u * mt)) * ((N + 32u * nt - 1u) / (32u * nt)); };
    GmTile t{2u, 2u, 1u};
    if (wgs(4u, 4u) >= 512u) t = {4u, 4u, 1u};
    else if (wgs(2u, 4u) >= 256u) t = {2u, 4u, 1u};
    if (!glu && t.nt == 2u && wgs(2u, 2u) <= kGmSplitWgs) t.splits = std::min(4u, std::max(1u, nkb / 8u));
    return t;
}

uint32_t gm_splits(uint32_t M, uint32_t N, uint32_t nkb) {
    return gm_use_rows(M, N, nkb) ? 1u : gm_tile_shape(M, N, nkb, false).splits;
}

template <int MT, int NT, int NS, bool GLU>
static int gm_launch_tile(const GmArgs& G, uint32_t splits, hipStream_t s) {
    GmArgs arg = G;
    void* args[] = {&arg};
    VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_gm_tile<MT, NT, NS, GLU>),
                                  dim3((G.N + 32u * NT - 1u) / (32u * NT), (G.M + 32u * MT - 1u) / (32u * MT), splits),
                                  dim3(256), args, 0, s));
    return VRT_OK;
}

template <int MT, int NT, int NW, int U, bool GLU>
static int gm_launch_rows(const GmArgs& G, hipStream_t s) {
    GmArgs arg = G;
    void* args[] = {&arg};
    VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_gm_rows<MT, NT, NW, U, GLU>),
                                  dim3((G.N + 16u * NT - 1u) / (16u * NT), (G.M + 16u * MT - 1u) / (16u * MT)),
                                  dim3(64 * NW), args, 0, s));
    return VRT_OK;
}

template <bool GLU>
static int gm_run_tile(const GmArgs& G, uint32_t splits, hipStream_t s) {
    const GmTile t = gm_tile_shape(G.M, G.N, G.nkb, GLU);
    if (t.mt == 4u) return gm_launch_tile<4, 4, 3, GLU>(G, splits, s);
    if (t.nt == 4u) return gm_launch_tile<2, 4, 3, GLU>(G, splits, s);
    return gm_launch_tile<2, 2, 4, GLU>(G, splits, s);
}

int gm_run(const GmArgs& G, uint32_t splits, bool glu, hipStream_t s) {
    if (splits > 1u || !gm_use_rows(G.M, G.N, G.nkb))
        return glu ? gm_run_tile<true>(G, 1u, s) : gm_run_tile<false>(G, splits, s);
    const uint32_t tiles = ((G.M + 15u) / 16u) * ((G.N + 15u) / 16u);   // 16 x 16
    // four waves for up to 24 K blocks (at most 6 per wave, five loaded at once), eight for more
    if (glu) return G.M <= 16u ? gm_launch_rows<1, 2, 4, 5, true>(G, s) : gm_launch_rows<2, 2, 4, 5, true>(G, s);
    if (G.nkb <= 24u) return tiles <= 384u ? gm_launch_rows<1, 1, 4, 5, false>(G, s) : gm_launch_rows<2, 2, 4, 5, false>(G, s);
    if (tiles <= 256u) return gm_launch_rows<1, 1, 8, 4, false>(G, s);
    return tiles <= 512u ? gm_launch_rows<2, 1, 8, 4, false>(G, s) : gm_launch_rows<2, 2, 8, 4, false>(G, s);
}

int gm_expand(const uint8_t* w0, const uint8_t* w1, const uint8_t* w2, uint32_t rows0, uint32_t rows1, uint32_t N,
              uint32_t nkb, bool glu, _Float16* wh, float* ws, hipStream_t s) {
    uint32_t npad = (N + kGmRowPad - 1u) / kGmRowPad * kGmRowPad, gl = glu ? 1u : 0u;
    void* args[] = {&w0, &w1, &w2, &rows0, &rows1, &N, &npad, &nkb, &gl, &wh, &ws};
    const uint64_t n = static_cast<uint64_t>(npad) * nkb;
    VRT_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void*>(&k_gm_expand),
                                  dim3(static_cast<uint32_t>((n + 255u) / 256u)), dim3(256), args, 0, s));
    return VRT_OK;
}

}  // namespace vrt
