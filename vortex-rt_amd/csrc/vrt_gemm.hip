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

// 1.0f / std::sqrt(float(sum_sq / n) + eps) (src/gemma3.cpp:967-983).
__device__ __forceinline__ float gm_rms_scale(double ss, uint32_t n, float eps) {
#pragma clang fp contract(off)
    return 1.0f / sqrtf(static_cast<float>(ss / static_cast<double>(n)) + eps);
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

// Output tile (row bm of nm, column bn of nx) of workgroup b, which runs on XCD b % 8. Each XCD takes a
// contiguous run of row tiles with all their columns, in passes of kGmPanels columns: the
// workgroups that run together read few rows and few columns, which stay in the XCD's 4 MB L2, and the
// rows stay for the next pass. (Column panels first, every XCD reads nearly all rows: 64% of the gate/up
// tile loads at 8192 rows missed L2.)
constexpr uint32_t kGmPanels = 8;
__device__ __forceinline__ void gm_tile_of(uint32_t b, uint32_t nx, uint32_t nm, uint32_t& bm, uint32_t& bn) {
    const uint32_t total = nx * nm, x = b & 7u, per = total >> 3, over = total & 7u;
    if ((nm & 7u) != 0u || nx <= kGmPanels) {   // a contiguous eighth of the tiles, columns innermost
        const uint32_t f = x * per + min(x, over) + (b >> 3);
        bm = f / nx;
        bn = f - bm * nx;
        return;
    }
    const uint32_t rows = nm >> 3, j = b >> 3, pass = j / (rows * kGmPanels), left = j - pass * rows * kGmPanels;
    const uint32_t w = min(kGmPanels, nx - pass * kGmPanels), r = left / w;
    bm = x * rows + r;
    bn = pass * kGmPanels + (left - r * w);
}

// Tiles of 32 MT rows x 32 NT columns, four waves of 16 MT x 16 NT each (2 x 2). K advances one
// Q8_0 block per step through NS LDS stages filled by direct global-to-LDS loads. A step's products
// run from registers while the next step's operands are read from LDS, so a stage is free one step
// after it arrives and NS - 1 later steps' loads are in flight; one barrier per step both hands over the
// stage that has arrived and frees the one read before it. Left to the scheduler, the operand reads
// gather at the top of the step with a full wait behind them (1650 cycles per 128 x 128 step, 512 of
// them products).
template <int MT, int NT, int NS, bool GLU>
__global__ void __launch_bounds__(256, 2) k_gm_tile(GmArgs G) {
    static_assert(NT % 2 == 0, "whole load slots");
    constexpr uint32_t kA = 4096u * MT, kW = 2048u * NT, kS = 128u * NT;   // stage bytes: A, W, scales
    constexpr uint32_t kStage = kA + kW + kS;
    constexpr uint32_t kLoads = MT + NT / 2u;    // 1 KB loads per wave and stage
    constexpr uint32_t kP = kLoads + 1u;         //   and one of scales
    __shared__ __align__(1024) unsigned char s_buf[NS * kStage];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t bm, bn;
    gm_tile_of(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x, gridDim.y, bm, bn);
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
    // One step's operands in registers: A as hi, lo, W and the scales of the wave's columns.
    struct Frag {
        half8 a[MT][2], w[NT];
        f4 sc[NT];
    };
    const uint32_t oa = wm * MT * 2048u + lane * 16u, ow = kA + wn * NT * 1024u + lane * 16u;
    const uint32_t os = kA + kW + wn * NT * 64u + (lane >> 4) * 16u;
    // the share of group i (of NT) of a stage's operand reads
    auto read = [&](Frag& F, const unsigned char* st, int i) {
        F.w[i] = *reinterpret_cast<const half8*>(st + ow + 1024 * i);
        F.sc[i] = *reinterpret_cast<const f4*>(st + os + 64 * i);
#pragma unroll
        for (int q = 2 * MT * i / NT; q < 2 * MT * (i + 1) / NT; ++q)
            F.a[q >> 1][q & 1] = *reinterpret_cast<const half8*>(st + oa + 1024 * q);
    };
    // Step k's products from F while step k + 1's operands are read into the other set, a group of
    // columns at a time (past the last step a stale stage is read and not used).
    uint32_t nbuf = 1u;   // stage of step k + 1
    auto step = [&](uint32_t k, const Frag& F, Frag& Fn) {
        // step k + 1 has arrived when only step k + 2's loads are in flight; every wave has read step k
        if (k + 2u < nsteps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(kP * (NS - 2u)) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (k + NS < nsteps) issue(nbuf == 0u ? NS - 1u : nbuf - 1u);
        const unsigned char* st = s_buf + nbuf * kStage;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            read(Fn, st, i);
            __builtin_amdgcn_sched_barrier(0);
            f4 p[MT];
#pragma unroll
            for (int j = 0; j < MT; ++j)
                p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(F.w[i], F.a[j][0], f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < MT; ++j) p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(F.w[i], F.a[j][1], p[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] += F.sc[i][r] * p[j][r];
        }
        nbuf = nbuf + 1u == NS ? 0u : nbuf + 1u;
    };
    static_assert(NS == 3, "the waits count two steps in flight");
#pragma unroll
    for (uint32_t j = 0; j < NS; ++j)
        if (j < nsteps) issue(j);
    if (nsteps >= NS) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(kP * (NS - 1u)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    Frag f0, f1;
#pragma unroll
    for (int i = 0; i < NT; ++i) read(f0, s_buf, i);
    for (uint32_t k = 0; k < nsteps; k += 2u) {
        step(k, f0, f1);
        if (k + 1u < nsteps) step(k + 1u, f1, f0);
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

// The NW waves' partial tiles s_red [NW][MT NT][256], added in wave order, into the output.
template <int MT, int NT, int NW, bool GLU>
__device__ __forceinline__ void gm_rows_out(const GmArgs& G, const float* s_red, uint32_t tid, uint32_t nt0, uint32_t mt0) {
    constexpr uint32_t kTiles = MT * NT;
    constexpr uint32_t kOut = GLU ? kTiles / 2u : kTiles;   // output tiles: gate/up pairs, or all
    for (uint32_t q = tid; q < kOut * 64u; q += 64u * NW) {
        const uint32_t t = q >> 6, l = q & 63u;
        const uint32_t i = GLU ? 2u * (t / MT) : t / MT, j = t % MT;
        const uint32_t m = 16u * (mt0 + j) + (l & 15u);
        auto total = [&](uint32_t tile) {
            f4 x = *reinterpret_cast<const f4*>(s_red + tile * 256u + l * 4u);
#pragma unroll
            for (uint32_t v = 1; v < NW; ++v) {
                const f4 y = *reinterpret_cast<const f4*>(s_red + (v * kTiles + tile) * 256u + l * 4u);
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

// Few rows: 16 MT rows x 16 NT columns per workgroup, the K blocks shared out over its NW waves
// (wave w takes blocks w, w + NW, ...), U blocks' operands loaded at once from memory to registers.
// Nothing is shared between the waves of the K loop, so there is no LDS stage and no barrier in
// it: at these sizes the time is one memory latency, not bandwidth. The waves' partial tiles are
// added in wave order through LDS.
template <int MT, int NT, int NW, int U, bool GLU>
__global__ void __launch_bounds__(64 * NW) k_gm_rows(GmArgs G) {
    __shared__ __align__(16) float s_red[NW][MT * NT][256];
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
    gm_rows_out<MT, NT, NW, GLU>(G, &s_red[0][0][0], tid, nt0, mt0);
}

// k_gm_rows for a projection that starts with a norm: every workgroup folds the previous sublayer's
// output into the residual of its 16 MT rows and norms them itself (the arithmetic of k_pf_norm_w: h = f *
// (scale(f) * w_post) + h, then (h * scale(h)) * w_next), straight into its LDS operand, instead of reading what
// a norm kernel left. The rows' 5 KB each come from L2 while the weights of the K blocks, loaded first, come from
// memory: a launch of 4 to 4.5 us per norm is saved for about 1 us here. The workgroups of column 0 write the
// new residual to h_out, another buffer than h (the others still read h), and flag a non-finite one.
template <int KR, int NT, int U, int NQ, bool GLU>
__global__ void __launch_bounds__(256) k_gm_norm_rows(GmArgs G, GmNorm R) {
#pragma clang fp contract(off)
    constexpr uint32_t NW = 4, kTiles = NT;
    extern __shared__ __align__(16) unsigned char s_x[];   // [nkb][hi, lo][1 KB], then the partial tiles
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nt0 = blockIdx.x * NT, K = 32u * G.nkb;
    half8 w[U][NT];
    f4 sc[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {   // clamped, in-bounds blocks; one past the end counts with scale 0
        const uint32_t kb = min(wave + NW * u, G.nkb - 1u);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            w[u][i] = *reinterpret_cast<const half8*>(G.w + (static_cast<uint64_t>(nt0 + i) * G.nkb + kb) * 512u + lane * 8u);
            sc[u][i] = *reinterpret_cast<const f4*>(G.ws + static_cast<uint64_t>(kb) * G.npad + 16u * (nt0 + i) + 4u * (lane >> 4));
        }
    }
    uint32_t ic[NQ];
    bool live[NQ];
    f4 wp[NQ], wn[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        live[k] = 4u * lane + 256u * k < K;
        ic[k] = min(4u * lane + 256u * k, K - 4u);
        wn[k] = *reinterpret_cast<const f4*>(R.w_next + ic[k]);
        wp[k] = R.f ? *reinterpret_cast<const f4*>(R.w_post + ic[k]) : wn[k];
    }
    constexpr uint32_t kRows = KR;   // this wave's rows: wave + 4 r (rows past M: copies of the last, not stored)
    {
        f4 hv[kRows][NQ], fv[kRows][NQ];
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            const uint64_t row = static_cast<uint64_t>(min(wave + NW * r, G.M - 1u)) * K;
#pragma unroll
            for (int k = 0; k < NQ; ++k) {
                hv[r][k] = *reinterpret_cast<const f4*>(R.h + row + ic[k]);
                fv[r][k] = R.f ? *reinterpret_cast<const f4*>(R.f + row + ic[k]) : f4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // all rows' loads in flight together
        if (R.f) {
            double ss[kRows];
#pragma unroll
            for (uint32_t r = 0; r < kRows; ++r) {
                ss[r] = 0.0;
#pragma unroll
                for (int k = 0; k < NQ; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss[r] += live[k] ? static_cast<double>(fv[r][k][e]) * static_cast<double>(fv[r][k][e]) : 0.0;
            }
#pragma unroll
            for (uint32_t r = 0; r < kRows; ++r) {
                const float s = gm_rms_scale(wave_red_sum_d(ss[r]), K, R.eps);
                const uint32_t m = wave + NW * r;
                int bad = 0;
#pragma unroll
                for (int k = 0; k < NQ; ++k) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        hv[r][k][e] = fv[r][k][e] * (s * wp[k][e]) + hv[r][k][e];
                        bad |= live[k] && !__builtin_isfinite(hv[r][k][e]);
                    }
                    if (blockIdx.x == 0u && live[k] && m < G.M)
                        *reinterpret_cast<f4*>(R.h_out + static_cast<uint64_t>(m) * K + ic[k]) = hv[r][k];
                }
                if (blockIdx.x == 0u && bad) atomicMin(R.nonfinite, R.code);
            }
        }
        double ss[kRows];
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            ss[r] = 0.0;
#pragma unroll
            for (int k = 0; k < NQ; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) ss[r] += live[k] ? static_cast<double>(hv[r][k][e]) * static_cast<double>(hv[r][k][e]) : 0.0;
        }
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            const float s = gm_rms_scale(wave_red_sum_d(ss[r]), K, R.eps);
#pragma unroll
            for (int k = 0; k < NQ; ++k) {
                f4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = (hv[r][k][e] * s) * wn[k][e];
                if (live[k]) gm_store_split(reinterpret_cast<_Float16*>(s_x), wave + NW * r, ic[k], G.nkb, y);
            }
        }
    }
    __syncthreads();
    f4 acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t kb = min(wave + NW * u, G.nkb - 1u);
        const bool on = wave + NW * u < G.nkb;
        const unsigned char* pa = s_x + kb * 2048u + lane * 16u;
        const half8 ah = *reinterpret_cast<const half8*>(pa), al = *reinterpret_cast<const half8*>(pa + 1024u);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][i], ah, f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][i], al, p, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][r] = __builtin_fmaf(on ? sc[u][i][r] : 0.0f, p[r], acc[i][r]);
        }
    }
    __syncthreads();   // every wave is done with the activations
    float* s_red = reinterpret_cast<float*>(s_x);   // [NW][kTiles][256]
#pragma unroll
    for (int i = 0; i < NT; ++i) *reinterpret_cast<f4*>(s_red + (wave * kTiles + i) * 256u + lane * 4u) = acc[i];
    __syncthreads();
    gm_rows_out<1, NT, NW, GLU>(G, s_red, tid, nt0, 0u);
}

// Logits of M rows against Q8_0 rows in their file layout (the tied embedding table), with each
// workgroup's greedy candidate per row. The table is streamed once per 16 GM rows (178 MB at the 270M shape),
// so its time is the floor, and what counts is bytes in flight. Tiles of 16 table rows, contiguous in the file,
// come in whole 1 KB direct-to-LDS loads, R - 1 tiles ahead (gm_wait counts up to 12 loads per wave: three tiles
// from 23 K blocks on, two from 31). At 20 K blocks one or four row tiles leave LDS for two workgroups per CU (74 and
// 76 KB each); two row tiles, with their deeper ring, for one (82 KB), and so do all from 23 K blocks on. The four
// waves share out the K blocks (wave w: w, w + 4, ...); a wave keeps its blocks' activations of all GM row tiles in
// registers, takes its blocks of the raw tile (lane l: quants k = 8 (l / 16) .. + 7 of row l % 16) and turns them
// into the MFMA's second operand in ten instructions (0x6400 | (q ^ 0x80) is the f16 1152 + q), once for all row
// tiles. The waves' partial tiles are added through LDS one pass later; one barrier per tile. Result r of lane l is
// logit [m = 4 (l / 16) + r][n = l % 16]; two tiles' logits leave together, 128 bytes per row and store. At 8 / 32 /
// 64 rows 48 / 92 / 88 us; before: the K loop of a 128-column GEMM and an argmax over its logits 109 + 5 at 8 rows,
// 130 + 25 at 64. Other forms, at 8 / 64 rows where this one then took 45 / 88: operands
// from memory straight to registers 68 / 152 (16 rows of addresses per load); one conversion per
// workgroup shared through LDS 85 (a second dependent LDS pass behind every barrier); row tiles dealt to the
// waves, each converting every block, 126 at 64. The table bypasses the caches as far as it can, so the blocks'
// weights stay in the last-level cache from step to step (O and down at 8 rows 5.2 -> 4.4 us).
__host__ __device__ __forceinline__ uint32_t gm_lm_units(uint32_t nkb) { return (nkb * 544u + 1023u) / 1024u; }
__host__ __device__ __forceinline__ uint32_t gm_lm_loads(uint32_t nkb) { return (gm_lm_units(nkb) + 3u) / 4u; }   // per wave
constexpr uint32_t gm_lm_ring(uint32_t gm) { return gm == 4u ? 4u : 6u; }
__host__ __device__ __forceinline__ uint32_t gm_lm_lds(uint32_t nkb, uint32_t gm) {
    return gm_lm_ring(gm) * gm_lm_units(nkb) * 1024u + 2u * gm * 4096u;
}

// Waits for the wave's memory operations but the last `left` (or fewer), then a barrier.
__device__ __forceinline__ void gm_wait(uint32_t left) {
#define VRT_GM_WAIT(N) asm volatile("s_waitcnt vmcnt(" #N ") lgkmcnt(0)\n\ts_barrier" ::: "memory")
    if (left >= 12u) VRT_GM_WAIT(12);
    else if (left >= 9u) VRT_GM_WAIT(9);
    else if (left >= 6u) VRT_GM_WAIT(6);
    else if (left >= 3u) VRT_GM_WAIT(3);
    else if (left >= 1u) VRT_GM_WAIT(1);
    else VRT_GM_WAIT(0);
#undef VRT_GM_WAIT
}

template <int GM, int N5>   // nkb <= 20 N5
__global__ void __launch_bounds__(256, 2) k_gm_lm(const uint8_t* table, uint32_t V, uint32_t nkb, const _Float16* x, uint32_t M,
                                                  uint32_t chunks, float* logits, GmBest* best) {
    constexpr uint32_t kQ = 5u * N5, R = gm_lm_ring(GM);   // K blocks per wave, stages
    static_assert(GM * kQ <= 20u, "activations in registers");
    extern __shared__ __align__(1024) unsigned char s_lm[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t units = gm_lm_units(nkb), loads = gm_lm_loads(nkb), raw = units * 1024u, row_bytes = nkb * 34u;
    float* s_red = reinterpret_cast<float*>(s_lm + R * raw);   // [2][row tile][wave][r][lane]
    // the row groups of a chunk are neighbours on one XCD (workgroup b runs on XCD b % 8) and read it together
    const uint32_t groups = gridDim.x / chunks, rest = blockIdx.x >> 3;
    const uint32_t grp = rest % groups, chunk = (rest / groups) * 8u + (blockIdx.x & 7u);
    const uint32_t tiles = (V + 15u) / 16u;
    const uint32_t t0 = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * chunk / chunks),
                   t1 = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * (chunk + 1u) / chunks);
    // this wave's activations, resident for the whole chunk
    half8 xa[GM][kQ][2];
#pragma unroll
    for (uint32_t o = 0; o < GM; ++o)
#pragma unroll
        for (uint32_t q = 0; q < kQ; ++q) {
            const uint32_t kb = min(wave + 4u * q, nkb - 1u);
            const _Float16* p = x + (static_cast<uint64_t>(grp * GM + o) * nkb + kb) * 1024u + lane * 8u;
            xa[o][q][0] = *reinterpret_cast<const half8*>(p);
            xa[o][q][1] = *reinterpret_cast<const half8*>(p + kGmLo);
        }
#pragma unroll
    for (uint32_t o = 0; o < GM; ++o)   // waited for here, not in the loop (its loads are counted by hand)
#pragma unroll
        for (uint32_t q = 0; q < kQ; ++q)
#pragma unroll
            for (uint32_t e = 0; e < 2u; ++e) asm volatile("" : "+v"(xa[o][q][e]));
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)s_lm));
    const uint64_t last16 = (static_cast<uint64_t>(V) * row_bytes - 1u) / 16u * 16u;   // the table's last 16-byte unit
    auto issue = [&](uint32_t t) {   // every wave issues `loads`; the last unit may be loaded twice
        const uint64_t at = static_cast<uint64_t>(t) * 16u * row_bytes;
        for (uint32_t j = 0; j < loads; ++j) {
            const uint32_t u = min(wave + 4u * j, units - 1u);
            const uint64_t o = min(at + u * 1024u + lane * 16u, last16);
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                         :: "v"(reinterpret_cast<uintptr_t>(table) + o), "s"(lds0 + (t % R) * raw + u * 1024u) : "memory", "m0");
        }
    };
    // this thread's outputs of a tile: result `wave` of its lane in every row tile
    float bv[GM], held[GM];
    uint32_t bi[GM];
#pragma unroll
    for (int o = 0; o < GM; ++o) {
        bv[o] = -INFINITY;
        bi[o] = 0xffffffffu;
        held[o] = 0.0f;
    }
    auto row_of = [&](int o, uint32_t group) { return 16u * (grp * GM + static_cast<uint32_t>(o)) + 4u * group + wave; };
    auto put = [&](float y, uint32_t m, uint32_t n) {
        if (n < V && m < M) logits[static_cast<uint64_t>(m) * V + n] = y;
    };
    // tile t: its logits are held until its neighbour's are there (the chunk's last may have none)
    auto emit = [&](uint32_t t) {
        const bool second = ((t - t0) & 1u) != 0u;   // wave-uniform
        uint32_t go = g;   // opaque: the rows' addresses are not kept across the passes
        asm volatile("" : "+v"(go));
#pragma unroll
        for (int o = 0; o < GM; ++o) {
            const float* red = s_red + ((t & 1u) * GM + o) * 1024u + wave * 64u + lane;
            float y = red[0];
#pragma unroll
            for (uint32_t k = 1; k < 4u; ++k) y += red[k * 256u];
            const uint32_t n = 16u * t + l16;
            if (n < V && am_better(y, n, bv[o], bi[o])) {   // columns in rising order: a tie keeps the lower
                bv[o] = y;
                bi[o] = n;
            }
            if (second) {   // 16-lane groups [0, 1, 2, 3] of both tiles: [a0, b0, a2, b2] and [a1, b1, a3, b3]
                const auto pr = __builtin_amdgcn_permlane16_swap(__float_as_uint(held[o]), __float_as_uint(y), false, false);
                const uint32_t c = 16u * (t - 1u + (go & 1u)) + l16;
                put(__uint_as_float(pr[0]), row_of(o, go & 2u), c);
                put(__uint_as_float(pr[1]), row_of(o, (go & 2u) + 1u), c);
            } else if (t + 1u == t1) {
                put(y, row_of(o, go), n);
            }
            held[o] = y;
        }
    };
    for (uint32_t t = t0; t < t0 + R - 1u && t < t1; ++t) issue(t);
    for (uint32_t t = t0; t <= t1; ++t) {   // pass t multiplies tile t and writes out tile t - 1
        // tile t has arrived once no more than the later tiles' loads are left (stores among them only wait longer)
        gm_wait(t < t1 ? min(t1 - 1u - t, R - 2u) * loads : 0u);
        if (t > t0) emit(t - 1u);
        if (t >= t1) break;
        if (t + R - 1u < t1) issue(t + R - 1u);   // into the stage that tile t - 1 left
        const unsigned char* src = s_lm + (t % R) * raw;
        uint32_t row = l16 * row_bytes;   // opaque: every block's offset kept across the passes would not fit the registers
        asm volatile("" : "+v"(row));
        f4 acc[GM];
#pragma unroll
        for (int o = 0; o < GM; ++o) acc[o] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        // five blocks at a time, in straight line: reads, conversions, products (a block past the end: the last
        // one again with scale 0)
#pragma unroll
        for (uint32_t q5 = 0; q5 < kQ / 5u; ++q5) {
            __builtin_amdgcn_sched_barrier(0);   // (two groups' operands at once do not fit either)
            uint32_t d[5][3];
            uint16_t sb[5];
#pragma unroll
            for (uint32_t e = 0; e < 5u; ++e) {
                const uint32_t b = row + 34u * min(wave + 4u * (5u * q5 + e), nkb - 1u);
                const uint32_t* p = reinterpret_cast<const uint32_t*>(src + ((b + 8u * g) & ~3u));
#pragma unroll
                for (int k = 0; k < 3; ++k) d[e][k] = p[k];
                sb[e] = *reinterpret_cast<const uint16_t*>(src + b);
            }
#pragma unroll
            for (uint32_t e = 0; e < 5u; ++e) {
                const uint32_t kb = min(wave + 4u * (5u * q5 + e), nkb - 1u);
                const bool odd = ((row + 34u * kb) & 2u) != 0u;   // the block starts two bytes past a dword
                const uint32_t q0 = (odd ? d[e][1] : __builtin_amdgcn_alignbyte(d[e][1], d[e][0], 2u)) ^ 0x80808080u;
                const uint32_t q1 = (odd ? d[e][2] : __builtin_amdgcn_alignbyte(d[e][2], d[e][1], 2u)) ^ 0x80808080u;
                typedef uint32_t u4 __attribute__((ext_vector_type(4)));
                const u4 h = {__builtin_amdgcn_perm(0x64646464u, q0, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, q0, 0x04030402u),
                              __builtin_amdgcn_perm(0x64646464u, q1, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, q1, 0x04030402u)};
                const _Float16 off = static_cast<_Float16>(1152.0f);
                const half8 w = __builtin_bit_cast(half8, h) - half8{off, off, off, off, off, off, off, off};
                const float sc = wave + 4u * (5u * q5 + e) < nkb ? half_bits_to_float(sb[e]) : 0.0f;
                f4 p[GM];
#pragma unroll
                for (int o = 0; o < GM; ++o)
                    p[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[o][5u * q5 + e][0], w, f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int o = 0; o < GM; ++o) p[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[o][5u * q5 + e][1], w, p[o], 0, 0, 0);
#pragma unroll
                for (int o = 0; o < GM; ++o)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[o][r] += sc * p[o][r];
                if constexpr (GM * kQ == 20u) __builtin_amdgcn_sched_barrier(0);   // one block's products at a time: registers
            }
        }
#pragma unroll
        for (int o = 0; o < GM; ++o)
#pragma unroll
            for (int r = 0; r < 4; ++r) s_red[((t & 1u) * GM + o) * 1024u + wave * 256u + r * 64u + lane] = acc[o][r];
    }
    // candidates of the 16 columns
#pragma unroll
    for (int o = 0; o < GM; ++o) {
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const float ov = __shfl_xor(bv[o], off);
            const uint32_t oi = static_cast<uint32_t>(__shfl_xor(static_cast<int>(bi[o]), off));
            if (am_better(ov, oi, bv[o], bi[o])) {
                bv[o] = ov;
                bi[o] = oi;
            }
        }
        const uint32_t m = row_of(o, g);
        if (l16 == 0u && m < M) best[static_cast<uint64_t>(m) * chunks + chunk] = {bv[o], bi[o]};
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

// Tile of k_gm_tile. 64 x 128 from two workgroups per CU on (below, 64 x 64: q|k|v at 2048 rows 15.7 against
// 16.7 us, gate/up at 512 rows 11.2 against 12.9, O at 4096 rows 20.9 against 22.8; above, O at 8192 rows 35.0
// against 31.3); 128 x 128 with the GELU epilogue, which it amortises (gate/up at 2048 rows 29.9 -> 27.6;
// q|k|v at 8192 rows 43.9 -> 47.1 on that card, not taken). Few 64 x 64 tiles split K in up to four (down at 512 rows
// 21.4 -> 9.6).
struct GmTile {
    uint32_t mt, nt, splits;
};
static GmTile gm_tile_shape(uint32_t M, uint32_t N, uint32_t nkb, bool glu) {
    auto wgs = [&](uint32_t mt, uint32_t nt) { return ((M + 32u * mt - 1u) / (32u * mt)) * ((N + 32u * nt - 1u) / (32u * nt)); };
    GmTile t{2u, 2u, 1u};
    if (glu && wgs(4u, 4u) >= 512u) t = {4u, 4u, 1u};
    else if (wgs(2u, 4u) >= 512u) t = {2u, 4u, 1u};
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
    if constexpr (GLU)
        if (t.mt == 4u) return gm_launch_tile<4, 4, 3, true>(G, splits, s);
    if (t.nt == 4u) return gm_launch_tile<2, 4, 3, GLU>(G, splits, s);
    return gm_launch_tile<2, 2, 3, GLU>(G, splits, s);
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

// One row tile and up to 24 K blocks (five or six per wave, their weights in registers before the norm; wider models
// keep the two launches). With more rows a wave norms several in turn and
// the launch that is saved costs more than it took (32 rows per workgroup: 13.8 us against 4.5 + 4.5).
bool gm_norm_fits(uint32_t M, uint32_t nkb) { return M <= 16u && nkb <= 24u; }

template <int NT, bool GLU>
static const void* gm_norm_fn(uint32_t M, uint32_t nkb) {
#define VRT_GM_NORM(KR, U, NQ) reinterpret_cast<const void*>(&k_gm_norm_rows<KR, NT, U, NQ, GLU>)
    if (nkb <= 16u) return M <= 8u ? VRT_GM_NORM(2, 4, 2) : VRT_GM_NORM(4, 4, 2);
    if (nkb <= 20u) return M <= 8u ? VRT_GM_NORM(2, 5, 3) : VRT_GM_NORM(4, 5, 3);
    return M <= 8u ? VRT_GM_NORM(2, 6, 3) : VRT_GM_NORM(4, 6, 3);
#undef VRT_GM_NORM
}

int gm_run_norm(const GmArgs& G, const GmNorm& R, bool glu, hipStream_t s) {
    if (!gm_norm_fits(G.M, G.nkb)) return set_error(VRT_ERR_INVALID, "normed projection: shape outside the kernel");
    const uint32_t nt = glu ? 2u : 1u;
    GmArgs a = G;
    GmNorm r = R;
    void* args[] = {&a, &r};
    const uint32_t lds = std::max(G.nkb * 2048u, 4u * nt * 1024u);
    VRT_HIP_CHECK(hipLaunchKernel(glu ? gm_norm_fn<2, true>(G.M, G.nkb) : gm_norm_fn<1, false>(G.M, G.nkb),
                                  dim3((G.N + 16u * nt - 1u) / (16u * nt)), dim3(256), args, lds, s));
    return VRT_OK;
}

// Row tiles per workgroup: as many as M has (1, 2, 4) while a wave's activations fit its registers.
static uint32_t gm_lm_tiles(uint32_t M, uint32_t nkb) {
    const uint32_t gm = M > 32u ? 4u : M > 16u ? 2u : 1u;
    return nkb > 20u ? std::min(gm, 2u) : gm;
}
static const void* gm_lm_fn(uint32_t gm, bool wide) {
    if (wide) return gm == 2u ? reinterpret_cast<const void*>(&k_gm_lm<2, 2>) : reinterpret_cast<const void*>(&k_gm_lm<1, 2>);
    return gm == 4u   ? reinterpret_cast<const void*>(&k_gm_lm<4, 1>)
           : gm == 2u ? reinterpret_cast<const void*>(&k_gm_lm<2, 1>)
                      : reinterpret_cast<const void*>(&k_gm_lm<1, 1>);
}

int gm_setup() {
    for (const void* fn : {gm_lm_fn(1u, false), gm_lm_fn(2u, false), gm_lm_fn(4u, false), gm_lm_fn(1u, true), gm_lm_fn(2u, true)})
        VRT_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kGmLdsMax)));
    return VRT_OK;
}

bool gm_lm_fits(const uint8_t* table, uint64_t readable, uint32_t V, uint32_t nkb) {
    const uint64_t bytes = static_cast<uint64_t>(V) * nkb * 34u;
    return (reinterpret_cast<uintptr_t>(table) & 15u) == 0u && readable >= (bytes + 15u) / 16u * 16u && gm_lm_lds(nkb, 2u) <= kGmLdsMax &&
           nkb <= 40u;
}

// 512 workgroups in all, two for each CU: 512 chunks of one row group, 256 of two. Where LDS holds one per CU (k_gm_lm)
// they run as two rounds.
uint32_t gm_lm_chunks(uint32_t M, uint32_t nkb) { return M <= 16u * gm_lm_tiles(M, nkb) ? kGmLmMaxChunks : kGmLmMaxChunks / 2u; }

int gm_lm(const uint8_t* table, uint32_t V, uint32_t nkb, const _Float16* x, uint32_t M, float* logits, GmBest* best,
          hipStream_t s) {
    const uint32_t gm = gm_lm_tiles(M, nkb), groups = (M + 16u * gm - 1u) / (16u * gm);
    uint32_t chunks = gm_lm_chunks(M, nkb);
    void* args[] = {&table, &V, &nkb, &x, &M, &chunks, &logits, &best};
    VRT_HIP_CHECK(hipLaunchKernel(gm_lm_fn(gm, nkb > 20u), dim3(chunks * groups), dim3(256), args, gm_lm_lds(nkb, gm), s));
    return VRT_OK;
}

}  // namespace vrt
