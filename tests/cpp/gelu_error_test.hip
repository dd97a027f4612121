// The row-batch GEMMs' gelu_tanh(gate) * up (gm_gelu_mul) against 64 bits: over gates of several spreads
// its error (2-norm) is no larger than that of the reference's expression with every operation in fp32, the
// form the standalone kernels keep (shaders/gelu_mul.comp:23-31). Far gates give 0 or the gate itself.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "vrt_gemm.hpp"

#define CHECK(e)                                                                  \
    do {                                                                          \
        const hipError_t r_ = (e);                                                \
        if (r_ != hipSuccess) {                                                   \
            std::printf("%s: %s\n", #e, hipGetErrorString(r_));                   \
            return 1;                                                             \
        }                                                                         \
    } while (0)

__global__ void k_both(const float* x, const float* up, float* y, float* ref, int n) {
#pragma clang fp contract(off)
    const int i = static_cast<int>(blockIdx.x * 256u + threadIdx.x);
    if (i >= n) return;
    const float cubic = x[i] * x[i] * x[i];
    ref[i] = 0.5f * x[i] * (1.0f + tanhf(0.7978845608028654f * (x[i] + 0.044715f * cubic))) * up[i];
    y[i] = vrt::gm_gelu_mul(x[i], up[i]);
}

int main() {
    const int n = 1 << 18;
    std::vector<float> x(n), up(n), y(n), ref(n);
    float* d[4];
    for (float*& p : d) CHECK(hipMalloc(reinterpret_cast<void**>(&p), n * 4));
    auto both = [&]() {
        CHECK(hipMemcpy(d[0], x.data(), n * 4, hipMemcpyHostToDevice));
        CHECK(hipMemcpy(d[1], up.data(), n * 4, hipMemcpyHostToDevice));
        k_both<<<n / 256, 256>>>(d[0], d[1], d[2], d[3], n);
        CHECK(hipGetLastError());
        CHECK(hipMemcpy(y.data(), d[2], n * 4, hipMemcpyDeviceToHost));
        CHECK(hipMemcpy(ref.data(), d[3], n * 4, hipMemcpyDeviceToHost));
        return 0;
    };
    int bad = 0;
    std::mt19937_64 gen(7);
    std::normal_distribution<double> N(0.0, 1.0);
    for (const double spread : {0.05, 0.5, 1.0, 3.0, 20.0}) {
        for (int i = 0; i < n; ++i) {
            x[i] = static_cast<float>(spread * N(gen));
            up[i] = static_cast<float>(N(gen));
        }
        if (both()) return 1;
        double se = 0.0, sr = 0.0, ss = 0.0;
        for (int i = 0; i < n; ++i) {
            const double g = x[i], u = 0.7978845608028654 * (g + 0.044715 * g * g * g);
            const double want = g / (1.0 + std::exp(-2.0 * u)) * up[i];
            se += (y[i] - want) * (y[i] - want);
            sr += (ref[i] - want) * (ref[i] - want);
            ss += want * want;
        }
        std::printf("gates N(0, %g^2): error %.3e, in the reference's order %.3e\n", spread, std::sqrt(se / ss), std::sqrt(sr / ss));
        bad += !(se <= sr);
    }
    const float far[] = {-10.2f, -10.4f, -1e5f, -1e20f, -3e38f, 12.0f, 1e5f, 1e20f, 3e38f, 0.0f};
    for (int i = 0; i < n; ++i) {
        x[i] = far[i % 10];
        up[i] = 1.0f;
    }
    if (both()) return 1;
    for (int i = 0; i < 10; ++i)
        if (!(std::fabs(y[i] - (far[i] > 0.0f ? far[i] : 0.0f)) <= 1e-30f)) {
            std::printf("far gate %g: %g\n", far[i], y[i]);
            ++bad;
        }
    for (float* p : d) CHECK(hipFree(p));
    if (bad) return 1;
    std::printf("gelu_error_test ok\n");
    return 0;
}
