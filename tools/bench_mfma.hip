// tools/bench_mfma.hip — issue-rate microbenchmark of the int8 and f16 MFMAs used by the prefill kernels (not part of the product).
// build: hipcc --offload-arch=gfx950 -O3 -Xclang -target-feature -Xclang -packed-fp32-ops tools/bench_mfma.hip -o tools/bin/bench_mfma
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <int NACC>
__global__ __launch_bounds__(256) void k_i8(int iters, int *sink) {
    i32x16 acc[NACC];
    for (int a = 0; a < NACC; a++) for (int r = 0; r < 16; r++) acc[a][r] = 0;
    i32x4 x = {(int)threadIdx.x, 1, 2, 3}, y = {4, 5, 6, (int)blockIdx.x};
    for (int i = 0; i < iters; i++) {
#pragma unroll
        for (int a = 0; a < NACC; a++) acc[a] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, y, acc[a], 0, 0, 0);
    }
    int s = 0;
    for (int a = 0; a < NACC; a++) for (int r = 0; r < 16; r++) s += acc[a][r];
    if (s == 0x12345678) *sink = s;
}
template <int NACC>
__global__ __launch_bounds__(256) void k_f16(int iters, float *sink) {
    f32x16 acc[NACC];
    for (int a = 0; a < NACC; a++) for (int r = 0; r < 16; r++) acc[a][r] = 0;
    f16x8 x, y;
    for (int i = 0; i < 8; i++) { x[i] = (_Float16)(threadIdx.x & 3); y[i] = (_Float16)(i & 1); }
    for (int i = 0; i < iters; i++) {
#pragma unroll
        for (int a = 0; a < NACC; a++) acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, acc[a], 0, 0, 0);
    }
    float s = 0;
    for (int a = 0; a < NACC; a++) for (int r = 0; r < 16; r++) s += acc[a][r];
    if (s == 1.2345f) *sink = s;
}
// pairs of int8 products of operands from memory (random or zero), and VALU f32 multiply-adds beside each pair: what the card's power leaves of the clock.
// clk: shader cycles and ticks of the 100 MHz clock of workgroup 0's loop
template <int VALU>
__global__ __launch_bounds__(256) void k_mix(int iters, const i32x4 *ops, unsigned long long *clk, float *sink) {
    i32x16 acc[4];
    for (int a = 0; a < 4; a++) for (int r = 0; r < 16; r++) acc[a][r] = 0;
    const i32x4 *o = ops + (blockIdx.x & 255) * 1024 + threadIdx.x;
    const i32x4 x0 = o[0], x1 = o[256], y0 = o[512], y1 = o[768];
    float f[16];
    for (int i = 0; i < 16; i++) f[i] = (float)x0.x * (1.0f + i);
    const float m = 0.9999f, c = (float)y0.x * 1e-9f;
    const unsigned long long r0 = __builtin_amdgcn_s_memrealtime(), t0 = __builtin_readcyclecounter();
    for (int i = 0; i < iters; i++) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            acc[2 * p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(p ? x1 : x0, y0, acc[2 * p], 0, 0, 0);
            acc[2 * p + 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(p ? x1 : x0, y1, acc[2 * p + 1], 0, 0, 0);
#pragma unroll
            for (int v = 0; v < VALU; v++) f[(p * 8 + v) & 15] = __builtin_fmaf(f[(p * 8 + v) & 15], m, c);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) { clk[0] = __builtin_readcyclecounter() - t0; clk[1] = __builtin_amdgcn_s_memrealtime() - r0; }
    int s = 0;
    float g = 0;
    for (int a = 0; a < 4; a++) for (int r = 0; r < 16; r++) s += acc[a][r];
    for (int i = 0; i < 16; i++) g += f[i];
    if (s == 0x12345678 || g == 1.2345f) *sink = g;
}
int main() {
    int *sink; hipMalloc(&sink, 16);
    hipDeviceProp_t p; hipGetDeviceProperties(&p, 0);
    const int cus = p.multiProcessorCount, iters = 20000;
    hipEvent_t e0, e1; hipEventCreate(&e0); hipEventCreate(&e1);
    auto run = [&](const char *name, auto launch, double ops_per_mfma, int nacc, int waves_per_simd) {
        launch(); hipDeviceSynchronize();
        hipEventRecord(e0); launch(); hipEventRecord(e1); hipEventSynchronize(e1);
        float ms; hipEventElapsedTime(&ms, e0, e1);
        const double n = (double)cus * 4 * waves_per_simd * iters * nacc;
        printf("%-28s acc=%d waves/SIMD=%d: %.1f TOP/s  (%.1f cycles per MFMA per SIMD at %.2f GHz)\n", name, nacc, waves_per_simd,
               n * ops_per_mfma / (ms * 1e-3) / 1e12, (ms * 1e-3) * p.clockRate * 1e3 / ((double)iters * nacc * waves_per_simd), p.clockRate / 1e6);
    };
    for (int w = 1; w <= 2; w++) {
        run("mfma_i32_32x32x32_i8", [&] { hipLaunchKernelGGL(k_i8<4>, dim3(cus * w), dim3(256), 0, nullptr, iters, sink); }, 2.0 * 32 * 32 * 32, 4, w);
        run("mfma_f32_32x32x16_f16", [&] { hipLaunchKernelGGL(k_f16<4>, dim3(cus * w), dim3(256), 0, nullptr, iters, (float *)sink); }, 2.0 * 32 * 32 * 16, 4, w);
    }
    run("mfma_i32_32x32x32_i8 (1 acc)", [&] { hipLaunchKernelGGL(k_i8<1>, dim3(cus), dim3(256), 0, nullptr, iters, sink); }, 2.0 * 32 * 32 * 32, 1, 1);
    i32x4 *ops; unsigned long long *clk, hc[2];
    const size_t ob = (size_t)256 * 1024 * 16;
    hipMalloc(&ops, ob); hipMalloc(&clk, 16);
    unsigned *h = (unsigned *)malloc(ob), seed = 1;
    for (int zero = 0; zero < 2; zero++) {
        for (size_t i = 0; i < ob / 4; i++) { seed = seed * 1664525u + 1013904223u; h[i] = zero ? 0u : seed ^ (seed >> 13); }
        hipMemcpy(ops, h, ob, hipMemcpyHostToDevice);
        auto mix = [&](int valu, auto launch) {
            float best = 1e9f;
            for (int r = 0; r < 3; r++) {
                hipEventRecord(e0); launch(); hipEventRecord(e1); hipEventSynchronize(e1);
                float ms; hipEventElapsedTime(&ms, e0, e1); best = ms < best ? ms : best;
            }
            hipMemcpy(hc, clk, 16, hipMemcpyDeviceToHost);
            printf("%s operands, %2d f32 multiply-adds a pair, 2 waves/SIMD: %.0f TOP/s, shader clock %.2f GHz\n", zero ? "zero  " : "random", valu, (double)cus * 8 * iters * 4 * 65536.0 / (best * 1e-3) / 1e12,
                   (double)hc[0] / hc[1] * 0.1);
        };
        mix(0, [&] { hipLaunchKernelGGL(k_mix<0>, dim3(cus * 2), dim3(256), 0, nullptr, iters, ops, clk, (float *)sink); });
        mix(5, [&] { hipLaunchKernelGGL(k_mix<5>, dim3(cus * 2), dim3(256), 0, nullptr, iters, ops, clk, (float *)sink); });
        mix(10, [&] { hipLaunchKernelGGL(k_mix<10>, dim3(cus * 2), dim3(256), 0, nullptr, iters, ops, clk, (float *)sink); });
    }
    return 0;
}
