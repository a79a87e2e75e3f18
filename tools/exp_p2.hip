// tools/exp_p2.hip — the prompt contraction on a tensor's plane set: per-lane planes kernel (256 x 32 and 128 x 128 tiles) against the kernel with the activations through LDS
// (128 x 256): bit-for-bit comparison on random GGUF rows, laid out as at load, and time per launch (HIP events; the launches read copies of the tensor in turn, more than the last
// level of cache holds).
// build: tools/build_exp_p2.sh; usage: exp_p2 [rows] [columns] [tokens] [type] [launches] [1: all operands zero]
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include <cmath>
#include <algorithm>
#include "kernels.h"
namespace mi355 {
void set_error(const char *, ...) {}
static int g_ncu = 256;
void set_num_cu(int n) { g_ncu = n; }
int num_cu() { return g_ncu; }
void mmq_set_tiles(int mt);
void mmq_set_split(int n);
}
using namespace mi355;
#define CK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { printf("%s failed: %s (line %d)\n", #x, hipGetErrorString(e_), __LINE__); exit(1); } } while (0)

static unsigned rs = 12345u;
static unsigned rnd() { rs = rs * 1664525u + 1013904223u; return rs >> 8; }
static uint16_t f2h_host(float f) { _Float16 h = (_Float16)f; uint16_t u; memcpy(&u, &h, 2); return u; }

__global__ void tick_kernel(unsigned long long *o) {          // s_memtime ticks per 100 us of the 100 MHz wall clock
    const unsigned long long r0 = __builtin_amdgcn_s_memrealtime(), t0 = __builtin_readcyclecounter();
    while (__builtin_amdgcn_s_memrealtime() - r0 < 10000) {}
    o[0] = __builtin_readcyclecounter() - t0;
}

int main(int argc, char **argv) {
    const int N = argc > 1 ? atoi(argv[1]) : 4096, K = argc > 2 ? atoi(argv[2]) : 4096, T = argc > 3 ? atoi(argv[3]) : 2048;
    const int type = argc > 4 ? atoi(argv[4]) : T_Q4_K, reps = argc > 5 ? atoi(argv[5]) : 20;
    const bool zeros = argc > 6 && atoi(argv[6]);
    const int nb = K / 256;
    const size_t rb = dev_row_bytes(type, K), pb = (mmq_planes_bytes(type, N, K) + 255) & ~(size_t)255;
    if (!pb) { printf("no planes of type %d\n", type); return 1; }
    std::vector<uint8_t> hw(rb * N);                            // device rows: any byte is a code, a scale or a min; the block scales are chosen
    for (auto &b : hw) b = zeros ? 0 : (uint8_t)rnd();
    for (int r = 0; r < N && !zeros; r++)
        for (int b = 0; b < nb; b++) {
            const uint16_t d = f2h_host(0.001f + (rnd() & 255) * 1e-5f), dmin = f2h_host(0.0005f + (rnd() & 255) * 1e-5f);
            uint8_t *row = hw.data() + rb * r;
            if (type == T_Q4_K || type == T_Q5_K) { uint8_t *blk = row + (size_t)b * (type == T_Q4_K ? 144 : 176); memcpy(blk, &d, 2); memcpy(blk + 2, &dmin, 2); }
            else if (type == T_Q6_K) memcpy(row + (size_t)nb * 208 + 2 * b, &d, 2);
            else { printf("Q4_K, Q5_K or Q6_K (%d, %d, %d)\n", T_Q4_K, T_Q5_K, T_Q6_K); return 1; }
        }
    const int copies = (int)std::max<size_t>(2, std::min<size_t>(64, ((size_t)600 << 20) / pb));
    uint8_t *w, *planes;
    CK(hipMalloc(&w, hw.size())); CK(hipMemcpy(w, hw.data(), hw.size(), hipMemcpyHostToDevice)); CK(hipMalloc(&planes, pb * copies));
    for (int i = 0; i < copies; i++) CK(launch_mmq_expand(type, w, rb, N, K, planes + pb * i, nullptr));
    std::vector<int8_t> haq((size_t)T * K); std::vector<float> had((size_t)T * nb); std::vector<int16_t> hbs((size_t)T * K / 16);
    for (auto &v : haq) v = zeros ? 0 : (int8_t)((int)(rnd() % 255) - 127);
    for (auto &v : had) v = 0.01f + (rnd() & 1023) * 1e-4f;
    for (size_t i = 0; i < hbs.size(); i++) { int sum = 0; for (int k = 0; k < 16; k++) sum += haq[i * 16 + k]; hbs[i] = (int16_t)sum; }
    ActQuant q{};
    CK(hipMalloc(&q.qs, haq.size())); CK(hipMemcpy(q.qs, haq.data(), haq.size(), hipMemcpyHostToDevice));
    CK(hipMalloc(&q.d, had.size() * 4)); CK(hipMemcpy(q.d, had.data(), had.size() * 4, hipMemcpyHostToDevice));
    CK(hipMalloc(&q.bsums, hbs.size() * 2)); CK(hipMemcpy(q.bsums, hbs.data(), hbs.size() * 2, hipMemcpyHostToDevice));
    int8_t *bh, *bl; CK(hipMalloc(&bh, mmq_prep_bytes(K, T))); CK(hipMalloc(&bl, mmq_prep_bytes(K, T)));
    CK(launch_mmq_prep(q, K, T, bh, bl, nullptr));
    float *o_old, *o_new; CK(hipMalloc(&o_old, (size_t)T * N * 4)); CK(hipMalloc(&o_new, (size_t)T * N * 4));
    CK(hipMemset(o_old, 0, (size_t)T * N * 4)); CK(hipMemset(o_new, 0xff, (size_t)T * N * 4));
    hipEvent_t e0, e1; CK(hipEventCreate(&e0)); CK(hipEventCreate(&e1));
    MMQWorkspace wsp; wsp.bytes = (size_t)4 * T * N * 4; CK(hipMalloc(&wsp.p, wsp.bytes));
    auto run = [&](int tiles, float *out, int split = 0) {
        mmq_set_tiles(tiles); mmq_set_split(split);
        for (int i = 0; i < copies; i++) CK(launch_mmq_planes(type, planes + pb * i, N, K, T, q, bh, bl, out, N, nullptr, nullptr, wsp));
        CK(hipDeviceSynchronize());
        CK(hipEventRecord(e0));
        for (int i = 0; i < reps; i++) CK(launch_mmq_planes(type, planes + pb * (i % copies), N, K, T, q, bh, bl, out, N, nullptr, nullptr, wsp));
        CK(hipEventRecord(e1)); CK(hipEventSynchronize(e1));
        float ms; CK(hipEventElapsedTime(&ms, e0, e1));
        return ms * 1e3f / reps;
    };
    const float us1 = run(1, o_old, 1), us2 = run(2, o_old, 1);
    const float us4 = run(4, o_new, 1);
    float *o_sk; CK(hipMalloc(&o_sk, (size_t)T * N * 4));
    float us_sk[5] = {0, 0, 0, 0, 0};
    for (int sp = 2; sp <= 4; sp++) us_sk[sp] = run(4, o_sk, sp);
    {
        std::vector<float> a((size_t)T * N), b((size_t)T * N);
        CK(hipMemcpy(a.data(), o_new, a.size() * 4, hipMemcpyDeviceToHost)); CK(hipMemcpy(b.data(), o_sk, b.size() * 4, hipMemcpyDeviceToHost));
        double md = 0, mx = 0; for (size_t i = 0; i < a.size(); i++) { md = std::max(md, (double)fabsf(a[i] - b[i])); mx = std::max(mx, (double)fabsf(a[i])); }
        printf("  split K (+ reduce): x2 %.1f us  x3 %.1f us  x4 %.1f us   max |diff| vs unsplit %.3g of max |y| %.3g\n", us_sk[2], us_sk[3], us_sk[4], md, mx);
    }
    std::vector<float> a((size_t)T * N), b((size_t)T * N);
    CK(hipMemcpy(a.data(), o_old, a.size() * 4, hipMemcpyDeviceToHost)); CK(hipMemcpy(b.data(), o_new, b.size() * 4, hipMemcpyDeviceToHost));
    size_t bad = 0; for (size_t i = 0; i < a.size(); i++) if (memcmp(&a[i], &b[i], 4)) bad++;
    const double top = 2.0 * N * K * T / 1e6;
    printf("N %d K %d T %d type %d: 256x32 %.1f us (%.0f TOP/s)  128x128 %.1f us (%.0f)  lds 128x256 %.1f us (%.0f)  mismatches %zu / %zu  sample %g\n",
           N, K, T, type, us1, top / us1, us2, top / us2, us4, top / us4, bad, a.size(), (double)b[12345 % b.size()]);
    return bad ? 1 : 0;
}
