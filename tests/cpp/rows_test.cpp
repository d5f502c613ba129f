// Every instance of the kernel for many rows (launch_rows), which the library's plans reach only for some sizes: planes
// 1 to 9 (an offset counts as one), two to four row tiles per workgroup, one and two k groups, with and without splits
// along k, with a partial last row tile, output batch, group of batches and k-block; results in rows of 8-byte and of
// 2-byte stores and in columns, with and without bias.  Results against double precision within the tolerance of the path
// (oracle/oracle.py), the same launch twice bit for bit, the bias as an addition to the fp16 result bit for bit, nothing
// written behind the results, and the arrival counts back at zero.
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../lut-gemm_amd/csrc/kernels.h"
#include "lutgemm_c.h"

namespace {

#define HIP_OK(call)                                                                   \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess) {                                                        \
            fprintf(stderr, "%s failed: %s\n", #call, hipGetErrorString(e_));          \
            exit(2);                                                                   \
        }                                                                              \
    } while (0)

constexpr int kK = 1664, kN = 300, kTs = 4, kNb = 10;   // the last k-block is a quarter, the last batch 12 outputs
constexpr int kMaxRows = 2 * 4 * 16;
constexpr int kGuard = 4096;                            // halves behind the results
const int kGroups[] = {128, 32, 832, 416, 64, 1664};    // one, four, two, four, two and one scale groups per 128 k

uint16_t bits(_Float16 v) { uint16_t b; memcpy(&b, &v, 2); return b; }

template <typename T>
T *to_device(const std::vector<T> &v)
{
    T *p = nullptr;
    HIP_OK(hipMalloc((void **)&p, v.size() * sizeof(T)));
    HIP_OK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
}

// y of one launch, element (row, output) at [row * n + output] whatever the layout on the device
std::vector<_Float16> launch(int planes, int rt, int kw, lutgemm_kernels::MatvecArgs a, lutgemm_kernels::RowsGrid g, bool cols)
{
    const size_t count = (size_t)a.rows * kN;
    std::vector<uint16_t> filled(count + kGuard, 0x7e01);
    uint16_t *y = to_device(filled);
    std::vector<unsigned long long> zeros((size_t)g.row_chunks * kNb);
    unsigned long long *counts = to_device(zeros);
    float *partials = nullptr;
    HIP_OK(hipMalloc((void **)&partials, (size_t)kNb * g.row_chunks * rt * a.k_splits * 512 * sizeof(float)));
    a.y = y;
    a.accum = counts;
    a.y_stride = cols ? a.rows : 1;
    a.y_row_stride = cols ? 1 : kN;
    g.partials = partials;
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(lutgemm_kernels::launch_rows(planes, rt, kw, a, g, nullptr));
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(hipMemcpy(filled.data(), y, filled.size() * 2, hipMemcpyDeviceToHost));
    HIP_OK(hipMemcpy(zeros.data(), counts, zeros.size() * 8, hipMemcpyDeviceToHost));
    HIP_OK(hipFree(y));
    HIP_OK(hipFree(counts));
    HIP_OK(hipFree(partials));
    for (size_t i = count; i < filled.size(); i++)
        if (filled[i] != 0x7e01) { printf("FAIL written behind the results\n"); exit(1); }
    for (unsigned long long c : zeros)
        if (c) { printf("FAIL a count is not back at zero\n"); exit(1); }
    std::vector<_Float16> out(count);
    for (int r = 0; r < a.rows; r++)
        for (int j = 0; j < kN; j++)
            memcpy(&out[(size_t)r * kN + j], &filled[cols ? (size_t)j * a.rows + r : (size_t)r * kN + j], 2);
    return out;
}

void run_weight(int q, bool offset, int group, int *variant)
{
    std::mt19937 rng(q * 2 + offset);
    std::normal_distribution<float> normal;
    const int planes = q + offset, groups = kK / group;
    std::vector<uint32_t> words((size_t)kK / 32 * q * kN);
    for (auto &w : words) w = rng();
    std::vector<_Float16> alpha((size_t)groups * q * kN), z((size_t)groups * kN), x((size_t)kMaxRows * kK), bias(kN);
    for (auto &v : alpha) v = (_Float16)std::fabs(0.02f * normal(rng));
    for (auto &v : z) v = (_Float16)(0.01f * normal(rng));
    for (auto &v : x) v = (_Float16)normal(rng);
    for (auto &v : bias) v = (_Float16)normal(rng);
    std::vector<double> truth((size_t)kMaxRows * kN), row(kN);
    for (int k = 0; k < kK; k++) {
        for (int j = 0; j < kN; j++) {
            double sum = offset ? (double)z[(size_t)(k / group) * kN + j] : 0.0;
            for (int b = 0; b < q; b++) {
                const double s = (double)alpha[((size_t)(k / group) * q + b) * kN + j];
                sum += words[((size_t)(k / 32) * q + b) * kN + j] >> (k % 32) & 1 ? s : -s;
            }
            row[j] = sum;
        }
        for (int r = 0; r < kMaxRows; r++) {
            const double v = (double)x[(size_t)r * kK + k];
            for (int j = 0; j < kN; j++) truth[(size_t)r * kN + j] += v * row[j];
        }
    }
    lutgemm_weight *w = nullptr;
    if (lutgemm_weight_create_f16(words.data(), reinterpret_cast<const uint16_t *>(alpha.data()),
                                  offset ? reinterpret_cast<const uint16_t *>(z.data()) : nullptr, kK, kN, q, groups, &w) != LUTGEMM_OK) {
        printf("FAIL %s\n", lutgemm_last_error());
        exit(1);
    }
    void *signs = nullptr, *scales = nullptr;
    lutgemm_weight_device_ptrs(w, &signs, &scales, nullptr);
    _Float16 *xd = to_device(x), *bd = to_device(bias);
    for (int rt = lutgemm_kernels::kRowsTilesMin; rt <= lutgemm_kernels::kRowsTilesMax; rt++)
        for (int kw = 1; kw <= 2; kw++)
            for (int bps : {4, 3, 1}) {   // no split; splits of three k-blocks and one; four splits
                const int v = (*variant)++, nw = lutgemm_kernels::kRowsWaves / kw;
                const bool cols = v % 3 == 2, wide = v % 3 == 0;
                lutgemm_kernels::MatvecArgs a{};
                a.signs = static_cast<const uint8_t *>(signs);
                a.scales = static_cast<const uint16_t *>(scales);
                a.x = xd;
                a.k = kK;
                a.n = kN;
                a.ts = kTs;
                a.nb = kNb;
                a.ntiles = (kNb + nw - 1) / nw;
                a.blocks_per_split = bps;
                a.k_splits = (kTs + bps - 1) / bps;
                a.rows = 16 * rt + (v % 2 ? 1 : 16 * rt - 5);   // two row chunks, the second of one row or all but five
                a.x_row_stride = kK;
                lutgemm_kernels::RowsGrid g{};
                g.row_chunks = 2;
                g.q = q;
                g.gsub = group % 128 == 0 ? 1 : group % 64 == 0 ? 2 : 4;
                g.wide_y = wide;
                printf("case rows instance planes %d offset %d group %d row tiles %d k groups %d splits %d rows %d\n", planes, offset, group,
                       rt, kw, a.k_splits, a.rows);
                fflush(stdout);
                const std::vector<_Float16> y = launch(planes, rt, kw, a, g, cols), again = launch(planes, rt, kw, a, g, cols);
                g.bias = bd;
                const std::vector<_Float16> plus = launch(planes, rt, kw, a, g, cols);
                for (size_t i = 0; i < y.size(); i++) {
                    const double t = truth[i], m = std::fmax(std::fabs(t), std::ldexp(1.0, -14));
                    const double bound = 2 * std::ldexp(1.0, (int)std::floor(std::log2(m)) - 10) + 1e-3;
                    const _Float16 sum = (_Float16)((float)y[i] + (float)bias[i % kN]);
                    if (!(std::fabs((double)y[i] - t) <= bound) || bits(again[i]) != bits(y[i]) || bits(plus[i]) != bits(sum)) {
                        printf("FAIL at %zu: %g, %g again, %g with bias %g, truth %g\n", i, (double)y[i], (double)again[i], (double)plus[i],
                               (double)bias[i % kN], t);
                        exit(1);
                    }
                }
            }
    HIP_OK(hipFree(xd));
    HIP_OK(hipFree(bd));
    lutgemm_weight_destroy(w);
}

}  // namespace

int main()
{
    int variant = 0;
    for (int q = 1; q <= 8; q++)
        for (int offset = 0; offset < 2; offset++) run_weight(q, offset, kGroups[(2 * q + offset) % 6], &variant);
    printf("ROWS OK %d\n", variant);
    return 0;
}
