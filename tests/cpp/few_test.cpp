// Every instance of the kernel for 3 to 16 rows (launch_few, and launch_few_multi as a list of two batches): planes, with and without an offset, scale groups of 128, 64 and 32 k, activations as rows (at most
// one and two per wavefront) and as columns, with and without splits along k, their sums by atomics and through memory, with a
// partial output batch, group of batches and k-block; results in rows of 8-byte and of 2-byte stores and in columns, with
// and without bias.  Results against double precision within the tolerance of the path (oracle/oracle.py), the same launch
// twice bit for bit, the bias as an addition to the fp16 result bit for bit, nothing written behind the results, the words for
// the splits back at zero, columns with the bits of rows, and the batches of a list with the bits of launches of their own.
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
constexpr int kMaxRows = lutgemm_kernels::kBatchRows;
constexpr int kGuard = 4096;                            // halves behind the results

uint16_t bits(_Float16 v) { uint16_t b; memcpy(&b, &v, 2); return b; }

template <typename T>
T *to_device(const std::vector<T> &v)
{
    T *p = nullptr;
    HIP_OK(hipMalloc((void **)&p, v.size() * sizeof(T)));
    HIP_OK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
}

// device memory of a batch's results and sums
struct Batch {
    size_t count;
    uint16_t *y;
    unsigned long long *words;
    float *partials;

    Batch(lutgemm_kernels::MatvecArgs *a, bool y_cols) : count((size_t)a->rows * kN)
    {
        y = to_device(std::vector<uint16_t>(count + kGuard, 0x7e01));
        words = to_device(std::vector<unsigned long long>((size_t)kMaxRows * kNb * 32));
        HIP_OK(hipMalloc((void **)&partials, (size_t)kNb * a->k_splits * 512 * sizeof(float)));
        a->y = y;
        a->accum = words;
        a->accum_row_stride = kNb * 32;
        a->y_stride = y_cols ? a->rows : 1;
        a->y_row_stride = y_cols ? 1 : kN;
    }

    // element (row, output) at [row * n + output] whatever the layout on the device; frees the memory
    std::vector<_Float16> results(int rows, bool y_cols)
    {
        std::vector<uint16_t> filled(count + kGuard);
        std::vector<unsigned long long> counts((size_t)kMaxRows * kNb * 32);
        HIP_OK(hipMemcpy(filled.data(), y, filled.size() * 2, hipMemcpyDeviceToHost));
        HIP_OK(hipMemcpy(counts.data(), words, counts.size() * 8, hipMemcpyDeviceToHost));
        HIP_OK(hipFree(y));
        HIP_OK(hipFree(words));
        HIP_OK(hipFree(partials));
        for (size_t i = count; i < filled.size(); i++)
            if (filled[i] != 0x7e01) { printf("FAIL written behind the results\n"); exit(1); }
        for (unsigned long long c : counts)
            if (c) { printf("FAIL a word is not back at zero\n"); exit(1); }
        std::vector<_Float16> out(count);
        for (int r = 0; r < rows; r++)
            for (int j = 0; j < kN; j++)
                memcpy(&out[(size_t)r * kN + j], &filled[y_cols ? (size_t)j * rows + r : (size_t)r * kN + j], 2);
        return out;
    }
};

// y of one launch
std::vector<_Float16> launch(int q, bool offset, int waves, bool atomics, lutgemm_kernels::MatvecArgs a, lutgemm_kernels::FewGrid g, bool y_cols)
{
    Batch batch(&a, y_cols);
    g.partials = atomics ? nullptr : batch.partials;
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(lutgemm_kernels::launch_few(q, offset, a, g, waves, nullptr));
    HIP_OK(hipDeviceSynchronize());
    return batch.results(a.rows, y_cols);
}

// A launch of a batch of `other` rows and one of a.rows as a list (sums by atomics); y of both, one behind the other
std::vector<_Float16> launch_list(int q, bool offset, int waves, lutgemm_kernels::MatvecArgs a, const lutgemm_kernels::FewGrid &g, int other)
{
    lutgemm_kernels::MultiMatvecArgs list{};
    list.count = 2;
    list.entry[0] = list.entry[1] = a;
    list.entry[0].rows = other;
    list.first_block[1] = a.ntiles * a.k_splits;
    Batch first(&list.entry[0], false), second(&list.entry[1], false);
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(lutgemm_kernels::launch_few_multi(q, offset, list, g, 2 * a.ntiles * a.k_splits, waves, nullptr));
    HIP_OK(hipDeviceSynchronize());
    std::vector<_Float16> y = first.results(other, false), more = second.results(a.rows, false);
    y.insert(y.end(), more.begin(), more.end());
    return y;
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
    const int wmax = lutgemm_kernels::few_waves_max(planes, 128 / group);
    uint16_t *xc = nullptr;   // the first rows of x as columns
    HIP_OK(hipMalloc((void **)&xc, (size_t)kK * kMaxRows * 2));
    for (int rows : {3, 8, 9, 16}) {
        std::vector<_Float16> columns((size_t)kK * rows);
        for (int r = 0; r < rows; r++)
            for (int k = 0; k < kK; k++) columns[(size_t)k * rows + r] = x[(size_t)r * kK + k];
        HIP_OK(hipMemcpy(xc, columns.data(), columns.size() * 2, hipMemcpyHostToDevice));
        for (int bps : {4, 3, 1})       // no split; splits of three k-blocks and one; four splits
            for (int end = 0; end < (bps == 4 ? 1 : 2); end++) {
                const int v = (*variant)++, waves = v % 2 ? lutgemm_kernels::kFewWavesMin : wmax;
                lutgemm_kernels::MatvecArgs a{};
                a.signs = static_cast<const uint8_t *>(signs);
                a.scales = static_cast<const uint16_t *>(scales);
                a.x = xd;
                a.k = kK;
                a.n = kN;
                a.ts = kTs;
                a.nb = kNb;
                a.ntiles = (kNb + waves - 1) / waves;
                a.blocks_per_split = bps;
                a.k_splits = (kTs + bps - 1) / bps;
                a.rows = rows;
                a.x_row_stride = kK;
                lutgemm_kernels::FewGrid g{};
                g.wide_y = v % 3 == 0;
                g.gsub = 128 / group;
                const bool y_cols = v % 3 == 2;
                printf("case few rows instance planes %d offset %d groups of %d rows %d wavefronts %d splits %d %s\n", planes, offset, group, rows, waves, a.k_splits,
                       end ? "atomics" : "memory");
                fflush(stdout);
                const std::vector<_Float16> y = launch(q, offset, waves, end, a, g, y_cols), again = launch(q, offset, waves, end, a, g, y_cols);
                g.bias = bd;
                const std::vector<_Float16> plus = launch(q, offset, waves, end, a, g, y_cols);
                lutgemm_kernels::MatvecArgs ac = a;
                ac.x = xc;
                ac.ntiles = (kNb + lutgemm_kernels::kFewWavesMin - 1) / lutgemm_kernels::kFewWavesMin;
                g.bias = nullptr;
                g.columns = 1;
                const std::vector<_Float16> from_columns = launch(q, offset, lutgemm_kernels::kFewWavesMin, end, ac, g, y_cols);
                if (end || a.k_splits == 1) {
                    g.columns = 0;
                    const int other = rows == 3 ? 8 : 24 - rows;   // lists with one row per wavefront at most and with two
                    lutgemm_kernels::MatvecArgs alone = a;
                    alone.rows = other;
                    std::vector<_Float16> each = launch(q, offset, waves, true, alone, g, false);
                    const std::vector<_Float16> last = y_cols ? launch(q, offset, waves, true, a, g, false) : y;
                    each.insert(each.end(), last.begin(), last.end());
                    const std::vector<_Float16> list = launch_list(q, offset, waves, a, g, other);
                    if (list.size() != each.size() || memcmp(list.data(), each.data(), each.size() * 2)) {
                        printf("FAIL the batches of a list are not those of launches of their own\n");
                        exit(1);
                    }
                }
                for (size_t i = 0; i < y.size(); i++) {
                    const double t = truth[i], m = std::fmax(std::fabs(t), std::ldexp(1.0, -14));
                    const double bound = 2 * std::ldexp(1.0, (int)std::floor(std::log2(m)) - 10) + 1e-3;
                    const _Float16 sum = (_Float16)((float)y[i] + (float)bias[i % kN]);
                    if (!(std::fabs((double)y[i] - t) <= bound) || bits(again[i]) != bits(y[i]) || bits(plus[i]) != bits(sum) ||
                        bits(from_columns[i]) != bits(y[i])) {
                        printf("FAIL at %zu: %g, %g again, %g with bias %g, %g from columns, truth %g\n", i, (double)y[i], (double)again[i],
                               (double)plus[i], (double)bias[i % kN], (double)from_columns[i], t);
                        exit(1);
                    }
                }
            }
    }
    HIP_OK(hipFree(xc));
    HIP_OK(hipFree(xd));
    HIP_OK(hipFree(bd));
    lutgemm_weight_destroy(w);
}

}  // namespace

int main()
{
    int variant = 0;
    for (int q = 1; q <= 8; q++)
        for (int offset = 0; offset < 2; offset++)
            for (int group : {128, 64, 32}) run_weight(q, offset, group, &variant);
    printf("FEW OK %d\n", variant);
    return 0;
}
