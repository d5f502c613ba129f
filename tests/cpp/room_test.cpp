// A handle whose device has no memory for the partial sums of 3 to 16 rows: this program's own hipMalloc refuses what it is told
// to.  A handle made without that room gets it with the first launch that needs it, where there is memory by then (the bits of a
// handle that has it); where there is none, sums go through the accumulators (within the tolerance of the path, oracle/oracle.py,
// the same bits from launch to launch, on a second stream too) until the workspace is reset.  The allocation-free entry point,
// whose room is its own, does not notice; and a handle that does not fit at all is refused.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "lutgemm_c.h"

namespace {
size_t g_most = SIZE_MAX, g_largest = 0;   // larger pieces are refused; the largest one since it was last cleared
}

extern "C" hipError_t hipMalloc(void **p, size_t bytes)
{
    typedef hipError_t (*Malloc)(void **, size_t);
    static Malloc next = reinterpret_cast<Malloc>(dlsym(RTLD_NEXT, "hipMalloc"));
    g_largest = std::max(g_largest, bytes);
    return bytes > g_most ? hipErrorOutOfMemory : next(p, bytes);
}

namespace {

#define CHECK(what)                                                                                            \
    do {                                                                                                       \
        if (!(what)) {                                                                                         \
            printf("FAIL line %d: %s (%s, %s)\n", __LINE__, #what, lutgemm_last_error(), hipGetErrorString(hipGetLastError())); \
            exit(1);                                                                                           \
        }                                                                                                      \
    } while (0)

constexpr int kK = 4096, kN = 2048, kQ = 2, kGroup = 128, kRows = 8;

size_t device_bytes(const lutgemm_weight *w)
{
    lutgemm_weight_info_t info;
    CHECK(lutgemm_weight_info(w, &info) == LUTGEMM_OK);
    return info.device_bytes;
}

template <typename Call>
std::vector<uint16_t> results(uint16_t *y, hipStream_t stream, Call call)
{
    std::vector<uint16_t> out((size_t)kRows * kN, 0x7e01);
    CHECK(hipMemcpy(y, out.data(), out.size() * 2, hipMemcpyHostToDevice) == hipSuccess && hipDeviceSynchronize() == hipSuccess);
    CHECK(call() == LUTGEMM_OK);
    CHECK(hipStreamSynchronize(stream) == hipSuccess);
    CHECK(hipMemcpy(out.data(), y, out.size() * 2, hipMemcpyDeviceToHost) == hipSuccess);
    return out;
}

}  // namespace

int main()
{
    std::mt19937 rng(3);
    std::normal_distribution<float> normal;
    std::vector<uint32_t> words((size_t)kK / 32 * kQ * kN);
    for (auto &w : words) w = rng();
    std::vector<_Float16> alpha((size_t)kK / kGroup * kQ * kN), x((size_t)kRows * kK);
    for (auto &v : alpha) v = (_Float16)std::fabs(0.02f * normal(rng));
    for (auto &v : x) v = (_Float16)normal(rng);
    std::vector<double> truth((size_t)kRows * kN), row(kN);
    for (int k = 0; k < kK; k++) {
        for (int j = 0; j < kN; j++) {
            row[j] = 0.0;
            for (int b = 0; b < kQ; b++) {
                const double s = (double)alpha[((size_t)(k / kGroup) * kQ + b) * kN + j];
                row[j] += words[((size_t)(k / 32) * kQ + b) * kN + j] >> (k % 32) & 1 ? s : -s;
            }
        }
        for (int r = 0; r < kRows; r++)
            for (int j = 0; j < kN; j++) truth[(size_t)r * kN + j] += (double)x[(size_t)r * kK + k] * row[j];
    }
    uint16_t *xd = nullptr, *y = nullptr;
    CHECK(hipMalloc((void **)&xd, x.size() * 2) == hipSuccess && hipMalloc((void **)&y, truth.size() * 2) == hipSuccess);
    CHECK(hipMemcpy(xd, x.data(), x.size() * 2, hipMemcpyHostToDevice) == hipSuccess);
    hipStream_t streams[2];
    for (hipStream_t &s : streams) CHECK(hipStreamCreate(&s) == hipSuccess);
    const uint16_t *scales = reinterpret_cast<const uint16_t *>(alpha.data());
    auto create = [&](lutgemm_weight **w) { return lutgemm_weight_create_f16(words.data(), scales, nullptr, kK, kN, kQ, kK / kGroup, w); };
    auto matvec = [&](lutgemm_weight *w, hipStream_t s) { return results(y, s, [&] { return lutgemm_matvec(w, xd, y, kRows, s); }); };
    auto right = [&](const std::vector<uint16_t> &got) {
        for (size_t i = 0; i < got.size(); i++) {
            _Float16 v;
            memcpy(&v, &got[i], 2);
            const double m = std::fmax(std::fabs(truth[i]), std::ldexp(1.0, -14));
            if (!(std::fabs((double)v - truth[i]) <= 2 * std::ldexp(1.0, (int)std::floor(std::log2(m)) - 10) + 1e-3)) return false;
        }
        return true;
    };

    printf("case room as it is made\n"), fflush(stdout);
    lutgemm_weight *w = nullptr;
    g_largest = 0;
    CHECK(create(&w) == LUTGEMM_OK);
    const size_t block = g_largest, whole = device_bytes(w);   // the tiles and the memory of the first stream
    int splits = 0;
    CHECK(lutgemm_weight_plan_for(w, kRows, nullptr, nullptr, &splits, nullptr) == LUTGEMM_OK && splits > 1);
    const std::vector<uint16_t> want = matvec(w, streams[0]);
    CHECK(right(want) && device_bytes(w) == whole);
    CHECK(lutgemm_weight_destroy(w) == LUTGEMM_OK);

    printf("case room with the first launch\n"), fflush(stdout);
    g_most = block - 1;
    CHECK(create(&w) == LUTGEMM_OK);
    const size_t without = device_bytes(w);
    CHECK(without < whole);
    CHECK(matvec(w, streams[0]) == want && device_bytes(w) > without);
    CHECK(lutgemm_weight_destroy(w) == LUTGEMM_OK);

    printf("case no room\n"), fflush(stdout);
    CHECK(create(&w) == LUTGEMM_OK && device_bytes(w) == without);
    g_most = 0;
    const std::vector<uint16_t> atomics = matvec(w, streams[0]);
    CHECK(right(atomics) && matvec(w, streams[0]) == atomics && device_bytes(w) == without);
    CHECK(results(y, streams[0], [&] { return lutgemm_matvec_static(w, xd, y, kRows, streams[0]); }) == want);
    CHECK(lutgemm_matvec(w, xd, y, kRows, streams[1]) == LUTGEMM_ERR_OUT_OF_MEMORY);   // no memory for a second stream's words
    g_most = (size_t)16 * (kN * sizeof(uint64_t) + kK * 2);                            // for those and the staged columns only
    CHECK(matvec(w, streams[1]) == atomics);
    g_most = SIZE_MAX;
    CHECK(matvec(w, streams[0]) == atomics && matvec(w, streams[1]) == atomics);       // the same call keeps its bits
    CHECK(lutgemm_weight_reset_workspace(w, streams[0]) == LUTGEMM_OK);
    CHECK(matvec(w, streams[0]) == want);
    CHECK(lutgemm_weight_destroy(w) == LUTGEMM_OK);

    printf("case no handle\n"), fflush(stdout);
    g_most = 4096;
    CHECK(create(&w) == LUTGEMM_ERR_OUT_OF_MEMORY && !w);
    g_most = SIZE_MAX;
    CHECK(create(&w) == LUTGEMM_OK && device_bytes(w) == whole && matvec(w, streams[1]) == want);
    CHECK(lutgemm_weight_destroy(w) == LUTGEMM_OK);
    for (hipStream_t s : streams) CHECK(hipStreamDestroy(s) == hipSuccess);
    CHECK(hipFree(xd) == hipSuccess && hipFree(y) == hipSuccess);
    printf("ROOM OK\n");
    return 0;
}
