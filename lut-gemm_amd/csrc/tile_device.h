// Device-side pieces shared by the matvec kernels (kernels.hip) and the kernels for 3 and more rows (*_body.h):
// the registers of one weight tile with their loads, and the split-k completion of an output.
#ifndef LUTGEMM_TILE_DEVICE_H
#define LUTGEMM_TILE_DEVICE_H

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "device_util.h"
#include "kernels.h"
#include "layout.h"

namespace lutgemm_kernels {
using namespace lutgemm_layout;

template <int Q, int QO, int GSUB>
struct TileRegs {
    u32x4 sign[2 * Q];
    uint32_t scale[GSUB * QO];
};

// Where the next tile's loads of a wavefront come from (all lanes the same dummy line when the
// workgroup has no next k-block, see tile_address).
struct NextTile {
    const u32x4 *sign;    // this lane's first sign vector
    size_t sign_stride;   // in u32x4 units between units
    const uint32_t *scale;
};

// Addresses of tile `tile` for this lane.  `real` is wave-uniform; when false every lane reads
// the first bytes of the arrays instead (one cached line).  Written with masks rather than
// conditionals so that no branch appears: with straight-line code the compiler's wait counts
// for the loads stay exact.
template <int Q, int QO, int GSUB>
__device__ __forceinline__ NextTile tile_address(const u32x4 *signs, const uint32_t *scales, size_t tile,
                                                 int lane, bool real)
{
    const size_t m = (size_t)0 - (size_t)real;  // all ones or zero
    NextTile n;
    n.scale = scales + (((tile * kLanes + lane) * (size_t)(GSUB * QO)) & m);
    n.sign = signs + ((tile * (size_t)(2 * Q * kLanes) + lane) & m);
    n.sign_stride = (size_t)kLanes & m;
    return n;
}

// The same for a kernel that can afford a whole tile of loads past the end of its range: the tile
// number becomes 0 there (tile 0 stays in the cache: every workgroup ends on it).  `tile` and
// `real` are wave-uniform, so an address is a uniform base plus a lane constant plus an immediate
// and the address arithmetic stays on the scalar unit.
template <int Q, int QO, int GSUB>
__device__ __forceinline__ NextTile tile_address_uniform(const u32x4 *signs, const uint32_t *scales, size_t tile,
                                                         int lane, bool real)
{
    const size_t t = real ? tile : (size_t)0;
    NextTile n;
    n.scale = scales + t * (size_t)(kLanes * GSUB * QO) + lane * (GSUB * QO);
    n.sign = signs + t * (size_t)(2 * Q * kLanes) + lane;
    n.sign_stride = (size_t)kLanes;
    return n;
}

template <int Q, int QO, int GSUB>
__device__ __forceinline__ void load_tile(TileRegs<Q, QO, GSUB> &r, const NextTile &n)
{
#pragma unroll
    for (int d = 0; d < GSUB * QO; d++) r.scale[d] = __builtin_nontemporal_load(n.scale + d);
#pragma unroll
    for (int u = 0; u < 2 * Q; u++) r.sign[u] = __builtin_nontemporal_load(n.sign + u * n.sign_stride);
}

// The output that `value` rounds to plus a bias, still to be rounded: what adding the bias to a finished output gives
__device__ __forceinline__ float plus_bias(float value, float bias) { return __half2float(__float2half_rn(value)) + bias; }

// plus_bias of output `out` (in the kernels that take a bias; BIAS is a template argument because even a test for
// its absence at the end of a workgroup cost the batch kernel 2 to 7 %)
template <bool BIAS>
__device__ __forceinline__ float add_bias(const __half *bias, float value, int out)
{
    if constexpr (BIAS) return plus_bias(value, __half2float(bias[out]));
    else return value;
}

// Lane pair (2j, 2j+1) of a wavefront holds the k-range total of output `out`; the even lane
// delivers it.  With one k-split it is the result.  Otherwise: one 64-bit atomic add per output,
// no barrier, no second pass.  The word holds an arrival count in its top 8 bits and the running
// sum below it, as a biased fixed-point integer (2^-24 units, bias 2^46 per addend so every
// addend is positive; at most 128 addends below 2^47 keep the sum below 2^54 and out of the
// flags and the count).  Integer addition is associative, so the total does not depend on the
// order in which the workgroups arrive: the result is deterministic.  The workgroup whose add
// returns count == k_splits-1 is the last one for that output: it holds the complete sum, writes
// y and puts the word back to zero for the next launch.
// A partial sum that is not finite cannot be expressed in fixed point.  Its workgroup first sets
// a flag in the same word (bit 54: +infinity seen, bit 55: -infinity seen, both: NaN) and then
// adds a zero contribution; the finishing workgroup turns the flags into the value IEEE
// arithmetic gives the sum: +-infinity, or NaN for a NaN or for infinities of both signs.  The
// flag store and the add are atomics of one thread on one address, so they take effect in
// program order.
constexpr unsigned long long kPosInfFlag = 1ull << 54, kNegInfFlag = 1ull << 55;
// The two halves of the completion, so that a wavefront that finishes several values per lane can
// issue all its atomics before it waits for the first answer.
struct Arrival {
    unsigned long long old, addend;
};

// First half: the split-k atomic (only with more than one k-split).  `valid` selects the lanes
// that deliver a value.
__device__ __forceinline__ Arrival arrive_output(float total, bool valid, unsigned long long *word)
{
    Arrival r{0ull, 0ull};
    if (!valid) return r;
    float scaled = total * 16777216.f;
    if (!(fabsf(scaled) < 7.0e13f)) {  // beyond 2^46 in fixed point, infinite or NaN
        const unsigned long long flags =
            total != total ? (kPosInfFlag | kNegInfFlag) : total > 0.f ? kPosInfFlag : kNegInfFlag;
        __hip_atomic_fetch_or(word, flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        scaled = 0.f;
    }
    r.addend = (unsigned long long)(__float2ll_rn(scaled) + (1ll << 46)) + (1ull << 56);
    r.old = __hip_atomic_fetch_add(word, r.addend, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return r;
}

// Second half: the lane whose add arrived last writes the output and clears the word.
// arrived_last only looks at the answer of the atomic; a wavefront that finishes several values per
// lane evaluates it for all of them before the first finish_last, so that no wait for an answer
// comes behind a store (the wait would then also wait for that store's round trip).
__device__ __forceinline__ bool arrived_last(const Arrival &r, bool valid, int k_splits)
{
    return valid && (r.old >> 56) == (unsigned long long)(k_splits - 1);
}

// `finish` makes the output's value of the sum
template <typename F>
__device__ __forceinline__ void finish_last(const Arrival &r, unsigned long long *word, __half *yout, int k_splits, F &&finish)
{
    const unsigned long long all = r.old + r.addend;
    const long long value = (long long)(all & (kPosInfFlag - 1)) - (long long)k_splits * (1ll << 46);
    float result = __ll2float_rn(value) * (1.f / 16777216.f);
    const unsigned long long flags = all & (kPosInfFlag | kNegInfFlag);
    if (flags)
        result = flags == kPosInfFlag ? __builtin_inff() : flags == kNegInfFlag ? -__builtin_inff() : __builtin_nanf("");
    *yout = __float2half_rn(finish(result));
    __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void finish_last(const Arrival &r, unsigned long long *word, __half *yout, int k_splits)
{
    finish_last(r, word, yout, k_splits, [](float sum) { return sum; });
}

template <bool BIAS>
__device__ __forceinline__ void finish_output(float total, bool active, int out, int lane, __half *y,
                                              unsigned long long *accum, const MatvecArgs &a, const __half *bias)
{
    const bool valid = active && (lane & 1) == 0 && out < a.n;
    if (a.k_splits == 1) {
        if (valid) y[(size_t)out * a.y_stride] = __float2half_rn(add_bias<BIAS>(bias, total, out));
        return;
    }
    const Arrival r = arrive_output(total, valid, accum + out);
    if (arrived_last(r, valid, a.k_splits))
        finish_last(r, accum + out, y + (size_t)out * a.y_stride, a.k_splits, [&](float sum) { return add_bias<BIAS>(bias, sum, out); });
}

// Split-k sums of a wavefront's N registers of four values through memory, for kernels that finish many values per
// lane: one 64-bit atomic per value (above) costs 8.7 us per million on the memory side, and a launch of 64 rows x
// 12288 outputs x 5 splits makes four million of them.  Here every wavefront writes its partial sums as they lie in
// its registers (1 KiB runs), counts itself in once, and the one that comes last adds up all partial sums in the
// order of their k ranges, so that the result does not depend on who that is; it returns true with the totals in the
// registers and the count back at zero.
// The XCDs' L2 caches are not coherent among each other: the stores and loads of the partial sums are device-scope (they
// go past the L2), and the count is raised only when the stores are acknowledged.  A lane moves 16 bytes at a time: as 8-byte
// halves of them, which the memory side gets as partial lines, the exchange of 8 MB took 5 us longer (4096 x 16384, three
// planes, 16 rows, 4 splits: 21.9 us).
// `partials`: k_splits blocks of N * 256 floats; `of(I)`: register I.
template <int N, typename F>
__device__ __forceinline__ bool sum_partials(float *partials, unsigned *count, int ks, int k_splits, int lane, F &&of)
{
    typedef float float4v __attribute__((ext_vector_type(4)));
    constexpr int kDeviceScope = 16;   // sc1: write through, and read past the L2
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)partials, (short)0, -1, 0x00020000);
    static_for<N>([&](auto I) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, (float4v)of(I)), rsrc, lane * 16, (ks * N + I) * 1024, kDeviceScope);
    });
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    unsigned before = 0;
    if (lane == 0) before = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = __builtin_amdgcn_readfirstlane(before);
    if (before != (unsigned)(k_splits - 1)) return false;
    asm volatile("" : : : "memory");
    static_for<N>([&](auto I) { auto &v = of(I); v[0] = v[1] = v[2] = v[3] = 0.f; });
    // Loads past the L2 take a microsecond, so as many partial sums as fit are on their way together; no more than there are,
    // since they also cost their bytes.
    constexpr int AHEAD = N <= 2 ? 8 : N <= 4 ? 4 : 2;
    for (int s = 0; s < k_splits; s += AHEAD) {
        u32x4 part[AHEAD][N];
        static_for<AHEAD>([&](auto J) {
            if (s + J < k_splits)   // uniform
                static_for<N>([&](auto I) {
                    part[J][I] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16, ((s + J) * N + I) * 1024, kDeviceScope));
                });
        });
        static_for<AHEAD>([&](auto J) {
            if (s + J < k_splits) static_for<N>([&](auto I) { of(I) += __builtin_bit_cast(float4v, part[J][I]); });
        });
    }
    if (lane == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

}  // namespace lutgemm_kernels
#endif
