// Re-tiling of a weight on the device: the arrays of the reference's layout (packer.cpp) as they were copied from the host
// become the sign and scale tiles of layout.h.
//
// A 4096 x 16384 weight of four planes with offset spent 9 ms in the host packer (byte gathers over 34 MB on eight threads) of
// the 13 ms that creating and expanding it took; here the raw words cross the link instead of the tiles, which have the
// same size, and both kernels together run at memory speed (about 40 us).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "device_util.h"
#include "kernels.h"
#include "layout.h"

namespace lutgemm_kernels {
using namespace lutgemm_layout;

namespace {

// One thread per 16 bytes of a sign tile: byte c % 4 of the words of 16 neighbouring outputs.  The four lanes of a word read the
// same 64 bytes (one line, served together); a wavefront writes 1 KiB.
__global__ __launch_bounds__(256) void pack_signs_kernel(PackArgs a)
{
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = (int)(idx & 63);
    const size_t unit = idx >> 6;
    const int units = 2 * a.q;
    if (unit >= (size_t)a.nb * a.ts * units) return;
    const int u = (int)(unit % units), b = u >> 1, h = u & 1;
    const size_t tile = unit / units;
    const int ts = (int)(tile % a.ts), nb = (int)(tile / a.ts);
    const int c = ts * kLanes + lane, n0 = nb * kBatch + h * 16;
    u32x4 out = u32x4{0u, 0u, 0u, 0u};
    if (c < a.k / kChunk && n0 < a.n) {
        const uint32_t *src = a.words + ((size_t)(c >> 2) * a.q + b) * a.n + n0;
        uint32_t w[16];
        if (n0 + 16 <= a.n && a.n % 4 == 0) {   // rows of words are 16-byte aligned
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32x4 v = reinterpret_cast<const u32x4 *>(src)[i];
                w[4 * i] = v.x;
                w[4 * i + 1] = v.y;
                w[4 * i + 2] = v.z;
                w[4 * i + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) w[i] = n0 + i < a.n ? src[i] : 0u;
        }
        const uint32_t sel = (uint32_t)(c & 3), pick = sel | ((4u + sel) << 8);   // byte c % 4 of either operand
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = __builtin_amdgcn_perm(w[4 * i + 1], w[4 * i], pick) & 0xffffu;
            const uint32_t hi = __builtin_amdgcn_perm(w[4 * i + 3], w[4 * i + 2], pick);
            out[i] = lo | (hi << 16);
        }
    }
    reinterpret_cast<u32x4 *>(a.signs)[idx] = out;
}

// fp32 -> fp16 bits, round to nearest even, every NaN the quiet one of its sign (what the host packer makes of it)
__device__ __forceinline__ uint16_t half_bits(float f)
{
    if (f != f) return (uint16_t)(((__builtin_bit_cast(uint32_t, f) >> 16) & 0x8000u) | 0x7e00u);
    return __half_as_ushort(__float2half_rn(f));
}

// One thread per fp16 of a scale tile; consecutive threads write consecutive halves.
template <bool HALF>
__global__ __launch_bounds__(256) void pack_scales_kernel(PackArgs a)
{
    const int qo = a.q + (a.offsets ? 1 : 0), lh = 2 * a.gsub * qo, subl = 16 / a.gsub;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)a.nb * a.ts * kLanes * lh) return;
    const int e = (int)(idx % lh), t = e / qo, bo = e % qo;
    const size_t rest = idx / lh;
    const int lane = (int)(rest % kLanes), ts = (int)(rest / kLanes % a.ts), nb = (int)(rest / kLanes / a.ts);
    const int j = lane & 15;
    const int kpos = ts * kBlockK + (lane >> 4) * 128 + (j / subl) * (128 / a.gsub);
    const int out = nb * kBatch + t * subl + j % subl;
    uint16_t v = 0;
    if (kpos < a.k && out < a.n) {
        const size_t group = (size_t)(kpos / a.group_size);
        const void *from = bo < a.q ? a.alpha : a.offsets;
        const size_t at = bo < a.q ? (group * a.q + bo) * a.n + out : group * a.n + out;
        v = HALF ? static_cast<const uint16_t *>(from)[at] : half_bits(static_cast<const float *>(from)[at]);
    }
    a.scales[idx] = v;
}

// Bound by reading the scales (4096 x 16384, four planes with offset: 5 MB, a few microseconds behind the kernels above).
__global__ __launch_bounds__(256) void find_non_finite_kernel(const u32x4 *halves, size_t pieces, unsigned long long *found)
{
    bool any = false;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < pieces; i += (size_t)gridDim.x * blockDim.x) {
        const u32x4 v = halves[i];
#pragma unroll
        for (int c = 0; c < 4; c++) any |= (v[c] & 0x7c00u) == 0x7c00u || (v[c] & 0x7c000000u) == 0x7c000000u;
    }
    if (any) *found = 1;   // every thread that stores stores the same
}

}  // namespace

hipError_t launch_find_non_finite(const uint16_t *halves, size_t pieces, unsigned long long *found, hipStream_t stream)
{
    const size_t blocks = (pieces + 255) / 256;
    hipLaunchKernelGGL(find_non_finite_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, stream,
                       reinterpret_cast<const u32x4 *>(halves), pieces, found);
    return hipGetLastError();
}

hipError_t launch_pack(const PackArgs &a, hipStream_t stream)
{
    const size_t sign_threads = (size_t)a.nb * a.ts * 2 * a.q * kLanes;
    const size_t halves = (size_t)a.nb * a.ts * kLanes * 2 * a.gsub * (a.q + (a.offsets ? 1 : 0));
    const size_t sign_blocks = (sign_threads + 255) / 256, scale_blocks = (halves + 255) / 256;
    if (sign_blocks > 0x7fffffu || scale_blocks > 0x7fffffu) return hipErrorInvalidValue;   // 2^31 threads
    hipLaunchKernelGGL(pack_signs_kernel, dim3((unsigned)sign_blocks), dim3(256), 0, stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.halves)
        hipLaunchKernelGGL((pack_scales_kernel<true>), dim3((unsigned)scale_blocks), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL((pack_scales_kernel<false>), dim3((unsigned)scale_blocks), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace lutgemm_kernels
