// gfx950 kernel for small batches, 3 to 16 activation rows against a packed BCQ weight in one pass over its tiles.
//
// The contraction is the batch kernel's (batch_body.h): v_smfmac_f32_16x16x64_f16 with every activation in LDS as the
// pair (-x, +x) and the sign bits as the index registers.  What bounds both is instruction issue: a matrix instruction
// holds the vector unit of its SIMD for 16 cycles, during which it takes ONE other vector instruction for nothing and every
// further one in 4 cycles more, whatever the number of wavefronts (measured: 16.3 / 20.3 / 24.3 / 28.4 cycles with 1 / 2 / 3 / 4
// v_perm_b32 per matrix instruction, with 1, 2 and 4 wavefronts per SIMD).  The batch kernel issues 179 others per 64 of them
// (two planes), most of them scale multiply-adds in a row.  Here they are 66, spread one behind each matrix instruction:
//  * The scales are the matrix operand (fp16, exact) and go from the lane that loads them straight into it: the lane groups
//    own 128 consecutive k each (kappa: row kappa of the tile), so a lane's scale words are those of its own output.  An
//    offset is one more plane whose index always picks +x.
//  * The index of step pair n + 1 is made while step pair n is contracted (sched_barrier keeps the order).
//  * With scale groups of 32 and 64 k (FINE) a lane's operands change from word to word.  The scales of a tile are 1 KiB per plane;
//    they go through LDS, loaded a k-block ahead, and an operand is made anew behind its last use.  Loaded word by word, a word
//    ahead, they were waited for: 12288 x 12288, two planes, groups of 64, 8 rows 20.0 us, now 17.4.
//  * Activations and tiles come by buffer loads: an offset beyond the weight's k reads zero, and addresses are scalar.  The bounds
//    check covers the vector and the immediate offset and is not promised for the scalar one, so what may lie beyond k has no scalar
//    offset (12 columns of 7168 x 28672: 29.6 us with and without it).
//  * Sums of a k-split go through memory (sum_partials): eight 64-bit atomics per lane took 3.5 to 5 us of a launch.
// Products of two fp16 numbers are exact in the fp32 sums, so a result differs from the batch kernel's by fp32 rounding.  All planes
// of an output share one accumulator: codes off the middle of their range and activations with a mean make plane sums that only
// cancel together.  With an accumulator per plane parity both grew over a workgroup's k and lost the bits of their difference (k = 49152,
// four planes and offset, codes around 4 of 15, x around 1: 33 % of the results not the nearest fp16 number, 1.3 % now, 2.9 % in the
// batch kernel), and the distance of two uses that it gave was not needed (block of 12288 at 8 rows 134.7 us, now 133.9).
// What bounds it now: power.  With the weight stream taken away the loop runs at the 10.7 ns a matrix instruction takes when all
// compute units issue nothing else (6.9 ns on a few of them); the stream comes on top.  Measured (us, batch kernel -> this one, the
// better plan of each): 12288 x 12288, two planes, 8 rows 20.3 -> 18.3; n = 36864 45.2 -> 36.4; n = 49152 50.1 -> 45.8; k = 49152
// 51.4 -> 45.9; 7168 x 28672, three planes, 12 rows 34.4 -> 28.8; 12288 x 12288, four planes, 16 rows 36.7 -> 32.1; groups of 64, 12288 x 12288, two planes, 8 rows 22.9 -> 17.4;
// groups of 32, 7168 x 7168, three planes, 16 rows 21.3 -> 16.0, 12288 x 36864, two planes, 8 rows 50.4 -> 45.5.
// Tried: transposing the next tile's signs during the steps (two sets of sign registers, three activation buffers, the barrier in
// the middle of a k-block): no faster, 30 to 100 more registers; two workgroups per compute unit: no faster.
#ifndef LUTGEMM_FEW_BODY_H
#define LUTGEMM_FEW_BODY_H

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "device_util.h"
#include "kernels.h"
#include "layout.h"
#include "tile_device.h"

namespace lutgemm_kernels {
using namespace lutgemm_layout;

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half16 __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) half8 lds_half8;
typedef __attribute__((address_space(3))) v2i lds_v2i;

// The activation block of a k-block in LDS: [lane group kb of the B operand][row][word w][step][half of the operand], 16 bytes
// each, as in rows_body.h with whole k-blocks.  Chunk (kappa, byte of the word) is in half kappa / 2 of lane group
// 2 (kappa % 2) + byte % 2, for the steps of byte / 2.  A row's pitch shifts its 16-byte slots, so the 16 lanes that a read
// serves together hit 16 of them.
constexpr int kFewGroup = kBatchRows * kFewPitch, kFewBuf = 4 * kFewGroup;
static_assert(few_lds_bytes(0) == 2 * kFewBuf && kFewGroup % 256 == 0, "kernels.h states the LDS of this kernel");

// How the activations of a k-block come: rows of k halves, one or two per wavefront, or columns of m halves (all m of a
// k side by side), a piece of 64 halves per instruction, which a workgroup of eight wavefronts cuts evenly
enum class FewInput { kOneRow, kTwoRows, kColumns };

// word (x[2i], x[2i+1]) -> (-x[2i], +x[2i]) (selector 0x01000100) or (-x[2i+1], +x[2i+1]) (0x03020302)
__device__ __forceinline__ uint32_t minus_plus(uint32_t pair, uint32_t selector)
{
    return __builtin_amdgcn_perm(pair, pair, selector) ^ 0x00008000u;
}

// the largest workgroup an instance is compiled for
constexpr int few_waves(int planes, FewInput in, bool fine) { return in == FewInput::kColumns ? kFewWavesMin : few_waves_max(planes, fine ? 2 : 1); }

// workgroup `block` of a launch of a.ntiles * a.k_splits
template <int Q, bool OFF, FewInput IN, bool FINE>
__device__ __forceinline__ void few_workgroup(const MatvecArgs &a, const FewGrid &g, unsigned block)
{
    constexpr int P = Q + (OFF ? 1 : 0);
    constexpr int PG = (P + 3) / 4;              // passes over the planes of a k-block
    constexpr int QP = (P + PG - 1) / PG;        // planes per pass
    constexpr int NU = 2 * QP;                   // operands per pass: plane b, output half h -> 2 b + h
    constexpr int AHEAD = 2;                     // steps whose activations are on their way
    constexpr bool COLS = IN == FewInput::kColumns;
    constexpr int NP = COLS ? kBatchRows : IN == FewInput::kTwoRows ? 2 : 1;   // pieces of a k-block per lane, at most
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_generic[];
    lds_byte *lds = (lds_byte *)lds_generic;

    const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kappa = lane >> 4, j = lane & 15;
    const int ntile = (int)(block % (unsigned)a.ntiles), ks = (int)(block / (unsigned)a.ntiles);
    const int nb = ntile * waves + wave;
    const bool active = nb < a.nb;
    const int ts0 = ks * a.blocks_per_split, ts1 = min(ts0 + a.blocks_per_split, a.ts);
    const size_t tile0 = (size_t)(active ? nb : 0) * a.ts;
    constexpr int kBufferFlags = 0x00020000;   // 32-bit elements, offsets in bytes

    // sign staging as in rows_body.h: lane c writes outputs 0..15 of chunk c, lane (kappa, j) reads output j of the chunks of kappa
    lds_byte *stage = lds + 2 * kFewBuf + wave * kFewStage;
    lds_u32x4 *stage_w = reinterpret_cast<lds_u32x4 *>(stage + 16 * (lane ^ ((lane >> 1) & 8)));
    const int r_off = 256 * kappa + 8 * j;
    lds_v2i *stage_r0 = reinterpret_cast<lds_v2i *>(stage + (r_off ^ ((kappa & 1) * 128)));
    lds_v2i *stage_r1 = reinterpret_cast<lds_v2i *>(stage + ((r_off + 128) ^ ((kappa & 1) * 128)));

    const int gsub = FINE ? g.gsub : 1, subl = 16 / gsub, lh = 2 * gsub * P;   // scales of a lane of a tile
    const auto sign_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(a.signs + tile0 * (size_t)(2 * Q * kUnitBytes)), (short)0, -1, kBufferFlags);
    const auto scale_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(a.scales + tile0 * (size_t)(kLanes * lh)), (short)0, a.ts * 2 * kLanes * lh, kBufferFlags);
    u32x4 sign[NU];
    auto load_signs = [&](int kb, auto Pc) {
        static_for<NU>([&](auto U) {
            if constexpr (Pc * QP + U / 2 < Q)
                sign[U] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(sign_rsrc, lane * 16, kb * (2 * Q * kUnitBytes) + (Pc * NU + U) * kUnitBytes, 2));
        });
    };
    uint32_t scale[P];   // of the next k-block: number h P + b is the scale of plane b, output 16 h + j
    auto load_scales = [&](int kb) {
        if constexpr (FINE) return;
        const int from = lane * (4 * P), tile = kb * (kLanes * 4 * P);
        static_for<(P + 3) / 4>([&](auto I) {
            constexpr int n = P - 4 * I < 4 ? P - 4 * I : 4;
            if constexpr (n == 4) {
                const u32x4 t = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(scale_rsrc, from + 16 * I, tile, 2));
                static_for<4>([&](auto J) { scale[4 * I + J] = t[(int)J]; });
            } else if constexpr (n == 3) {
                const u32x3 t = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(scale_rsrc, from + 16 * I, tile, 2));
                static_for<3>([&](auto J) { scale[4 * I + J] = t[(int)J]; });
            } else if constexpr (n == 2) {
                const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(scale_rsrc, from + 16 * I, tile, 2));
                static_for<2>([&](auto J) { scale[4 * I + J] = t[(int)J]; });
            } else {
                scale[4 * I] = __builtin_amdgcn_raw_buffer_load_b32(scale_rsrc, from + 16 * I, tile, 2);
            }
        });
    };

    // FINE: the scales of a tile lie in LDS, from where a word's go into its operands; those of the next k-block are on their way
    // while one is contracted, and take its place when its last word's have been read.
    lds_byte *scale_area = lds + 2 * kFewBuf + waves * kFewStage + wave * few_scale_area(P);
    u32x4 fine[P];
    auto load_fine = [&](int kb) {
        static_for<P>([&](auto I) {
            if (4 * I < gsub * P) fine[I] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(scale_rsrc, lane * 16, kb * (2 * kLanes * lh) + I * 1024, 2));
        });
    };
    auto store_fine = [&]() {
        static_for<P>([&](auto I) {
            if (4 * I < gsub * P) *reinterpret_cast<lds_u32x4 *>(scale_area + I * 1024 + lane * 16) = fine[I];
        });
    };
    const lds_byte *scale_at = scale_area + 2 * ((kappa * 16 + j % subl) * lh + (j / subl) * P);
    uint32_t word_scale[NU];   // of word w for the units of pass Pc
    auto read_word_scales = [&](int w, auto Pc) {
        static_for<NU>([&](auto U) {
            constexpr int b = Pc * QP + U / 2, h = U % 2;
            if constexpr (b < P) word_scale[U] = *reinterpret_cast<const __attribute__((address_space(3))) uint16_t *>(scale_at + (w * gsub / 4) * (2 * subl * lh) + h * lh + 2 * b);
        });
    };
    half8 A[NU];
    auto make_word_operand = [&](auto U) {
        const uint32_t s = __builtin_amdgcn_perm(word_scale[U], word_scale[U], 0x01000100u);
        A[U] = __builtin_bit_cast(half8, u32x4{s, s, s, s});
    };

    // Activations.  Rows: a wavefront moves one row (and the one `waves` further on) of a k-block, a lane one chunk of 16 bytes,
    // which becomes a 16-byte block of each parity of k.  A lane's chunk, and the parity it writes first, are chosen so that the
    // 16 lanes that a write serves together (quads 0, 3, 5, 6 and 1, 2, 4, 7 of a half wavefront) hit 16 slots.
    // Columns: instruction i moves the halves 512 i + 64 wave + lane of the k-block; each goes to its place as a pair of its own.
    // k beyond the weight is beyond the buffer and reads as zero; rows beyond the batch stay zero from the start.
    const __half *x = reinterpret_cast<const __half *>(a.x);
    const int c_byte = lane & 3, c_kappa = ((lane >> 2) & 1) | ((lane >> 3) & 2), c_w = ((lane >> 3) & 1) | ((lane >> 4) & 2);
    const int first = lane & 1;
    const uint32_t sel_a = first ? 0x03020302u : 0x01000100u, sel_b = first ? 0x01000100u : 0x03020302u;
    lds_byte *piece_at = lds + (2 * (c_kappa & 1) + (c_byte & 1)) * kFewGroup + wave * kFewPitch + c_w * 128 + (c_byte >> 1) * 64 + (c_kappa >> 1) * 16 + 32 * first;
    const int to_other = 32 - 64 * first;
    const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, (int)((unsigned)a.k * (unsigned)a.rows * 2u), kBufferFlags);
    auto row_rsrc = [&](int row) {   // rows beyond the batch read its last one, and do not store it
        return __builtin_amdgcn_make_buffer_rsrc((void *)(x + (size_t)min(row, a.rows - 1) * (size_t)a.x_row_stride), (short)0, (int)((unsigned)a.k * 2u), kBufferFlags);
    };
    uint32_t x_off = COLS ? (uint32_t)(ts0 * kBlockK * a.rows + tid) * 2u
                          : (uint32_t)(ts0 * kBlockK + (16 * c_kappa + 4 * c_w + c_byte) * kChunk) * 2u;
    u32x4 piece[COLS ? 1 : NP];
    uint16_t half_of[COLS ? NP : 1];
    uint32_t half_at[COLS ? NP : 1];   // LDS offsets in an activation buffer
    if constexpr (COLS) {
        int kk = tid / a.rows, r = tid % a.rows;
        const int k_step = 512 / a.rows, r_step = 512 % a.rows;
        static_for<NP>([&](auto I) {
            half_at[I] = (uint32_t)((2 * ((kk >> 7) & 1) + ((kk >> 3) & 1)) * kFewGroup + r * kFewPitch + ((kk >> 5) & 3) * 128 + ((kk >> 4) & 1) * 64 +
                                    (kk & 1) * 32 + ((kk >> 8) & 1) * 16 + ((kk >> 1) & 3) * 4);
            kk += k_step;
            r += r_step;
            if (r >= a.rows) {
                r -= a.rows;
                kk++;
            }
        });
    }
    auto load_pieces = [&]() {
        if constexpr (COLS) {
            static_for<NP>([&](auto I) {
                if (I < a.rows) half_of[I] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(x_rsrc, (int)x_off + I * 1024, 0, 0);
            });
            x_off += (uint32_t)(kBlockK * 2) * (uint32_t)a.rows;
        } else {
            static_for<NP>([&](auto I) { piece[I] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(row_rsrc(wave + I * waves), (int)x_off, 0, 0)); });
            x_off += kBlockK * 2;
        }
    };
    auto store_pieces = [&](int buf) {
        static_for<NP>([&](auto I) {
            if constexpr (COLS) {
                if (I < a.rows)
                    *reinterpret_cast<lds_u32 *>(lds + buf * kFewBuf + half_at[I]) = ((uint32_t)half_of[I] * 0x10001u) ^ 0x00008000u;
            } else if (wave + I * waves < a.rows) {
                lds_byte *at = piece_at + buf * kFewBuf + I * waves * kFewPitch;
                const u32x4 v = piece[I];
                *reinterpret_cast<lds_u32x4 *>(at) = u32x4{minus_plus(v.x, sel_a), minus_plus(v.y, sel_a), minus_plus(v.z, sel_a), minus_plus(v.w, sel_a)};
                *reinterpret_cast<lds_u32x4 *>(at + to_other) = u32x4{minus_plus(v.x, sel_b), minus_plus(v.y, sel_b), minus_plus(v.z, sel_b), minus_plus(v.w, sel_b)};
            }
        });
    };

    float4v acc[2];   // output half: every plane's products, so that they cancel where the planes do (the top of this file)
    static_for<2>([&](auto H) { acc[H] = float4v{0.f, 0.f, 0.f, 0.f}; });
    const lds_byte *xlane = lds + kappa * kFewGroup + j * kFewPitch;
    uint32_t mask55 = 0x55555555u, high88 = 0x88888888u;   // in registers, so that the mask and the OR are one v_and_or_b32
    asm("" : "+s"(mask55));
    asm("" : "+v"(high88));
    constexpr int kAlwaysPlus = (int)0xddddddddu;

    load_pieces();
    load_scales(ts0);
    if constexpr (FINE) load_fine(ts0);
    load_signs(ts0, std::integral_constant<int, 0>{});
    {
        constexpr int slots = 4 * (kFewPitch / 16);   // of a row, all lane groups
        const int missing = (kBatchRows - a.rows) * 2 * slots;
        for (int i = tid; i < missing; i += waves * kLanes) {
            const int row = a.rows + i / (2 * slots), s = i % (2 * slots), group = s / (kFewPitch / 16);   // 0..7: both buffers
            *reinterpret_cast<lds_u32x4 *>(lds + group * kFewGroup + row * kFewPitch + (s % (kFewPitch / 16)) * 16) = u32x4{0u, 0u, 0u, 0u};
        }
    }
    store_pieces(0);
    if constexpr (FINE) {
        store_fine();
        read_word_scales(0, std::integral_constant<int, 0>{});
        static_for<NU>([&](auto U) {
            if constexpr (U / 2 < P) make_word_operand(U);
        });
    }
    __syncthreads();
    int buf = 0;
    for (int kb = ts0; kb < ts1; kb++) {
        const int next = kb + 1 < ts1 ? kb + 1 : ts0;   // past the end a tile that is there
        load_pieces();
        uint32_t sc[P];
        if constexpr (!FINE) static_for<P>([&](auto I) { sc[I] = scale[I]; });
        else load_fine(next);
        static_for<PG>([&](auto Pc) {
            constexpr int b0 = Pc * QP;
            u32x4 R[NU];   // sign bits of output j: word w are the 32 k 128 kappa + 32 w
            static_for<NU>([&](auto U) {
                if constexpr (b0 + U / 2 < Q) {
                    *stage_w = sign[U];
                    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(stage_r0);
                    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(stage_r1);
                    R[U] = u32x4{(uint32_t)lo.x, (uint32_t)lo.y, (uint32_t)hi.x, (uint32_t)hi.y};
                }
            });
            static_for<NU>([&](auto U) {
                constexpr int b = b0 + U / 2, number = (U % 2) * P + b;
                if constexpr (b < P && !FINE) {
                    const uint32_t s = __builtin_amdgcn_perm(sc[number / 2], sc[number / 2], number % 2 ? 0x03020302u : 0x01000100u);
                    A[U] = __builtin_bit_cast(half8, u32x4{s, s, s, s});
                }
            });
            if constexpr (Pc + 1 == PG) {
                load_scales(next);
                load_signs(next, std::integral_constant<int, 0>{});
            } else {
                load_signs(kb, std::integral_constant<int, (Pc + 1) % PG>{});
            }
            // Steps g: word w, parity p of k, half hh of the index register.  One index serves the two steps of (w, p).
            const lds_byte *xr = xlane + buf * kFewBuf;
            half16 B[AHEAD + 1];
            auto read_step = [&](auto Gc) {
                constexpr int w = Gc / 4, p = (Gc / 2) % 2, hh = Gc % 2;
                const lds_byte *at = xr + w * 128 + (2 * hh + p) * 32;
                const half8 b0 = *reinterpret_cast<const lds_half8 *>(at);
                const half8 b1 = *reinterpret_cast<const lds_half8 *>(at + 16);
                B[Gc % (AHEAD + 1)] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
            };
            static_for<AHEAD>(read_step);
            uint32_t index[2][NU], shifted[NU];
            static_for<NU>([&](auto U) {
                if constexpr (b0 + U / 2 < Q) index[0][U] = (R[U][0] & mask55) | high88;
            });
            __builtin_amdgcn_sched_barrier(0);
            static_for<16>([&](auto Gc) {
                constexpr int step = Gc, w = step / 4, p = (step / 2) % 2, hh = step % 2, pair = step / 2;
                constexpr int pass_next = w == 3 ? (Pc + 1) % PG : (int)Pc;   // whose word comes behind this one
                if constexpr (FINE && step % 4 == 0) {
                    if constexpr (w == 3 && Pc + 1 == PG) store_fine();
                    read_word_scales((w + 1) % 4, std::integral_constant<int, pass_next>{});
                }
                if constexpr (step + AHEAD < 16) read_step(std::integral_constant<int, (step + AHEAD < 16 ? step + AHEAD : 0)>{});
                __builtin_amdgcn_sched_barrier(0);
                static_for<NU>([&](auto U) {
                    constexpr int b = b0 + U / 2;
                    if constexpr (b < P) {
                        const int picks = b < Q ? (int)index[pair % 2][U] : kAlwaysPlus;
                        acc[U % 2] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A[U], B[step % (AHEAD + 1)], acc[U % 2], picks, 0, hh);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    // behind it one instruction of the next pair's indices: two per unit for odd k, one for even k
                    constexpr int slot = hh * NU + U;
                    if constexpr (p == 0) {
                        constexpr int u = slot / 2;
                        if constexpr (b0 + u / 2 < Q) {
                            if constexpr (slot % 2 == 0) shifted[u] = R[u][w] >> 1;
                            else index[(pair + 1) % 2][u] = (shifted[u] & mask55) | high88;
                        }
                    } else if constexpr (w < 3 && slot < NU) {
                        if constexpr (b0 + slot / 2 < Q) index[(pair + 1) % 2][slot] = (R[slot % NU][(w + 1) % 4] & mask55) | high88;
                    }
                    if constexpr (FINE && step % 4 == 3 && pass_next * QP + U / 2 < P) make_word_operand(U);   // its last use was this one
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
        });
        store_pieces(buf ^ 1);
        __syncthreads();   // the next activation block is in place; this one is no longer read
        buf ^= 1;
    }

    __half *y = reinterpret_cast<__half *>(a.y);
    const __half *bias = static_cast<const __half *>(g.bias);
    if (a.k_splits > 1 && !g.partials) {
        // One atomic per value.  Each 16 x 16 tile is turned through the staging area first, so that the lanes hold the outputs of
        // a row side by side (one cache line per row): acc[h][v] becomes activation row 4 kappa + v, output 16 h + j.
        typedef __attribute__((address_space(3))) float lds_float;
        lds_float *turn = reinterpret_cast<lds_float *>(stage);
        static_for<2>([&](auto H) {
            asm volatile("" ::: "memory");   // the reads before are done with (LDS operations of a wavefront execute in order)
            static_for<4>([&](auto V) { turn[(4 * kappa + V) * 16 + j] = acc[H][(int)V]; });
            asm volatile("" ::: "memory");
            acc[H] = *reinterpret_cast<__attribute__((address_space(3))) float4v *>(turn + j * 16 + 4 * kappa);
        });
        Arrival arrival[8];
        bool valid[8];
        unsigned long long *word[8];
        static_for<8>([&](auto I) {
            const int row = 4 * kappa + I % 4, out = nb * kBatch + 16 * (I / 4) + j;
            valid[I] = active && row < a.rows && out < a.n;
            word[I] = a.accum + (size_t)row * a.accum_row_stride + out;
            arrival[I] = arrive_output(acc[I / 4][I % 4], valid[I], word[I]);
        });
        // all answers are looked at before the first output is stored: a wait behind a store would wait for the store as well
        unsigned last = 0;
        static_for<8>([&](auto I) { last |= (unsigned)arrived_last(arrival[I], valid[I], a.k_splits) << I; });
        asm volatile("" : "+v"(last) : : "memory");
        static_for<8>([&](auto I) {
            const int row = 4 * kappa + I % 4, out = nb * kBatch + 16 * (I / 4) + j;
            if (last >> I & 1)
                finish_last(arrival[I], word[I], y + (size_t)row * a.y_row_stride + (size_t)out * a.y_stride, a.k_splits,
                            [&](float sum) { return bias ? plus_bias(sum, __half2float(bias[out])) : sum; });
        });
        return;
    }
    // acc[h][v]: activation row j, output nb * 32 + 16 h + 4 kappa + v
    if (!active || j >= a.rows) return;
    if (a.k_splits > 1 &&
        !sum_partials<2>(g.partials + (size_t)nb * a.k_splits * 512, reinterpret_cast<unsigned *>(a.accum + nb), ks, a.k_splits, lane,
                         [&](auto I) -> float4v & { return acc[I]; }))
        return;
    static_for<2>([&](auto H) {
        const int out = nb * kBatch + 16 * H + 4 * kappa;
        float4v &v = acc[H];
        if (bias)
            static_for<4>([&](auto V) {
                if (out + V < a.n) v[(int)V] = plus_bias(v[(int)V], __half2float(bias[out + V]));
            });
        __half *at = y + (size_t)j * a.y_row_stride + (size_t)out * a.y_stride;
        if (g.wide_y && out + 3 < a.n) {
            const __half2 lo = __floats2half2_rn(v[0], v[1]), hi = __floats2half2_rn(v[2], v[3]);
            *reinterpret_cast<uint2 *>(at) = uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
        } else {
            static_for<4>([&](auto V) {
                if (out + V < a.n) at[(size_t)V * a.y_stride] = __float2half_rn(v[(int)V]);
            });
        }
    });
}

template <int Q, bool OFF, FewInput IN, bool FINE>
__global__ __launch_bounds__(few_waves(Q + OFF, IN, FINE) * 64) void lut_few_kernel(MatvecArgs a, FewGrid g)
{
    few_workgroup<Q, OFF, IN, FINE>(a, g, blockIdx.x);
}

// A work list (like lut_matvec_multi_kernel): entry i owns the workgroups first_block[i] .. first_block[i + 1] - 1.  A kernel of its
// own beside the one for a single batch, since the larger kernel arguments cost a launch one to two microseconds.
template <int Q, bool OFF, FewInput IN, bool FINE>
__global__ __launch_bounds__(few_waves(Q + OFF, IN, FINE) * 64) void lut_few_multi_kernel(MultiMatvecArgs m, FewGrid g)
{
    int i = 0;
    while (i + 1 < m.count && (int)blockIdx.x >= m.first_block[i + 1]) i++;   // scalar: at most 31 steps
    few_workgroup<Q, OFF, IN, FINE>(m.entry[i], g, blockIdx.x - (unsigned)m.first_block[i]);
}

template <int Q, bool OFF, FewInput IN, bool FINE>
hipError_t allow_few_lds(const void *kernel, std::atomic<unsigned long long> &allowed)
{
    constexpr int W = few_waves(Q + OFF, IN, FINE);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (allowed.load(std::memory_order_relaxed) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, few_lds_bytes(W) + (FINE ? W * few_scale_area(Q + OFF) : 0));
    if (e == hipSuccess) allowed.fetch_or(bit, std::memory_order_relaxed);
    return e;
}

template <int Q, bool OFF, FewInput IN, bool FINE>
hipError_t launch_few_one(const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t stream)
{
    static std::atomic<unsigned long long> allowed{0};
    const hipError_t e = allow_few_lds<Q, OFF, IN, FINE>(reinterpret_cast<const void *>(&lut_few_kernel<Q, OFF, IN, FINE>), allowed);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((lut_few_kernel<Q, OFF, IN, FINE>), dim3((unsigned)(a.ntiles * a.k_splits)), dim3(waves * kLanes),
                       few_lds_bytes(waves) + (FINE ? waves * few_scale_area(Q + OFF) : 0), stream, a, g);
    return hipGetLastError();
}

// `workgroups`: of all entries
template <int Q, bool OFF, FewInput IN, bool FINE>
hipError_t launch_few_list(const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t stream)
{
    static std::atomic<unsigned long long> allowed{0};
    const hipError_t e = allow_few_lds<Q, OFF, IN, FINE>(reinterpret_cast<const void *>(&lut_few_multi_kernel<Q, OFF, IN, FINE>), allowed);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((lut_few_multi_kernel<Q, OFF, IN, FINE>), dim3((unsigned)workgroups), dim3(waves * kLanes),
                       few_lds_bytes(waves) + (FINE ? waves * few_scale_area(Q + OFF) : 0), stream, m, g);
    return hipGetLastError();
}

// launch(planes, offset) for the weight's
template <typename Launch>
hipError_t by_planes(int q, int has_offset, Launch launch)
{
    auto by_offset = [&](auto Qc) -> hipError_t { return has_offset ? launch(Qc, std::true_type{}) : launch(Qc, std::false_type{}); };
    switch (q) {
        case 1: return by_offset(std::integral_constant<int, 1>{});
        case 2: return by_offset(std::integral_constant<int, 2>{});
        case 3: return by_offset(std::integral_constant<int, 3>{});
        case 4: return by_offset(std::integral_constant<int, 4>{});
        case 5: return by_offset(std::integral_constant<int, 5>{});
        case 6: return by_offset(std::integral_constant<int, 6>{});
        case 7: return by_offset(std::integral_constant<int, 7>{});
        case 8: return by_offset(std::integral_constant<int, 8>{});
        default: return hipErrorInvalidValue;
    }
}

template <FewInput IN, bool FINE>
hipError_t launch_few_input(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t s)
{
    return by_planes(q, has_offset, [&](auto Qc, auto Off) { return launch_few_one<Qc, Off, IN, FINE>(a, g, waves, s); });
}

template <FewInput IN, bool FINE>
hipError_t launch_few_list_input(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t s)
{
    return by_planes(q, has_offset, [&](auto Qc, auto Off) { return launch_few_list<Qc, Off, IN, FINE>(m, g, workgroups, waves, s); });
}

}  // namespace
}  // namespace lutgemm_kernels
#endif
