// gfx950 kernel for many activation rows (17 and more) against a packed BCQ weight in one launch.
//
// The contraction is the batch kernel's (batch_body.h): v_smfmac_f32_16x16x64_f16 with every activation in LDS as the
// pair (-x, +x) and the sign bits as the index registers.  What differs is what many rows make worthwhile:
//  * A sign vector is transposed and turned into index registers once and contracted with RT = 2 to 4 row tiles of
//    16 rows (a workgroup of the batch kernel has one, so a call of m rows read and transposed the weight m / 16 times).
//  * The scales are the matrix operand (fp16, exact), where the batch kernel uses 1.0 and multiplies afterwards: with RT row tiles
//    the multiplications, and a set of partial accumulators for each plane, would cost more than the matrix unit
//    loses by operands that vary (measured: 1.67 against 1.90 PFLOP/s of signed sums).  Sums are fp32 throughout, products
//    of two fp16 numbers are exact in them, so a result differs from the batch kernel's by fp32 rounding only.
//  * The chunks of a lane group kappa are the 128 k of row kappa of the tile (layout.h): word w of a lane are the 32
//    consecutive k 128 kappa + 32 w, which belong to one scale group whatever its size, so an operand of a lane is one scale
//    repeated, and one kernel serves every group size.  An offset is one more plane, whose signs are all plus.
//  * LDS reads of a step run a step ahead (the compiler keeps counted waits), global loads a stage ahead.
//  * A matrix instruction holds the vector unit of its SIMD for 16 cycles and takes one other vector instruction for nothing,
//    every further one in 4 cycles (few_body.h), so indices and activations are made one instruction behind each matrix
//    instruction, and addresses are scalar (buffer loads).
// What bounds it: power.  7168 x 7168, 3 planes, 256 rows (RT = 2, KW = 1): 4.8 million matrix instructions in 73 to 75 us; a loop of
// nothing but them with such operands takes 50 us on the whole device (10.7 ns each and SIMD, 6.9 on a few compute units), and
// the compute units that the plan leaves idle, start and end the rest.  Before the instructions were spread: 82 to 89 us; 12288 x
// 12288, 3 planes, 48 rows (RT = 3, five splits): 58 -> 49 us.  The launch replaced 16 of the batch kernel: 257 us.
// Tried: a staging area for each sign vector, written a pass ahead and read when the words before are done with, so that no
// transposition is waited for: no faster.
// Registers: up to 256 (two wavefronts share a SIMD).  One instance spills: P = 8, RT = 4, KW = 2 (36 bytes per lane).
//
// A workgroup is eight wavefronts, each with one batch of 32 outputs; KW = 2 makes them two groups of four that share out
// the k-blocks and add their sums through LDS at the end (more workgroups for a narrow weight, no exchange between them).
// Splits along k beyond that exchange their sums through memory (sum_partials).
#ifndef LUTGEMM_ROWS_BODY_H
#define LUTGEMM_ROWS_BODY_H

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
typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) half8 lds_half8;
typedef __attribute__((address_space(3))) v2i lds_v2i;

constexpr int kStageBytes = 1024;   // per wavefront: one sign vector of a tile

// P planes (an offset counts as one whose signs are all plus), RT row tiles of 16 activation rows per workgroup,
// KW groups of wavefronts that take every KW-th k-block.
template <int P, int RT, int KW>
__global__ __launch_bounds__(kRowsWaves * 64) void lut_rows_kernel(MatvecArgs a, RowsGrid g)
{
    constexpr int PG = (P + 3) / 4;            // passes over the planes of a k-block
    constexpr int QP = (P + PG - 1) / PG;      // planes per pass
    constexpr int NU = 2 * QP;                 // sign vectors per pass: plane b, output half h -> 2 b + h
    constexpr int NW = kRowsWaves / KW;        // output batches of the workgroup
    constexpr int WS = rows_stage_words(RT);   // words of 32 k per lane group staged at a time
    constexpr int PITCH = rows_pitch(RT);
    constexpr int ROWS = NW * 64 / (16 * WS);               // rows the wavefronts of a k group stage at a time
    constexpr int PIECES = (16 * RT + ROWS - 1) / ROWS;     // 16-byte pieces of a stage per thread
    constexpr int GROUP = rows_staged(RT, KW) * PITCH;      // bytes of a lane group's share of a stage
    constexpr int XBUF = 4 * GROUP;
    constexpr bool SPREAD = PIECES < 4;   // activations are converted between the matrix instructions (four pieces: registers)
    static_assert(GROUP % 256 == 0, "no shift of the banks from group to group");
    static_assert(PIECES * ROWS == rows_staged(RT, KW), "kernels.h states the LDS of this kernel");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_generic[];
    lds_byte *lds = (lds_byte *)lds_generic;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / NW, nw = wave % NW;       // k group, output batch of this wavefront
    const int kappa = lane >> 4, j = lane & 15;

    // the row chunks of one weight tile follow each other on one XCD (workgroups go round robin over the eight)
    const unsigned xcd = blockIdx.x & 7u, local = blockIdx.x >> 3;
    const unsigned rc = local % (unsigned)g.row_chunks, tile_id = (local / (unsigned)g.row_chunks) * 8u + xcd;
    if (tile_id >= (unsigned)(a.ntiles * a.k_splits)) return;
    const int ntile = (int)(tile_id % (unsigned)a.ntiles), ks = (int)(tile_id / (unsigned)a.ntiles);
    const int row0 = (int)rc * (16 * RT);
    const int nb = ntile * NW + nw;
    const bool active = nb < a.nb;
    const int ts0 = ks * a.blocks_per_split, ts1 = min(ts0 + a.blocks_per_split, a.ts);
    const int iterations = (ts1 - ts0 + KW - 1) / KW;

    const size_t tile0 = (size_t)(active ? nb : 0) * a.ts;
    constexpr int kBufferFlags = 0x00020000;   // 32-bit elements, offsets in bytes

    lds_byte *xbuf = lds + (size_t)kw * 2 * XBUF;
    lds_byte *stage = lds + (size_t)KW * 2 * XBUF + wave * kStageBytes;

    // sign staging: lane c writes its 16 bytes (outputs 0..15 of chunk c) to a slot; ds_read_b64_tr_b8 hands lane
    // (kappa, j) the bytes of output j for eight chunks.  Chunks 16 kappa + 4 w .. + 3 make word w of the lane.
    lds_u32x4 *stage_w = reinterpret_cast<lds_u32x4 *>(stage + 16 * (lane ^ ((lane >> 1) & 8)));
    const int r_off = 256 * kappa + 8 * j;
    lds_v2i *stage_r0 = reinterpret_cast<lds_v2i *>(stage + (r_off ^ ((kappa & 1) * 128)));
    lds_v2i *stage_r1 = reinterpret_cast<lds_v2i *>(stage + ((r_off + 128) ^ ((kappa & 1) * 128)));

    // scales of output j (both halves) for the group of word w, in bytes
    const int subl = 16 / g.gsub, lh = 2 * g.gsub * P;
    const int sc_lane = 2 * ((kappa * 16 + j % subl) * lh + (j / subl) * P), sc_sub = 2 * subl * lh, sc_h = 2 * g.gsub * P;
    const bool one_group = g.gsub == 1;   // of a lane in a tile: the four words have the same scales

    // Activation pieces (16 bytes: one chunk of one row) of this thread.  Rows beyond the batch read its last row: a row
    // is a column of the matrix product, and theirs are never stored; k beyond the weight reads zero (an offset beyond the
    // buffer).  A wavefront moves, per piece, the 16 chunks of one
    // word w in four rows: lane bits 0-1 the byte of the word, 2-3 the row, 4-5 the lane group kappa of the chunk.
    // In LDS a stage is [B lane group kb][row][w][step][half of the B operand], 16 bytes each: chunk (kappa, byte) is
    // in half kappa / 2 of lane group 2 (kappa % 2) + byte % 2, for the steps of byte / 2.  The rows' pitch shifts their
    // 16-byte slots (of the 256 bytes the LDS banks span), the lane groups lie whole multiples of 256 bytes apart, so
    // the 16 lanes a read serves together, which differ in the row, hit 16 slots.  Rows 0, 1, 8 and 9 of a
    // write and the parity its lanes start with are chosen so that a write does, too.
    const int c_byte = lane & 3, c_kappa = lane >> 4;
    const int piece_w = nw % WS, piece_row = 16 * (nw / (4 * WS)) + 2 * ((nw / WS) & 3) + ((lane >> 2) & 1) + (lane & 8);
    const int piece_k = (16 * c_kappa + 4 * piece_w + c_byte) * kChunk;
    auto piece_row_step = [](int i) constexpr { return 16 * (i * NW / (4 * WS)) + 2 * ((i * NW / WS) & 3); };
    const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc(   // of this workgroup's rows: at most 64 of 2^24 halves, 2^31 bytes
        (void *)(reinterpret_cast<const __half *>(a.x) + (size_t)row0 * (size_t)a.x_row_stride), (short)0,
        (int)((uint32_t)min(a.rows - row0, 16 * RT) * (uint32_t)a.x_row_stride * 2u), kBufferFlags);
    uint32_t piece_off[PIECES];   // of the row, in bytes
    static_for<PIECES>([&](auto I) {
        piece_off[I] = (uint32_t)min(piece_row + piece_row_step(I), a.rows - 1 - row0) * (uint32_t)a.x_row_stride * 2u;
    });
    const int first = c_byte & 1;
    const uint32_t sel_a = first ? 0x03020302u : 0x01000100u, sel_b = first ? 0x01000100u : 0x03020302u;
    lds_byte *piece_at = xbuf + (2 * (c_kappa & 1) + (c_byte & 1)) * GROUP + piece_row * PITCH + piece_w * 128 + (c_byte >> 1) * 64 +
                         (c_kappa >> 1) * 16 + 32 * first;
    const int to_other = 32 - 64 * first;
    u32x4 piece[PIECES];
    // words w0 .. w0 + WS - 1 of k-block kb
    auto load_pieces = [&](int kb, int w0) {
        const int kpos = kb * kBlockK + 32 * w0 + piece_k, limit = kb < ts1 ? a.k : 0;
        const uint32_t at = (uint32_t)kpos * 2u, beyond = kpos < limit ? 0u : 0xffffff00u;
        static_for<PIECES>([&](auto I) {
            piece[I] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, (int)((piece_off[I] + at) | beyond), 0, 0));
        });
    };
    // A piece becomes a 16-byte block of each parity of k, [-x, +x] x 4: instruction N of 16 for piece I (with a write behind the
    // eighth and the last)
    constexpr int PIECE_OPS = 16;
    uint32_t block[PIECES][4];
    auto piece_op = [&](auto I, auto N, int buf) {
        constexpr int second = N / 8, d = (N % 8) / 2;
        if constexpr (N % 2 == 0) block[I][d] = __builtin_amdgcn_perm(piece[I][d], piece[I][d], second ? sel_b : sel_a);
        else block[I][d] ^= 0x00008000u;
        if constexpr (N % 8 == 7)
            *reinterpret_cast<lds_u32x4 *>(piece_at + buf * XBUF + piece_row_step(I) * PITCH + (second ? to_other : 0)) =
                u32x4{block[I][0], block[I][1], block[I][2], block[I][3]};
    };
    auto store_pieces = [&](int buf) {
        static_for<PIECES * PIECE_OPS>([&](auto N) { piece_op(std::integral_constant<int, N / PIECE_OPS>{}, std::integral_constant<int, N % PIECE_OPS>{}, buf); });
    };

    float4v acc[2][RT];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int t = 0; t < RT; t++) acc[h][t] = float4v{0.f, 0.f, 0.f, 0.f};

    const int xlane = kappa * GROUP + j * PITCH;
    uint32_t mask55 = 0x55555555u, high88 = 0x88888888u;
    asm("" : "+s"(mask55));
    asm("" : "+v"(high88));

    auto block_of = [&](int it) {   // k-block of this wavefront's iteration `it`, a valid one past the end
        const int kb = ts0 + it * KW + kw;
        return kb < ts1 ? kb : ts0;
    };
    const auto sign_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(a.signs + tile0 * (size_t)(2 * g.q * kUnitBytes)), (short)0, -1, kBufferFlags);
    const auto scale_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(a.scales + tile0 * (size_t)(kLanes * lh)), (short)0, -1, kBufferFlags);
    u32x4 sign[NU];
    auto load_signs = [&](int kb, auto Pc) {
        static_for<NU>([&](auto U) {
            constexpr int unit = Pc * NU + U;
            if constexpr (unit < 2 * P)
                sign[U] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(sign_rsrc, lane * 16, (kb * 2 * g.q + (unit < 2 * g.q ? unit : 0)) * kUnitBytes, 2));
        });
    };
    uint32_t scale[NU];   // raw scales of the units whose operands are made next
    auto load_scales = [&](int kb, int w, auto Pc) {
        const int at = kb * (2 * kLanes * lh) + (w * g.gsub / 4) * sc_sub;
        static_for<NU>([&](auto U) {
            constexpr int b = Pc * QP + U / 2, h = U % 2;
            if constexpr (b < P) scale[U] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(scale_rsrc, sc_lane, at + h * sc_h + 2 * b, 0);
        });
    };
    half8 A[NU];
    auto make_operands = [&](uint32_t vmask, auto Pc) {
        static_for<NU>([&](auto U) {
            if constexpr (Pc * QP + U / 2 < P) {
                const uint32_t s = scale[U] * vmask;
                A[U] = __builtin_bit_cast(half8, u32x4{s, s, s, s});
            }
        });
    };
    // signs of the last plane when that is the offset
    const uint32_t all_plus = g.q < P ? 0xffffffffu : 0u;

    load_pieces(ts0 + kw, 0);
    load_signs(block_of(0), std::integral_constant<int, 0>{});
    load_scales(block_of(0), 0, std::integral_constant<int, 0>{});
    store_pieces(0);
    __syncthreads();

    int buf = 0;
    for (int it = 0; it < iterations; it++) {
        const int kb = ts0 + it * KW + kw;
        const int cur = block_of(it), next = block_of(it + 1);
        const uint32_t vmask = kb < ts1 ? 0x10001u : 0u;
        static_for<PG>([&](auto Pc) {
            constexpr int pg = Pc, b0 = pg * QP;
            constexpr int ACTIVE = 2 * (P - b0 < QP ? P - b0 : QP);   // units of this pass
            constexpr bool last_pass = pg + 1 == PG;
            constexpr int pg_next = (pg + 1) % PG;
            make_operands(vmask, Pc);
            // this pass's sign bits of output j, refill of the registers behind it
            u32x4 R[NU];
            static_for<NU>([&](auto U) {
                constexpr int b = b0 + U / 2;
                if constexpr (b < P) {
                    *stage_w = sign[U];
                    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(stage_r0);
                    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(stage_r1);
                    R[U] = u32x4{(uint32_t)lo.x, (uint32_t)lo.y, (uint32_t)hi.x, (uint32_t)hi.y};
                    if constexpr (b == P - 1) {
                        R[U].x |= all_plus;
                        R[U].y |= all_plus;
                        R[U].z |= all_plus;
                        R[U].w |= all_plus;
                    }
                }
            });
            // Index registers.  With two row tiles those of the next pair of steps are made while one is contracted; with more,
            // those of the next unit, again for each step of a pair (two of them at a time, so that the registers do).
            constexpr bool BY_UNIT = RT > 2;
            uint32_t index[2][BY_UNIT ? 1 : NU], shifted;
            auto even_index = [&](auto U, auto W) { return (R[U][(int)W] & mask55) | high88; };
            static_for<BY_UNIT ? 1 : ACTIVE>([&](auto U) { index[0][U] = even_index(U, std::integral_constant<int, 0>{}); });
            static_for<4 / WS>([&](auto Sc) {
                constexpr int w0 = Sc * WS;
                constexpr bool last_stage = w0 + WS == 4;
                // the activations of the next stage
                if constexpr (!last_stage) load_pieces(kb, w0 + WS);
                else if constexpr (!last_pass) load_pieces(kb, 0);
                else load_pieces(kb + KW, 0);
                if constexpr (Sc == 0) load_signs(last_pass ? next : cur, std::integral_constant<int, pg_next>{});
                const lds_byte *xr = xbuf + buf * XBUF + xlane;
                half16 B[2][RT];
                // step: word, parity p of k, half hh of the index register; one index serves the two steps of (w, p)
                auto read_step = [&](auto Gc) {
                    constexpr int wl = Gc / 4, p = (Gc / 2) % 2, hh = Gc % 2;
                    static_for<RT>([&](auto T) {
                        const lds_byte *at = xr + T * (16 * PITCH) + wl * 128 + (2 * hh + p) * 32;
                        const half8 b0 = *reinterpret_cast<const lds_half8 *>(at);
                        const half8 b1 = *reinterpret_cast<const lds_half8 *>(at + 16);
                        B[Gc % 2][T] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
                    });
                };
                read_step(std::integral_constant<int, 0>{});
                __builtin_amdgcn_sched_barrier(0);
                static_for<4 * WS>([&](auto Gc) {
                    constexpr int w = w0 + Gc / 4, p = (Gc / 2) % 2, hh = Gc % 2, pair = 2 * w + p;
                    constexpr bool last_word = w == 3, stage_end = Gc / 4 == WS - 1;
                    if constexpr (Gc % 4 == 0) {   // scales of the next word
                        if constexpr (!last_word) {
                            if (!one_group) load_scales(cur, w + 1, Pc);
                        } else {
                            load_scales(last_pass ? next : cur, 0, std::integral_constant<int, pg_next>{});
                        }
                    }
                    if constexpr (Gc + 1 < 4 * WS) read_step(std::integral_constant<int, (Gc + 1 < 4 * WS ? Gc + 1 : 0)>{});
                    __builtin_amdgcn_sched_barrier(0);   // the reads of the next step go out ahead of this one's products
                    static_for<ACTIVE * RT>([&](auto Sl) {
                        constexpr int U = Sl / RT, T = Sl % RT;
                        const int picks = (int)(BY_UNIT ? index[U % 2][0] : index[pair % 2][BY_UNIT ? 0 : U]);
                        acc[U % 2][T] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A[U], B[Gc % 2][T], acc[U % 2][T], picks, 0, hh);
                        __builtin_amdgcn_sched_barrier(0);
                        // Behind each matrix instruction one other, for nothing: the indices (for even k one instruction, for odd k
                        // two), and in the last steps of a stage the next stage's activations.
                        constexpr int step_slots = BY_UNIT ? ACTIVE * (RT - 2) : ACTIVE * RT;
                        constexpr int made = BY_UNIT || last_word || p == 0 ? 0 : ACTIVE;   // slots of the pair taken by indices
                        constexpr int slot = hh * step_slots + (BY_UNIT ? U * (RT - 2) + T - 2 : Sl);
                        if constexpr (BY_UNIT) {
                            constexpr bool wraps = U + 1 == ACTIVE;   // the next unit is the first one of the next step
                            constexpr int nu = wraps ? 0 : U + 1, np = wraps && hh ? 1 - p : p, nw_ = wraps && hh && p ? w + 1 : w;
                            if constexpr (nw_ < 4) {
                                if constexpr (np == 0 && T == 0) index[nu % 2][0] = even_index(std::integral_constant<int, nu>{}, std::integral_constant<int, nw_ % 4>{});
                                if constexpr (np == 1 && T == 0) shifted = R[nu][nw_ % 4] >> 1;
                                if constexpr (np == 1 && T == 1) index[nu % 2][0] = (shifted & mask55) | high88;
                            }
                        } else if constexpr (p == 0) {
                            if constexpr (slot < 2 * ACTIVE) {
                                if constexpr (slot % 2 == 0) shifted = R[slot / 2 % NU][w] >> 1;
                                else index[(pair + 1) % 2][slot / 2 % NU] = (shifted & mask55) | high88;
                            }
                        } else if constexpr (slot < made) {
                            index[(pair + 1) % 2][slot % NU] = even_index(std::integral_constant<int, slot % NU>{}, std::integral_constant<int, (w + 1) % 4>{});
                        }
                        if constexpr (SPREAD && p == 1 && stage_end && (BY_UNIT ? T >= 2 : slot >= made)) {
                            constexpr int total = PIECES * PIECE_OPS, slots = 2 * step_slots - made, per = (total + slots - 1) / slots;
                            static_for<per>([&](auto N) {
                                constexpr int n = (slot - made) * per + N;
                                if constexpr (n < total) piece_op(std::integral_constant<int, n / PIECE_OPS>{}, std::integral_constant<int, n % PIECE_OPS>{}, buf ^ 1);
                            });
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    if constexpr (Gc % 4 == 3 && !last_word) {
                        if (!one_group) make_operands(vmask, Pc);
                    }
                });
                if constexpr (!SPREAD) store_pieces(buf ^ 1);
                __syncthreads();
                buf ^= 1;
            });
        });
    }

    // acc[h][t][v]: activation row row0 + 16 t + j, output nb * 32 + 16 h + 4 kappa + v
    if constexpr (KW == 2) {   // the second k group hands its sums over (the activation buffers are free)
        lds_byte *hand = lds + (size_t)nw * (RT * 2 * 1024) + lane * 16;
        if (kw == 1)
            static_for<2 * RT>([&](auto I) { *reinterpret_cast<__attribute__((address_space(3))) float4v *>(hand + I * 1024) = acc[I % 2][I / 2]; });
        __syncthreads();
        if (kw == 1) return;
        static_for<2 * RT>([&](auto I) { acc[I % 2][I / 2] += *reinterpret_cast<__attribute__((address_space(3))) float4v *>(hand + I * 1024); });
    }
    if (!active) return;
    if (a.k_splits > 1) {
        // sums over the workgroups of the tile in the order of their k ranges, by the wavefront that comes last
        const size_t unit = ((size_t)rc * a.nb + nb) * a.k_splits;
        if (!sum_partials<2 * RT>(g.partials + unit * (2 * RT * 256), reinterpret_cast<unsigned *>(a.accum + ((size_t)rc * a.nb + nb)), ks,
                                  a.k_splits, lane, [&](auto I) -> float4v & { return acc[I % 2][I / 2]; }))
            return;
    }
    __half *y = reinterpret_cast<__half *>(a.y);
    if (g.bias)
        static_for<8>([&](auto I) {
            constexpr int h = I / 4, v = I % 4;
            const int out = nb * kBatch + 16 * h + 4 * kappa + v;
            const float bias = out < a.n ? __half2float(static_cast<const __half *>(g.bias)[out]) : 0.f;
#pragma unroll
            for (int t = 0; t < RT; t++) acc[h][t][v] = plus_bias(acc[h][t][v], bias);
        });
    static_for<2 * RT>([&](auto I) {
        constexpr int h = I % 2, t = I / 2;
        const int row = row0 + 16 * t + j, out = nb * kBatch + 16 * h + 4 * kappa;
        if (row >= a.rows) return;
        __half *at = y + (size_t)row * a.y_row_stride + (size_t)out * a.y_stride;
        if (g.wide_y && out + 3 < a.n) {
            const __half2 lo = __floats2half2_rn(acc[h][t][0], acc[h][t][1]), hi = __floats2half2_rn(acc[h][t][2], acc[h][t][3]);
            *reinterpret_cast<uint2 *>(at) = uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (out + v < a.n) at[(size_t)v * a.y_stride] = __float2half_rn(acc[h][t][v]);
        }
    });
}

template <int P, int RT, int KW>
hipError_t launch_rows_one(const MatvecArgs &a, const RowsGrid &g, hipStream_t stream)
{
    static std::atomic<unsigned long long> allowed{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (!(allowed.load(std::memory_order_relaxed) & bit)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&lut_rows_kernel<P, RT, KW>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                rows_lds_bytes(RT, KW));
        if (e != hipSuccess) return e;
        allowed.fetch_or(bit, std::memory_order_relaxed);
    }
    const unsigned blocks = (unsigned)div_up(a.ntiles * a.k_splits, 8) * 8u * (unsigned)g.row_chunks;
    hipLaunchKernelGGL((lut_rows_kernel<P, RT, KW>), dim3(blocks), dim3(kRowsWaves * kLanes), rows_lds_bytes(RT, KW), stream, a, g);
    return hipGetLastError();
}

template <int P, int KW>
hipError_t launch_rows_p(int rt, const MatvecArgs &a, const RowsGrid &g, hipStream_t s)
{
    switch (rt) {
        case 2: return launch_rows_one<P, 2, KW>(a, g, s);
        case 3: return launch_rows_one<P, 3, KW>(a, g, s);
        case 4: return launch_rows_one<P, 4, KW>(a, g, s);
        default: return hipErrorInvalidValue;
    }
}

template <int KW>
hipError_t launch_rows_kw(int planes, int rt, const MatvecArgs &a, const RowsGrid &g, hipStream_t s)
{
    switch (planes) {
        case 1: return launch_rows_p<1, KW>(rt, a, g, s);
        case 2: return launch_rows_p<2, KW>(rt, a, g, s);
        case 3: return launch_rows_p<3, KW>(rt, a, g, s);
        case 4: return launch_rows_p<4, KW>(rt, a, g, s);
        case 5: return launch_rows_p<5, KW>(rt, a, g, s);
        case 6: return launch_rows_p<6, KW>(rt, a, g, s);
        case 7: return launch_rows_p<7, KW>(rt, a, g, s);
        case 8: return launch_rows_p<8, KW>(rt, a, g, s);
        case 9: return launch_rows_p<9, KW>(rt, a, g, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace lutgemm_kernels
#endif
