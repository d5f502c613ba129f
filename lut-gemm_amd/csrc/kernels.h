// Launch interface between the C ABI host layer and the gfx950 kernels.
#ifndef LUTGEMM_KERNELS_H
#define LUTGEMM_KERNELS_H

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace lutgemm_kernels {

struct MatvecArgs {
    const uint8_t *signs;   // sign tiles (layout.h)
    const uint16_t *scales; // scale tiles (layout.h)
    const void *x;          // fp16 activations, contiguous, 16-byte aligned
    void *y;                // fp16 outputs, element j at y[j * y_stride]
    unsigned long long *accum;  // [rows][nb*32] split-k accumulators (count | flags | fixed-point sum), zero
                                // between launches; used when k_splits > 1 (launch_rows: only counts)
    int k, n;
    int ts, nb;             // k-blocks, output batches
    int ntiles;             // column tiles = ceil(nb / waves)
    int k_splits;           // workgroups along k
    int blocks_per_split;   // k-blocks per workgroup
    int y_stride;           // output j goes to y[j * y_stride]
    // rows == 2: a second activation row at x + x_row_stride goes to y + y_row_stride in the
    // same pass (strides in fp16 elements), with its accumulators at accum + accum_row_stride
    int rows;               // 1 or 2 activation rows (0 selects the read probe); 1..kBatchRows for launch_few and launch_batch
    long long x_row_stride, y_row_stride, accum_row_stride;
};

// Activation rows the kernel for few rows and the batch kernel take in one pass over the weight (rows r at x + r * x_row_stride
// go to y + r * y_row_stride, with split-k accumulators at accum + r * accum_row_stride).
constexpr int kBatchRows = 16;

// Up to kMaxFused independent one-row matvecs for one launch: entry i owns the workgroups
// first_block[i] .. first_block[i+1]-1 of the grid (the last entry up to the end).
constexpr int kMaxFused = 32;
struct MultiMatvecArgs {
    int count;
    int first_block[kMaxFused];
    MatvecArgs entry[kMaxFused];
};

// Device copies of the arrays a weight is created from (packer.h's layout) and the tiles to make of them.
struct PackArgs {
    const uint32_t *words;  // [k/32][q][n]
    const void *alpha;      // [groups][q][n], fp16 bits or fp32
    const void *offsets;    // [groups][n], null for a weight without
    int halves;             // the scales are fp16 bits
    uint8_t *signs;
    uint16_t *scales;
    int k, n, q, gsub, group_size, ts, nb;
};

struct DequantArgs {
    const uint8_t *signs;
    const uint16_t *scales;
    void *out;              // fp16 [k][n] or [n][k]
    int k, n, q, has_offset, gsub, ts;
    int transposed;
};

// workgroups = ntiles * k_splits, `waves` wavefronts of 64 lanes per workgroup.  `bias` (one row only): fp16 [n] added to
// the rounded sum of an output, which is rounded again.
hipError_t launch_matvec(int q, int has_offset, int gsub, const MatvecArgs &a, int workgroups,
                         int waves, hipStream_t stream, const void *bias = nullptr);

// entries that all have one row or all have two, sharing q, has_offset, gsub and the wavefronts per workgroup
hipError_t launch_matvec_multi(int q, int has_offset, int gsub, const MultiMatvecArgs &m, int workgroups, int waves,
                               hipStream_t stream);

// 1..kBatchRows activation rows in one pass (matrix cores), any number of planes up to kBatchMaxPlanes.
// A workgroup has kBatchWavesMin .. kBatchWaves wavefronts: wavefront w stages activation rows w and
// w + wavefronts, so eight cover the 16 rows of a pass.  A tile of more than kBatchWidePlanes planes
// needs more than 128 registers per lane, so such weights run with exactly kBatchWavesMin wavefronts
// (which may then use 256 registers each).
constexpr int kBatchMaxPlanes = 8;
constexpr int kBatchWidePlanes = 4;
constexpr int kBatchWaves = 16;
constexpr int kBatchWavesMin = 8;
// LDS of a workgroup of the batch kernel: two activation blocks of 17 rows of 2064 bytes (every
// activation as the pair -x, +x), and per wavefront a 1 KiB staging area plus the scales of its tile
// for the matrix lanes (64 bytes per (scale group of the k-block, plane or offset)).  A compute
// unit has 160 KiB, which bounds the wavefronts of a workgroup when there are four groups per 128 k.
constexpr int batch_scale_area_bytes(int gsub, int qo) { return 256 * gsub * qo; }
constexpr int batch_lds_bytes(int waves, int gsub, int qo)
{
    return 2 * 17 * 2064 + waves * (1024 + batch_scale_area_bytes(gsub, qo));
}
constexpr int batch_waves_max(int gsub, int q, int qo)
{
    int w = q > kBatchWidePlanes ? kBatchWavesMin : kBatchWaves;
    while (w > kBatchWavesMin && batch_lds_bytes(w, gsub, qo) > 160 * 1024) w--;
    return w;
}
static_assert(batch_lds_bytes(kBatchWavesMin, 4, kBatchMaxPlanes + 1) <= 160 * 1024, "LDS of a compute unit");
hipError_t launch_batch(int q, int has_offset, int gsub, const MatvecArgs &a, int workgroups, int waves, hipStream_t stream);
// A work list of independent batches in one launch: entries sharing q, has_offset, gsub and the
// wavefronts per workgroup, each with 1..kBatchRows rows and its own ntiles / k_splits / blocks_per_split;
// workgroups = sum of the entries' ntiles * k_splits, entry i starting at first_block[i].
hipError_t launch_batch_multi(int q, int has_offset, int gsub, const MultiMatvecArgs &m, int workgroups, int waves,
                              hipStream_t stream);

// 3 to kBatchRows activation rows (few_body.h): kFewWavesMin .. few_waves_max
// wavefronts per workgroup (two planes and fewer take 128 registers per lane, three 168, more up to 256; one plane less each with
// scale groups of 32 and 64 k), one output batch
// each; with activations as columns (x [k][rows]) exactly kFewWavesMin.
constexpr int kFewWavesMin = 8;
constexpr int few_waves_max(int planes, int gsub)
{
    return gsub == 1 ? (planes <= 2 ? 16 : planes == 3 ? 12 : 8) : planes == 1 ? 16 : planes == 2 ? 12 : 8;
}
// a quarter of an activation row of a k-block, every value as the pair (-x, +x), with 16 bytes of padding; the sign staging of
// a wavefront; two activation blocks and the staging of all wavefronts
constexpr int kFewPitch = 4 * 128 + 16, kFewStage = 1024;
constexpr int few_lds_bytes(int waves) { return 2 * 4 * kBatchRows * kFewPitch + waves * kFewStage; }
// and, for scale groups of 32 and 64 k, the scales of a wavefront's tile
constexpr int few_scale_area(int planes) { return 1024 * planes; }
static_assert(few_lds_bytes(16) + 16 * few_scale_area(1) <= 160 * 1024 && few_lds_bytes(12) + 12 * few_scale_area(2) <= 160 * 1024 &&
              few_lds_bytes(8) + 8 * few_scale_area(kBatchMaxPlanes + 1) <= 160 * 1024, "LDS of a compute unit");
struct FewGrid {
    const void *bias;  // fp16 [n] added to the rounded sum of an output, which is rounded again; null for none
    float *partials;   // k_splits > 1: 512 floats per (output batch, split) (no initial value); counts in accum[batch]
    int columns;       // x is [k][rows]
    int wide_y;        // four neighbouring outputs of a row are 8-byte aligned in y
    int gsub;          // scale groups per 128 k: 1, 2 or 4
};
hipError_t launch_few(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t stream);
hipError_t launch_few_two_rows(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t stream);   // rows > waves
hipError_t launch_few_columns(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, hipStream_t stream);
hipError_t launch_few_fine(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t stream);   // gsub > 1
hipError_t launch_few_fine_two_rows(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t stream);
// A work list of independent batches in one launch, as launch_batch_multi; sums of a k-split go through the accumulators
// (g.partials null), and activations come as rows.
hipError_t launch_few_multi(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t stream);
hipError_t launch_few_multi_two_rows(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t stream);
hipError_t launch_few_fine_multi(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t stream);
hipError_t launch_few_fine_multi_two_rows(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t stream);
hipError_t launch_few_fine_columns(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, hipStream_t stream);

// Many activation rows in one launch (rows_body.h): a workgroup of kRowsWaves wavefronts takes 16 rt rows and
// kRowsWaves / kw output batches, its wavefronts in kw groups that share out the k-blocks; row_chunks workgroups share
// a weight tile.  `planes` is q, one more with an offset (1 to 9); rt kRowsTilesMin .. kRowsTilesMax; kw 1 or 2.
constexpr int kRowsWaves = 8;
constexpr int kRowsTilesMin = 2, kRowsTilesMax = 4;
struct RowsGrid {
    int row_chunks;
    int q, gsub;
    const void *bias;  // fp16 [n] added to the rounded sum of an output, which is rounded again; null for none
    float *partials;   // k_splits > 1: partial sums (no initial value)
    int wide_y;   // four neighbouring outputs of a row are 8-byte aligned in y
};
// words of 32 k (for each of the four lane groups) that are staged in LDS at a time
constexpr int rows_stage_words(int rt) { return rt == 2 ? 2 : 1; }
// bytes of a quarter of one activation row of a stage: every value as the pair (-x, +x), 16 bytes of padding
constexpr int rows_pitch(int rt) { return rows_stage_words(rt) * 128 + 16; }
// rows staged by a k group: whole rounds of its wavefronts
constexpr int rows_staged(int rt, int kw)
{
    const int per_round = kRowsWaves / kw * 64 / (16 * rows_stage_words(rt));
    return (16 * rt + per_round - 1) / per_round * per_round;
}
// LDS of a workgroup: two stage buffers per k group and the sign staging of its wavefronts
constexpr int rows_lds_bytes(int rt, int kw) { return kw * 2 * 4 * rows_staged(rt, kw) * rows_pitch(rt) + kRowsWaves * 1024; }
static_assert(rows_lds_bytes(2, 2) <= 160 * 1024 && rows_lds_bytes(3, 2) <= 160 * 1024 && rows_lds_bytes(4, 2) <= 160 * 1024, "LDS of a compute unit");
hipError_t launch_rows(int planes, int rt, int kw, const MatvecArgs &a, const RowsGrid &g, hipStream_t stream);
hipError_t launch_rows_two_groups(int planes, int rt, const MatvecArgs &a, const RowsGrid &g, hipStream_t stream);   // kw == 2

// words[0..count) = 0 (a fill kernel rather than a memset node, so that it can be captured)
hipError_t launch_fill_zero(unsigned long long *words, size_t count, hipStream_t stream);

// Split-k words of the allocation-free entry point: a static device array of kStaticSplitKWords
// 64-bit words (8 MiB on every device the library runs on, enough for 65,536 outputs per
// activation row of a pass of kBatchRows rows), zero at load and zero again after every completed
// launch; and the room for the partial sums of launch_rows (16 MiB, as much as any plan needs).
// static_workspace gives their device addresses on `device`, which must be the current device (0 <= device <
// kMaxDevices); looked up once per device.
constexpr size_t kStaticSplitKWords = (size_t)1 << 20, kStaticPartials = (size_t)1 << 22;
struct StaticWorkspace {
    unsigned long long *words;
    float *partials;
};
constexpr int kMaxDevices = 64;
hipError_t static_workspace(int device, StaticWorkspace *out);

// y [m][n] += bias [n], fp16
hipError_t launch_add_bias(void *y, const void *bias, int m, int n, hipStream_t stream);

// fp16 [k][m] -> [m][k]
hipError_t launch_gather_columns(const void *cols, void *rows, int k, int m, hipStream_t stream);

// hipErrorInvalidValue for a weight beyond the kernels' grids (2^31 threads)
hipError_t launch_pack(const PackArgs &a, hipStream_t stream);

// *found = 1 if one of the halves in 16 * `pieces` bytes is an infinity or a NaN, else as it was
hipError_t launch_find_non_finite(const uint16_t *halves, size_t pieces, unsigned long long *found, hipStream_t stream);

hipError_t launch_dequantize(const DequantArgs &a, hipStream_t stream);

// The matvec's loads without its arithmetic (same grid and arguments; x, y and accum unused):
// nothing is written.
hipError_t launch_read_probe(int q, int has_offset, int gsub, const MatvecArgs &a, int workgroups, int waves,
                             hipStream_t stream);

// Dense fp16 comparator: y[n] = sum_k W^T[n][k] x[k]; k a multiple of 8, pointers 16-byte aligned.
hipError_t launch_dense_gemv(const void *wt, const void *x, void *y, int k, int n, int compute_units,
                             hipStream_t stream);

}  // namespace lutgemm_kernels
#endif
