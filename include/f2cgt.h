/*
 * f2cgt.h — C ABI of libf2cgt_hip.so: hand-written gfx950 (MI355X) kernels for the
 * fused feature-decompression + neighbour-aggregation path of F2CGT.
 *
 * Conventions
 *   - every pointer is a DEVICE pointer to a dense row-major buffer unless stated;
 *   - `stream` is a hipStream_t passed as void* (NULL = the null stream); every call
 *     only enqueues work on that stream: no device-wide synchronisation, no host
 *     read-back, no allocation (outputs are caller-allocated);
 *   - return value 0 = success, < 0 = rejected arguments (F2CGT_E_*), > 0 = hipError_t
 *     of a failed launch; f2cgt_last_error() gives the message of the calling thread's
 *     last failure;
 *   - dtype arguments take the F2CGT_DT_* tags below;
 *   - CSC = indptr[num_rows + 1], indices[num_edges], both of `idx_dtype`
 *     (F2CGT_DT_I32 or F2CGT_DT_I64).  Source ids are clamped to [0, num_src_rows) and
 *     edge offsets to [0, num_edges], so malformed graphs give wrong sums, not faults.
 *
 * Each entry point names the reference interface (file:line under the reference
 * checkout) whose device work it replaces.
 */
#ifndef F2CGT_H_
#define F2CGT_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
  F2CGT_DT_U8 = 0,
  F2CGT_DT_I8 = 1,
  F2CGT_DT_I16 = 2,
  F2CGT_DT_I32 = 3,
  F2CGT_DT_I64 = 4,
  F2CGT_DT_F16 = 5,
  F2CGT_DT_F32 = 6,
  F2CGT_DT_F64 = 7
};

enum {
  F2CGT_OK = 0,
  F2CGT_E_INVALID = -1,     /* bad size / null pointer / misaligned buffer */
  F2CGT_E_UNSUPPORTED = -2, /* dtype, target_bits or shape the kernels do not cover */
  F2CGT_E_DEVICE = -3       /* no usable gfx950 device */
};

enum { F2CGT_METRIC_L2 = 0, F2CGT_METRIC_COSINE = 1 };

/* Library version (major * 100 + minor). */
int f2cgt_version(void);

/* Message of the calling thread's most recent failure ("" if none). */
const char* f2cgt_last_error(void);

/* Number of compute units of the current device (the kernels size their grids by it). */
int f2cgt_num_cus(void);

/* How the row-block aggregation kernels (the SQ and affine-SQ fused operators) write their output
 * (no counterpart in the reference, whose kernels use plain stores, src/fusion_spmm.cu:173-236).
 *   F2CGT_STORE_AUTO    (default) outputs above 220 MB (above 140 MB when the output rows are whole
 *                       128-byte lines or the graph has six or more edges per row) are streamed past
 *                       the caches with non-temporal stores, smaller ones are written with plain stores
 *   F2CGT_STORE_STREAM  always streamed: the launch time no longer depends on what the caches hold
 *   F2CGT_STORE_CACHED  never streamed
 * Plain stores are fastest when the same output buffer is written again before the last-level cache
 * (256 MB) has been turned over, as in a loop over one buffer; a caller whose outputs are written
 * once and consumed later (a training step with other large kernels in between) is better off
 * streaming.  The fused VQ operator streams its output, in whole lines, in every mode.
 * Results are identical in every mode.  Process-wide; returns the previous mode, or
 * F2CGT_E_INVALID for a value that is none of the three (the mode is then unchanged). */
#define F2CGT_STORE_AUTO 0
#define F2CGT_STORE_STREAM 1
#define F2CGT_STORE_CACHED 2
int f2cgt_set_store_mode(int mode);

/* Dry runs of the fused aggregation entry points (no counterpart in the reference; for tests and
 * tools that want to know what a shape dispatches to, with or without a GPU).  While switched on
 * for the calling thread, f2cgt_spmm_csr and the f2cgt_*_spmm_csr operators validate their
 * arguments and choose kernel and launch geometry exactly as usual, then return 0 without touching
 * the device or dereferencing any pointer (pointers only need the alignment of the real buffers;
 * the device is taken to have 256 compute units).  f2cgt_last_plan copies the last choice:
 * grid / block / lds_bytes of the launch, destination rows per workgroup (0 = not row-blocked),
 * and kernel-specific numbers in aux[]: lane-group counts (every one of them must be >= 1 for the kernel's
 * loops to advance); of vq_wave_kernel the float4 per lane and edge, the rows of a mini-block, 1 where the columns are no
 * multiple of four and 1 where codes are read byte by byte.  f2cgt_set_plan_only returns the previous setting. */
typedef struct {
  char kernel[48];
  int64_t grid;
  int32_t block;
  int64_t lds_bytes;
  int32_t rows_per_block;
  int32_t aux[4];
} f2cgt_plan;
int f2cgt_set_plan_only(int on);
int f2cgt_last_plan(f2cgt_plan* out);

/* ---- bit packing ------------------------------------------------------------- */

/* Replaces packbits(), src/packbits.cu:44-64 (kernel :6-42).
 * unpack uint8 [rows, unpack_dim] -> pack uint8 [rows, ceil(unpack_dim / (8/bits))];
 * element i of a group goes to bits [bits*i, bits*(i+1)); target_bits in {1,2,4}. */
int f2cgt_packbits(const uint8_t* unpack, uint8_t* pack, int64_t rows, int64_t unpack_dim,
                   int target_bits, void* stream);

/* Replaces unpackbits(), src/packbits.cu:96-114 (kernel :66-94).
 * pack uint8 [rows, pack_dim] -> unpack uint8 [rows, unpack_dim]. */
int f2cgt_unpackbits(const uint8_t* pack, uint8_t* unpack, int64_t rows, int64_t pack_dim,
                     int64_t unpack_dim, int target_bits, void* stream);

/* ---- scalar quantisation (log domain, the reference's SQ) ---------------------- */

/* Replaces sq_compress(), src/sq_quantization.cu:65-83 (kernel :5-63).
 * src fp32 [rows, feat_dim] -> dst fp32 [rows, feat_dim] of integer-valued codes;
 * codebooks fp32 [num_codebooks, 5] = fmin,fmax,emin,emax,mean; column j uses
 * codebook j / column_slice; target_bits in {1,2,4,8,16}. */
int f2cgt_sq_compress(const float* src, float* dst, const float* codebooks, int64_t rows,
                      int64_t feat_dim, int64_t num_codebooks, int target_bits,
                      int64_t column_slice, void* stream);

/* One-pass form of the three calls every caller of sq_compress() makes next
 * (examples/process_compress.py:128-139: sq_compress -> cast -> packbits): writes the storage
 * tensor directly.  dst: uint8 [rows, ceil(feat_dim * bits / 8)] packed low bits first for
 * bits in {1,2,4}; int8 [rows, feat_dim] for 8; int16 [rows, feat_dim] for 16.  Bit for bit what
 * f2cgt_sq_compress + integer cast + f2cgt_packbits give. */
int f2cgt_sq_encode(const float* src, void* dst, const float* codebooks, int64_t rows,
                    int64_t feat_dim, int64_t num_codebooks, int target_bits, int64_t column_slice,
                    void* stream);

/* Replaces sq_decompress(), src/sq_quantization.cu:158-182 (kernel :85-156).
 * codes [rows, src_dim] of code_dtype (U8/I8 packed bytes for bits < 8, I8 for 8, I16 for 16)
 * -> out fp32 [rows, feat_dim].  Codebook per OUTPUT column.  8-bit codes are signed; U8 with
 * target_bits 8 is refused (F2CGT_E_UNSUPPORTED): the reference's dtype dispatch
 * (src/common.h:68-82) would read such a tensor as 0..255, which its encoder never writes. */
int f2cgt_sq_decompress(const void* codes, int code_dtype, float* out, const float* codebooks,
                        int64_t rows, int64_t src_dim, int64_t feat_dim,
                        int64_t num_codebooks, int target_bits, int64_t column_slice,
                        void* stream);

/* Per-column affine SQ decode (no counterpart in the reference; defined by the
 * benchmark configurations): out[r][c] = params[c] + code * params[feat_dim_stride + c]
 * with params fp32 [2, param_stride] (row 0 = min, row 1 = scale), unsigned codes,
 * sub-byte codes packed low bits first; target_bits in {1,2,4,8}. */
int f2cgt_sq_affine_decompress(const uint8_t* codes, float* out, const float* params,
                               int64_t param_stride, int64_t rows, int64_t src_dim,
                               int64_t feat_dim, int target_bits, void* stream);

/* ---- vector quantisation decode ---------------------------------------------- */

/* Replaces vq_decompress(), src/vq_quantization.cu:35-60 (kernel :5-33).
 * codes [rows, num_codebooks] (U8/I8/I16), codebooks [num_codebooks, K, width]
 * (F32 or F16) -> out fp32 [rows, feat_dim], feat_dim <= num_codebooks * width. */
int f2cgt_vq_decompress(const void* codes, int code_dtype, const void* codebooks, int cb_dtype,
                        float* out, int64_t rows, int64_t feat_dim, int64_t num_codebooks,
                        int64_t K, int64_t width, void* stream);

/* ---- CSC mean aggregation ---------------------------------------------------- */

/* Replaces SpMMCsr(), src/fusion_spmm.cu:45-70 (kernel :13-43).
 * feat [num_src_rows, feat_dim] of feat_dtype (F32/F16/F64) -> out same dtype
 * [num_rows, feat_dim]; out[r] = sum(feat[indices[e]]) / max(deg, 1). */
int f2cgt_spmm_csr(const void* feat, int feat_dtype, void* out, const void* indptr,
                   const void* indices, int idx_dtype, int64_t num_rows, int64_t num_edges,
                   int64_t num_src_rows, int64_t feat_dim, void* stream);

/* Replaces VqDecompressSpMMFusionCsr(), src/fusion_spmm.cu:107-141 (kernel :72-105,
 * decode src/cuda_utils.cuh:48-58).  fp32 codebooks; out fp32 [num_rows, feat_dim]. */
int f2cgt_vq_decompress_spmm_csr(const void* codes, int code_dtype, const float* codebooks,
                                 const void* indptr, const void* indices, int idx_dtype,
                                 float* out, int64_t num_rows, int64_t num_edges,
                                 int64_t num_src_rows, int64_t feat_dim,
                                 int64_t num_codebooks, int64_t K, int64_t width,
                                 void* stream);

/* Replaces SqDecompressSpMMFusionCsr(), src/fusion_spmm.cu:240-272 (kernel :143-238).
 * Codebook per PACKED BYTE (:180): byte j uses codebook j*(8/bits) / column_slice, which
 * equals the per-column choice of f2cgt_sq_decompress iff column_slice % (8/bits) == 0.
 * Code dtypes as for f2cgt_sq_decompress (8-bit codes must be I8). */
int f2cgt_sq_decompress_spmm_csr(const void* codes, int code_dtype, const float* codebooks,
                                 const void* indptr, const void* indices, int idx_dtype,
                                 float* out, int64_t num_rows, int64_t num_edges,
                                 int64_t num_src_rows, int64_t src_dim, int64_t feat_dim,
                                 int64_t num_codebooks, int target_bits, int64_t column_slice,
                                 void* stream);

/* Fused per-column affine SQ decode + mean aggregation (benchmark-defined extension;
 * argument order follows f2cgt_sq_decompress_spmm_csr). */
int f2cgt_sq_affine_decompress_spmm_csr(const uint8_t* codes, const float* params,
                                        int64_t param_stride, const void* indptr,
                                        const void* indices, int idx_dtype, float* out,
                                        int64_t num_rows, int64_t num_edges,
                                        int64_t num_src_rows, int64_t src_dim,
                                        int64_t feat_dim, int target_bits, void* stream);

/* Two-table fused decode + mean aggregation (benchmark-defined extension; the reference's
 * two-level mode, examples/compress.py:39-54,74-106, never mixes tables in one call).
 * row_map int32 [num_src_rows]: m >= 0 -> row m of the 8-bit affine SQ table
 * (sq_codes uint8 [num_sq_rows, feat_dim], sq_params fp32 [2, param_stride]);
 * m < 0 -> row -m-1 of the VQ table (vq_codes uint8 [num_vq_rows, num_codebooks],
 * vq_codebooks fp32 [num_codebooks, K, width]). */
int f2cgt_hybrid_decompress_spmm_csr(const int32_t* row_map, const uint8_t* sq_codes,
                                     const float* sq_params, int64_t param_stride,
                                     const uint8_t* vq_codes, const float* vq_codebooks,
                                     const void* indptr, const void* indices, int idx_dtype,
                                     float* out, int64_t num_rows, int64_t num_edges,
                                     int64_t num_src_rows, int64_t num_sq_rows,
                                     int64_t num_vq_rows, int64_t feat_dim,
                                     int64_t num_codebooks, int64_t K, int64_t width,
                                     void* stream);

/* ---- row fetch in front of the operators -------------------------------------- */

/* Replaces TensorCache.__getitem__, examples/tensor_cache.py:49-58: shmtensor.capi.uva_fetch
 * (slot_map NULL) and shmtensor.capi.cache_fetch (hot table + id -> slot map; the reference
 * keeps a GPU hash map, examples/tensor_cache.py:80-86, here a dense int32 array).
 * Tables hold opaque rows of row_bytes bytes each (code rows or plain feature rows).
 * out[i, :] = hot[slot_map[id], :] if slot_map && 0 <= slot_map[id] < num_hot_rows
 *            else table[id, :],   id = index[i] clamped to [0, num_rows).
 * `table` may be pinned host memory mapped into the device address space (its rows then
 * cross the host link); hot, slot_map [num_rows], index [num_index] and out
 * [num_index, row_bytes] are device buffers.  No alignment is required of any of them. */
int f2cgt_fetch_rows(const void* table, const void* hot, const int32_t* slot_map,
                     const void* index, int idx_dtype, void* out, int64_t num_index,
                     int64_t row_bytes, int64_t num_rows, int64_t num_hot_rows, void* stream);

/* Decode through a row list: out[i] = the decoded row index[i] of a table in device memory, as f2cgt_fetch_rows followed
 * by f2cgt_vq_decompress / f2cgt_sq_decompress, without the copy of the code rows.  F2CGT_E_UNSUPPORTED, with nothing
 * launched, for the shapes left to those (the caller falls back).
 * f2cgt_vq_decompress_rows: uint8 codes [num_rows, num_codebooks], fp32 codebooks; widths that divide 128 (4 and more),
 * K <= 256, even feat_dim >= 64, at least 1024 rows, out 16-byte aligned.
 * f2cgt_sq_decompress_rows: 1, 2, 4 or 8-bit codes, even feat_dim from 8 to 8192, out 16-byte aligned, the decode table
 * in LDS.  slot_map (int32 [num_slots], may be NULL): row slot_map[index[i]] instead; an id below zero counts from the end
 * of the map.  bad (int32, device-accessible host memory, may be NULL; zero on entry): 1 when the map has no row
 * (a negative entry) for an id, 2 when an id lies outside it; such rows are decoded from some row of the table. */
int f2cgt_vq_decompress_rows(const uint8_t* table, const void* index, int idx_dtype, const float* codebooks, float* out,
                             int64_t num_index, int64_t num_rows, int64_t feat_dim, int64_t num_codebooks, int64_t K,
                             int64_t width, void* stream);
int f2cgt_sq_decompress_rows(const void* table, int code_dtype, const void* index, int idx_dtype, const int32_t* slot_map,
                             int64_t num_slots, int32_t* bad, const float* codebooks, float* out, int64_t num_index,
                             int64_t num_rows, int64_t src_dim, int64_t feat_dim, int64_t num_codebooks, int target_bits,
                             int64_t column_slice, void* stream);

/* ---- codebook statistics ------------------------------------------------------- */

/* The statistics behind an SQ codebook (examples/process_compress.py:45-68), of the absolute values of every column
 * slice of a sample: x fp32 [num_rows, cols] with row stride ld; rows int64 [m] (device) lists the sample's rows (negative
 * ones count from the end; others outside the table are clamped to it and reported), NULL takes rows [0, m).  ranks (host,
 * 8 values): four ranks (0 = smallest) among the m * column_slice values of a full slice, then four among those of the
 * last slice.  out fp64 [ceil(cols / column_slice), 6] (device): the exact |x| at the four ranks, the sum of |x| (fp64),
 * and the sum of 1 when a NaN was among the values and 2 when rows held an id outside the table.  workspace: device scratch, 256-byte aligned, contents irrelevant. */
int64_t f2cgt_abs_order_stats_workspace_bytes(int64_t m, int64_t cols, int64_t column_slice);
int f2cgt_abs_order_stats(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                          int64_t column_slice, const int64_t* ranks, void* workspace, int64_t workspace_bytes,
                          double* out, void* stream);

/* The same with the SQ codebooks themselves (fp32 [slices, 5] on the device: fmin, fmax, emin, emax, mean): ranks below and
 * above the lower percentile, then those of the upper one; weights (host, 4 values): how far each percentile lies from its
 * rank below to the one above, in a full slice and in the last one.  The log2 are correctly rounded. */
int f2cgt_sq_codebooks(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                       int64_t column_slice, const int64_t* ranks, const float* weights, void* workspace,
                       int64_t workspace_bytes, double* stats, float* codebooks, void* stream);
/* The same; the first kernel also sets *bad_row (host memory that the device can write, e.g. hipHostMalloc'ed, cleared by the
 * caller) where an id of rows lies outside the table, and the event `checked` (a hipEvent_t) is recorded behind it, so that a
 * caller can wait for the ids alone. */
int f2cgt_sq_codebooks_checked(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                               int64_t column_slice, const int64_t* ranks, const float* weights, void* workspace,
                               int64_t workspace_bytes, double* stats, float* codebooks, int32_t* bad_row, void* checked,
                               void* stream);

/* ---- VQ encode ---------------------------------------------------------------- */

/* Replaces pairwise_distance(), src/kmeans.cu:102-118 (raft L2Unexpanded /
 * CosineExpanded).  x fp32 [m,k], y fp32 [n,k] -> dist fp32 [m,n]; metric L2 is the
 * squared distance sum((x-y)^2). */
int f2cgt_pairwise_distance(const float* x, const float* y, float* dist, int64_t m, int64_t n,
                            int64_t k, int metric, void* stream);

/* Replaces KMeans::predict(), src/kmeans.cu:77-98 (raft kmeans_predict) and the argmin
 * the callers run on pairwise_distance (examples/my_kmeans.py:116-125).
 * x fp32 [m,k], centers fp32 [n,k], n <= 65536.  Writes the index of the nearest centre
 * (first minimum) to labels_i64 [m] and/or labels_u8 [m] (either may be NULL; labels_u8
 * needs n <= 256).  The distance matrix is never materialised.  Cosine: the nearest by direction; the 1e-8 below which
 * f2cgt_pairwise_distance does not let |x||y| fall counts only between centres whose directions are equally near to
 * rounding. */
int f2cgt_kmeans_predict(const float* x, const float* centers, int64_t* labels_i64,
                         uint8_t* labels_u8, int64_t m, int64_t n, int64_t k, int metric,
                         void* stream);

/* Codes of a whole feature table in one launch: column slice s (columns [s k, s k + k) of the rows; the last slice may
 * have fewer, which count as zeros) against its own centres, as f2cgt_kmeans_predict labels it
 * (examples/process_compress.py:234-292, one slice at a time).  x: row r starts ldx floats after row r - 1, ldx >=
 * feat_dim; codebooks fp32 [slices, n, k]; codes uint8, row r at r * code_stride, code_stride >= slices.
 * f2cgt_vq_encode_slices_covers: 1 where the shape is taken (n <= 256, k <= 64, centres within 96 KB of LDS), else 0. */
int f2cgt_vq_encode_slices_covers(int64_t n, int64_t k);
int f2cgt_vq_encode_slices(const float* x, int64_t ldx, int64_t feat_dim, const float* codebooks, uint8_t* codes,
                           int64_t code_stride, int64_t m, int64_t slices, int64_t n, int64_t k, int metric, void* stream);

/* One Lloyd iteration's centre update, after f2cgt_kmeans_predict has produced the labels.
 * Replaces the update half of the reference's two training loops: compute_new_centers and the
 * centre-shift test of examples/my_kmeans.py:87-113,128-147 (plain mean whatever the metric, a centre
 * without members keeps its value) and the loop inside raft::cluster::kmeans::fit, src/kmeans.cu:61-75.
 * x fp32 [m,k]; labels int64 [m] or uint8 [m] (exactly one non-NULL; values clamped to [0,n));
 * centers fp32 [n,k], updated in place; shift fp32 [2] (device) receives sum_c |dc| and sum_c |dc|^2.
 * stop (device int32, may be NULL): when it is nonzero on entry the call does nothing, and the call
 * sets it when stop_rule says the centres are final (1: sum_c |dc|^2 < tol, raft's rule; 2:
 * (sum_c |dc|)^2 < tol, the rule of examples/my_kmeans.py:105; 0: never) -- a training loop can then
 * run without reading anything back per iteration.  workspace: device scratch for the partial sums,
 * f2cgt_kmeans_update_workspace_bytes(n, k) bytes, 16-byte aligned, contents irrelevant (4 (n k + n) bytes, rounded up
 * to 256, are enough for the form that adds into one set of sums, which is slower for most shapes that ask for more).
 * The sums are fp32.  With one set of them all rows are added atomically, in device memory; with a set per workgroup the
 * rows of a workgroup are, in LDS, and the sets are then added in a fixed order.  Either way the last bits depend on the
 * order the hardware takes the atomic adds in. */
int64_t f2cgt_kmeans_update_workspace_bytes(int64_t n, int64_t k);
int f2cgt_kmeans_update(const float* x, const int64_t* labels_i64, const uint8_t* labels_u8, float* centers,
                        float* shift, int32_t* stop, int stop_rule, float tol, void* workspace,
                        int64_t workspace_bytes, int64_t m, int64_t n, int64_t k, void* stream);

/* f2cgt_kmeans_update without a workspace and without any allocation (no counterpart in the
 * reference: it is for callers that cannot allocate device memory -- code under HIP graph capture,
 * tight serving loops, harnesses that forbid hipMalloc).  The partial sums live in a device array
 * inside the library (272 KB per device, kept until the process ends), so the problem is limited to
 * n * k <= 65536 sums and n <= 4096 centres; larger ones return F2CGT_E_UNSUPPORTED.  Same arguments,
 * results and stop-flag behaviour as f2cgt_kmeans_update.  Every call on a device uses that device's
 * one array: calls that overlap on one GPU (two streams, two threads) race; calls on one stream do not.
 * The first call on each device looks the array's address up (hipGetSymbolAddress, which may load
 * the code object): make that first call outside any stream capture; later calls only launch kernels. */
int f2cgt_kmeans_update_static(const float* x, const int64_t* labels_i64, const uint8_t* labels_u8,
                               float* centers, float* shift, int32_t* stop, int stop_rule, float tol,
                               int64_t m, int64_t n, int64_t k, void* stream);

/* Codebook training of all column slices of a sample at once (examples/process_compress.py:147-182, one slice at a time).
 *
 * f2cgt_slice_rows: the sample, slice by slice.  x: row r starts ld floats after row r - 1; rows int64 [m] (NULL: rows
 * [0, m)), negative ids count from the end; slice s has the columns [s k, s k + k), zeros after the last one (k <= 64).
 * out fp32 [slices, m, k]; norms fp32 [m, slices]; bad_row (device int32): set where an id lies outside the table (the row
 * read is then another one of it).
 *
 * f2cgt_keep_rows: which rows take part, the ones at least as long as a quantile of their slice's lengths.  stats fp64
 * [slices, 6] as f2cgt_abs_order_stats leaves them for norms: the lengths below and above the quantile and, last, flags
 * (a slice with NaN keeps no row); weight, weight_last: where between the two it lies (of a slice, and of the last one).
 * keep uint32 [slices, ceil(m / 32)]: bit r % 32 of word r / 32.
 *
 * f2cgt_kmeans_slices_step: one Lloyd iteration of every slice whose stop flag is zero, as f2cgt_kmeans_predict and
 * f2cgt_kmeans_update would make it from the rows kept: x fp32 [slices, m, k], keep as above or NULL (all), centers fp32
 * [slices, n, k] updated in place, stop int32 [slices] (device) with stop_rule and tol as in f2cgt_kmeans_update,
 * and 3 where no row takes part.  A label
 * is the true first minimum.  Sums: a workgroup's rows in fp64 (LDS), each workgroup's set rounded to fp32 once, the sets
 * added in fp64 in a fixed order.
 * workspace: f2cgt_kmeans_slices_workspace_bytes, 16-byte aligned.  f2cgt_kmeans_slices_covers: 1 where the shape is
 * taken (operands and sums of a slice in LDS, up to 256 slices, 512 centres, 64 columns), else 0. */
int f2cgt_slice_rows(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols, int64_t k,
                     float* out, float* norms, int32_t* bad_row, void* stream);
int f2cgt_keep_rows(const float* norms, const double* stats, float weight, float weight_last, int64_t m, int64_t slices,
                    uint32_t* keep, void* stream);
int f2cgt_kmeans_slices_covers(int64_t slices, int64_t n, int64_t k);
int64_t f2cgt_kmeans_slices_workspace_bytes(int64_t m, int64_t slices, int64_t n, int64_t k);
int f2cgt_kmeans_slices_step(const float* x, const uint32_t* keep, float* centers, int32_t* stop, int stop_rule, float tol,
                             void* workspace, int64_t workspace_bytes, int64_t m, int64_t slices, int64_t n, int64_t k,
                             int metric, void* stream);
/* out [slices, n, k] = every centre divided by its length and multiplied by its slice's mean length
 * (examples/process_compress.py:16-18).  flags int32 [slices + 2] (device): word `slices` becomes *bad_row (device; NULL: is
 * left), word slices + 1 is set where a value of out is no number; the others are left alone. */
int f2cgt_kmeans_rescale(const float* centers, float* out, int64_t n, int64_t k, int64_t slices, const int32_t* bad_row,
                         int32_t* flags, void* stream);

/* The dense part of a GraphSAGE layer (examples/conv.py:68-76) at the sizes of a minibatch, fp32 throughout.
 *
 * f2cgt_sage_linear: out[m, n] = x0 w0^T + x1 w1^T + bias, through max(., 0) where relu is nonzero (a NaN stays one).
 * x0 [m, k0], w0 [n, k0], x1 [m, k1], w1 [n, k1], bias [n] or NULL, all dense; k0 and k1 multiples of four and the buffers
 * 16-byte aligned (others: F2CGT_E_UNSUPPORTED).
 *
 * f2cgt_sage_linear_grad: dw0 = g^T x0, dw1 = g^T x1, db = column sums of g, each left out where NULL, with g = grad, or
 * (out given: the values f2cgt_sage_linear wrote with relu) grad where out is not <= 0 and 0 elsewhere.  The sums are made
 * in a fixed order.  workspace: f2cgt_sage_linear_grad_workspace_bytes (0 up to 1024 rows), contents irrelevant. */
int f2cgt_sage_linear(const float* x0, const float* w0, const float* x1, const float* w1, const float* bias, float* out,
                      int64_t m, int64_t n, int64_t k0, int64_t k1, int relu, void* stream);
int64_t f2cgt_sage_linear_grad_workspace_bytes(int64_t m, int64_t n, int64_t k0, int64_t k1);
int f2cgt_sage_linear_grad(const float* grad, const float* out, const float* x0, const float* x1, float* dw0, float* dw1,
                           float* db, void* workspace, int64_t workspace_bytes, int64_t m, int64_t n, int64_t k0, int64_t k1,
                           void* stream);
/* Which of the two a caller with a library's products beside them takes: bits of F2CGT_SAGE_FORWARD (f2cgt_sage_linear in a
 * pass that is not differentiated), F2CGT_SAGE_STEP (f2cgt_sage_linear in a pass whose gradients f2cgt_sage_linear_grad makes)
 * and F2CGT_SAGE_GRAD (f2cgt_sage_linear_grad).  The first two are set only where f2cgt_sage_linear adds in the order in
 * which rocBLAS and hipBLASLt of ROCm 7.0 were seen to. */
#define F2CGT_SAGE_FORWARD 1
#define F2CGT_SAGE_STEP 2
#define F2CGT_SAGE_GRAD 4
int f2cgt_sage_linear_ahead(int64_t m, int64_t n, int64_t k0, int64_t k1);

#ifdef __cplusplus
}
#endif
#endif /* F2CGT_H_ */
