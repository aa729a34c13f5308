// One Lloyd iteration's centre update (codebook training), after the assignment kernel of
// assign.hip has produced the labels:
//   sums[c]   = sum of the rows assigned to centre c,  count[c] = how many
//   centre[c] = sums[c] / count[c]   (a centre without members keeps its value)
//   shift     = how far the centres moved, in the two forms the reference's two trainers test
// Follows examples/my_kmeans.py:128-147 (compute_new_centers: plain mean whatever the metric,
// empty clusters keep the previous centre) and :100-111 (centre shift and stopping rule);
// raft's kmeans::fit (src/kmeans.cu:61-75) stops on the squared form of the same shift.
//
// The partial sums are scratch memory beyond inputs and outputs.  f2cgt_kmeans_update takes them from a
// workspace the caller passes: up to 256 workgroups each leave their own n * k sums and n counters there, which
// one workgroup per centre adds up, moves the centre and counts itself in; the last one to arrive decides about
// the stop.  f2cgt_kmeans_update_static uses a device array of this file (for callers that cannot allocate),
// which has room for one set of sums: all workgroups add into it in memory, as they do from a workspace where a
// set per workgroup does not pay (km_by_parts).
//
// f2cgt_kmeans_slices_step makes the whole iteration of several column slices in two launches, of the kernel that labels
// (assign.hip) and of one that merges; slice_rows and keep_rows make its input.  Eight iterations of six slices of 16
// columns, 150 000 rows, 256 centres, with a sort for each slice's quantile: 4.65 ms slice by slice, 0.75 now (of it
// the steps 0.52, the sample's slices 0.02, their quantiles 0.06).
#include "assign.hpp"

namespace f2cgt {
namespace {

constexpr int kKmThreads = 256;
constexpr int kKmLdsFloats = 12 * 1024;   // per-workgroup partial sums kept in LDS up to this many entries
constexpr int kKmParts = 256;             // sets of partial sums in a workspace: one workgroup per CU
constexpr int kKmPartThreads = 1024;
constexpr int kKmBatch = 8;               // values per thread in flight
constexpr int kKmMergeThreads = 1024;

// Scratch of the allocation-free entry point: 65536 sums and 4096 counters, 272 KB that every device
// the library runs on holds until the process ends.  The name is a host-side stand-in, not a device
// address: host code only ever uses the pointer hipGetSymbolAddress returns for the current device.
constexpr int64_t kStaticSums = 65536;
constexpr int64_t kStaticCenters = 4096;
static __device__ __align__(256) unsigned char scratch[(kStaticSums + kStaticCenters) * 4];

struct KmArgs {
  const float* x;
  const int64_t* labels_i64;
  const uint8_t* labels_u8;
  float* centers;
  float* shift;         // [2]: sum_c |dc|, sum_c |dc|^2
  int32_t* stop;        // may be null; nonzero = the centres are final, the step does nothing (1: rule met, 2: shift is NaN)
  float* sums;          // [n * k]
  uint32_t* counts;     // [n]
  int64_t m;
  int n, k;
  int rule;             // 0: never stop; 1: stop when sum |dc|^2 < tol; 2: stop when (sum |dc|)^2 < tol
  float tol;
  int rows_per_block;
};

__device__ __forceinline__ bool km_stopped(const KmArgs& a) { return a.stop != nullptr && *a.stop != 0; }

__global__ __launch_bounds__(kKmThreads) void km_clear_kernel(KmArgs a) {
  if (km_stopped(a)) return;
  const int64_t words = (int64_t)a.n * a.k + a.n;
  uint32_t* w = reinterpret_cast<uint32_t*>(a.sums);   // sums and counts are one block of the scratch
  for (int64_t i = (int64_t)blockIdx.x * kKmThreads + threadIdx.x; i < words; i += (int64_t)gridDim.x * kKmThreads)
    w[i] = 0u;
  if (blockIdx.x == 0 && threadIdx.x < 2) a.shift[threadIdx.x] = 0.f;
}

// fp32 add in memory: the LDS unit's own add, or the L2's (device memory: never a compare-and-swap loop)
template <bool LDS>
__device__ __forceinline__ void add_f32(float* p, float v) {
  if (LDS) atomicAdd(p, v);
  else unsafeAtomicAdd(p, v);
}

__device__ __forceinline__ int km_label(const KmArgs& a, int64_t row) {
  const int64_t l = a.labels_i64 ? a.labels_i64[row] : (int64_t)a.labels_u8[row];
  return (int)(l < 0 ? 0 : (l >= a.n ? a.n - 1 : l));
}

// A workgroup adds its rows into partial sums (LDS when n * k fits, else straight into the
// scratch) and then adds the partial sums into the scratch.
template <bool LDS>
__global__ __launch_bounds__(kKmThreads) void km_accumulate_kernel(KmArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (km_stopped(a)) return;
  float* s_sum = reinterpret_cast<float*>(smem);
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_sum + (LDS ? a.n * a.k : 0));
  const int entries = a.n * a.k;
  if (LDS) {
    for (int i = threadIdx.x; i < entries + a.n; i += kKmThreads) reinterpret_cast<uint32_t*>(smem)[i] = 0u;
    __syncthreads();
  }
  const int64_t row0 = (int64_t)blockIdx.x * a.rows_per_block;
  const int64_t left = a.m - row0;
  const int nrows = (int)(left < a.rows_per_block ? left : a.rows_per_block);
  const int64_t items = (int64_t)nrows * a.k;
  float* sums = LDS ? s_sum : a.sums;
  uint32_t* counts = LDS ? s_cnt : a.counts;
  for (int64_t e = threadIdx.x; e < items; e += kKmThreads) {
    const int r = (int)(e / a.k), col = (int)(e - (int64_t)r * a.k);
    const int c = km_label(a, row0 + r);
    add_f32<LDS>(sums + c * a.k + col, a.x[(row0 + r) * a.k + col]);
    if (col == 0) atomicAdd(counts + c, 1u);
  }
  if (LDS) {
    __syncthreads();
    for (int i = threadIdx.x; i < entries; i += kKmThreads) {
      const float v = s_sum[i];
      if (v != 0.f) add_f32<false>(a.sums + i, v);
    }
    for (int i = threadIdx.x; i < a.n; i += kKmThreads) {
      const uint32_t v = s_cnt[i];
      if (v != 0u) atomicAdd(a.counts + i, v);
    }
  }
}

// One wave per centre: the new centre, and its share of the shift.
__global__ __launch_bounds__(kKmThreads) void km_finalize_kernel(KmArgs a) {
  if (km_stopped(a)) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int c = blockIdx.x * (kKmThreads / kWave) + (threadIdx.x / kWave);
  if (c >= a.n) return;
  const uint32_t cnt = a.counts[c];
  float d2 = 0.f;
  if (cnt > 0u) {
    const float members = (float)cnt;
    for (int j = lane; j < a.k; j += kWave) {
      const float old = a.centers[(int64_t)c * a.k + j];
      const float now = a.sums[(int64_t)c * a.k + j] / members;
      const float d = now - old;
      d2 += d * d;
      a.centers[(int64_t)c * a.k + j] = now;
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) d2 += __shfl_xor(d2, off);
  if (lane == 0 && !(d2 <= 0.f)) {   // a NaN shift is added too: the decide kernel has to see it
    add_f32<false>(a.shift, sqrtf(d2));
    add_f32<false>(a.shift + 1, d2);
  }
}

// Decides, on the device, whether the centres just written are final (so that a training loop
// needs no host read-back per iteration: every later step sees the flag and does nothing).
__device__ void km_decide(const KmArgs& a, float sum, float sq) {
  if (a.stop == nullptr || *a.stop != 0 || a.rule == 0) return;
  const float s = a.rule == 1 ? sq : sum * sum;
  // a shift that is not a number never passes `s < tol`: flag it (2) so that the loop ends and the
  // caller can tell (examples/my_kmeans.py:108-109 gives up on such a fit)
  if (s != s) *a.stop = 2;
  else if (s < a.tol) *a.stop = 1;
}

__global__ void km_decide_kernel(KmArgs a) { km_decide(a, a.shift[0], a.shift[1]); }

// Partial sums of a workgroup's rows, left in the workspace: set blockIdx.x of n * k sums and n counters.
// The kernel is a latency chain (label, value, LDS add), not bandwidth: 1024 threads with eight values each in
// flight take a workgroup's share of a 150 000 x 16 step (256 centres) in two rounds, and plain stores of the sums
// replace the 138 device-wide adds per sum that the workgroups used to queue for.  Clear and accumulate 40 us
// before, 18 now; finalize and decide 13.7, km_merge_kernel 11.5.
__global__ __launch_bounds__(kKmPartThreads) void km_partial_kernel(KmArgs a, uint32_t* arrived) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (km_stopped(a)) return;
  float* s_sum = reinterpret_cast<float*>(smem);
  const int entries = a.n * a.k, words = entries + a.n;
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_sum + entries);
  if (blockIdx.x == 0 && threadIdx.x == 0) *arrived = 0u;
  for (int i = threadIdx.x; i < words; i += kKmPartThreads) reinterpret_cast<uint32_t*>(smem)[i] = 0u;
  __syncthreads();
  const int64_t row0 = (int64_t)blockIdx.x * a.rows_per_block;
  const int64_t left = a.m - row0;
  const int nrows = (int)(left < a.rows_per_block ? (left > 0 ? left : 0) : a.rows_per_block);
  const float* x = a.x + row0 * a.k;
  const int step_r = kKmPartThreads / a.k, step_c = kKmPartThreads - step_r * a.k;
  int r = threadIdx.x / a.k, col = threadIdx.x - r * a.k;
  while (r < nrows) {
    float v[kKmBatch];
    int at[kKmBatch], cnt_at[kKmBatch];
#pragma unroll
    for (int u = 0; u < kKmBatch; ++u) {
      const bool in = r < nrows;
      const int rr = in ? r : 0;                       // row 0 of the share: there is one, the loop has begun
      const int c = km_label(a, row0 + rr);
      v[u] = x[(int64_t)rr * a.k + col];
      at[u] = in ? c * a.k + col : -1;
      cnt_at[u] = in && col == 0 ? c : -1;
      r += step_r;
      col += step_c;
      if (col >= a.k) { col -= a.k; ++r; }
    }
#pragma unroll
    for (int u = 0; u < kKmBatch; ++u) {
      if (at[u] >= 0) add_f32<true>(s_sum + at[u], v[u]);
      if (cnt_at[u] >= 0) atomicAdd(s_cnt + cnt_at[u], 1u);
    }
  }
  __syncthreads();
  uint32_t* part = reinterpret_cast<uint32_t*>(a.sums) + (int64_t)blockIdx.x * words;
  for (int i = threadIdx.x; i < words; i += kKmPartThreads) part[i] = reinterpret_cast<const uint32_t*>(smem)[i];
}

// One workgroup per centre: adds up its sums over the `parts` sets, writes the new centre and its squared shift;
// the workgroup that arrives last adds the shifts in order and applies the stop rule.
__global__ __launch_bounds__(kKmThreads) void km_merge_kernel(KmArgs a, int parts, float* moves, uint32_t* arrived) {
  if (km_stopped(a)) return;
  __shared__ float s_part[kKmThreads];
  __shared__ float s_d2[kKmThreads / kWave];
  __shared__ uint32_t s_cnt[kKmThreads / kWave];
  __shared__ int s_last;
  const int c = blockIdx.x, t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave;
  const int64_t words = (int64_t)a.n * a.k + a.n;
  uint32_t cnt = 0;
  for (int p = t; p < parts; p += kKmThreads) cnt += reinterpret_cast<const uint32_t*>(a.sums)[p * words + (int64_t)a.n * a.k + c];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off);
  if (lane == 0) s_cnt[wv] = cnt;
  __syncthreads();
  cnt = 0;
#pragma unroll
  for (int w = 0; w < kKmThreads / kWave; ++w) cnt += s_cnt[w];
  const float members = (float)cnt;
  const int side = kKmThreads / a.k;                    // sets read side by side (k <= kKmThreads)
  const int col = t % a.k, p0 = t / a.k;
  float d2 = 0.f, s = 0.f;
  if (p0 < side) {
    const float* from = a.sums + (int64_t)c * a.k + col;
#pragma unroll 8
    for (int p = p0; p < parts; p += side) s += from[p * words];
  }
  s_part[t] = s;
  __syncthreads();
  if (t < a.k && cnt > 0u) {
    float sum = 0.f;
    for (int q = 0; q < side; ++q) sum += s_part[q * a.k + t];
    float* centre = a.centers + (int64_t)c * a.k + t;
    const float now = sum / members;
    d2 = (now - *centre) * (now - *centre);
    *centre = now;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) d2 += __shfl_xor(d2, off);
  if (lane == 0) s_d2[wv] = d2;
  __syncthreads();
  if (t == 0) {
    d2 = 0.f;
    for (int w = 0; w < kKmThreads / kWave; ++w) d2 += s_d2[w];
    // device-wide: the workgroup that reads the shifts may run behind another L2
    __hip_atomic_store(moves + c, d2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)a.n - 1u;
  }
  __syncthreads();
  if (!s_last || t >= kWave) return;
  float sum = 0.f, sq = 0.f;
  for (int i = lane; i < a.n; i += kWave) {
    const float m2 = __hip_atomic_load(moves + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sum += sqrtf(m2);
    sq += m2;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off);
    sq += __shfl_xor(sq, off);
  }
  if (lane == 0) {
    a.shift[0] = sum;
    a.shift[1] = sq;
    km_decide(a, sum, sq);
  }
}

// The same for the sets of a step of several column slices (blockIdx.y: the slice, with sums, centres, shifts, counter and
// flag of its own one behind the other).  A workgroup takes as many whole centres as VALUES values hold, over 1024 / VALUES
// sets side by side: both the chain of loads per thread and the workgroups at the counter count, whose release has the L2
// write back.  With a workgroup per centre six slices of 256 centres of 16 columns, 40 sets, took 35 us, with 256 values
// per workgroup 10.8, with all reads of a thread in one round 8.2; one slice of 200 sets takes 32 with 256 values, 10.7
// with 64 and 7.3 in one round.  fp64 sums: a set is rounded once, the sum of the sets once more.
template <int VALUES>
__global__ __launch_bounds__(kKmMergeThreads) void km_merge_slices_kernel(KmArgs a, int parts, float* moves, uint32_t* arrived) {
  const int slice = blockIdx.y;
  const int words = a.n * a.k + a.n;
  a.sums += (int64_t)slice * parts * words;
  a.centers += (int64_t)slice * a.n * a.k;
  a.shift += 2 * slice;
  if (a.stop != nullptr) a.stop += slice;
  moves += (int64_t)slice * a.n;
  arrived += slice;
  if (km_stopped(a)) return;
  constexpr int kSide = kKmMergeThreads / VALUES;
  __shared__ double s_part[kSide][VALUES];
  __shared__ uint32_t s_cnt[kSide][VALUES];
  __shared__ float s_d2[VALUES];
  __shared__ int s_last;
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int at = t % VALUES, q = t / VALUES;
  const int held = VALUES / a.k, c0 = blockIdx.x * held;   // centres of the workgroup (k <= VALUES)
  const int mine = at / a.k, c = c0 + mine, col = at - mine * a.k;
  const bool on = mine < held && c < a.n;
  double total = 0.0;
  uint32_t cnt = 0;
  if (on) {
    // Sixteen sets in flight per thread: another CU of another die wrote them, and a second round of reads is 2 us.  A
    // place beyond the last set reads the first one's and adds nothing; the members are counted by a centre's first lane.
    constexpr int U = 16;
    const float* from = a.sums + (int64_t)c * a.k + col;
    const uint32_t* count = reinterpret_cast<const uint32_t*>(a.sums) + (int64_t)a.n * a.k + c;
    for (int p0 = q; p0 < parts; p0 += kSide * U) {
      float v[U];
      uint32_t m[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int p = p0 + u * kSide;
        v[u] = from[(int64_t)(p < parts ? p : q) * words];
        m[u] = 0u;
        if (col == 0) m[u] = count[(int64_t)(p < parts ? p : q) * words];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = p0 + u * kSide < parts;
        total += in ? (double)v[u] : 0.0;
        cnt += in ? m[u] : 0u;
      }
    }
  }
  s_part[q][at] = total;
  s_cnt[q][at] = cnt;
  __syncthreads();
  if (q == 0) {
    float d2 = -0.f;
    cnt = 0u;
#pragma unroll
    for (int w = 1; w < kSide; ++w) total += s_part[w][at];
#pragma unroll
    for (int w = 0; w < kSide; ++w) cnt += s_cnt[w][at - col];
    if (on && cnt > 0u) {
      float* centre = a.centers + (int64_t)c * a.k + col;
      const float now = (float)total / (float)cnt;
      d2 = (now - *centre) * (now - *centre);
      *centre = now;
    }
    s_d2[at] = d2;
  }
  __syncthreads();
  if (t < held && c0 + t < a.n) {
    float d2 = s_d2[t * a.k];               // (-0 from all columns where the centre has no member)
    for (int i = 1; i < a.k; ++i) d2 += s_d2[t * a.k + i];
    // device-wide: the workgroup that reads the shifts may run behind another L2
    __hip_atomic_store(moves + c0 + t, d2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (t == 0) s_last = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u;
  __syncthreads();
  if (!s_last || t >= kWave) return;
  float sum = 0.f, sq = 0.f;
  bool members = false;
  for (int i = lane; i < a.n; i += kWave) {
    const float m2 = __hip_atomic_load(moves + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sum += sqrtf(m2);
    sq += m2;
    members = members || __float_as_uint(m2) != 0x80000000u;
  }
  members = __any(members);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off);
    sq += __shfl_xor(sq, off);
  }
  if (lane == 0) {
    a.shift[0] = sum;
    a.shift[1] = sq;
    if (!members && a.stop != nullptr) *a.stop = 3;
    else km_decide(a, sum, sq);
  }
}

// A slice's centres rescaled to their mean length (examples/process_compress.py:16-18), by one workgroup: divide, then
// multiply, the lengths and their mean summed in fp64 and rounded.  flags[slices]: the rows' bad_row; flags[slices + 1]: set
// where a rescaled value is no number.  Six small operators and two reads of flags by the host, 60 us behind a training
// run, come down to this launch (7 us) and the read of the stop flags.
__global__ __launch_bounds__(kKmMergeThreads) void km_rescale_kernel(const float* __restrict__ centers, float* __restrict__ out,
                                                                     int n, int k, int slices, const int32_t* bad_row,
                                                                     int32_t* flags) {
  constexpr int kWaves = kKmMergeThreads / kWave;
  extern __shared__ float s_len[];                          // [n]
  __shared__ double s_sum[kWaves];
  const int t = threadIdx.x, slice = blockIdx.x;
  centers += (int64_t)slice * n * k;
  out += (int64_t)slice * n * k;
  double sum = 0.0;
  for (int c = t; c < n; c += kKmMergeThreads) {
    double sq = 0.0;
#pragma unroll 8
    for (int i = 0; i < k; ++i) sq += (double)centers[c * k + i] * (double)centers[c * k + i];
    const float len = (float)sqrt(sq);
    s_len[c] = len;
    sum += (double)len;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if ((t & (kWave - 1)) == 0) s_sum[t / kWave] = sum;
  __syncthreads();
  sum = 0.0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum += s_sum[w];
  const float mean = (float)(sum / (double)n);
  bool nan = false;
  for (int i = t; i < n * k; i += kKmMergeThreads) {
    const float v = __fdiv_rn(centers[i], s_len[i / k]) * mean;
    nan = nan || v != v;
    out[i] = v;
  }
  if (nan) atomicOr(flags + slices + 1, 1);
  if (slice == 0 && t == 0 && bad_row != nullptr) flags[slices] = *bad_row;
}

// Rows of a sample, column slice by column slice: out[s][i] = columns [s k, s k + k) of row rows[i] (zeros after the
// table's last column), norms[i][s] its length.  LANES lanes of four columns each per row and slice, the slices of a row
// side by side, so that a row is read as one run.
template <int LANES>
__global__ __launch_bounds__(kKmThreads) void slice_rows_kernel(const float* __restrict__ x, int64_t ld,
                                                                const int64_t* __restrict__ rows, int64_t m,
                                                                int64_t num_rows, int cols, int k, int slices,
                                                                float* __restrict__ out, float* __restrict__ norms,
                                                                int32_t* bad) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef f4 f4_dword __attribute__((aligned(4)));
  const int64_t unit = ((int64_t)blockIdx.x * kKmThreads + threadIdx.x) / LANES;
  const int c = 4 * (threadIdx.x % LANES);
  const int64_t i = unit / slices;
  const int s = (int)(unit - i * slices);
  const bool on = i < m;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (on) {
    int64_t id = i;
    if (rows != nullptr) {
      const int64_t want = rows[i] < 0 ? rows[i] + num_rows : rows[i];
      id = clamp_idx(want, num_rows);
      if (id != want) atomicOr(bad, 1);
    }
    const int left = (cols - s * k < k ? cols - s * k : k) - c;
    const float* from = x + id * ld + s * k + c;
    if (left >= 4) {
      const f4 q = *reinterpret_cast<const f4_dword*>(from);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = q[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = e < left ? from[e] : 0.f;
    }
    float* to = out + ((int64_t)s * m + i) * k + c;
    if (c + 4 <= k) {
      const f4 q = {v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f4_dword*>(to) = q;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < k) to[e] = v[e];
    }
  }
  float sq = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) sq += __shfl_xor(sq, off);
  if (on && c == 0) norms[unit] = sqrtf(sq);
}

// Bit r % 32 of word r / 32 of a slice's mask: its row r is at least as long as the quantile between two of the lengths
// (stats[s]: the two and, sixth, their flags), `weight` of the way from the lower to the upper one.
__global__ __launch_bounds__(kKmThreads) void keep_rows_kernel(const float* __restrict__ norms, const double* __restrict__ stats,
                                                               float weight, float weight_last, int64_t m, int slices,
                                                               uint32_t* __restrict__ keep, int64_t words) {
  const int s = blockIdx.y, lane = threadIdx.x & (kWave - 1);
  const int64_t r0 = ((int64_t)blockIdx.x * kKmThreads + threadIdx.x) - lane;
  if (r0 >= m) return;
  const float lo = (float)stats[6 * s], hi = (float)stats[6 * s + 1];
  const float w = s == slices - 1 ? weight_last : weight;
  const float gap = hi - lo;
  const float rim = w < 0.5f ? lo + w * gap : hi - gap * (1.f - w);   // from the nearer of the two
  const bool number = stats[6 * s + 5] == 0.0;                        // a quantile of NaN keeps no row
  const uint64_t bits = __ballot(r0 + lane < m && number && norms[(r0 + lane < m ? r0 + lane : 0) * slices + s] >= rim);
  if (lane == 0) {
    keep[s * words + r0 / 32] = (uint32_t)bits;
    if (r0 / 32 + 1 < words) keep[s * words + r0 / 32 + 1] = (uint32_t)(bits >> 32);
  }
}

int km_check(const char* what, const float* x, const int64_t* l64, const uint8_t* l8, float* centers, float* shift,
             int64_t m, int64_t n, int64_t k, int rule) {
  F2CGT_REQUIRE(m >= 0 && n > 0 && k > 0, F2CGT_E_INVALID, "%s: sizes must be m >= 0, n > 0, k > 0", what);
  F2CGT_REQUIRE(n <= 65536 && k <= 65536 && n * k < (1ll << 30), F2CGT_E_UNSUPPORTED, "%s: centre set too large", what);
  F2CGT_REQUIRE(rule >= 0 && rule <= 2, F2CGT_E_INVALID, "%s: stop rule must be 0, 1 or 2", what);
  F2CGT_REQUIRE((l64 != nullptr) != (l8 != nullptr), F2CGT_E_INVALID, "%s: give int64 labels or uint8 labels", what);
  F2CGT_REQUIRE(l8 == nullptr || n <= 256, F2CGT_E_INVALID, "%s: uint8 labels need n <= 256", what);
  F2CGT_REQUIRE(centers != nullptr && shift != nullptr && (m == 0 || x != nullptr), F2CGT_E_INVALID,
                "%s: null buffer", what);
  return 0;
}

// Shapes with a set of sums per workgroup: what fits LDS, with the columns of a centre in one pass of km_merge_kernel
// (wider ones leave its few workgroups a long chain of sets: 2 centres of 1000 columns, 2000 rows, 29 us with one set, 96
// by parts) and not so many centres that their arrivals at one counter take longer than the sums (2000 x 4, 8000 rows: 53
// and 70 us; 6000 x 1: 23 and 189; 500 x 4: 22.5 and 21.4).
bool km_parts_shape(int64_t n, int64_t k) { return n * k + n <= kKmLdsFloats && n <= 512 && k <= kKmThreads; }

// And the rows that pay for the sets: hundreds of centres need a few rows each (500 x 4: 500 rows 11.3 us with one set,
// 17.4 by parts; 2000 rows 19.4 and 19.6), a few wide ones more parts than 64 rows make (2 x 128: 2000 rows 14.0 and
// 18.1, 8000 rows 32 and 22; 8 x 128: 8000 rows 19.4 and 22.3; 16 x 128: 2000 rows 20.5 and 18.9).  Narrower ones are level
// on the device, with two launches for four.
bool km_by_parts(int64_t m, int64_t n, int64_t k) {
  return km_parts_shape(n, k) && (n < 256 || m >= 4 * n) && (k <= 64 || n >= 12 || m >= 2500 * n);
}

int64_t km_bytes(int64_t words) { return (words * 4 + 255) / 256 * 256; }

// The workspace of km_run_parts: kKmParts sets of sums and counters, the centres' shifts, the arrival counter.
int64_t km_parts_words(int64_t n, int64_t k) { return kKmParts * (n * k + n) + n + 1; }

int km_run_parts(const char* what, KmArgs a, hipStream_t st) {
  const int64_t words = (int64_t)a.n * a.k + a.n;
  // a set of sums for every 64 rows at least: fewer cost more to add up than to find
  int64_t rpb = ceil_div(a.m, (int64_t)kKmParts);
  rpb = rpb < 64 ? 64 : rpb;
  if (rpb > 0x7fffffff / 2) return fail(F2CGT_E_UNSUPPORTED, "%s: too many rows", what);
  a.rows_per_block = (int)rpb;
  const int parts = (int)(a.m > 0 ? ceil_div(a.m, rpb) : 1);
  float* moves = a.sums + kKmParts * words;
  uint32_t* arrived = reinterpret_cast<uint32_t*>(moves + a.n);
  km_partial_kernel<<<parts, kKmPartThreads, (size_t)words * 4, st>>>(a, arrived);
  km_merge_kernel<<<(unsigned)a.n, kKmThreads, 0, st>>>(a, parts, moves, arrived);
  return launch_status(what);
}

int km_run(const char* what, KmArgs a, hipStream_t st) {
  const int64_t words = (int64_t)a.n * a.k + a.n;
  const int cus = num_cus();
  int64_t clear_grid = ceil_div(words, kKmThreads * 4);
  clear_grid = clear_grid < 1 ? 1 : (clear_grid > cus * 4 ? cus * 4 : clear_grid);
  km_clear_kernel<<<(unsigned)clear_grid, kKmThreads, 0, st>>>(a);
  if (a.m > 0) {
    // rows per workgroup: enough of them to pay for flushing the partial sums, yet a grid that fills the device
    const bool lds = words <= kKmLdsFloats;
    int64_t rpb = ceil_div(a.m, (int64_t)cus * 8);
    const int64_t floor = lds ? ceil_div(4 * words, a.k) : 64;
    rpb = rpb < floor ? floor : rpb;
    rpb = rpb > (1 << 20) ? (1 << 20) : rpb;
    a.rows_per_block = (int)rpb;
    const int64_t grid = ceil_div(a.m, rpb);
    if (grid > 0x7fffffffll) return fail(F2CGT_E_UNSUPPORTED, "%s: too many rows", what);
    if (lds) km_accumulate_kernel<true><<<(unsigned)grid, kKmThreads, (size_t)words * 4, st>>>(a);
    else km_accumulate_kernel<false><<<(unsigned)grid, kKmThreads, 0, st>>>(a);
  }
  km_finalize_kernel<<<(unsigned)ceil_div(a.n, kKmThreads / kWave), kKmThreads, 0, st>>>(a);
  km_decide_kernel<<<1, 1, 0, st>>>(a);
  return launch_status(what);
}

}  // namespace
}  // namespace f2cgt

using namespace f2cgt;

extern "C" int64_t f2cgt_kmeans_update_workspace_bytes(int64_t n, int64_t k) {
  if (n <= 0 || k <= 0) return 0;
  return km_bytes(km_parts_shape(n, k) ? km_parts_words(n, k) : n * k + n);
}

extern "C" int f2cgt_kmeans_update(const float* x, const int64_t* labels_i64, const uint8_t* labels_u8,
                                   float* centers, float* shift, int32_t* stop, int stop_rule, float tol,
                                   void* workspace, int64_t workspace_bytes, int64_t m, int64_t n, int64_t k,
                                   void* stream) {
  const char* what = "kmeans_update";
  if (int rc = km_check(what, x, labels_i64, labels_u8, centers, shift, m, n, k, stop_rule)) return rc;
  // room for one set of sums is enough: all workgroups then add into it
  F2CGT_REQUIRE(workspace != nullptr && workspace_bytes >= km_bytes(n * k + n) && aligned(workspace, 16),
                F2CGT_E_INVALID, "%s: workspace of %lld bytes (16-byte aligned) needed", what,
                (long long)km_bytes(n * k + n));
  KmArgs a{};
  a.x = x; a.labels_i64 = labels_i64; a.labels_u8 = labels_u8; a.centers = centers; a.shift = shift; a.stop = stop;
  a.sums = static_cast<float*>(workspace);
  a.counts = reinterpret_cast<uint32_t*>(a.sums + n * k);
  a.m = m; a.n = (int)n; a.k = (int)k; a.rule = stop_rule; a.tol = tol;
  if (km_by_parts(m, n, k) && workspace_bytes >= f2cgt_kmeans_update_workspace_bytes(n, k)) return km_run_parts(what, a, as_stream(stream));
  return km_run(what, a, as_stream(stream));
}

extern "C" int f2cgt_kmeans_update_static(const float* x, const int64_t* labels_i64, const uint8_t* labels_u8,
                                          float* centers, float* shift, int32_t* stop, int stop_rule, float tol,
                                          int64_t m, int64_t n, int64_t k, void* stream) {
  const char* what = "kmeans_update_static";
  if (int rc = km_check(what, x, labels_i64, labels_u8, centers, shift, m, n, k, stop_rule)) return rc;
  F2CGT_REQUIRE(n * k <= kStaticSums && n <= kStaticCenters, F2CGT_E_UNSUPPORTED,
                "%s: at most %lld sums (n * k) and %lld centres fit the built-in scratch (got %lld and %lld); "
                "use f2cgt_kmeans_update with a workspace",
                what, (long long)kStaticSums, (long long)kStaticCenters, (long long)(n * k), (long long)n);
  // the device address of the scratch array, looked up once per device (every device has its own copy)
  static void* scratch_of[64] = {nullptr};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64) return fail(F2CGT_E_DEVICE, "%s: no current device", what);
  void* base = __atomic_load_n(&scratch_of[dev], __ATOMIC_ACQUIRE);
  if (base == nullptr) {
    e = hipGetSymbolAddress(&base, HIP_SYMBOL(scratch));
    if (e != hipSuccess || base == nullptr)
      return fail((int)(e != hipSuccess ? e : hipErrorInvalidSymbol), "%s: cannot resolve the scratch array: %s", what,
                  hipGetErrorString(e));
    __atomic_store_n(&scratch_of[dev], base, __ATOMIC_RELEASE);
  }
  KmArgs a{};
  a.x = x; a.labels_i64 = labels_i64; a.labels_u8 = labels_u8; a.centers = centers; a.shift = shift; a.stop = stop;
  a.sums = static_cast<float*>(base);
  a.counts = reinterpret_cast<uint32_t*>(a.sums + n * k);
  a.m = m; a.n = (int)n; a.k = (int)k; a.rule = stop_rule; a.tol = tol;
  return km_run(what, a, as_stream(stream));
}

extern "C" int f2cgt_slice_rows(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                                int64_t k, float* out, float* norms, int32_t* bad_row, void* stream) {
  const char* what = "slice_rows";
  F2CGT_REQUIRE(m >= 0 && num_rows > 0 && cols > 0 && k > 0 && k <= 64, F2CGT_E_INVALID, "%s: sizes must be positive, k <= 64", what);
  F2CGT_REQUIRE(ld >= cols && (rows != nullptr || m <= num_rows), F2CGT_E_INVALID, "%s: the rows do not fit the table", what);
  const int64_t slices = ceil_div(cols, k);
  F2CGT_REQUIRE(cols < (1 << 24), F2CGT_E_UNSUPPORTED, "%s: too many columns", what);
  if (m == 0) return 0;
  F2CGT_REQUIRE(x && out && norms && bad_row, F2CGT_E_INVALID, "%s: null buffer", what);
  const int lanes = pow2_ceil((int)ceil_div(k, (int64_t)4));
  const int64_t grid = ceil_div(m * slices, (int64_t)(kKmThreads / lanes));
  F2CGT_REQUIRE(grid <= 0x7fffffffll, F2CGT_E_UNSUPPORTED, "%s: too many rows", what);
  hipStream_t st = as_stream(stream);
#define F2CGT_SLICE_ROWS(L) slice_rows_kernel<L><<<(unsigned)grid, kKmThreads, 0, st>>>(x, ld, rows, m, num_rows, (int)cols, \
                                                                                       (int)k, (int)slices, out, norms, bad_row)
  switch (lanes) {
    case 1: F2CGT_SLICE_ROWS(1); break;
    case 2: F2CGT_SLICE_ROWS(2); break;
    case 4: F2CGT_SLICE_ROWS(4); break;
    case 8: F2CGT_SLICE_ROWS(8); break;
    default: F2CGT_SLICE_ROWS(16); break;
  }
#undef F2CGT_SLICE_ROWS
  return launch_status(what);
}

extern "C" int f2cgt_keep_rows(const float* norms, const double* stats, float weight, float weight_last, int64_t m,
                               int64_t slices, uint32_t* keep, void* stream) {
  const char* what = "keep_rows";
  F2CGT_REQUIRE(m >= 0 && slices > 0 && slices <= 65535, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  if (m == 0) return 0;
  F2CGT_REQUIRE(norms && stats && keep, F2CGT_E_INVALID, "%s: null buffer", what);
  const int64_t grid = ceil_div(m, (int64_t)kKmThreads);
  F2CGT_REQUIRE(grid <= 0x7fffffffll, F2CGT_E_UNSUPPORTED, "%s: too many rows", what);
  keep_rows_kernel<<<dim3((unsigned)grid, (unsigned)slices), kKmThreads, 0, as_stream(stream)>>>(
      norms, stats, weight, weight_last, m, (int)slices, keep, ceil_div(m, (int64_t)32));
  return launch_status(what);
}

extern "C" int f2cgt_kmeans_slices_covers(int64_t slices, int64_t n, int64_t k) {
  return n > 0 && k > 0 && km_parts_shape(n, k) && assign_sums_fits(slices, n, k) ? 1 : 0;
}

extern "C" int64_t f2cgt_kmeans_slices_workspace_bytes(int64_t m, int64_t slices, int64_t n, int64_t k) {
  if (m <= 0 || !f2cgt_kmeans_slices_covers(slices, n, k)) return 0;
  return km_bytes(slices * (assign_sums_shares(m, slices, k) * (n * k + n) + n + 3));
}

extern "C" int f2cgt_kmeans_slices_step(const float* x, const uint32_t* keep, float* centers, int32_t* stop, int stop_rule,
                                        float tol, void* workspace, int64_t workspace_bytes, int64_t m, int64_t slices,
                                        int64_t n, int64_t k, int metric, void* stream) {
  const char* what = "kmeans_slices_step";
  F2CGT_REQUIRE(m > 0 && slices > 0 && n > 0 && k > 0, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  F2CGT_REQUIRE(f2cgt_kmeans_slices_covers(slices, n, k), F2CGT_E_UNSUPPORTED,
                "%s: %lld slices of %lld centres of %lld columns are left to kmeans_predict and kmeans_update", what,
                (long long)slices, (long long)n, (long long)k);
  F2CGT_REQUIRE(metric == F2CGT_METRIC_L2 || metric == F2CGT_METRIC_COSINE, F2CGT_E_INVALID, "%s: unknown metric %d", what,
                metric);
  F2CGT_REQUIRE(stop_rule >= 0 && stop_rule <= 2, F2CGT_E_INVALID, "%s: stop rule must be 0, 1 or 2", what);
  F2CGT_REQUIRE(x && centers && stop && workspace && aligned(workspace, 16) &&
                    workspace_bytes >= f2cgt_kmeans_slices_workspace_bytes(m, slices, n, k),
                F2CGT_E_INVALID, "%s: null buffer, or workspace misaligned or too small", what);
  const int parts = (int)assign_sums_shares(m, slices, k);
  float* sums = static_cast<float*>(workspace);
  float* moves = sums + slices * parts * (n * k + n);
  float* shift = moves + slices * n;
  uint32_t* arrived = reinterpret_cast<uint32_t*>(shift + 2 * slices);
  hipStream_t st = as_stream(stream);
  if (int rc = assign_sums(x, m * k, keep, ceil_div(m, (int64_t)32), centers, stop, sums, arrived, m, (int)slices, (int)n, (int)k,
                           metric, st))
    return rc;
  KmArgs a{};
  a.centers = centers; a.shift = shift; a.stop = stop; a.sums = sums; a.m = m; a.n = (int)n; a.k = (int)k;
  a.rule = stop_rule; a.tol = tol;
  const int values = parts <= 64 ? 256 : parts <= 128 ? 128 : 64;
  const dim3 grid((unsigned)ceil_div(n, values / k), (unsigned)slices);
  if (parts <= 64) km_merge_slices_kernel<256><<<grid, kKmMergeThreads, 0, st>>>(a, parts, moves, arrived);
  else if (parts <= 128) km_merge_slices_kernel<128><<<grid, kKmMergeThreads, 0, st>>>(a, parts, moves, arrived);
  else km_merge_slices_kernel<64><<<grid, kKmMergeThreads, 0, st>>>(a, parts, moves, arrived);
  return launch_status(what);
}

extern "C" int f2cgt_kmeans_rescale(const float* centers, float* out, int64_t n, int64_t k, int64_t slices, const int32_t* bad_row,
                                    int32_t* flags, void* stream) {
  const char* what = "kmeans_rescale";
  F2CGT_REQUIRE(n > 0 && k > 0 && slices > 0, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  F2CGT_REQUIRE(n <= 8192 && k <= 4096 && slices <= 65535, F2CGT_E_UNSUPPORTED, "%s: too many centres, columns or slices", what);
  F2CGT_REQUIRE(centers && out && flags, F2CGT_E_INVALID, "%s: null buffer", what);
  km_rescale_kernel<<<(unsigned)slices, kKmMergeThreads, (size_t)n * 4, as_stream(stream)>>>(centers, out, (int)n, (int)k, (int)slices,
                                                                                             bad_row, flags);
  return launch_status(what);
}
