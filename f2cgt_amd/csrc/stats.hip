// Order statistics and mean of |x| over column slices of a (sampled) feature table: what the scalar quantiser's codebook
// is made of (examples/process_compress.py:45-68: two percentiles and the mean of the absolute values of a slice).
//
// The statistics are exact: the requested ranks are found by a radix selection on the bit pattern of |x| (for
// non-negative floats the order of the values is the order of the bit patterns), three digits of 12, 10 and 9 bits.  A pass
// counts the next digit of the values that share the digits found so far with a wanted rank, in LDS, and the next pass finds
// the digit from the sums in its prologue.  Nothing is sorted and nothing is copied but the few values that a pass keeps for
// the next one (see stat_pass_kernel); the rows are read through the sample's row list.
//   The first pass shares no counter between workgroups: the hot bins of a normal distribution lie in a dozen cache lines, on
// which device-wide atomics of 256 workgroups would queue up.  Each writes its counts and a small kernel adds them.  What the
// second and the third pass count are a few hundred values a workgroup, which go to the sums by atomics as they are.
//
// What bounds it: one read of the sample (15 us at 120 000 x 100 values, 3.2 TB/s through the row list, as long on its LDS
// counters and sums as on its loads; 22 with the values that it keeps for the second pass), the sum behind it (4 us) and two
// passes over what was kept, 9 and 10 us, the last with the outputs.  The codebook is made by the last workgroup of the last
// pass, so that the encoder can follow at once, and the ids' check is on the host as soon as the first pass is done, so that a
// caller does not wait for the rest.  The four launches take 44 us; six, with sums of all counters behind the second and third
// pass too, 49, with a second read of the sample 52, a third 66 (the host 195 ms on a copy of the sample, np.percentile).
// Likewise 100 000 x 602 values 151 -> 101 -> 96 us (second read saved, sums saved), 60 000 x 1030 203 -> 130 -> 125, 1 000 000 x 128
// 238 -> 151 -> 146, 1000 x 64 31 -> 27 (25 with more workgroups).  Tables on which a workgroup has to read its rows again lose up to 6 % by what it kept in
// vain and gain the sums (120 000 x 100: all values equal 369 us before and after, 80 % zeros 180, rows of very different
// lengths 52 -> 48).
#include "common.hpp"

namespace f2cgt {
namespace {

constexpr int kStatThreads = 1024;
constexpr int kBins = 4096;          // counters of a pass: 4096, 4 x 1024 or 4 x 512
constexpr int kReplicas = 4;         // copies of the first pass's counters in LDS, by lane: its hot bins are few
constexpr int kMaxBlocks = 256;      // workgroups per pass over all slices (one per CU)
constexpr int kStatWaves = kStatThreads / kWave;
constexpr int kKept = 1024;          // values a wave of a pass can hand to the next one
constexpr int kRoomBlocks = 256;     // more workgroups than that in all hand over half as many per wave,
constexpr int kKeepBlocks = 1024;    // and more than that none (32 KB of workspace each)

constexpr int kInFlight = 8;         // rows that a lane reads at a time

constexpr uint32_t kSawNan = 1u, kSawBadRow = 2u;   // a NaN among the values; a row id outside the table

struct StatState {                   // per slice, written by the first workgroup of the second pass for the third
  uint32_t prefix[4];                // digits found so far of the value at each wanted rank
  uint32_t pad[4];
  uint64_t rank[4];                  // its rank among the values that share them
};

struct StatArgs {
  const float* x;
  const int64_t* rows;               // row list of the sample; null: rows [0, m)
  int64_t m, num_rows, ld;
  int cols, slice, n_slices;
  int blocks;                        // workgroups per slice
  uint64_t ranks[8];                 // wanted ranks of a full slice, and of the last one
  uint32_t* partial;                 // [n_slices][blocks][kBins]: of the first pass
  uint32_t* hist;                    // [3][n_slices][kBins]: the passes' counters
  StatState* state;                  // [n_slices]: after the first digit
  double* sums;                      // [n_slices][blocks]
  uint32_t* flags;                   // [n_slices][blocks]: kSawNan, kSawBadRow
  int keep;                          // kKept, or 0 where there is no room for them
  int ahead;                         // the first pass keeps values for the second
  // [n_slices][blocks][kStatWaves][keep]: the values of a workgroup's windows, then those that share the first digit of a
  // wanted rank
  uint32_t* kept;
  uint32_t* n_kept;                  // [n_slices][blocks][kStatWaves]: how many; more than `keep`: not all of them are there
  uint32_t* windows;                 // [n_slices][blocks][2]: the digits between these two are not kept
  double* out;                       // [n_slices][6]
  uint32_t* arrived;                 // [n_slices]: workgroups of the last pass that are done with a slice
  int32_t* bad;                      // host memory: set by the first pass where a row id lies outside the table; or null
  float* books;                      // [n_slices][5], or null
  float weights[4];                  // lower and upper percentile of a slice, and of the last one: where between its ranks
};

// Finds, in `groups` runs of kBins / groups counters, the counter that holds rank[t] (run t, or the only run), for all
// four ranks, by the whole workgroup: digit[t] is the counter's place in its run and rank[t] becomes the rank inside it.
// counter(i): the i-th one.
template <int GROUPS, int USED, typename Counter>
__device__ __forceinline__ void find_digits(Counter counter, const uint64_t (&rank)[4],
                                            uint64_t* s_scan, uint32_t* s_digit, uint64_t* s_rest) {
  constexpr int PER = USED / (kStatThreads / GROUPS);   // counters per thread
  static_assert(PER >= 1, "a thread owns at least one counter");
  const int t = threadIdx.x;
  const int group = t / (kStatThreads / GROUPS), at = t % (kStatThreads / GROUPS);
  uint32_t c[PER];
  uint64_t own = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c[i] = counter(group * USED + at * PER + i);
    own += c[i];
  }
  uint64_t run = own;                                   // inclusive sum over the wave
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t other = __shfl_up(run, off);
    run += (t & (kWave - 1)) >= off ? other : 0;
  }
  if ((t & (kWave - 1)) == kWave - 1) s_scan[t / kWave] = run;
  if (t < 4) { s_digit[t] = 0; s_rest[t] = 0; }
  __syncthreads();
  constexpr int WPG = kStatThreads / kWave / GROUPS;    // waves per run
  uint64_t before = run - own;
  for (int w = group * WPG; w < t / kWave; ++w) before += s_scan[w];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (GROUPS > 1 && k != group) continue;
    const uint64_t want = rank[k];
    if (want < before || want >= before + own) continue;
    uint64_t lo = before;
    int found = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (want >= lo && want < lo + c[i]) { found = i; s_rest[k] = want - lo; }
      lo += c[i];
    }
    s_digit[k] = (uint32_t)(at * PER + found);
  }
  __syncthreads();
}

__device__ __forceinline__ void wanted_ranks(const StatArgs& a, int slice, uint64_t (&rank)[4]) {
  const int base = slice == a.n_slices - 1 ? 4 : 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) rank[k] = a.ranks[base + k];
}

// The digits known after pass PASS - 1 (prefix of every wanted rank, rank inside it), by every workgroup from the summed
// counters of that pass.
template <int PASS>
__device__ __forceinline__ void known_digits(const StatArgs& a, int slice, uint64_t* s_scan, uint32_t* s_digit,
                                             uint64_t* s_rest, uint32_t (&prefix)[4], uint64_t (&rank)[4]) {
  const uint32_t* __restrict__ hist = a.hist + ((int64_t)(PASS - 1) * a.n_slices + slice) * kBins;
  auto counter = [&](int i) { return hist[i]; };
  if (PASS == 1) {
    wanted_ranks(a, slice, rank);
    find_digits<1, 4096>(counter, rank, s_scan, s_digit, s_rest);
#pragma unroll
    for (int k = 0; k < 4; ++k) prefix[k] = s_digit[k];
  } else {
    const StatState& st = a.state[slice];
#pragma unroll
    for (int k = 0; k < 4; ++k) rank[k] = st.rank[k];
    find_digits<4, 1024>(counter, rank, s_scan, s_digit, s_rest);
#pragma unroll
    for (int k = 0; k < 4; ++k) prefix[k] = (st.prefix[k] << 10) | s_digit[k];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) rank[k] = s_rest[k];
}

// The quantiser's codebook of a slice (fmin, fmax, emin, emax, mean) from its statistics: percentiles interpolated in
// float32 from the nearer rank, floored at 1e-5 and 2e-5, their log2 correctly rounded, and the mean, lifted by 0.1 where
// it is below 0.1 (examples/process_compress.py:45-68).  A NaN stays one.
__device__ void sq_codebook(const StatArgs& a, int slice, const float (&at)[4], double total, uint32_t flags) {
  const bool last = slice == a.n_slices - 1;
  auto between = [](float below, float above, float w) {
    const float gap = above - below;
    return w < 0.5f ? below + gap * w : above - gap * (1.f - w);
  };
  float lo = between(at[0], at[1], a.weights[last ? 2 : 0]), hi = between(at[2], at[3], a.weights[last ? 3 : 1]);
  if (flags & kSawNan) lo = hi = __uint_as_float(0x7fc00000u);
  const float floor = 1e-5f;
  lo = floor > lo ? floor : lo;
  hi = 2e-5f > hi ? 2e-5f : hi;
  const int64_t width = last ? a.cols - (int64_t)slice * a.slice : a.slice;
  float level = (float)(total / (double)(a.m * width));
  level = level < 0.1f ? level + 0.1f : level;
  float* book = a.books + slice * 5;
  book[0] = lo;
  book[1] = hi;
  book[2] = log2_cr(lo);
  book[3] = log2_cr(hi) + floor;
  book[4] = level;
}

// Last digit, and the outputs of a slice: the values at the four ranks, the sum, the flags; by one workgroup.
__device__ void stat_finish(const StatArgs& a, int slice, uint64_t* s_scan, uint32_t* s_digit, uint64_t* s_rest,
                            uint32_t (&prefix)[4], const uint64_t (&rank)[4]) {
  const int t = threadIdx.x;
  uint32_t* hist = a.hist + ((int64_t)2 * a.n_slices + slice) * kBins;
  find_digits<4, 512>([&](int i) { return __hip_atomic_load(hist + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }, rank,
                      s_scan, s_digit, s_rest);
#pragma unroll
  for (int k = 0; k < 4; ++k) prefix[k] = (prefix[k] << 9) | s_digit[k];
  if (t < 4) a.out[slice * 6 + t] = (double)__uint_as_float(t == 0 ? prefix[0] : t == 1 ? prefix[1] : t == 2 ? prefix[2] : prefix[3]);
  if (t >= kWave && t < 2 * kWave) {                    // the second wave
    double total = 0.0;
    uint32_t flags = 0;
    for (int b = t - kWave; b < a.blocks; b += kWave) {
      total += a.sums[(int64_t)slice * a.blocks + b];
      flags |= a.flags[(int64_t)slice * a.blocks + b];
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      total += __shfl_xor(total, off);
      flags |= __shfl_xor(flags, off);
    }
    if (t == kWave) {
      a.out[slice * 6 + 4] = total;
      a.out[slice * 6 + 5] = (double)flags;
      if (a.books != nullptr) {
        const float at[4] = {__uint_as_float(prefix[0]), __uint_as_float(prefix[1]), __uint_as_float(prefix[2]),
                             __uint_as_float(prefix[3])};
        sq_codebook(a, slice, at, total, flags);
      }
    }
  }
}

// One pass over the sample.  A thread keeps its place in the row (a V-wide column group) and walks rows; eight rows are in
// flight at a time, and the ids of the eight after them.
//
// A later pass needs only the values that share the digits found so far with a wanted rank, one in a few hundred of a
// feature table, so the pass before keeps them, wave by wave, and the sample is read once.
//   The second pass knows the first digits and keeps what the third will count.
//   The first pass does not know them yet.  Its workgroups take the first rows that they count for a sample of the sample:
//   a wanted rank lies, with six standard deviations to either side, between two of its ranks, and the values between these
//   two (a window of first digits; one or two of a hundred values at the percentiles 0.5 and 99.5) are kept.  The second
//   pass holds the true digits against the windows.
// A workgroup whose windows missed a digit (rows in an order that its first ones say nothing about), or with a wave that
// met more than `keep` of the values (a table of few different values), reads its rows again.
template <int PASS, int V>
__global__ __launch_bounds__(kStatThreads) void stat_pass_kernel(StatArgs a) {
  __shared__ __align__(16) uint32_t s_hist[PASS == 0 ? kBins * kReplicas : kBins];
  __shared__ uint64_t s_scan[kStatThreads / kWave];
  __shared__ uint32_t s_digit[4];
  __shared__ uint64_t s_rest[4];
  __shared__ double s_sum[kStatThreads / kWave];
  __shared__ uint32_t s_flags;
  __shared__ uint32_t s_kept[PASS < 2 ? kStatWaves * kKept : 1];
  __shared__ uint32_t s_n_kept[kStatWaves];
  const int t = threadIdx.x, slice = blockIdx.y, wave = t / kWave;
  constexpr int LDS_BINS = PASS == 0 ? kBins * kReplicas : kBins;
  for (int i = t; i < LDS_BINS / 4; i += kStatThreads) reinterpret_cast<uint4*>(s_hist)[i] = make_uint4(0u, 0u, 0u, 0u);
  if (t == 0) s_flags = 0u;
  if (t < kStatWaves) s_n_kept[t] = 0u;
  uint32_t prefix[4] = {0u, 0u, 0u, 0u};
  uint64_t rank[4] = {0u, 0u, 0u, 0u};
  if constexpr (PASS > 0) {
    known_digits<PASS>(a, slice, s_scan, s_digit, s_rest, prefix, rank);
#pragma unroll
    for (int k = 0; k < 4; ++k) prefix[k] = __builtin_amdgcn_readfirstlane(prefix[k]);
    if (PASS == 1 && blockIdx.x == 0 && t == 0) {
      StatState& st = a.state[slice];
#pragma unroll
      for (int k = 0; k < 4; ++k) { st.prefix[k] = prefix[k]; st.rank[k] = rank[k]; }
    }
  }
  __syncthreads();

  const int col0 = slice * a.slice;
  const int width = a.cols - col0 < a.slice ? a.cols - col0 : a.slice;
  const int groups = width / V;
  const int cg = groups < kStatThreads ? groups : kStatThreads;
  const int rpp = kStatThreads / cg;                    // rows per pass of the workgroup
  const int r0 = t / cg, c0 = t - r0 * cg;
  const int64_t step = (int64_t)a.blocks * rpp;
  double sum = 0.0;
  uint32_t flags = 0u;
  auto take = [&](float v) {
    const uint32_t mag = __float_as_uint(v) & 0x7fffffffu;
    if constexpr (PASS == 0) {
      sum += (double)__uint_as_float(mag);
      flags |= mag > 0x7f800000u ? kSawNan : 0u;
      atomicAdd(&s_hist[(mag >> 19) * kReplicas + (t & (kReplicas - 1))], 1u);
    } else if constexpr (PASS == 1) {
      const uint32_t digit = mag >> 19;
      if ((digit == prefix[0]) | (digit == prefix[1]) | (digit == prefix[2]) | (digit == prefix[3])) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (digit == prefix[k]) atomicAdd(&s_hist[k * 1024 + ((mag >> 9) & 1023u)], 1u);
        // a place for every lane that is here, by one addition for the wave
        const uint64_t all = __ballot(true);
        const uint32_t before = __popcll(all & ((1ull << (t & (kWave - 1))) - 1));
        uint32_t at = before == 0 ? atomicAdd(&s_n_kept[wave], (uint32_t)__popcll(all)) : 0u;
        at = __builtin_amdgcn_readfirstlane(at) + before;
        if (at < (uint32_t)a.keep) s_kept[wave * kKept + at] = mag;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if ((mag >> 9) == prefix[k]) atomicAdd(&s_hist[k * 512 + (mag & 511u)], 1u);
    }
  };
  const int64_t place = (int64_t)slice * a.blocks + blockIdx.x;
  bool read_rows = true;
  if (PASS == 2 || (PASS == 1 && a.ahead)) {
    uint32_t most = 0;
#pragma unroll
    for (int w = 0; w < kStatWaves; ++w) {
      const uint32_t n = a.n_kept[place * kStatWaves + w];
      most = n > most ? n : most;
    }
    bool whole = most <= (uint32_t)a.keep;
    if (PASS == 1) {
      const uint32_t* between = a.windows + place * 2;
#pragma unroll
      for (int k = 0; k < 4; ++k) whole &= prefix[k] <= between[0] || prefix[k] >= between[1];
    }
    if (whole) {
      read_rows = false;
      const uint32_t n = a.n_kept[place * kStatWaves + wave];
      const uint32_t* kept = a.kept + (place * kStatWaves + wave) * a.keep;
      for (uint32_t i = t & (kWave - 1); i < n; i += kWave) take(__uint_as_float(kept[i]));
    }
  }
  constexpr int U = kInFlight;
  if constexpr (PASS == 0) {
    if (a.ahead) {
      // All lanes walk together, as many rounds as the first row has; rows that a lane has not are its first, and not counted.
      read_rows = false;
      const int64_t base = (int64_t)blockIdx.x * rpp;
      const int64_t first = base + r0 < a.m ? base + r0 : 0;
      const int rounds = base < a.m ? (int)((a.m - base + step * U - 1) / (step * U)) : 0;
      int mine = r0 < rpp && base + r0 < a.m ? (int)((a.m - base - r0 + step - 1) / step) : 0;   // rows of this lane left
      int64_t id[U], row = base + r0;
      auto row_ids = [&](int have) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t ru = u < have ? row + u * step : first;
          id[u] = a.rows != nullptr ? a.rows[ru] : ru;
        }
      };
      uint32_t from = 0u, span = 0x80000000u, kept = 0u;   // magnitudes that are not kept; what the wave has kept
      auto keep = [&](float v, bool counts) {
        const uint32_t mag = __float_as_uint(v) & 0x7fffffffu;
        if (kept > (uint32_t)a.keep) return;                // (the same for the wave)
        const bool in = counts && mag - from >= span;
        const uint64_t all = __ballot(in);
        if (all == 0) return;
        const uint32_t at = kept + __builtin_amdgcn_mbcnt_hi((uint32_t)(all >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)all, 0u));
        if (in && at < (uint32_t)a.keep) s_kept[wave * kKept + at] = mag;
        kept += (uint32_t)__popcll(all);
      };
      row_ids(mine);
      for (int round = 0; round < rounds; ++round) {
        float v[U][V];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t want = id[u] < 0 ? id[u] + a.num_rows : id[u];
          const int64_t at = clamp_idx(want, a.num_rows);
          flags |= at != want ? kSawBadRow : 0u;
          const float* p = a.x + at * a.ld + col0 + c0 * V;
          if constexpr (V == 4) {
            const float4 q = *reinterpret_cast<const float4*>(p);
            v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
          } else if constexpr (V == 2) {
            const float2 q = *reinterpret_cast<const float2*>(p);
            v[u][0] = q.x; v[u][1] = q.y;
          } else {
            v[u][0] = *p;
          }
        }
        row += step * U;
        if (round + 1 < rounds) row_ids(mine - U);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (u < mine)
#pragma unroll
            for (int i = 0; i < V; ++i) take(v[u][i]);
        if (round == 0) {
          int64_t rows = 0;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t left = a.m - (base + u * step);
            rows += left < 0 ? 0 : left < rpp ? left : rpp;
          }
          const float n = (float)(rows * width), all = (float)a.m * (float)width;
          uint64_t edge[4] = {0u, 0u, (uint64_t)n - 1u, 0u};
          wanted_ranks(a, slice, rank);
          uint64_t low = rank[0] > rank[1] ? rank[0] : rank[1], high = rank[2] < rank[3] ? rank[2] : rank[3];
          const float p = (float)low / all, q = (float)high / all;
          const float below = n * p + 6.f * __builtin_amdgcn_sqrtf(n * p * (1.f - p)) + 4.f;
          const float above = n * q - 6.f * __builtin_amdgcn_sqrtf(n * q * (1.f - q)) - 4.f;
          edge[0] = below < n - 1.f ? (uint64_t)below : (uint64_t)n - 1u;
          edge[1] = above > 0.f ? (uint64_t)above : 0u;
          __syncthreads();
          auto counter = [&](int i) {
            const uint4 c = *reinterpret_cast<const uint4*>(s_hist + i * kReplicas);
            return c.x + c.y + c.z + c.w;
          };
          find_digits<1, 4096>(counter, edge, s_scan, s_digit, s_rest);
          // kept: digits up to the one that `below` of the sample's values reach, and from the one that `above` do
          const uint32_t lo = __builtin_amdgcn_readfirstlane(s_digit[0]), hi = __builtin_amdgcn_readfirstlane(s_digit[1]);
          from = (lo + 1) << 19;
          span = hi > lo ? (hi - lo - 1) << 19 : 0u;
          if (t == 0) {
            a.windows[place * 2] = lo;
            a.windows[place * 2 + 1] = hi;
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int i = 0; i < V; ++i) keep(v[u][i], u < mine);
        mine -= U;
      }
      if ((t & (kWave - 1)) == 0) s_n_kept[wave] = kept;
      if (rounds == 0 && t < 2) a.windows[place * 2 + t] = t == 0 ? kBins : 0u;   // nothing that could be left out
    }
  }
  if (read_rows && r0 < rpp) {
    int64_t id[U];
    // the rows r, r + step, ...: a place beyond the sample takes row r again, which the sample has
    auto row_ids = [&](int64_t r, int64_t (&id)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t ru = r + u * step < a.m ? r + u * step : r;
        id[u] = a.rows != nullptr ? a.rows[ru] : ru;
      }
    };
    const int64_t first = (int64_t)blockIdx.x * rpp + r0;
    if (first < a.m) row_ids(first, id);
    for (int64_t r = first; r < a.m; r += step * U) {
      const float* p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t want = id[u] < 0 ? id[u] + a.num_rows : id[u];
        const int64_t at = clamp_idx(want, a.num_rows);
        if (PASS == 0) flags |= at != want ? kSawBadRow : 0u;
        p[u] = a.x + at * a.ld + col0;
      }
      if (r + step * U < a.m) row_ids(r + step * U, id);
      for (int c = c0; c < groups; c += cg) {
        float v[U][V];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if constexpr (V == 4) {
            const float4 q = *reinterpret_cast<const float4*>(p[u] + c * V);
            v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
          } else if constexpr (V == 2) {
            const float2 q = *reinterpret_cast<const float2*>(p[u] + c * V);
            v[u][0] = q.x; v[u][1] = q.y;
          } else {
            v[u][0] = p[u][c];
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (u > 0 && r + u * step >= a.m) break;
#pragma unroll
          for (int i = 0; i < V; ++i) take(v[u][i]);
        }
      }
    }
  }
  if constexpr (PASS == 0) {
    if (flags) atomicOr(&s_flags, flags);
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if ((t & (kWave - 1)) == 0) s_sum[t / kWave] = sum;
  }
  __syncthreads();
  if (PASS == 1 || (PASS == 0 && a.ahead)) {
    const uint32_t n = s_n_kept[wave];
    if ((t & (kWave - 1)) == 0) a.n_kept[place * kStatWaves + wave] = n;
    uint32_t* kept = a.kept + (place * kStatWaves + wave) * a.keep;
    for (uint32_t i = t & (kWave - 1); i < (n < (uint32_t)a.keep ? n : (uint32_t)a.keep); i += kWave) kept[i] = s_kept[wave * kKept + i];
  }
  if constexpr (PASS == 0) {
    uint32_t* dst = a.partial + place * kBins;
    for (int i = t; i < kBins; i += kStatThreads) {
      uint32_t c = 0;
#pragma unroll
      for (int k = 0; k < kReplicas; ++k) c += s_hist[i * kReplicas + k];
      dst[i] = c;
    }
    // the counters of the passes after this one
    for (int i = blockIdx.x * kStatThreads + t; i < 2 * kBins; i += a.blocks * kStatThreads)
      a.hist[((int64_t)(1 + i / kBins) * a.n_slices + slice) * kBins + i % kBins] = 0u;
  } else {
    // A few hundred values of a workgroup share the digits of a wanted rank: its counters go to the slice's one by one.
    uint32_t* dst = a.hist + ((int64_t)PASS * a.n_slices + slice) * kBins;
    for (int i = t; i < (PASS == 2 ? 2048 : kBins); i += kStatThreads) {
      const uint32_t c = s_hist[i];
      if (c != 0) __hip_atomic_fetch_add(dst + i, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if constexpr (PASS == 2) {
    // The workgroup that finishes a slice goes on to its last digit and outputs, a launch less (3.8 us of 55).
    __shared__ int s_last;
    // Each wave's additions have reached the memory before the workgroup arrives, and nothing else that the last one reads
    // was written in this launch: no cache has to be written back (as a fence of each wave, that took 65 us).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0) s_last = __hip_atomic_fetch_add(a.arrived + slice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u;
    __syncthreads();
    if (s_last) stat_finish(a, slice, s_scan, s_digit, s_rest, prefix, rank);
  }
  if (PASS == 0 && t == 0) {
    if (blockIdx.x == 0) a.arrived[slice] = 0u;
    if (a.bad != nullptr && (s_flags & kSawBadRow)) *a.bad = 1;
    double total = 0.0;
    for (int w = 0; w < kStatThreads / kWave; ++w) total += s_sum[w];
    a.sums[place] = total;
    a.flags[place] = s_flags;
  }
}

// The first pass's counts: hist[bin] = sum of the workgroups'.  A wave reads 64 neighbouring bins of every sixteenth workgroup, all its
// reads in flight at once (with four waves to 64 bins, four rounds of reads each, the kernel took 9 us instead of 4).
__global__ __launch_bounds__(kStatThreads) void stat_reduce_kernel(StatArgs a) {
  constexpr int WAVES = kStatThreads / kWave;
  __shared__ uint32_t s_part[WAVES][kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int bin = blockIdx.x * kWave + lane, slice = blockIdx.y;
  const uint32_t* src = a.partial + (int64_t)slice * a.blocks * kBins + bin;
  uint32_t c = 0;
#pragma unroll 16
  for (int b = wave; b < a.blocks; b += WAVES) c += src[(int64_t)b * kBins];
  s_part[wave][lane] = c;
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 1; w < WAVES; ++w) c += s_part[w][lane];
    a.hist[(int64_t)slice * kBins + bin] = c;
  }
}

// Workgroups per slice: one per CU over all slices, each with at least four rows per lane of what a lane reads of a row at a
// time.  A short sample is the length of its chains, the counters' additions in LDS most of all, not the sum of its workgroups
// (32 values per lane / four rows: 150 000 x 6 in slices of one column 88 / 37 us, 5000 x 75 39 / 26, 3000 x 50 31 / 25, 1000 x 64 27 /
// 25, 50 000 x 128 in slices of 32 level; two rows of four columns lose: 10 000 x 128 28 / 30).
int stat_blocks(int64_t m, int64_t cols, int64_t slice, int64_t n_slices) {
  const int64_t width = cols < slice ? cols : slice;
  const int64_t least = width % 4 == 0 ? 16 : width % 2 == 0 ? 8 : 4;
  int64_t b = ceil_div(m * width, (int64_t)kStatThreads * least);
  const int64_t cap = n_slices >= kMaxBlocks / 4 ? 4 : kMaxBlocks / n_slices;
  b = b > cap ? cap : b;
  return (int)(b < 1 ? 1 : b);
}

int64_t round256(int64_t v) { return (v + 255) / 256 * 256; }

int stat_keep(int64_t blocks, int64_t n_slices) {
  return n_slices * blocks <= kRoomBlocks ? kKept : n_slices * blocks <= kKeepBlocks ? kKept / 2 : 0;
}

// Whether the first pass keeps values for the second: where they are expected to fit, with a lane's column group the same in
// every row (the first rows are a sample of all columns then), and from three million values on.  Finding the window takes
// the first pass 3 us, and a smaller sample is read as quickly again (10 000 x 128: 33 us, 35 with the window; 50 000 x 75
// 56 and 48).
bool stat_ahead(const StatArgs& a, int v) {
  const int64_t width = a.slice, groups = width / v;
  if (a.keep == 0 || groups > kStatThreads) return false;
  const double all = (double)a.m * (double)width, own = all / a.blocks;              // values of a slice, of a workgroup
  double n = (double)kInFlight * (double)(kStatThreads / groups) * (double)width;                  // of its first round
  n = n < own ? n : own;
  const double p = (double)(a.ranks[0] > a.ranks[1] ? a.ranks[0] : a.ranks[1]) / all;
  const double q = (double)(a.ranks[2] < a.ranks[3] ? a.ranks[2] : a.ranks[3]) / all;
  const double part = p + (6.0 * sqrt(n * p * (1.0 - p)) + 4.0) / n + 1.0 - q + (6.0 * sqrt(n * q * (1.0 - q)) + 4.0) / n + 0.005;
  return a.m * a.cols >= 3000000 && 1.3 * part * own / kStatWaves <= (double)a.keep;
}

struct StatLayout { int64_t hist, state, sums, flags, kept, n_kept, arrived, windows, total; };
StatLayout stat_layout(int64_t blocks, int64_t n_slices) {
  StatLayout l;
  l.hist = round256(n_slices * blocks * kBins * 4);
  l.state = l.hist + round256(3 * n_slices * kBins * 4);
  l.sums = l.state + round256(n_slices * (int64_t)sizeof(StatState));
  l.flags = l.sums + round256(n_slices * blocks * 8);
  l.kept = l.flags + round256(n_slices * blocks * 4);
  l.n_kept = l.kept + round256(n_slices * blocks * kStatWaves * stat_keep(blocks, n_slices) * 4);
  l.arrived = l.n_kept + round256(n_slices * blocks * kStatWaves * 4);
  l.windows = l.arrived + round256(n_slices * 4);
  l.total = l.windows + round256(n_slices * blocks * 2 * 4);
  return l;
}

// checked: recorded behind the first pass, which has then reported the row ids outside the table; or null.
template <int V>
hipError_t stat_launch(const StatArgs& a, hipEvent_t checked, hipStream_t st) {
  const dim3 grid((unsigned)a.blocks, (unsigned)a.n_slices), rgrid(kBins / kWave, (unsigned)a.n_slices);
  stat_pass_kernel<0, V><<<grid, kStatThreads, 0, st>>>(a);
  const hipError_t e = checked != nullptr ? hipEventRecord(checked, st) : hipSuccess;
  stat_reduce_kernel<<<rgrid, kStatThreads, 0, st>>>(a);
  stat_pass_kernel<1, V><<<grid, kStatThreads, 0, st>>>(a);
  stat_pass_kernel<2, V><<<grid, kStatThreads, 0, st>>>(a);
  return e;
}

int stat_check(const char* what, int64_t m, int64_t cols, int64_t slice) {
  F2CGT_REQUIRE(m > 0 && cols > 0 && slice > 0, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  F2CGT_REQUIRE(cols < (1ll << 24) && ceil_div(cols, slice) <= 65535, F2CGT_E_UNSUPPORTED, "%s: too many columns or slices", what);
  return 0;
}

}  // namespace
}  // namespace f2cgt

using namespace f2cgt;

extern "C" int64_t f2cgt_abs_order_stats_workspace_bytes(int64_t m, int64_t cols, int64_t column_slice) {
  if (m <= 0 || cols <= 0 || column_slice <= 0) return 0;
  const int64_t n_slices = ceil_div(cols, column_slice);
  return stat_layout(stat_blocks(m, cols, column_slice, n_slices), n_slices).total;
}

namespace {
int order_stats(const char* what, const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                int64_t column_slice, const int64_t* ranks, const float* weights, void* workspace, int64_t workspace_bytes,
                double* out, float* books, int32_t* bad, void* checked, void* stream) {
  if (int rc = stat_check(what, m, cols, column_slice)) return rc;
  F2CGT_REQUIRE(ld >= cols && num_rows > 0 && (rows != nullptr || m <= num_rows), F2CGT_E_INVALID,
                "%s: the sample does not fit the table", what);
  F2CGT_REQUIRE(x && ranks && workspace && out && aligned(workspace, 256), F2CGT_E_INVALID,
                "%s: null buffer or misaligned workspace", what);
  F2CGT_REQUIRE(workspace_bytes >= f2cgt_abs_order_stats_workspace_bytes(m, cols, column_slice), F2CGT_E_INVALID,
                "%s: workspace too small", what);
  const int64_t n_slices = ceil_div(cols, column_slice);
  const int64_t full = (cols < column_slice ? cols : column_slice) * m, last = (cols - (n_slices - 1) * column_slice) * m;
  F2CGT_REQUIRE(full < (1ll << 32), F2CGT_E_UNSUPPORTED, "%s: a slice of the sample has more than 2^32 values", what);
  for (int k = 0; k < 8; ++k) {
    F2CGT_REQUIRE(ranks[k] >= 0 && ranks[k] < (k < 4 ? full : last), F2CGT_E_INVALID, "%s: rank %lld out of range", what,
                  (long long)ranks[k]);
  }
  StatArgs a{};
  a.x = x; a.rows = rows; a.m = m; a.num_rows = num_rows; a.ld = ld;
  a.cols = (int)cols; a.slice = (int)(column_slice < cols ? column_slice : cols); a.n_slices = (int)n_slices;
  a.blocks = stat_blocks(m, cols, column_slice, n_slices);
  for (int k = 0; k < 8; ++k) a.ranks[k] = (uint64_t)ranks[k];
  const StatLayout l = stat_layout(a.blocks, n_slices);
  char* ws = static_cast<char*>(workspace);
  a.partial = reinterpret_cast<uint32_t*>(ws);
  a.hist = reinterpret_cast<uint32_t*>(ws + l.hist);
  a.state = reinterpret_cast<StatState*>(ws + l.state);
  a.sums = reinterpret_cast<double*>(ws + l.sums);
  a.flags = reinterpret_cast<uint32_t*>(ws + l.flags);
  a.keep = stat_keep(a.blocks, n_slices);
  a.kept = reinterpret_cast<uint32_t*>(ws + l.kept);
  a.n_kept = reinterpret_cast<uint32_t*>(ws + l.n_kept);
  a.arrived = reinterpret_cast<uint32_t*>(ws + l.arrived);
  a.windows = reinterpret_cast<uint32_t*>(ws + l.windows);
  a.bad = bad;
  a.out = out;
  a.books = books;
  if (books != nullptr)
    for (int k = 0; k < 4; ++k) a.weights[k] = weights[k];
  // widest access that every slice of every row is a multiple of
  const int64_t last_width = cols - (n_slices - 1) * column_slice;
  auto fits = [&](int v) {
    return ld % v == 0 && (n_slices == 1 || column_slice % v == 0) && last_width % v == 0 && aligned(x, 4 * v);
  };
  hipStream_t st = as_stream(stream);
  hipEvent_t ev = static_cast<hipEvent_t>(checked);
  a.ahead = stat_ahead(a, fits(4) ? 4 : fits(2) ? 2 : 1) ? 1 : 0;
  const hipError_t e = fits(4) ? stat_launch<4>(a, ev, st) : fits(2) ? stat_launch<2>(a, ev, st) : stat_launch<1>(a, ev, st);
  if (e != hipSuccess) return fail((int)e, "%s: cannot record the event: %s", what, hipGetErrorString(e));
  return launch_status(what);
}
}  // namespace

extern "C" int f2cgt_abs_order_stats(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows,
                                     int64_t cols, int64_t column_slice, const int64_t* ranks, void* workspace,
                                     int64_t workspace_bytes, double* out, void* stream) {
  return order_stats("abs_order_stats", x, ld, rows, m, num_rows, cols, column_slice, ranks, nullptr, workspace,
                     workspace_bytes, out, nullptr, nullptr, nullptr, stream);
}

extern "C" int f2cgt_sq_codebooks(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                                  int64_t column_slice, const int64_t* ranks, const float* weights, void* workspace,
                                  int64_t workspace_bytes, double* stats, float* codebooks, void* stream) {
  F2CGT_REQUIRE(weights && codebooks, F2CGT_E_INVALID, "sq_codebooks: null buffer");
  return order_stats("sq_codebooks", x, ld, rows, m, num_rows, cols, column_slice, ranks, weights, workspace,
                     workspace_bytes, stats, codebooks, nullptr, nullptr, stream);
}

extern "C" int f2cgt_sq_codebooks_checked(const float* x, int64_t ld, const int64_t* rows, int64_t m, int64_t num_rows, int64_t cols,
                                          int64_t column_slice, const int64_t* ranks, const float* weights, void* workspace,
                                          int64_t workspace_bytes, double* stats, float* codebooks, int32_t* bad_row, void* checked,
                                          void* stream) {
  F2CGT_REQUIRE(weights && codebooks && bad_row && checked, F2CGT_E_INVALID, "sq_codebooks_checked: null buffer or event");
  return order_stats("sq_codebooks_checked", x, ld, rows, m, num_rows, cols, column_slice, ranks, weights, workspace,
                     workspace_bytes, stats, codebooks, bad_row, checked, stream);
}
