// Nearest-centre labels on the matrix cores: kmeans_predict up to 64 dimensions, the codes of all column slices
// of a table in one launch (vq_encode_slices), and the training step of all slices of a sample (kmeans_slices_step,
// which adds the rows up by label instead of writing the labels).
//
// The distances are never written.  For L2 the kernel works on x - mu and c - mu (mu = mean of the centres) where that
// matters: a common offset of the data then costs nothing.  For cosine the normalised centres lose their mean direction
// m when |m| > 1/2 (argmin -x . c^ = argmin -x . (c^ - m)): the scores then resolve the differences between the centres'
// directions, which is all that data far from the origin leaves.  Scores use the expanded form (|c|^2 - 2 x.c, the row
// constant |x|^2 dropped).
//
// x . c comes from two fp16 pieces per fp32 value: x and the centres are scaled by powers of two (a row by its own norm,
// the centres by the largest) so that every norm lies near 2^14; then the leading piece has 11 significant bits, the
// second one 11 more or an absolute error below 2^-14, i.e. 2^-27 of the norm, and of the four piece products the three of
// relative size >= 2^-11 are evaluated.  What is dropped (2^-22 of |x||c|) is less than what the matrix core's alignment
// cuts from the leading products.  (Three bf16 pieces, six products, were exact to the last bit and no better after that
// cut, at twice the matrix instructions, 1.6 times the conversions and half as much LDS again.)
//
// What bounds it: the issue of vector and matrix instructions, which hardly run side by side on a SIMD (measured with two
// waves on it: six of the matrix instructions 194 clocks, 96 v_fma 220, both 396), behind that the staging of a launch, 4 us
// at 16 dimensions and 7 at 32 by time stamps: centres from memory, their means, norms and pieces.
// Against three bf16 pieces with (best, second) kept per tile: 1e6 x 32, 256 centres, L2 121 -> 79 us; 1e6 x 16 cosine
// 69 -> 47, 150 000 x 16 26 -> 17.5; 1e6 x 16 against 1024 centres 430 -> 154; 500 000 x 128 in slices of 16 229 -> 149.
// A wave owns 32 rows of x at a time and walks the centres a 32 x 32 tile at a time, A = centre tile (LDS), B = x tile (registers),
// so that a lane holds 16 scores of ONE row per tile.  It does not look for the best two of them: it keeps, over the T
// tiles of a chunk, the minimum of every slot (a class of T centres), half an instruction per score, and only the 16
// minima of a chunk go through the (best, second) tree.  The T centres of the winning class are evaluated again at the
// end (their dot products as v_dot2 on the same pieces, each half of the wave its own dimensions), which finds the label
// and the runner-up inside the class.  Rows whose two best scores are closer than the rounding bound of these evaluations
// are decided exactly: fp32 narrows the centres down, float64 decides on the original arrays, so the label is the true
// first minimum (cosine: of the directions; the clamp of |x||c| at 1e-8 counts only among those that float64 decides).
// 4.3e6 rows of 4 to 48 dimensions, 40 mixtures of sizes, offsets, grids and scales: no label away from float64's but the
// 1534 that the clamp makes, as many as with three bf16 pieces.
#include "assign.hpp"
#include "assign_exact.hpp"

namespace f2cgt {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4_dword __attribute__((ext_vector_type(4), aligned(4)));   // loaded from any float's address
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

// Absolute part of the near-tie bound: products that fall below the smallest normal fp32 number, which the relative
// bound does not see.  A few hundred such terms stay below this.
constexpr float kTinyGap = 1e-33f;

// One workgroup per CU, of as many waves as the registers allow (168 at three per SIMD): its waves share one copy of the
// centres and one counter.
constexpr int assign_threads(int steps) { return steps <= 3 ? 768 : 512; }
constexpr size_t kAssignLds = 96 * 1024;

struct AssignArgs {
  const float* x;
  const float* centers;
  int64_t* lab64;
  uint8_t* lab8;
  int64_t m;
  int n, k, metric, n_pad;
  // several column slices of a table, each against its own centres (slices == 1: rows of ldx floats, labels
  // label_stride apart); the grid is a multiple of 8 * slices workgroups then
  int slices;
  int feat_dim;            // columns of the table; the last slice may have fewer than k
  int64_t ldx, label_stride, slice_step;   // slice_step: from a row of a slice to the same row of the next, in floats
  // training step: the rows' sums and counts by label instead of the labels
  const int32_t* stop;     // [slices]: nonzero = the slice's centres are final
  const uint32_t* keep;    // [slices][keep_words]: bit r % 32 of word r / 32 = row r takes part; null: all do
  int64_t keep_words;
  float* sums;             // [slices][shares][n * k + n]
  uint32_t* arrived;       // [slices]: cleared for the merging kernel
};

// Minima and maxima that keep a NaN (v_minimum3, v_maximum3): no instruction to quieten the operands first, and a row with
// a score that is no number ends in the exact evaluation.
__device__ __forceinline__ float min2(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float min3(float a, float b, float c) { return min2(min2(a, b), c); }

// Running (best, second) over 16 class minima.  A minimum carries its slot in its four lowest bits (one v_and_or, a
// change below 2^-19 of it that the near-tie bound includes), so that the index needs no compare and select of its own
// and the rest is a tree of three-way minima and medians: 39 instructions where compare, two selects and a median took
// 64.  An infinity with a slot in its low bits is a NaN: the caller evaluates rows whose scores could overflow exactly.
__device__ __forceinline__ void update_packed(const floatx16& mn, int ct, float& best, float& second, int& bct) {
  float p[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) p[v] = __int_as_float((__float_as_int(mn[v]) & ~15) | v);
  float lo[6], mid[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    lo[i] = min3(p[3 * i], p[3 * i + 1], p[3 * i + 2]);
    mid[i] = __builtin_amdgcn_fmed3f(p[3 * i], p[3 * i + 1], p[3 * i + 2]);
  }
  lo[5] = p[15];
  const float lo_a = min3(lo[0], lo[1], lo[2]), mid_a = __builtin_amdgcn_fmed3f(lo[0], lo[1], lo[2]);
  const float lo_b = min3(lo[3], lo[4], lo[5]), mid_b = __builtin_amdgcn_fmed3f(lo[3], lo[4], lo[5]);
  const float before = best;
  const float behind_a = max2(best, lo_a);
  best = min2(best, lo_a);
  const float behind_b = max2(best, lo_b);
  best = min2(best, lo_b);
  const float s0 = min3(mid[0], mid[1], mid[2]), s1 = min3(mid[3], mid[4], mid_a);
  second = min3(second, s0, s1);
  second = min3(second, mid_b, min2(behind_a, behind_b));
  bct = best < before ? ct : bct;
}

// The same with the slot kept beside the minimum.
__device__ __forceinline__ void update_plain(const floatx16& mn, int ct, float& best, float& second, int& bv, int& bct) {
  const float before = best;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float s = mn[v];
    const bool lt = s < best;
    second = __builtin_amdgcn_fmed3f(best, second, s);
    bv = lt ? v : bv;
    best = lt ? s : best;
  }
  bct = best < before ? ct : bct;
}

// What the lane of the lower and of the upper half of the wave holds, in both of them.
struct Halves { uint32_t lo, hi; };
__device__ __forceinline__ Halves halves(uint32_t v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return {r[0], r[1]};
}
__device__ __forceinline__ float add_halves(float v) {
  const Halves h = halves(__float_as_uint(v));
  return __uint_as_float(h.lo) + __uint_as_float(h.hi);
}

// Scale of a vector of squared norm `norm2`: the power of two that takes the norm to [2^13, 2^14).
__device__ __forceinline__ int norm_shift(float norm2) {
  return 13 - (((int)(__float_as_uint(norm2) >> 23) - 127) >> 1);
}
__device__ __forceinline__ float pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }   // -126 <= e <= 127

__device__ __forceinline__ void split2(float v, _Float16& hi, _Float16& lo) {
  hi = (_Float16)v;
  lo = (_Float16)(v - (float)hi);      // the difference is exact
}

// Exact assignment of one row by a whole wave.  The distances from the centre pieces in LDS, in fp32, leave the centres
// that can be the nearest one, usually two; float64 decides between those on the original arrays.
//   L2: unexpanded sum of (x' - c')^2 of the centred values, relative error (k + 3) 2^-24; a piece sum is within 2^-22
//   of its centre, which moves d^2 by at most 2^-21 d |c| <= 2^-22 (d^2 + |c|^2) <= 3 * 2^-22 (|x'|^2 + |c'|^2), and the
//   rounding of the centring by 2^-22 (|x'|^2 + |c'|^2): 4 * 2^-22 (9.6e-7) for each of two distances.
//   Cosine: -x . d with |d| <= cdev; fp32 sum, roundings of the normalisation and of m ((k + 2) cdev + 3) 2^-24 |x|, the
//   pieces 2^-22 |x| cdev, for each of two scores; products below the smallest normal float lose 2^-150 each (64 twice: 9e-44).
//   Where fp32 has no number for a distance (a centre beyond the range of the pieces, which |c|^2 beyond the largest float
//   admits; sums that overflow) it leaves nothing out: such a distance passes, and where it makes the limit no number, or
//   a row's dot products may overflow (|x| >= 1e38), every centre does.
template <int S>
__device__ __forceinline__ int exact_row(const AssignArgs& a, const float* __restrict__ xrow,
                                         const float* __restrict__ centers, float* xs, const half8* ap, const float* inv,
                                         int kx, int lane, const float* mu, float unscale, float cmax, float cdev) {
  const bool cosine = a.metric == F2CGT_METRIC_COSINE;
  const int n = a.n, k = a.k, piece = (a.n_pad >> 5) * S * 64;
  // The row goes through a wave-private LDS slot (16 S floats, zero padded), centred and as it is, and the loops over
  // the 8-dimension chunks stay rolled: this rare path must not raise the kernel's register count.  It is a chain of
  // latencies that a whole workgroup may wait for at the end, so what can be in flight together is.
  float* xo = xs + 16 * S;
  float own = 0.f;
  if (lane < 16 * S) {
    own = lane < kx ? xrow[lane] : 0.f;
    xo[lane] = own;
    own = cosine || lane >= k ? own : own - mu[lane];
    xs[lane] = own;
  }
  __builtin_amdgcn_wave_barrier();                       // LDS operations of one wave execute in order
  // distances of centres c0, c0 + 64, ... to the row (cosine: -x . c)
  constexpr int kKeep = 4;
  auto measure = [&](int c0, float (&d)[kKeep]) {
    const half8* q[kKeep];
#pragma unroll
    for (int i = 0; i < kKeep; ++i) {
      const int c = c0 + i * kWave < n ? c0 + i * kWave : 0;
      q[i] = ap + (c >> 5) * S * 64 + (c & 31);
      d[i] = 0.f;
    }
#pragma nounroll
    for (int ch = 0; ch < 2 * S; ++ch) {
      const float4 xa = *reinterpret_cast<const float4*>(xs + 8 * ch);
      const float4 xb = *reinterpret_cast<const float4*>(xs + 8 * ch + 4);
      const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
      for (int i = 0; i < kKeep; ++i) {
        const half8 p0 = q[i][ch * 32], p1 = q[i][piece + ch * 32];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float cv = ((float)p0[e] + (float)p1[e]) * unscale;
          const float df = cosine ? -cv : xv[e] - cv;    // dimensions >= k hold zeros on both sides
          d[i] = __fmaf_rn(cosine ? xv[e] : df, df, d[i]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kKeep; ++i) {
      const int c = c0 + i * kWave;
      d[i] = c < n && inv[c < n ? c : 0] != 0.f ? d[i] : INFINITY;   // (zero: no number)
    }
  };
  float keep[kKeep], d[kKeep];           // the first 256 centres' distances stay in registers
  measure(lane, keep);
  float nearest = fminf(fminf(keep[0], keep[1]), fminf(keep[2], keep[3]));
  for (int c = lane + kKeep * kWave; c < n; c += kKeep * kWave) {
    measure(c, d);
    nearest = fminf(nearest, fminf(fminf(d[0], d[1]), fminf(d[2], d[3])));
  }
  float xnorm2 = own * own;
  double xn = lane < 16 * S ? (double)xo[lane] * (double)xo[lane] : 0.0;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    nearest = fminf(nearest, __shfl_xor(nearest, off));
    xnorm2 += __shfl_xor(xnorm2, off);
    xn += __shfl_xor(xn, off);
  }
  // (cosine: |x| from the fp64 sum, its square may vanish in fp32)
  float limit = cosine ? nearest + (1.1920929e-7f * ((float)(k + 4) * cdev + 3.f) + 4.9e-7f * cdev) * (float)sqrt(xn) * 1.001f + 1e-43f
                       : nearest * (1.f + 1.1920929e-7f * (float)(k + 4)) + 1e-37f + 2.1e-6f * (xnorm2 + cmax);
  if (cosine && !(xn < 1e76)) limit = INFINITY;
  double bestv = DBL_MAX;
  int besti = INT_MAX;
  for (int c0 = lane; c0 < n; c0 += kKeep * kWave) {
    if (c0 != lane) measure(c0, d);
#pragma nounroll
    for (int i = 0; i < kKeep; ++i) {
      const int c = c0 + i * kWave;
      float di = c0 == lane ? keep[0] : d[0];
#pragma unroll
      for (int q = 1; q < kKeep; ++q) di = i == q ? (c0 == lane ? keep[q] : d[q]) : di;
      if (di > limit || c >= n) continue;                // (passes what is no number)
      // float64 on the original values, eight of the centre's in flight
      const float* cr = centers + (int64_t)c * k;
      double dot = 0.0, cn = 0.0;
#pragma nounroll
      for (int t0 = 0; t0 < k; t0 += 8) {
        float cv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) cv[e] = cr[t0 + e < k ? t0 + e : 0];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (t0 + e >= k) break;
          const double xv = xo[t0 + e], v = cv[e];
          if (cosine) {
            dot += xv * v;
            cn += v * v;
          } else {
            dot += (xv - v) * (xv - v);
          }
        }
      }
      if (cosine) {
        double den = sqrt(xn) * sqrt(cn);
        den = den > 1e-8 ? den : 1e-8;
        dot = 1.0 - dot / den;
      }
      if (dot < bestv) { bestv = dot; besti = c; }
    }
  }
  return first_minimum(bestv, besti);
}

// S: steps of 16 dimensions.  T: tiles of a chunk (a class has T centres).  PACKED: update_packed.  SUMS: the training
// step, which adds the rows up by label in LDS (n * (16 S + 1) doubles) and leaves a set of sums per workgroup.
// METRIC: the launch's, where it is fixed when the kernel is chosen, or kEither.
constexpr int kEither = -1;
template <int S, int T, bool PACKED, bool SUMS, int METRIC>
__global__ __launch_bounds__(assign_threads(S), S <= 3 ? 3 : 2) void assign_kernel(AssignArgs a) {
  constexpr int kThreads = assign_threads(S), kWaves = kThreads / kWave;
  constexpr int U = T == 1 ? 1 : 2;                              // tiles a step
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const float* __restrict__ x = a.x;
  const float* __restrict__ centers = a.centers;
  uint8_t* __restrict__ lab8 = a.lab8;
  const int64_t m = a.m;
  const int n = a.n, k = a.k, n_pad = a.n_pad;
  int64_t share = blockIdx.x, shares = gridDim.x;
  int slice = 0;
  if (a.slices > 1) {
    // Workgroups go round-robin to the 8 XCDs: with 8 shares side by side, the slices of a share run on one
    // XCD, whose L2 then serves the lines of x that two slices have in common and joins their code bytes.
    shares = gridDim.x / a.slices;
    if (shares & 7) {
      slice = blockIdx.x % a.slices;
      share = blockIdx.x / a.slices;
    } else {
      const int turn = blockIdx.x / (8 * a.slices), at = blockIdx.x % (8 * a.slices);
      slice = at >> 3;
      share = turn * 8 + (at & 7);
    }
    x += slice * a.slice_step;
    centers += (int64_t)slice * n * k;
    lab8 += slice;
  }
  if (SUMS && a.stop[slice] != 0) return;
  int kx = a.feat_dim - slice * k;                               // dimensions the rows have (zeros after them)
  kx = kx < k ? kx : k;
  const int64_t ldx = a.ldx, ldl = a.label_stride;
  const int n_ct = (n + 31) >> 5;                                // 32-centre tiles
  const int piece = (n_pad >> 5) * S * 64;                             // operands per piece
  half8* ap = reinterpret_cast<half8*>(smem_raw);                // [2][n_pad / 32][S][64]
  double* norm2 = reinterpret_cast<double*>(smem_raw + (size_t)2 * piece * 16);   // [n_pad] |c|^2
  float* bias = reinterpret_cast<float*>(norm2 + n_pad);         // [n_pad]
  float* inv = bias + n_pad;                                     // [n_pad] 1 / |c| (cosine) or 1; 0: no number
  int* flags = reinterpret_cast<int*>(inv + n_pad);              // max |c|^2, degenerate centre, draws, mean in use
  float* mu = reinterpret_cast<float*>(flags + 4);               // [16 S]
  float* psum = mu + 16 * S;                                     // [2][kThreads]
  float* xs = psum + 2 * kThreads + (threadIdx.x >> 6) * 32 * S;   // one row of x per wave, centred and as it is
  constexpr int kPitch = 16 * S + 1;                             // (odd: the centres' sums start in different banks)
  // SUMS: [n][kPitch] sums, then [n] counts.  In fp64: the LDS adds a float in 178 clocks per wave and CU, a double in 19
  // (measured, addresses as here; 32-bit integers 6): a step of six slices of 150 000 x 16 rows took 110 us, now 56.
  double* sums = reinterpret_cast<double*>(psum + 2 * kThreads + kWaves * 32 * S);
  uint32_t* counts = reinterpret_cast<uint32_t*>(sums + n * kPitch);
  const bool cosine = METRIC == kEither ? a.metric == F2CGT_METRIC_COSINE : METRIC == F2CGT_METRIC_COSINE;
  const int lane = threadIdx.x & 63;
  const int j = lane & 31;
  const int g = lane >> 5;
  const int64_t n_groups = (m + 31) / 32;
  // A workgroup owns a contiguous share of the row groups; its waves start with one each and draw the others through
  // a counter in LDS: a wave held up by exact re-evaluations simply takes fewer groups.
  const int64_t per_wg = (n_groups + shares - 1) / shares;
  const int64_t wg_lo = share * per_wg;
  const int64_t wg_hi = wg_lo + per_wg < n_groups ? wg_lo + per_wg : n_groups;
  if (!SUMS && wg_lo >= wg_hi) return;                           // the whole workgroup

  // Staging.  The centres are read once, into the places where their pieces go: item (centre c, chunk ch of 8 dimensions)
  // is operand lane (c % 32) + 32 (ch % 2) of step ch / 2 of tile c / 32, and its first four values lie where its leading
  // pieces go, the others where its second pieces go.  Column sums, norms and the conversion work there.  Dimensions from
  // k on and centres from n on are zeros.  The loops stay rolled: in a kernel that starts with cold instruction caches
  // straight-line code is what the staging waits for.
  constexpr int kChunks = 2 * S, kWidth = 16 * S;
  float4* lo4 = reinterpret_cast<float4*>(smem_raw);
  float4* hi4 = lo4 + piece;
  auto raw = [&](int c, int d) -> float {
    const int at = ((c >> 5) * S + (d >> 4)) * 64 + ((d >> 3) & 1) * 32 + (c & 31);
    return reinterpret_cast<const float*>((d & 4) ? hi4 + at : lo4 + at)[d & 3];
  };
  {
    const bool cvec = (k % 8 == 0) && ((reinterpret_cast<uintptr_t>(centers) & 15) == 0);
#pragma unroll 4
    for (int at = threadIdx.x; at < piece; at += kThreads) {
      const int c = at / (64 * S) * 32 + (at & 31), d0 = (at / 64 % S) * 16 + (at & 32) / 4;
      const bool in = c < n && d0 < k;
      const float* cr = centers + (in ? (int64_t)c * k + d0 : 0);
      float4 p = make_float4(0.f, 0.f, 0.f, 0.f), w = p;
      if (cvec) {
        p = reinterpret_cast<const float4*>(cr)[0];
        w = reinterpret_cast<const float4*>(cr)[1];
        if (!in) p = w = make_float4(0.f, 0.f, 0.f, 0.f);
      } else if (in) {
        p.x = cr[0];
        if (d0 + 1 < k) p.y = cr[1];
        if (d0 + 2 < k) p.z = cr[2];
        if (d0 + 3 < k) p.w = cr[3];
        if (d0 + 4 < k) w.x = cr[4];
        if (d0 + 5 < k) w.y = cr[5];
        if (d0 + 6 < k) w.z = cr[6];
        if (d0 + 7 < k) w.w = cr[7];
      }
      lo4[at] = p;
      hi4[at] = w;
    }
  }
  const bool ragged = kx < kWidth;          // there are operand places without a dimension
  float q[S][8] = {};                       // this lane's share of a row: dimensions 16 st + 8 g + e
  // Loads of a group's rows, issued always: two 16-byte loads per step, which take any float's address, from one address
  // for the group and an offset for the lane.  A row of fewer than 16 S values is read past its end, into the rows after
  // it (the places without a dimension are cleared before they are used): the groups whose last row has enough of them
  // behind it.  The others' step that a row ends in is read in pieces that the row's length is a multiple of (four, two or
  // one value).  Lanes past the last row read the group's first.
  const int64_t behind = ragged ? (kWidth + ldx - 1) / ldx : 0;
  const int64_t whole_groups = ldx >= (1 << 24) ? 0 : !ragged ? n_groups : m > behind ? (m - behind) / 32 : 0;
  const uint32_t row_at = 4u * ((uint32_t)j * (uint32_t)ldx + 8u * (uint32_t)g);   // bytes (below 4 GB: ldx < 2^24)
  auto load_rows = [&](int64_t grp) {
    const int64_t left = m - grp * 32;
    if (grp < whole_groups) {
      const char* group = reinterpret_cast<const char*>(x + grp * 32 * ldx);
      const uint32_t at = j < left ? row_at : 32u * (uint32_t)g;
#pragma unroll
      for (int st = 0; st < S; ++st) {
        const floatx4_dword u = *reinterpret_cast<const floatx4_dword*>(group + (at + 64 * st));
        const floatx4_dword w = *reinterpret_cast<const floatx4_dword*>(group + (at + 64 * st + 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) { q[st][e] = u[e]; q[st][4 + e] = w[e]; }
      }
    } else {
      int from = 8 * g;                     // (opaque: the places below are not worth registers over the loop)
      asm volatile("" : "+v"(from));
      const float* __restrict__ xr = x + (grp * 32 + (j < left ? j : 0)) * ldx;
      int now = kx;
      asm volatile("" : "+s"(now));
      auto pieces = [&](int st, auto width) {
        constexpr int V = decltype(width)::value;
        typedef float piece __attribute__((ext_vector_type(V), aligned(4)));
#pragma unroll
        for (int i = 0; i < 8; i += V) {
          const int c = from + 16 * st + i;
          const piece u = *reinterpret_cast<const piece*>(xr + (c < now ? c : 0));
#pragma unroll
          for (int e = 0; e < V; ++e) q[st][i + e] = u[e];
        }
      };
#pragma unroll
      for (int st = 0; st < S; ++st) {
        if (16 * st >= now) continue;
        // value by value throughout, these rows' reads were most of a short call: 33 rows of 40 dimensions 12.6 -> 17.8 us
        if (16 * st + 16 <= now || now % 4 == 0) pieces(st, std::integral_constant<int, 4>{});
        else if (now % 2 == 0) pieces(st, std::integral_constant<int, 2>{});
        else pieces(st, std::integral_constant<int, 1>{});
      }
    }
  };
  int64_t grp = wg_lo + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  load_rows(grp < wg_hi ? grp : wg_lo < n_groups ? wg_lo : 0);
  if constexpr (SUMS) {
    for (int i = threadIdx.x; i < n * kPitch; i += kThreads) sums[i] = 0.0;
    for (int i = threadIdx.x; i < n; i += kThreads) counts[i] = 0u;
    if (share == 0 && threadIdx.x == 0) a.arrived[slice] = 0u;
  }
  for (int c = threadIdx.x; c < n_pad; c += kThreads) norm2[c] = 0.0;
  if (threadIdx.x < 4) flags[threadIdx.x] = threadIdx.x == 2 ? kWaves : 0;
  // Column sums of raw * weight (and of the squares), a thread per column and row class; then the mean by the first wave.
  auto column_mean = [&](bool weighted) {
    constexpr int kParts = kThreads / kWidth;
    const int col = threadIdx.x % kWidth, part = threadIdx.x / kWidth;
    float sum = 0.f, sq = 0.f;
    if (part < kParts) {
#pragma unroll 4
      for (int c = part; c < n; c += kParts) {
        const float v = raw(c, col);
        sum = weighted ? __fmaf_rn(v, inv[c], sum) : sum + v;
        sq = __fmaf_rn(v, v, sq);
      }
    }
    psum[threadIdx.x] = sum;
    psum[kThreads + threadIdx.x] = sq;
    __syncthreads();
    if (threadIdx.x < 64) {                                      // the first wave, all of it
      float mt = 0.f, st = 0.f;
      constexpr int kSide = 64 / kWidth;                         // lanes to a column
      if (lane < kSide * kWidth)
#pragma unroll
        for (int q = 0; q < (kParts + kSide - 1) / kSide; ++q) {
          const int from = (q * kSide + lane / kWidth) * kWidth + lane % kWidth;
          if (from < kParts * kWidth) {
            mt += psum[from];
            st += psum[kThreads + from];
          }
        }
      if constexpr (kSide >= 2) { mt += __shfl_xor(mt, 32); st += __shfl_xor(st, 32); }
      if constexpr (kSide == 4) { mt += __shfl_xor(mt, 16); st += __shfl_xor(st, 16); }
      if (lane >= kWidth) mt = st = 0.f;
      mt /= (float)n;
      st /= (float)n;
      float m2 = mt * mt, var = st - mt * mt;                    // dimensions from k on hold zeros
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        m2 += __shfl_xor(m2, off);
        var += __shfl_xor(var, off);
      }
      const bool use = m2 < INFINITY && (weighted ? m2 > 0.25f : m2 > 2.f * (var > 0.f ? var : 0.f));
      if (lane < kWidth) mu[lane] = use ? mt : 0.f;
      if (lane == 0) flags[3] = use ? 1 : 0;
    }
    __syncthreads();
  };
  __syncthreads();
  // L2: mu[t] = mean of the centres in dimension t, subtracted from every centre and every x (the
  // distances do not change, the cancellation of the expanded form does).  It is used only when it
  // matters, |mu|^2 above twice the summed variance of the centres (otherwise mu is zero and the
  // subtraction of the hot loop is skipped).
  if (!cosine) column_mean(false);
  // Norms, in fp64 (1 / |c| must be good to a rounding or two): a thread per chunk, then a thread per centre.
#pragma nounroll
  for (int at = threadIdx.x; at < piece; at += kThreads) {
    const int c = at / (64 * S) * 32 + (at & 31), d0 = (at / 64 % S) * 16 + (at & 32) / 4;
    const float4 p = lo4[at], w = hi4[at];
    float v[8] = {p.x, p.y, p.z, p.w, w.x, w.y, w.z, w.w};
    double sq = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (!cosine) v[e] -= mu[d0 + e];
      sq += (double)v[e] * (double)v[e];
    }
    unsafeAtomicAdd(norm2 + c, sq);
  }
  __syncthreads();
  float top = 0.f;
  for (int c = threadIdx.x; c < n_pad; c += kThreads) {
    const double cn64 = norm2[c];
    const float cn = (float)cn64;
    float sc = 1.f;
    if (cosine) sc = (float)(1.0 / sqrt(cn64 > 1e-60 ? cn64 : 1e-60));
    // A centre that is no number has no distance that compares and never wins; its operands are zeros and its bias that
    // of the padding: a minimum of the classes below is NaN as soon as one of its scores is.
    const bool number = cn64 < INFINITY;
    inv[c] = number ? sc : 0.f;
    // padding: finite where the lowest bits of a class minimum are its slot
    bias[c] = c >= n || !number ? FLT_MAX : (cosine ? 0.f : cn);
    if (c < n && !cosine && number) top = fmaxf(top, cn);
    // a centre without a direction, or (cosine) none that is a number
    if (c < n && cosine && !(cn > 1e-12f)) atomicOr(flags + 1, 1);
    if (c < n && cosine && !number) atomicOr(flags + 1, 2);
  }
  if (!cosine) {                                                 // one LDS atomic per wave
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    if (lane == 0) atomicMax(flags, __float_as_int(top));
  }
  __syncthreads();
  // Cosine: argmin_c -x . c^ = argmin_c -x . (c^ - m) for any m, and with m the mean of
  // the normalised centres c^ the operands of the matrix core shrink to the spread of the centres'
  // directions: what data far from the origin leaves of the evaluation's resolution goes to the
  // differences between centres.  Used when |m| > 1/2; mu[] then holds m (zeros otherwise).
  const bool degenerate = flags[1] != 0;         // centres without a direction: no candidate filter for cosine
  if (cosine && !degenerate) {
    column_mean(true);
  } else if (cosine) {
    if (threadIdx.x < kWidth) mu[threadIdx.x] = 0.f;
    __syncthreads();
  }
  // all the centres share one scale: cosine operands are at most 1, or 2 without their mean
  const int c_shift = cosine ? 13 : norm_shift(__int_as_float(flags[0]));
  const float c_scale = pow2(c_shift);
  float dev2max = 0.f;
#pragma nounroll
  for (int at = threadIdx.x; at < piece; at += kThreads) {
    const int c = at / (64 * S) * 32 + (at & 31), d0 = (at / 64 % S) * 16 + (at & 32) / 4;
    const float4 p = lo4[at], w = hi4[at];
    const float v[8] = {p.x, p.y, p.z, p.w, w.x, w.y, w.z, w.w};
    const float sc = inv[c];
    half8 p0, p1;
    float dev2 = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool in = c < n && d0 + e < k && sc != 0.f;
      const float val = in ? (cosine ? v[e] * sc : v[e]) - mu[d0 + e] : 0.f;
      dev2 = __fmaf_rn(val, val, dev2);
      _Float16 a0, a1;
      split2(val * c_scale, a0, a1);
      p0[e] = a0; p1[e] = a1;
    }
    dev2max = fmaxf(dev2max, dev2);                              // largest 8-dimension share of |c^ - m|^2
    ap[at] = p0;
    ap[piece + at] = p1;
  }
  if (cosine && flags[3] == 1) {                                 // one LDS atomic per wave
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) dev2max = fmaxf(dev2max, __shfl_xor(dev2max, off));
    if (lane == 0) atomicMax(flags, __float_as_int(dev2max));
  }
  __syncthreads();
  const float cmax = __int_as_float(flags[0]);
  const bool use_mu = !cosine && __builtin_amdgcn_readfirstlane(flags[3]) != 0;
  // cosine: upper bound of |c^ - m| over the centres (1 without the mean; never above 2)
  float cdev = 1.f;
  if (cosine && !degenerate && flags[3] == 1) {
    cdev = sqrtf((float)kChunks * cmax) * 1.0001f;
    cdev = cdev < 2.f ? cdev : 2.f;
  }
  cdev = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(cdev)));
  const int biased_from = (flags[1] & 2) ? 0 : n >> 5;           // cosine: the first tile with biases

  // Error bound of one score in units of 2^-24 (|x|^2 + max |c|^2), which is >= 2 |x||c| = P and
  // >= |c|^2: each of the S leading instructions cuts its 17 addends at 2^-22 of the largest
  // (<= P): 68 S; the small pairs (2^-11 P and below) together stay below 1; the pieces of x and c
  // stop at 2^-22 of the value (4 P each way in these units, on half of P) and the dropped pair is
  // as large: 6; below the smallest normal half 1; the bias sum k + 1; its addition 2; the rounding
  // of x - mu and c - mu 4 (L2: 2^-22 (|x|^2 + |c|^2)); 2 spare.  A class is decided by fp32 sums of
  // the same pieces (3 * 8 S roundings of partial sums <= P / 2: 24 S), which stays below.  Doubled
  // for the two scores of a gap.
  const float unit = 5.9604645e-8f * (float)(2 * (68 * S + k + 17));
  // Packed minima have to be finite.  An L2 score |c|^2 - 2 x . c is at most 2 (|x|^2 + |c|^2), which may exceed the
  // largest float (3.4e38) while the bound above is finite; cosine has |x . c^| <= |x|, below 2e19 wherever |x|^2 is finite.
  const float finite_below = cosine ? INFINITY : 1.6e38f;
  int label = 0;
  int64_t labelled = -1;                    // the group whose labels are still to be stored
  auto store_labels = [&]() {
    const int64_t row = labelled * 32 + j;
    if (row < m && g == 0) {
      if (a.lab64) a.lab64[row * ldl] = label;
      if (lab8) lab8[row * ldl] = (uint8_t)label;
    }
  };
  while (grp < wg_hi) {
    int drawn = 0;
    if (lane == 0) drawn = atomicAdd(flags + 2, 1);
    uint32_t kept = ~0u;                    // the group's rows that take part
    if (SUMS && a.keep != nullptr) kept = a.keep[slice * a.keep_words + grp];
    half8 xp[S][2];
    float own[SUMS ? S : 1][8];
    if constexpr (SUMS) {
#pragma unroll
      for (int st = 0; st < S; ++st)
#pragma unroll
        for (int e = 0; e < 8; ++e) own[st][e] = q[st][e];
    }
    if (ragged) {
      int has = kx - 8 * g;                 // compared here: as lane masks kept over the loop these were spilled scalars
      asm volatile("" : "+v"(has));
#pragma unroll
      for (int st = 0; st < S; ++st)
#pragma unroll
        for (int e = 0; e < 8; ++e) q[st][e] = 16 * st + e < has ? q[st][e] : 0.f;
    }
    if (use_mu) {                           // (zero from dimension k on)
#pragma unroll
      for (int st = 0; st < S; ++st) {
        const float4* mu4 = reinterpret_cast<const float4*>(mu + 16 * st + 8 * g);
        const float4 u = mu4[0], w = mu4[1];
        q[st][0] -= u.x; q[st][1] -= u.y; q[st][2] -= u.z; q[st][3] -= u.w;
        q[st][4] -= w.x; q[st][5] -= w.y; q[st][6] -= w.z; q[st][7] -= w.w;
      }
    }
    float sum = 0.f;
#pragma unroll
    for (int st = 0; st < S; ++st)
#pragma unroll
      for (int e = 0; e < 8; ++e) sum = __fmaf_rn(q[st][e], q[st][e], sum);
    const float xn = add_halves(sum);
    const int x_shift = norm_shift(xn);
    const float x_scale = -pow2(x_shift);
    // what takes a scaled product to -x . c (cosine) or -2 x . c
    const float back = ldexpf(cosine ? 1.f : 2.f, -(x_shift + c_shift));
    // The leading pieces, two with one conversion, rounded as one by one (cut off they would leave the second ones to end at
    // 2^-22 of the value instead of 2^-23, at the same cost).
#pragma unroll
    for (int st = 0; st < S; ++st)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const floatx2 scaled = {q[st][e] * x_scale, q[st][e + 1] * x_scale};
        const half2v lead = __builtin_convertvector(scaled, half2v);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          xp[st][0][e + i] = lead[i];
          xp[st][1][e + i] = (_Float16)__fmaf_rn(q[st][e + i], x_scale, -(float)lead[i]);   // (exact before the rounding)
        }
      }
    // The next rows travel while these are scored, behind the last ones' labels: the wait for the rows is one for every
    // access before them too, and a store that has just been issued takes as long as the rows.
    if (!SUMS && labelled >= 0) store_labels();
    const int64_t next = wg_lo + __builtin_amdgcn_readfirstlane(drawn);
    load_rows(next < wg_hi ? next : grp);
    asm volatile("" ::: "memory");

    float best = INFINITY, second = INFINITY;
    int bv = 0, bct = 0;
    for (int ct0 = 0; ct0 < n_ct; ct0 += T) {
      floatx16 mn;
#pragma unroll
      for (int tp = 0; tp < T; tp += U) {
        if (tp > 0 && ct0 + tp >= n_ct) break;
        // an odd last tile counts twice: its minima do not change
        int ct[U];
#pragma unroll
        for (int u = 0; u < U; ++u) ct[u] = ct0 + tp + u < n_ct ? ct0 + tp + u : ct0 + tp;
        half8 op[U][2][S];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int st = 0; st < S; ++st) op[u][h][st] = ap[h * piece + (ct[u] * S + st) * 64 + lane];
        // Piece pairs (x piece, centre piece).  The matrix core aligns the 16 products and C of an
        // instruction to the largest of them and keeps about 24 bits below it (measured: a unit
        // product next to +-2^24 survives, next to +-2^28 it does not), so the small pairs are
        // summed first, from zero, the leading pair last, and the bias, as large as the whole dot
        // product, is added on the vector ALU: the leading products are then cut at 2^-22 of their
        // own size, not of |c|^2 plus the running sum.
        constexpr int px[3] = {1, 0, 0};
        constexpr int pc[3] = {0, 1, 0};
        floatx16 zero, acc[U];
#pragma unroll
        for (int v = 0; v < 16; ++v) zero[v] = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u)
          acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(op[u][pc[0]][0], xp[0][px[0]], zero, 0, 0, 0);
#pragma unroll
        for (int term = 0; term < 3; ++term)
#pragma unroll
          for (int st = 0; st < S; ++st) {
            if (term == 0 && st == 0) continue;
#pragma unroll
            for (int u = 0; u < U; ++u)
              acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(op[u][pc[term]][st], xp[st][px[term]], acc[u], 0, 0, 0);
          }
        // L2: the score.  Cosine: a scaled product is as good for comparing (the best two are scaled back below), and
        // only padding has a bias, the largest float.
        if (!cosine || ct[U - 1] >= biased_from) {
          const float to_score = cosine ? 1.f : back;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const float* bp = bias + ct[u] * 32 + 4 * g;
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
              const float4 t4 = *reinterpret_cast<const float4*>(bp + 8 * v4);
              acc[u][4 * v4] = __fmaf_rn(acc[u][4 * v4], to_score, t4.x);
              acc[u][4 * v4 + 1] = __fmaf_rn(acc[u][4 * v4 + 1], to_score, t4.y);
              acc[u][4 * v4 + 2] = __fmaf_rn(acc[u][4 * v4 + 2], to_score, t4.z);
              acc[u][4 * v4 + 3] = __fmaf_rn(acc[u][4 * v4 + 3], to_score, t4.w);
            }
          }
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          mn[v] = U == 1 ? acc[0][v] : tp > 0 ? min3(acc[0][v], acc[U - 1][v], mn[v]) : min2(acc[0][v], acc[U - 1][v]);
        }
      }
      if constexpr (PACKED) update_packed(mn, ct0, best, second, bct);
      else update_plain(mn, ct0, best, second, bv, bct);
    }
    // the two halves of the wave have the same row and other classes; both go on with the winner
    const int slot = PACKED ? __float_as_int(best) & 15 : bv;
    int cls = bct * 32 + 8 * (slot >> 2) + 4 * g + (slot & 3);   // the class's centre in its chunk's first tile
    const Halves hb = halves(__float_as_uint(best)), hs = halves(__float_as_uint(second)), hc = halves((uint32_t)cls);
    const float b0 = __uint_as_float(hb.lo), b1 = __uint_as_float(hb.hi);
    cls = (int)(b1 < b0 ? hc.hi : hc.lo);
    float runner = min3(max2(b0, b1), __uint_as_float(hs.lo), __uint_as_float(hs.hi));
    if (cosine) runner = min2(runner * back, FLT_MAX);
    // the slot in a class minimum: 2^-19 of it
    const float slack = PACKED ? 1.92e-6f * fabsf(runner) : 0.f;
    // The class's centres one by one (a class of the last chunk may reach into the padding): each half of the wave takes
    // the dimensions that it has of the row.
    float dots[T];
    const half8* cand = ap + (cls >> 5) * S * 64 + g * 32 + (cls & 31);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float dot = 0.f;
#pragma unroll
      for (int st = 0; st < S; ++st) {
        const half8 c0 = cand[(t * S + st) * 64], c1 = cand[piece + (t * S + st) * 64];
        const half8 x0 = xp[st][0], x1 = xp[st][1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const half2v ch = {c0[2 * e], c0[2 * e + 1]}, cl = {c1[2 * e], c1[2 * e + 1]};
          const half2v xh = {x0[2 * e], x0[2 * e + 1]}, xl = {x1[2 * e], x1[2 * e + 1]};
          dot = __builtin_amdgcn_fdot2(xl, ch, dot, false);
          dot = __builtin_amdgcn_fdot2(xh, cl, dot, false);
          dot = __builtin_amdgcn_fdot2(xh, ch, dot, false);
        }
      }
      dots[t] = dot;
    }
    // The halves of a dot product meet: with one swap for two of them the lower half of the wave gets the even centre's
    // sum and the upper half the odd one's, each takes the best of its own, and then of both.
    float bs, other = INFINITY;
    int bt = 0;
    if constexpr (T == 1) {
      bs = __fmaf_rn(add_halves(dots[0]), back, bias[cls]);
    } else {
      bs = INFINITY;
#pragma unroll
      for (int t = 0; t < T; t += 2) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(dots[t]), __float_as_uint(dots[t + 1]), false, false);
        const float sc = __fmaf_rn(__uint_as_float(r[0]) + __uint_as_float(r[1]), back, bias[cls + 32 * (t + g)]);
        other = t == 0 ? other : min2(other, max2(bs, sc));
        bt = sc < bs ? t + g : bt;
        bs = t == 0 ? sc : min2(bs, sc);
      }
      const Halves b2 = halves(__float_as_uint(bs)), o2 = halves(__float_as_uint(other)), t2 = halves((uint32_t)bt);
      const float b0 = __uint_as_float(b2.lo), b1 = __uint_as_float(b2.hi);
      bs = min2(b0, b1);
      bt = (int)(b1 < b0 ? t2.hi : t2.lo);
      runner = min3(runner, max2(b0, b1), min2(__uint_as_float(o2.lo), __uint_as_float(o2.hi)));
    }
    int besti = cls + 32 * bt;
    // cosine: the evaluation's share shrinks with the operands, the rounding of c / |c| (norm in
    // fp64, one rounding for 1 / |c|, one for the product, one for - m: 3 units, doubled) does not
    const float scale = cosine ? __builtin_amdgcn_sqrtf(xn) * (cdev + 3.5762787e-7f / unit) : xn + cmax;
    const float bound = unit * scale + kTinyGap + slack;
    // Padding leads where no real score is a number.  A row whose square is below the smallest normal float has pieces of
    // too few bits and no norm to bound that by (scored 2^100 times as long it would not need float64, at 2 % of the time of
    // every other row); L2 has the centres' norm, or products below kTinyGap.
    const bool ask = besti >= n || !(scale < finite_below) || !((runner - bs) > bound) || (cosine && xn < FLT_MIN);
    // exact evaluation of the flagged rows (of a training step, of those that take part: the rows left out are the shortest
    // ones, and a row of zeros ties with every centre)
    uint64_t todo = __ballot(grp * 32 + j < m && g == 0 && ask) & kept;
    while (todo) {
      const int src = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const float* xr = x + (grp * 32 + src) * ldx;
      const int exact = cosine && degenerate ? exact_argmin_row(xr, centers, n, k, kx, a.metric, lane)
                                             : exact_row<S>(a, xr, centers, xs, ap, inv, kx, lane, mu, pow2(-c_shift), cmax, cdev);
      besti = lane == src ? exact : besti;
    }
    if constexpr (SUMS) {
      const int to = (int)halves((uint32_t)besti).lo;            // the exact evaluation's label is in the lower half
      const bool in = grp * 32 + j < m && (kept >> j & 1u);
      if (in) {
        int has = kx - 8 * g;
        asm volatile("" : "+v"(has));       // (as above)
        double* centre = sums + to * kPitch + 8 * g;
#pragma unroll
        for (int st = 0; st < S; ++st)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (!ragged || 16 * st + e < has) unsafeAtomicAdd(centre + 16 * st + e, (double)own[st][e]);
        if (g == 0) atomicAdd(counts + to, 1u);
      }
    }
    label = besti;
    labelled = grp;
    grp = next;
  }
  if constexpr (SUMS) {
    __syncthreads();
    const int words = n * k + n;
    float* part = a.sums + ((int64_t)slice * shares + share) * words;
    for (int i = threadIdx.x; i < n * k; i += kThreads) part[i] = (float)sums[i / k * kPitch + i % k];
    for (int i = threadIdx.x; i < n; i += kThreads) reinterpret_cast<uint32_t*>(part)[n * k + i] = counts[i];
  } else {
    if (labelled >= 0) store_labels();
  }
}

// Two pieces, norms, biases, 1 / |c|, flags, the mean, column sums and a row per wave.
// Tiles of a chunk: longer ones halve the updates and double the centres of the class that is evaluated again, whose cost
// goes with the dimensions; up to 64 centres there are only one or two tiles.
int assign_chunk(int64_t n, int64_t k) { return n <= 32 ? 1 : n <= 64 || k > 32 ? 2 : 4; }
int64_t assign_pad(int64_t n, int64_t k) { return ceil_div(n, 32 * assign_chunk(n, k)) * 32 * assign_chunk(n, k); }
size_t assign_lds(int64_t n, int64_t k) {
  const int64_t steps = ceil_div(k, 16), n_pad = assign_pad(n, k);
  const int64_t pieces = 2 * (n_pad / 32) * steps * 64 * 16, threads = assign_threads((int)steps);
  return (size_t)(pieces + 4 * n_pad * 4 + 16 + (1 + 2 * threads / kWave) * 16 * steps * 4 + 2 * threads * 4);
}

// Workgroups per slice: what takes the `resident` ones the fewest turns, with the staging of a workgroup about as long as
// two groups of rows of each of its waves.  A multiple of eight, which keeps the slices of a row on one XCD, is taken while
// it costs no more than a tenth (18 slices of 8 columns, 92 000 rows: 86 us with eight workgroups each, 144 in all, 61
// with fourteen).
int64_t assign_shares(int64_t m, int64_t slices, int64_t resident, int waves) {
  const int64_t groups = ceil_div(m, 32), most = groups < 4 * resident ? groups : 4 * resident;
  int64_t best = 1, best8 = 0, least = 0, least8 = 0;
  for (int64_t s = 1; s <= most && (s == 1 || s * slices <= 4 * resident); ++s) {
    const int64_t cost = ceil_div(s * slices, resident) * (2 + ceil_div(groups, s * waves));
    if (s == 1 || cost < least) { least = cost; best = s; }
    if (s % 8 == 0 && (best8 == 0 || cost < least8)) { least8 = cost; best8 = s; }
  }
  return best8 != 0 && 10 * least8 <= 11 * least ? best8 : best;
}
size_t assign_sums_lds(int64_t n, int64_t k) { return assign_lds(n, k) + (size_t)(n * (16 * ceil_div(k, 16) + 1) * 8 + n * 4); }

template <int S, int T, bool PACKED, bool SUMS, int METRIC>
int launch_assign(AssignArgs a, size_t lds, hipStream_t st) {
  auto kern = assign_kernel<S, T, PACKED, SUMS, METRIC>;
  constexpr int threads = assign_threads(S);
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail((int)e, "kmeans_predict: cannot reserve %zu B of LDS", lds);
  }
  // A grid that is resident all at once (a workgroup that starts late does its whole share after the others have
  // finished), from the occupancy that the registers and LDS of this instantiation really allow.
  static thread_local size_t cached_lds = 0;
  static thread_local int cached_per_cu = 0;
  if (cached_per_cu == 0 || cached_lds != lds) {
    int v = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, reinterpret_cast<const void*>(kern), threads, lds) !=
            hipSuccess || v < 1)
      v = 1;
    cached_per_cu = v;
    cached_lds = lds;
  }
  const int64_t need = ceil_div(a.m, 32);             // a group per workgroup at least
  const int64_t cap = (int64_t)num_cus() * cached_per_cu;
  int64_t grid = need < cap ? need : cap;
  if (SUMS || a.slices > 1) grid = assign_shares(a.m, a.slices, SUMS ? num_cus() : cap, threads / kWave) * a.slices;
  kern<<<(int)grid, threads, lds, st>>>(a);
  return launch_status("kmeans_predict");
}

// Up to 32 columns and more than 64 centres, what the encoder is run with, have a kernel for each metric: the general one
// asks for it in every tile of every group of rows.
template <int S, int T, bool SUMS>
int assign_metric(const AssignArgs& a, size_t lds, hipStream_t st) {
  if constexpr (S <= 2 && T == 4)
    return a.metric == F2CGT_METRIC_COSINE ? launch_assign<S, T, true, SUMS, F2CGT_METRIC_COSINE>(a, lds, st)
                                           : launch_assign<S, T, true, SUMS, F2CGT_METRIC_L2>(a, lds, st);
  else
    return launch_assign<S, T, true, SUMS, kEither>(a, lds, st);
}

template <int S, int T>
int assign_pick(const AssignArgs& a, size_t lds, hipStream_t st) {
  if (a.sums != nullptr) return assign_metric<S, T, true>(a, lds, st);
  if constexpr (S == 1) {
    // In fewer than four dimensions so many centres are close to a row that the slots' share of the near-tie bound
    // sends more rows to the exact evaluation than the packed update saves.
    if (a.k < 4) return launch_assign<1, T, false, false, kEither>(a, lds, st);
  }
  return assign_metric<S, T, false>(a, lds, st);
}

template <int S>
int assign_chunks(const AssignArgs& a, size_t lds, hipStream_t st) {
  switch (assign_chunk(a.n, a.k)) {
    case 1: return assign_pick<S, 1>(a, lds, st);
    case 2: return assign_pick<S, 2>(a, lds, st);
    default:
      if constexpr (S <= 2) return assign_pick<S, 4>(a, lds, st);
      else return fail(F2CGT_E_UNSUPPORTED, "kmeans_predict: no chunks of four tiles at this width");
  }
}

int assign_dispatch(AssignArgs a, hipStream_t st) {
  a.n_pad = (int)assign_pad(a.n, a.k);
  const size_t lds = a.sums != nullptr ? assign_sums_lds(a.n, a.k) : assign_lds(a.n, a.k);
  switch (ceil_div(a.k, 16)) {
    case 1: return assign_chunks<1>(a, lds, st);
    case 2: return assign_chunks<2>(a, lds, st);
    case 3: return assign_chunks<3>(a, lds, st);
    default: return assign_chunks<4>(a, lds, st);
  }
}

}  // namespace

bool assign_fits(int64_t n, int64_t k) { return k <= 64 && n <= 65536 && assign_lds(n, k) <= kAssignLds; }

int assign_rows(const float* x, const float* centers, int64_t* lab64, uint8_t* lab8, int64_t m, int n, int k, int metric,
                hipStream_t st) {
  AssignArgs a{};
  a.x = x; a.centers = centers; a.lab64 = lab64; a.lab8 = lab8; a.m = m; a.n = n; a.k = k; a.metric = metric;
  a.slices = 1; a.feat_dim = k; a.ldx = k; a.label_stride = 1;
  return assign_dispatch(a, st);
}

// The sums take LDS beside the operands, in a workgroup that has a CU to itself; as many slices as CUs.
bool assign_sums_fits(int64_t slices, int64_t n, int64_t k) {
  return slices >= 1 && slices <= 256 && assign_fits(n, k) && assign_sums_lds(n, k) <= 160 * 1024;
}

int64_t assign_sums_shares(int64_t m, int64_t slices, int64_t k) {
  return assign_shares(m, slices, num_cus(), assign_threads((int)ceil_div(k, (int64_t)16)) / kWave);
}

int assign_sums(const float* x, int64_t slice_step, const uint32_t* keep, int64_t keep_words, const float* centers,
                const int32_t* stop, float* sums, uint32_t* arrived, int64_t m, int slices, int n, int k, int metric,
                hipStream_t st) {
  AssignArgs a{};
  a.x = x; a.centers = centers; a.m = m; a.n = n; a.k = k; a.metric = metric;
  a.slices = slices; a.feat_dim = slices * k; a.ldx = k; a.slice_step = slice_step;
  a.stop = stop; a.keep = keep; a.keep_words = keep_words; a.sums = sums; a.arrived = arrived;
  return assign_dispatch(a, st);
}

}  // namespace f2cgt

using namespace f2cgt;

extern "C" int f2cgt_vq_encode_slices_covers(int64_t n, int64_t k) {
  return n > 0 && n <= 256 && k > 0 && assign_fits(n, k) ? 1 : 0;
}

extern "C" int f2cgt_vq_encode_slices(const float* x, int64_t ldx, int64_t feat_dim, const float* codebooks, uint8_t* codes,
                                      int64_t code_stride, int64_t m, int64_t slices, int64_t n, int64_t k, int metric,
                                      void* stream) {
  const char* what = "vq_encode_slices";
  F2CGT_REQUIRE(m >= 0 && slices > 0 && n > 0 && k > 0 && feat_dim > 0, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  F2CGT_REQUIRE(f2cgt_vq_encode_slices_covers(n, k), F2CGT_E_UNSUPPORTED,
                "%s: %lld centres of %lld columns are left to kmeans_predict, one slice at a time", what, (long long)n,
                (long long)k);
  F2CGT_REQUIRE(slices <= 65536 && feat_dim < (1 << 22), F2CGT_E_UNSUPPORTED, "%s: table too wide", what);
  F2CGT_REQUIRE((slices - 1) * k < feat_dim, F2CGT_E_INVALID, "%s: a slice without columns", what);
  F2CGT_REQUIRE(ldx >= feat_dim && code_stride >= slices, F2CGT_E_INVALID, "%s: rows overlap", what);
  F2CGT_REQUIRE(metric == F2CGT_METRIC_L2 || metric == F2CGT_METRIC_COSINE, F2CGT_E_INVALID, "%s: unknown metric %d", what,
                metric);
  if (m == 0) return 0;
  F2CGT_REQUIRE(x && codebooks && codes, F2CGT_E_INVALID, "%s: null buffer", what);
  AssignArgs a{};
  a.x = x; a.centers = codebooks; a.lab8 = codes; a.m = m; a.n = (int)n; a.k = (int)k; a.metric = metric;
  a.slices = (int)slices; a.feat_dim = (int)feat_dim; a.ldx = ldx; a.label_stride = code_stride;
  a.slice_step = k;
  return assign_dispatch(a, as_stream(stream));
}
