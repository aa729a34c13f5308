// The dense part of a GraphSAGE layer on a minibatch (examples/conv.py:68-76): fc_self(h_self) + fc_neigh(h_neigh), with
// bias and ReLU, and the gradients of its parameters, each one launch on the fp32 matrix instructions.
//
// What bounds it: at a minibatch's sizes (a thousand destination rows, 128 + 128 columns, 256 outputs: 67 million
// multiply-adds, half a microsecond of matrix time) launches and host time; two library products, an addition and an
// activation forward and two products, a reduction and a mask backward cost the host 200 us a step.  Hence one kernel each
// way, with tiles small enough that a launch of that size still covers the chip.
#include "common.hpp"

namespace f2cgt {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 32;            // rows and outputs of a tile: one 32 x 32 x 2 matrix instruction
constexpr int kForwardWaves = 4;     // a quarter of a tile each
constexpr int kGradWaves = 16;       // they share a tile's rows

struct SageArgs {
  const float* x[2];                 // h_self, h_neigh: [m, k[s]]
  const float* w[2];                 // [n, k[s]]
  const float* bias;                 // [n] or null
  float* out;                        // [m, n]
  int64_t m;
  int n, k[2], relu;
};

// out = (x0 w0^T + bias) + x1 w1^T, a 32 x 32 tile per workgroup and 16 x 16 of it per wave, so that 1024 rows and 256 outputs
// make 1024 waves, one per SIMD, of which a wave's chain of loads and matrix instructions is the time: 11 us at 128 + 128 columns (12 with
// 128 columns in flight; 6.8 with the columns shared among four waves, which adds in another order).
//
// A product is one chain of 16 x 16 x 4 instructions over its columns, of every eight the even ones and then the odd ones, four
// after four behind the last whole 16, and the two products meet behind it: the order in which the library behind torch's
// operators adds at the sizes that library_order below admits, as its results show.  A ReLU's gradient is why that matters: a
// value next to zero that another order puts on the other side of it, one in 10^7, passes its whole gradient or none of it.
// (A library that adds in another order leaves both as good as they were, but no longer equal: the tests compare the bits.)
__global__ __launch_bounds__(kForwardWaves * kWave) void sage_linear_kernel(SageArgs a) {
  constexpr int U = 8;                                  // blocks of eight columns in flight, and as many more on their way
  const int t = threadIdx.x, wave = t / kWave, lane = t & (kWave - 1), at = lane & 15, part = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * kTile + 16 * (wave & 1);
  const int n0 = blockIdx.y * kTile + 16 * (wave >> 1);
  if (m0 >= a.m || n0 >= a.n) return;
  const int64_t row = m0 + at < a.m ? m0 + at : a.m - 1;
  const int col = n0 + at < a.n ? n0 + at : a.n - 1;
  const int batches0 = (a.k[0] + 8 * U - 1) / (8 * U), batches = batches0 + (a.k[1] + 8 * U - 1) / (8 * U);
  float2 x[U], w[U];
  // Lane part p has columns 2 p and 2 p + 1 of a block; behind the last whole 16 columns it has p and, of eight, 4 + p.
  auto load = [&](int b) {
    const int s = b >= batches0 ? 1 : 0;
    const int k = a.k[s], from = (b - (s ? batches0 : 0)) * 8 * U;
    const float* xr = a.x[s] + row * k;
    const float* wr = a.w[s] + (int64_t)col * k;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = from + 8 * u;
      if (c < (k & ~15)) {
        x[u] = *reinterpret_cast<const float2*>(xr + c + 2 * part);
        w[u] = *reinterpret_cast<const float2*>(wr + c + 2 * part);
      } else if (c < k) {
        const int second = c + 8 <= k ? c + 4 + part : c + part;
        x[u] = make_float2(xr[c + part], xr[second]);
        w[u] = make_float2(wr[c + part], wr[second]);
      }
    }
  };
  floatx4 acc = {0.f, 0.f, 0.f, 0.f}, self = acc;
  load(0);
  for (int b = 0; b < batches; ++b) {
    float2 xc[U], wc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) { xc[u] = x[u]; wc[u] = w[u]; }
    if (b + 1 < batches) load(b + 1);
    if (b == batches0) {
      self = acc;
      acc = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    const int left = b >= batches0 ? a.k[1] - (b - batches0) * 8 * U : a.k[0] - b * 8 * U;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (8 * u >= left) break;
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[u].x, wc[u].x, acc, 0, 0, 0);
      if (8 * u + 4 < left) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[u].y, wc[u].y, acc, 0, 0, 0);
    }
  }
  const float bias = a.bias != nullptr ? a.bias[col] : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t r = m0 + 4 * part + i;
    float v = a.bias != nullptr ? self[i] + bias : self[i];
    v += acc[i];
    if (a.relu && v <= 0.f) v = 0.f;                    // (a NaN stays one)
    if (r < a.m && n0 + at < a.n) a.out[r * a.n + n0 + at] = v;
  }
}

struct SageGradArgs {
  const float* grad;                 // [m, n]
  const float* out;                  // [m, n] for the ReLU's mask, or null
  const float* x[2];
  float* dw[2];                      // [n, k[s]]
  float* db;                         // [n]
  float* part;                       // [splits][n * (k0 + k1) + n], or null: straight into dw and db
  int64_t m, rows_per_split;
  int n, k[2];
};

// dw[s] = (grad masked)^T x[s], db = column sums of it: a 32 x 32 tile of a weight per workgroup, whose sixteen waves share
// the rows and add their tiles in LDS in a fixed order; many rows are split over the grid too, the parts added afterwards.
__global__ __launch_bounds__(kGradWaves * kWave) void sage_grad_kernel(SageGradArgs a) {
  __shared__ float s_tile[kGradWaves / 2][kTile][kTile];
  __shared__ float s_bias[kGradWaves][kTile];
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / kWave), lane = t & (kWave - 1), at = lane & 31, side = lane >> 5;
  const int n0 = blockIdx.x * kTile;
  const int tiles0 = (a.k[0] + kTile - 1) / kTile;
  const int s = (int)blockIdx.y >= tiles0 ? 1 : 0;
  const int k = a.k[s], k0 = ((int)blockIdx.y - (s ? tiles0 : 0)) * kTile;
  const bool bias = blockIdx.y == 0;
  const bool n_in = n0 + at < a.n, k_in = k0 + at < k;
  const float* __restrict__ g = a.grad + (n_in ? n0 + at : a.n - 1);
  const float* __restrict__ o = a.out != nullptr ? a.out + (n_in ? n0 + at : a.n - 1) : nullptr;
  const float* __restrict__ x = a.x[s] + (k_in ? k0 + at : k - 1);
  const int64_t first = (int64_t)blockIdx.z * a.rows_per_split;
  const int64_t end = first + a.rows_per_split < a.m ? first + a.rows_per_split : a.m;
  constexpr int U = 8;                                     // row pairs in flight
  floatx16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  // The columns' sums in four chains per lane and pairs of waves: in one chain each they were further from float64 than the
  // operators' (relative error at 1024 rows 1.33e-7, theirs 1.04e-7, these 0.93e-7; no slower).
  float sums[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t r0 = first + wave * (2 * U); r0 < end; r0 += kGradWaves * 2 * U) {
    float gv[U], ov[U], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int64_t r = r0 + 2 * u + side;
      r = r < end ? r : end - 1;
      gv[u] = g[r * a.n];
      xv[u] = x[r * k];
      if (o != nullptr) ov[u] = o[r * a.n];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = r0 + 2 * u + side < end;
      float v = in && n_in ? gv[u] : 0.f;
      if (o != nullptr) v = ov[u] <= 0.f ? 0.f : v;        // (as the ReLU's own gradient: a NaN passes it on)
      sums[u & 3] += v;
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(v, in && k_in ? xv[u] : 0.f, acc, 0, 0, 0);
    }
  }
  if (wave >= kGradWaves / 2) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s_tile[wave - kGradWaves / 2][8 * (v / 4) + 4 * side + v % 4][at] = acc[v];
  }
  float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
  sum += __shfl_xor(sum, 32);
  if (side == 0) s_bias[wave][at] = sum;
  __syncthreads();
  if (wave < kGradWaves / 2) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s_tile[wave][8 * (v / 4) + 4 * side + v % 4][at] += acc[v];
  }
  __syncthreads();
  const int64_t words = (int64_t)a.n * (a.k[0] + a.k[1]) + a.n;
  float* dw = a.part != nullptr ? a.part + blockIdx.z * words + (s ? (int64_t)a.n * a.k[0] : 0) : a.dw[s];
  float* db = a.part != nullptr ? a.part + blockIdx.z * words + (int64_t)a.n * (a.k[0] + a.k[1]) : a.db;
  const int r = t / kTile, c = t % kTile;                  // a value per thread
  if (n0 + r < a.n && k0 + c < k && dw != nullptr) {
    float v = s_tile[0][r][c];
#pragma unroll
    for (int i = 1; i < kGradWaves / 2; ++i) v += s_tile[i][r][c];
    dw[(int64_t)(n0 + r) * k + k0 + c] = v;
  }
  if (bias && t < kTile && n0 + t < a.n && db != nullptr) {
    float v[kGradWaves];
#pragma unroll
    for (int i = 0; i < kGradWaves; ++i) v[i] = s_bias[i][t];
#pragma unroll
    for (int by = 1; by < kGradWaves; by *= 2)
#pragma unroll
      for (int i = 0; i < kGradWaves; i += 2 * by) v[i] += v[i + by];
    db[n0 + t] = v[0];
  }
}

__global__ __launch_bounds__(256) void sage_grad_add_kernel(SageGradArgs a, int splits) {
  const int64_t words0 = (int64_t)a.n * a.k[0], words1 = (int64_t)a.n * a.k[1], words = words0 + words1 + a.n;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= words) return;
  float v = 0.f;
#pragma unroll 8
  for (int p = 0; p < splits; ++p) v += a.part[p * words + i];
  if (i < words0) { if (a.dw[0] != nullptr) a.dw[0][i] = v; }
  else if (i < words0 + words1) { if (a.dw[1] != nullptr) a.dw[1][i - words0] = v; }
  else if (a.db != nullptr) a.db[i - words0 - words1] = v;
}

int sage_check(const char* what, int64_t m, int64_t n, int64_t k0, int64_t k1) {
  F2CGT_REQUIRE(m > 0 && n > 0 && k0 > 0 && k1 > 0, F2CGT_E_INVALID, "%s: sizes must be positive", what);
  F2CGT_REQUIRE(m < (1ll << 31) && n < (1 << 20) && k0 < (1 << 20) && k1 < (1 << 20), F2CGT_E_UNSUPPORTED,
                "%s: too many rows or columns", what);
  return 0;
}

int64_t sage_splits(int64_t m, int64_t n, int64_t k0, int64_t k1) {
  const int64_t tiles = ceil_div(n, kTile) * (ceil_div(k0, kTile) + ceil_div(k1, kTile));
  const int64_t most = ceil_div(m, 1024), want = ceil_div(2 * (int64_t)num_cus(), tiles);
  return most < want ? most : want;
}

}  // namespace
}  // namespace f2cgt

using namespace f2cgt;

extern "C" int f2cgt_sage_linear(const float* x0, const float* w0, const float* x1, const float* w1, const float* bias, float* out,
                                 int64_t m, int64_t n, int64_t k0, int64_t k1, int relu, void* stream) {
  const char* what = "sage_linear";
  if (int rc = sage_check(what, m, n, k0, k1)) return rc;
  F2CGT_REQUIRE(x0 && w0 && x1 && w1 && out, F2CGT_E_INVALID, "%s: null buffer", what);
  F2CGT_REQUIRE(k0 % 4 == 0 && k1 % 4 == 0 && aligned(x0, 16) && aligned(w0, 16) && aligned(x1, 16) && aligned(w1, 16) &&
                    aligned(out, 16), F2CGT_E_UNSUPPORTED, "%s: rows of whole 16-byte pieces only", what);
  SageArgs a{};
  a.x[0] = x0; a.x[1] = x1; a.w[0] = w0; a.w[1] = w1; a.bias = bias; a.out = out;
  a.m = m; a.n = (int)n; a.k[0] = (int)k0; a.k[1] = (int)k1; a.relu = relu;
  const dim3 grid((unsigned)ceil_div(m, kTile), (unsigned)ceil_div(n, kTile));
  sage_linear_kernel<<<grid, kForwardWaves * kWave, 0, as_stream(stream)>>>(a);
  return launch_status(what);
}

// Where the forward kernel has the library's bits: its order is that of the library's kernels for products of some size.
// Few rows, few outputs and very large products go to others, which split the columns.  Compared over 1 to 4096 rows, 1 to
// 600 outputs and every multiple of four up to 128 columns: the products differ at 16 outputs or fewer, at
// 256 rows or fewer and from 684 000 outputs in all, there not at multiples of 32 up to 256 outputs per row.  Of 300 000
// sizes drawn from the admitted ones none differs.
bool library_order(int64_t m, int64_t n, int64_t k0, int64_t k1) {
  return k0 <= 128 && k1 <= 128 && m > 256 && n > 16 && (m <= (1ll << 19) / n || (m <= 4096 && n <= 256 && n % 32 == 0));
}

// FORWARD, up to 2^27 multiply-adds: a tile of 32 outputs reads its rows and weights once per tile of the other side, which a
// library's larger tiles do half as often.  Device time of the two products, their sum and the ReLU, operators -> this, us
// (128 + 128 -> 256 means two inputs of 128 columns and 256 outputs), and what the host takes, 47 -> 5 us:
//   128 + 128 -> 256: 1024 rows 13.9 -> 10.3, 2048 15.8 -> 17.1, 4096 23.1 -> 31.6, 8192 33 -> 60, 60 000 131 -> 423
//   128 + 128 -> 128: 1024 rows 12.8 -> 10.0, 4096 17.8 -> 17.2, 8192 21 -> 32;  128 + 128 -> 47: 8192 15.4 -> 13.7
//   100 + 100 -> 128: 1024 rows 13.0 -> 7.0, 4096 18.4 -> 11.3;  64 + 64 -> 256: 4096 rows 20.0 -> 17.6, 8192 29 -> 33
// STEP, GRAD: forward and backward, 185 -> 65 us of the host's time with both kernels and 115 with the backward one alone.
// Device time:
//   128 + 128 -> 256: 300 rows 102 -> 16, 1024 44 -> 23, 2048 60 -> 33, 4096 93 -> 49;  100 + 100 -> 128: 4096 82 -> 29
//   the backward kernel behind the library's products: 256 + 256 -> 256: 1024 rows 47 -> 30, 4096 99 -> 57;
//   600 + 600 -> 16: 1024 38 -> 29, 4096 65 -> 35;  1000 + 1000 -> 64: 1024 56 -> 36, 4096 107 -> 58;
//   512 + 512 -> 512: 300 rows 49 -> 28, 1024 57 -> 49 (the backward alone 33 -> 25);  384 + 384 -> 256: 2048 65 -> 49
// Up to 4096 rows: the sums over the rows are closer to float64 than the library's at any size (relative error at
// 128 + 128 -> 256, 1024 rows 4.4e-7 -> 1.3e-7, 4096 9.0e-7 -> 1.4e-7) and differ from them by the library's error, which grows with
// the rows (2.1e-6 at 60 000).  Gradients of a layer that is given more rows than that stay bit for bit the operators'.
extern "C" int f2cgt_sage_linear_ahead(int64_t m, int64_t n, int64_t k0, int64_t k1) {
  if (m <= 0 || n <= 0 || k0 <= 0 || k1 <= 0 || m >= (1ll << 31) || n >= (1 << 20) || k0 >= (1 << 20) || k1 >= (1 << 20)) return 0;
  const int64_t weights = n * (k0 + k1);
  int take = 0;
  if (library_order(m, n, k0, k1)) take |= F2CGT_SAGE_STEP | (weights <= (1ll << 27) / m ? F2CGT_SAGE_FORWARD : 0);
  if (m <= 4096 && (weights <= 131072 || weights <= (1ll << 29) / m)) take |= F2CGT_SAGE_GRAD;
  return take;
}

extern "C" int64_t f2cgt_sage_linear_grad_workspace_bytes(int64_t m, int64_t n, int64_t k0, int64_t k1) {
  if (m <= 0 || n <= 0 || k0 <= 0 || k1 <= 0) return 0;
  const int64_t splits = sage_splits(m, n, k0, k1);
  return splits > 1 ? splits * (n * (k0 + k1) + n) * 4 : 0;
}

extern "C" int f2cgt_sage_linear_grad(const float* grad, const float* out, const float* x0, const float* x1, float* dw0, float* dw1,
                                      float* db, void* workspace, int64_t workspace_bytes, int64_t m, int64_t n, int64_t k0,
                                      int64_t k1, void* stream) {
  const char* what = "sage_linear_grad";
  if (int rc = sage_check(what, m, n, k0, k1)) return rc;
  F2CGT_REQUIRE(grad && x0 && x1, F2CGT_E_INVALID, "%s: null buffer", what);
  const int64_t splits = sage_splits(m, n, k0, k1);
  F2CGT_REQUIRE(splits == 1 || (workspace && workspace_bytes >= f2cgt_sage_linear_grad_workspace_bytes(m, n, k0, k1)),
                F2CGT_E_INVALID, "%s: workspace too small", what);
  SageGradArgs a{};
  a.grad = grad; a.out = out; a.x[0] = x0; a.x[1] = x1; a.dw[0] = dw0; a.dw[1] = dw1; a.db = db;
  a.part = splits > 1 ? static_cast<float*>(workspace) : nullptr;
  a.m = m; a.n = (int)n; a.k[0] = (int)k0; a.k[1] = (int)k1;
  a.rows_per_split = ceil_div(m, splits);
  const dim3 grid((unsigned)ceil_div(n, kTile), (unsigned)(ceil_div(k0, kTile) + ceil_div(k1, kTile)),
                  (unsigned)ceil_div(m, a.rows_per_split));
  F2CGT_REQUIRE(grid.y <= 65535 && grid.z <= 65535, F2CGT_E_UNSUPPORTED, "%s: too many tiles", what);
  hipStream_t st = as_stream(stream);
  sage_grad_kernel<<<grid, kGradWaves * kWave, 0, st>>>(a);
  if (a.part != nullptr)
    sage_grad_add_kernel<<<(unsigned)ceil_div(n * (k0 + k1) + n, (int64_t)256), 256, 0, st>>>(a, (int)grid.z);
  return launch_status(what);
}
