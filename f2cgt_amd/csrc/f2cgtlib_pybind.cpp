// Python module `F2CGTLib`: the operator surface of the reference's pybind module
// (src/pybind.cu:7-48: same function names, keyword names, argument order, tensor
// layouts and return types) on top of the C ABI of libf2cgt_hip.so.
//
// This file holds no device code.  It validates arguments (TORCH_CHECK -> RuntimeError
// where the reference aborts or reads out of bounds), allocates the result with torch,
// picks up torch's current HIP stream and forwards raw pointers.
#include <pybind11/pybind11.h>
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/f2cgt.h"

namespace py = pybind11;

namespace {

void* current_stream() { return static_cast<void*>(c10::hip::getCurrentHIPStream().stream()); }

void check_rc(int rc, const char* op) {
  TORCH_CHECK(rc == 0, op, " failed (", rc, "): ", f2cgt_last_error());
}

torch::Tensor dev_contig(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.defined(), name, " is undefined");
  TORCH_CHECK(t.device().is_cuda(), name, " must be a GPU tensor");
  return t.contiguous();
}

int dtype_tag(const torch::Tensor& t, const char* name) {
  switch (t.scalar_type()) {
    case torch::kUInt8: return F2CGT_DT_U8;
    case torch::kInt8: return F2CGT_DT_I8;
    case torch::kInt16: return F2CGT_DT_I16;
    case torch::kInt32: return F2CGT_DT_I32;
    case torch::kInt64: return F2CGT_DT_I64;
    case torch::kFloat16: return F2CGT_DT_F16;
    case torch::kFloat32: return F2CGT_DT_F32;
    case torch::kFloat64: return F2CGT_DT_F64;
    default: TORCH_CHECK(false, name, " has an unsupported dtype ", t.scalar_type());
  }
  return -1;
}

// CSC index tensors: int32/int64 go straight through; the narrower integer types the
// reference also dispatches on (src/common.h:33-53) are widened to int32 first.
struct Graph {
  torch::Tensor indptr, indices;
  int tag;
  int64_t rows, edges;
};

Graph graph_of(const torch::Tensor& indptr_in, const torch::Tensor& indices_in) {
  Graph g;
  g.indptr = dev_contig(indptr_in, "indptr");
  g.indices = dev_contig(indices_in, "indices");
  TORCH_CHECK(g.indptr.dim() == 1 && g.indptr.numel() >= 1, "indptr must be 1-D with at least one entry");
  TORCH_CHECK(g.indices.dim() == 1, "indices must be 1-D");
  TORCH_CHECK(g.indptr.scalar_type() == g.indices.scalar_type(),
              "indptr and indices must share one integer dtype");
  auto st = g.indptr.scalar_type();
  TORCH_CHECK(st == torch::kInt64 || st == torch::kInt32 || st == torch::kInt16 || st == torch::kInt8 ||
                  st == torch::kUInt8,
              "indptr/indices must be int64, int32, int16, int8 or uint8");
  if (st != torch::kInt64 && st != torch::kInt32) {
    g.indptr = g.indptr.to(torch::kInt32);
    g.indices = g.indices.to(torch::kInt32);
  }
  g.tag = g.indptr.scalar_type() == torch::kInt64 ? F2CGT_DT_I64 : F2CGT_DT_I32;
  g.rows = g.indptr.numel() - 1;
  g.edges = g.indices.numel();
  return g;
}

torch::Tensor empty_f32(std::initializer_list<int64_t> shape, const torch::Tensor& like) {
  return torch::empty(shape, torch::TensorOptions().dtype(torch::kFloat32).device(like.device()));
}

int metric_tag(const std::string& metric) {
  // "cosine" selects cosine; every other string selects squared L2 (src/kmeans.cu:108-112).
  return metric == "cosine" ? F2CGT_METRIC_COSINE : F2CGT_METRIC_L2;
}

// ---- reference operator surface -----------------------------------------------------

torch::Tensor packbits(torch::Tensor unpack, int64_t target_bits) {
  unpack = dev_contig(unpack, "unpack");
  TORCH_CHECK(unpack.dim() == 2, "unpack must be 2-D");
  TORCH_CHECK(unpack.scalar_type() == torch::kUInt8 || unpack.scalar_type() == torch::kInt8,
              "unpack must be uint8");
  TORCH_CHECK(target_bits == 1 || target_bits == 2 || target_bits == 4,
              "packbits: target_bits must be 1, 2 or 4");
  c10::DeviceGuard guard(unpack.device());
  const int64_t per = 8 / target_bits;
  const int64_t pack_dim = (unpack.size(1) + per - 1) / per;
  auto pack = torch::empty({unpack.size(0), pack_dim},
                           torch::TensorOptions().dtype(torch::kUInt8).device(unpack.device()));
  check_rc(f2cgt_packbits(static_cast<const uint8_t*>(unpack.data_ptr()),
                          static_cast<uint8_t*>(pack.data_ptr()), unpack.size(0), unpack.size(1),
                          (int)target_bits, current_stream()),
           "packbits");
  return pack;
}

torch::Tensor unpackbits(torch::Tensor pack, int64_t target_bits, int64_t unpack_dim) {
  pack = dev_contig(pack, "pack");
  TORCH_CHECK(pack.dim() == 2, "pack must be 2-D");
  TORCH_CHECK(pack.scalar_type() == torch::kUInt8 || pack.scalar_type() == torch::kInt8,
              "pack must be uint8");
  TORCH_CHECK(target_bits == 1 || target_bits == 2 || target_bits == 4,
              "unpackbits: target_bits must be 1, 2 or 4");
  TORCH_CHECK(unpack_dim >= 0 && unpack_dim <= pack.size(1) * (8 / target_bits),
              "unpackbits: unpack_dim does not fit the packed row");
  c10::DeviceGuard guard(pack.device());
  auto unpack = torch::empty({pack.size(0), unpack_dim},
                             torch::TensorOptions().dtype(torch::kUInt8).device(pack.device()));
  check_rc(f2cgt_unpackbits(static_cast<const uint8_t*>(pack.data_ptr()),
                            static_cast<uint8_t*>(unpack.data_ptr()), pack.size(0), pack.size(1),
                            unpack_dim, (int)target_bits, current_stream()),
           "unpackbits");
  return unpack;
}

// Codebooks on another device than the data would be read through a pointer of that device.
torch::Tensor beside(torch::Tensor codebooks, const torch::Tensor& data, const char* name = "codebooks") {
  codebooks = dev_contig(codebooks, name);
  TORCH_CHECK(codebooks.device() == data.device(), name, " are on ", codebooks.device(), ", the data on ", data.device());
  return codebooks;
}

torch::Tensor sq_codebooks_checked(torch::Tensor codebooks, const torch::Tensor& data) {
  codebooks = beside(codebooks, data);
  TORCH_CHECK(codebooks.scalar_type() == torch::kFloat32, "codebooks must be float32");
  TORCH_CHECK(codebooks.dim() == 2 && codebooks.size(1) == 5 && codebooks.size(0) >= 1,
              "SQ codebooks must be [n_codebooks, 5] = fmin,fmax,emin,emax,mean");
  return codebooks;
}

torch::Tensor sq_compress(torch::Tensor src, torch::Tensor codebooks, int64_t target_bits,
                          int64_t column_slice) {
  src = dev_contig(src, "src");
  TORCH_CHECK(src.dim() == 2 && src.scalar_type() == torch::kFloat32, "src must be float32 [rows, feat_dim]");
  codebooks = sq_codebooks_checked(codebooks, src);
  c10::DeviceGuard guard(src.device());
  auto out = torch::empty_like(src);
  check_rc(f2cgt_sq_compress(src.data_ptr<float>(), out.data_ptr<float>(), codebooks.data_ptr<float>(),
                             src.size(0), src.size(1), codebooks.size(0), (int)target_bits, column_slice,
                             current_stream()),
           "sq_compress");
  return out;
}

// Extension: the storage tensor in one pass (= sq_compress -> cast -> packbits of the callers).
// `out`: where to put it (a contiguous [rows, words] block of a larger table), instead of a new tensor.
torch::Tensor sq_encode(torch::Tensor src, torch::Tensor codebooks, int64_t target_bits, int64_t column_slice,
                        c10::optional<torch::Tensor> into) {
  src = dev_contig(src, "src");
  TORCH_CHECK(src.dim() == 2 && src.scalar_type() == torch::kFloat32, "src must be float32 [rows, feat_dim]");
  TORCH_CHECK(target_bits == 1 || target_bits == 2 || target_bits == 4 || target_bits == 8 || target_bits == 16,
              "target_bits must be 1, 2, 4, 8 or 16");
  codebooks = sq_codebooks_checked(codebooks, src);
  c10::DeviceGuard guard(src.device());
  const int64_t d = src.size(1);
  const int64_t words = target_bits < 8 ? (d * target_bits + 7) / 8 : d;
  const auto dtype = target_bits <= 8 ? torch::kInt8 : torch::kInt16;
  torch::Tensor out;
  if (into.has_value()) {
    out = *into;
    TORCH_CHECK(out.device() == src.device() && out.scalar_type() == dtype && out.dim() == 2 && out.is_contiguous() &&
                    out.size(0) == src.size(0) && out.size(1) == words,
                "out must be a contiguous ", dtype, " GPU tensor [", src.size(0), ", ", words, "]");
  } else {
    out = torch::empty({src.size(0), words}, src.options().dtype(dtype));
  }
  check_rc(f2cgt_sq_encode(src.data_ptr<float>(), out.data_ptr(), codebooks.data_ptr<float>(), src.size(0), d,
                           codebooks.size(0), (int)target_bits, column_slice, current_stream()),
           "sq_encode");
  return out;
}

// A flag in pinned memory that a kernel may still set, and the event behind that kernel.
class PendingFlag {
 public:
  PendingFlag() : word_(torch::empty({1}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true))) {
    *word_.data_ptr<int32_t>() = 0;
    const hipError_t e = hipEventCreateWithFlags(&event_, hipEventDisableTiming);
    TORCH_CHECK(e == hipSuccess, "cannot create an event: ", hipGetErrorString(e));
  }
  PendingFlag(const PendingFlag&) = delete;
  PendingFlag& operator=(const PendingFlag&) = delete;
  ~PendingFlag() {                 // the word goes back to its pool only when the kernel is done with it
    (void)hipEventSynchronize(event_);
    (void)hipEventDestroy(event_);
  }
  // Waits for the kernel.  -> whether it set the flag
  bool wait() {
    py::gil_scoped_release unlocked;
    const hipError_t e = hipEventSynchronize(event_);
    TORCH_CHECK(e == hipSuccess, "waiting for a check failed: ", hipGetErrorString(e));
    return *const_cast<volatile int32_t*>(word_.data_ptr<int32_t>()) != 0;
  }
  int32_t* word() { return word_.data_ptr<int32_t>(); }
  void* event() { return static_cast<void*>(event_); }

 private:
  torch::Tensor word_;
  hipEvent_t event_ = nullptr;
};

// Extension: order statistics, sum and flags (1: a NaN, 2: a row id outside the table) of |x| per column slice of the rows
// `rows` (None: all of them), for the codebooks of sq_encode.  ranks: four ranks in a full slice, four in the last one.
// -> (float64 [n_slices, 6], the codebooks fp32 [n_slices, 5] where weights are given), on the GPU; pending: the check of the
// row ids, on its way to the host.
std::tuple<torch::Tensor, torch::Tensor> order_stats(torch::Tensor x, c10::optional<torch::Tensor> rows, int64_t column_slice,
                                                     const std::vector<int64_t>& ranks, const std::vector<float>* weights,
                                                     std::shared_ptr<PendingFlag>* pending = nullptr) {
  TORCH_CHECK(x.defined() && x.device().is_cuda(), "x must be a GPU tensor");
  TORCH_CHECK(x.dim() == 2 && x.scalar_type() == torch::kFloat32, "x must be float32 [rows, feat_dim]");
  // columns apart, or rows that overlap (an expanded row): a copy.  The stride of a single row may be anything.
  if (x.stride(1) != 1 || x.stride(0) < x.size(1)) x = x.contiguous();
  const int64_t ld = x.size(0) > 1 ? x.stride(0) : x.size(1);
  TORCH_CHECK(ranks.size() == 8, "ranks must hold eight values");
  TORCH_CHECK(weights == nullptr || weights->size() == 4, "weights must hold four values");
  TORCH_CHECK(column_slice > 0, "column_slice must be positive");
  torch::Tensor r;
  if (rows.has_value()) {
    r = dev_contig(*rows, "rows");
    TORCH_CHECK(r.dim() == 1 && r.scalar_type() == torch::kInt64 && r.device() == x.device(),
                "rows must be int64 [m] on the device of x");
  }
  c10::DeviceGuard guard(x.device());
  const int64_t m = r.defined() ? r.numel() : x.size(0), cols = x.size(1);
  const int64_t slices = (cols + column_slice - 1) / column_slice;
  auto opts = torch::TensorOptions().device(x.device());
  auto out = torch::empty({slices, 6}, opts.dtype(torch::kFloat64));
  auto ws = torch::empty({f2cgt_abs_order_stats_workspace_bytes(m, cols, column_slice)}, opts.dtype(torch::kUInt8));
  const int64_t* list = r.defined() ? r.data_ptr<int64_t>() : nullptr;
  torch::Tensor books;
  if (weights != nullptr) {
    books = torch::empty({slices, 5}, opts.dtype(torch::kFloat32));
    if (pending != nullptr) {
      *pending = std::make_shared<PendingFlag>();
      check_rc(f2cgt_sq_codebooks_checked(x.data_ptr<float>(), ld, list, m, x.size(0), cols, column_slice, ranks.data(),
                                          weights->data(), ws.data_ptr(), ws.numel(), out.data_ptr<double>(),
                                          books.data_ptr<float>(), (*pending)->word(), (*pending)->event(), current_stream()),
               "sq_codebooks_checked");
      return {out, books};
    }
    check_rc(f2cgt_sq_codebooks(x.data_ptr<float>(), ld, list, m, x.size(0), cols, column_slice, ranks.data(), weights->data(),
                                ws.data_ptr(), ws.numel(), out.data_ptr<double>(), books.data_ptr<float>(), current_stream()),
             "sq_codebooks");
  } else {
    check_rc(f2cgt_abs_order_stats(x.data_ptr<float>(), ld, list, m, x.size(0), cols, column_slice, ranks.data(),
                                   ws.data_ptr(), ws.numel(), out.data_ptr<double>(), current_stream()),
             "abs_order_stats");
  }
  return {out, books};
}

torch::Tensor abs_order_stats(torch::Tensor x, c10::optional<torch::Tensor> rows, int64_t column_slice,
                              const std::vector<int64_t>& ranks) {
  return std::get<0>(order_stats(x, rows, column_slice, ranks, nullptr));
}

// -> (codebooks fp32 [slices, 5], the statistics they were made from fp64 [slices, 6]), both on the device.  With a row list,
// outside a graph's capture, the check of its ids is on its way to the host: the statistics carry it as `bad_rows`, a
// PendingFlag.
std::tuple<torch::Tensor, py::object> sq_codebooks(torch::Tensor x, c10::optional<torch::Tensor> rows, int64_t column_slice,
                                                   const std::vector<int64_t>& ranks, const std::vector<float>& weights) {
  TORCH_CHECK(x.defined() && x.device().is_cuda(), "x must be a GPU tensor");
  c10::DeviceGuard guard(x.device());      // the stream that is asked below is the one that is worked on
  std::shared_ptr<PendingFlag> pending;
  const bool check = rows.has_value() && c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
  auto both = order_stats(x, rows, column_slice, ranks, &weights, check ? &pending : nullptr);
  py::object stats = py::cast(std::get<0>(both));
  if (check) stats.attr("bad_rows") = py::cast(pending);
  return {std::get<1>(both), stats};
}

torch::Tensor sq_decompress(torch::Tensor compress_data, torch::Tensor codebooks, int64_t target_bits,
                            int64_t column_slice, int64_t feat_dim) {
  compress_data = dev_contig(compress_data, "compress_data");
  TORCH_CHECK(compress_data.dim() == 2, "compress_data must be 2-D");
  codebooks = sq_codebooks_checked(codebooks, compress_data);
  c10::DeviceGuard guard(compress_data.device());
  auto out = empty_f32({compress_data.size(0), feat_dim}, compress_data);
  check_rc(f2cgt_sq_decompress(compress_data.data_ptr(), dtype_tag(compress_data, "compress_data"),
                               out.data_ptr<float>(), codebooks.data_ptr<float>(), compress_data.size(0),
                               compress_data.size(1), feat_dim, codebooks.size(0), (int)target_bits,
                               column_slice, current_stream()),
           "sq_decompress");
  return out;
}

torch::Tensor vq_decompress(torch::Tensor index_tensor, torch::Tensor codebooks, int64_t feat_dim) {
  index_tensor = dev_contig(index_tensor, "index_tensor");
  codebooks = beside(codebooks, index_tensor);
  TORCH_CHECK(index_tensor.dim() == 2, "index_tensor must be [rows, n_codebooks]");
  TORCH_CHECK(codebooks.dim() == 3, "VQ codebooks must be [n_codebooks, K, width]");
  TORCH_CHECK(index_tensor.size(1) == codebooks.size(0), "index_tensor has ", index_tensor.size(1),
              " columns but there are ", codebooks.size(0), " codebooks");
  c10::DeviceGuard guard(index_tensor.device());
  auto out = empty_f32({index_tensor.size(0), feat_dim}, index_tensor);
  check_rc(f2cgt_vq_decompress(index_tensor.data_ptr(), dtype_tag(index_tensor, "index_tensor"),
                               codebooks.data_ptr(), dtype_tag(codebooks, "codebooks"),
                               out.data_ptr<float>(), index_tensor.size(0), feat_dim, codebooks.size(0),
                               codebooks.size(1), codebooks.size(2), current_stream()),
           "vq_decompress");
  return out;
}

torch::Tensor spmm_csr(torch::Tensor feat, torch::Tensor indptr, torch::Tensor indices) {
  feat = dev_contig(feat, "feat");
  TORCH_CHECK(feat.dim() == 2, "feat must be 2-D");
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(feat.device());
  auto out = torch::empty({g.rows, feat.size(1)}, feat.options());
  check_rc(f2cgt_spmm_csr(feat.data_ptr(), dtype_tag(feat, "feat"), out.data_ptr(), g.indptr.data_ptr(),
                          g.indices.data_ptr(), g.tag, g.rows, g.edges, feat.size(0), feat.size(1),
                          current_stream()),
           "spmm_csr");
  return out;
}

torch::Tensor vq_decompress_spmm_csr(torch::Tensor compress_feat, torch::Tensor codebooks,
                                     torch::Tensor indptr, torch::Tensor indices, int64_t feat_dim) {
  compress_feat = dev_contig(compress_feat, "compress_feat");
  codebooks = beside(codebooks, compress_feat);
  TORCH_CHECK(compress_feat.dim() == 2, "compress_feat must be [rows, n_codebooks]");
  TORCH_CHECK(codebooks.dim() == 3 && codebooks.scalar_type() == torch::kFloat32,
              "VQ codebooks must be float32 [n_codebooks, K, width]");
  TORCH_CHECK(compress_feat.size(1) == codebooks.size(0), "compress_feat has ", compress_feat.size(1),
              " columns but there are ", codebooks.size(0), " codebooks");
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(compress_feat.device());
  auto out = empty_f32({g.rows, feat_dim}, compress_feat);
  check_rc(f2cgt_vq_decompress_spmm_csr(compress_feat.data_ptr(), dtype_tag(compress_feat, "compress_feat"),
                                        codebooks.data_ptr<float>(), g.indptr.data_ptr(),
                                        g.indices.data_ptr(), g.tag, out.data_ptr<float>(), g.rows, g.edges,
                                        compress_feat.size(0), feat_dim, codebooks.size(0),
                                        codebooks.size(1), codebooks.size(2), current_stream()),
           "vq_decompress_spmm_csr");
  return out;
}

torch::Tensor sq_decompress_spmm_csr(torch::Tensor compress_feat, torch::Tensor codebooks,
                                     torch::Tensor indptr, torch::Tensor indices, int64_t target_bit,
                                     int64_t column_slice, int64_t feat_dim) {
  compress_feat = dev_contig(compress_feat, "compress_feat");
  TORCH_CHECK(compress_feat.dim() == 2, "compress_feat must be 2-D");
  codebooks = sq_codebooks_checked(codebooks, compress_feat);
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(compress_feat.device());
  auto out = empty_f32({g.rows, feat_dim}, compress_feat);
  check_rc(f2cgt_sq_decompress_spmm_csr(compress_feat.data_ptr(), dtype_tag(compress_feat, "compress_feat"),
                                        codebooks.data_ptr<float>(), g.indptr.data_ptr(),
                                        g.indices.data_ptr(), g.tag, out.data_ptr<float>(), g.rows, g.edges,
                                        compress_feat.size(0), compress_feat.size(1), feat_dim,
                                        codebooks.size(0), (int)target_bit, column_slice, current_stream()),
           "sq_decompress_spmm_csr");
  return out;
}

torch::Tensor kmeans_predict_impl(torch::Tensor x, torch::Tensor centers, const std::string& metric,
                                  bool as_u8) {
  x = dev_contig(x, "data");
  centers = dev_contig(centers, "centers");
  TORCH_CHECK(x.dim() == 2 && centers.dim() == 2 && x.size(1) == centers.size(1),
              "data [m,k] and centers [n,k] must share k");
  TORCH_CHECK(x.scalar_type() == torch::kFloat32 && centers.scalar_type() == torch::kFloat32,
              "data and centers must be float32");
  c10::DeviceGuard guard(x.device());
  auto labels = torch::empty({x.size(0)}, torch::TensorOptions()
                                              .dtype(as_u8 ? torch::kUInt8 : torch::kInt64)
                                              .device(x.device()));
  check_rc(f2cgt_kmeans_predict(x.data_ptr<float>(), centers.data_ptr<float>(),
                                as_u8 ? nullptr : labels.data_ptr<int64_t>(),
                                as_u8 ? static_cast<uint8_t*>(labels.data_ptr()) : nullptr, x.size(0),
                                centers.size(0), x.size(1), metric_tag(metric), current_stream()),
           "kmeans_predict");
  return labels;
}

torch::Tensor pairwise_distance(torch::Tensor x, torch::Tensor y, std::string metric) {
  x = dev_contig(x, "x");
  y = dev_contig(y, "y");
  TORCH_CHECK(x.dim() == 2 && y.dim() == 2 && x.size(1) == y.size(1), "x [m,k] and y [n,k] must share k");
  TORCH_CHECK(x.scalar_type() == torch::kFloat32 && y.scalar_type() == torch::kFloat32,
              "x and y must be float32");
  c10::DeviceGuard guard(x.device());
  auto dist = empty_f32({x.size(0), y.size(0)}, x);
  check_rc(f2cgt_pairwise_distance(x.data_ptr<float>(), y.data_ptr<float>(), dist.data_ptr<float>(),
                                   x.size(0), y.size(0), x.size(1), metric_tag(metric), current_stream()),
           "pairwise_distance");
  return dist;
}

// Extension: one Lloyd centre update in place (the update half of examples/my_kmeans.py:87-113).
// -> shift fp32 [2] on the device = (sum_c |dc|, sum_c |dc|^2).  `stop` (int32 [1] on the device, optional)
// freezes the centres once `rule` is met (1: sum |dc|^2 < tol; 2: (sum |dc|)^2 < tol), see include/f2cgt.h.
torch::Tensor kmeans_update(torch::Tensor x, torch::Tensor labels, torch::Tensor centers,
                            c10::optional<torch::Tensor> stop, int64_t rule, double tol) {
  x = dev_contig(x, "data");
  labels = dev_contig(labels, "labels");
  TORCH_CHECK(centers.is_cuda() && centers.is_contiguous() && centers.scalar_type() == torch::kFloat32 &&
                  centers.dim() == 2,
              "centers must be a contiguous float32 GPU tensor [n, k] (it is updated in place)");
  TORCH_CHECK(x.dim() == 2 && x.scalar_type() == torch::kFloat32 && x.size(1) == centers.size(1),
              "data must be float32 [m, k]");
  TORCH_CHECK(labels.dim() == 1 && labels.size(0) == x.size(0) &&
                  (labels.scalar_type() == torch::kInt64 || labels.scalar_type() == torch::kUInt8),
              "labels must be int64 or uint8 [m]");
  int32_t* stop_ptr = nullptr;
  if (stop.has_value()) {
    TORCH_CHECK(stop->is_cuda() && stop->scalar_type() == torch::kInt32 && stop->numel() == 1,
                "stop must be an int32 GPU tensor with one element");
    stop_ptr = stop->data_ptr<int32_t>();
  }
  c10::DeviceGuard guard(x.device());
  const int64_t n = centers.size(0), k = centers.size(1);
  auto ws = torch::empty({f2cgt_kmeans_update_workspace_bytes(n, k)},
                         torch::TensorOptions().dtype(torch::kUInt8).device(x.device()));
  auto shift = empty_f32({2}, x);
  const bool u8 = labels.scalar_type() == torch::kUInt8;
  check_rc(f2cgt_kmeans_update(x.data_ptr<float>(), u8 ? nullptr : labels.data_ptr<int64_t>(),
                               u8 ? static_cast<const uint8_t*>(labels.data_ptr()) : nullptr,
                               centers.data_ptr<float>(), shift.data_ptr<float>(), stop_ptr, (int)rule, (float)tol,
                               ws.data_ptr(), ws.numel(), x.size(0), n, k, current_stream()),
           "kmeans_update");
  return shift;
}

// The rows of a sample, column slice by column slice: (rows fp32 [slices, m, k], their lengths fp32 [m, slices], flag
// int32 [1] on the device: an id lies outside the table).
std::tuple<torch::Tensor, torch::Tensor, torch::Tensor> slice_rows(torch::Tensor x, c10::optional<torch::Tensor> rows,
                                                                   int64_t column_slice) {
  TORCH_CHECK(x.defined() && x.is_cuda() && x.dim() == 2 && x.scalar_type() == torch::kFloat32,
              "x must be a float32 GPU tensor [rows, feat_dim]");
  TORCH_CHECK(x.size(0) > 0 && x.size(1) > 0 && column_slice > 0, "x and column_slice must not be empty");
  if (x.stride(1) != 1 || x.stride(0) < x.size(1)) x = x.contiguous();
  const int64_t ld = x.size(0) > 1 ? x.stride(0) : x.size(1);
  torch::Tensor r;
  if (rows.has_value()) {
    r = dev_contig(*rows, "rows");
    TORCH_CHECK(r.dim() == 1 && r.scalar_type() == torch::kInt64 && r.device() == x.device(),
                "rows must be int64 [m] on the device of x");
  }
  c10::DeviceGuard guard(x.device());
  const int64_t m = r.defined() ? r.numel() : x.size(0), cols = x.size(1), slices = (cols + column_slice - 1) / column_slice;
  auto out = empty_f32({slices, m, column_slice}, x);
  auto norms = empty_f32({m, slices}, x);
  auto bad = torch::zeros({1}, torch::TensorOptions().dtype(torch::kInt32).device(x.device()));
  check_rc(f2cgt_slice_rows(x.data_ptr<float>(), ld, r.defined() ? r.data_ptr<int64_t>() : nullptr, m, x.size(0), cols,
                            column_slice, out.data_ptr<float>(), norms.data_ptr<float>(), bad.data_ptr<int32_t>(),
                            current_stream()),
           "slice_rows");
  return {out, norms, bad};
}

// Bits (int32 [slices, ceil(m / 32)]) of the rows that are as long as a quantile of their slice's lengths, from the order
// statistics of `norms` on both sides of it.
torch::Tensor keep_rows(torch::Tensor norms, torch::Tensor stats, double weight, double weight_last) {
  norms = dev_contig(norms, "norms");
  stats = dev_contig(stats, "stats");
  TORCH_CHECK(norms.dim() == 2 && norms.scalar_type() == torch::kFloat32, "norms must be float32 [m, slices]");
  TORCH_CHECK(stats.dim() == 2 && stats.size(0) == norms.size(1) && stats.size(1) == 6 &&
                  stats.scalar_type() == torch::kFloat64 && stats.device() == norms.device(),
              "stats must be float64 [slices, 6] on the device of norms");
  c10::DeviceGuard guard(norms.device());
  auto keep = torch::empty({norms.size(1), (norms.size(0) + 31) / 32},
                           torch::TensorOptions().dtype(torch::kInt32).device(norms.device()));
  check_rc(f2cgt_keep_rows(norms.data_ptr<float>(), stats.data_ptr<double>(), (float)weight, (float)weight_last, norms.size(0),
                           norms.size(1), reinterpret_cast<uint32_t*>(keep.data_ptr<int32_t>()), current_stream()),
           "keep_rows");
  return keep;
}

bool kmeans_slices_covers(int64_t slices, int64_t n, int64_t k) { return f2cgt_kmeans_slices_covers(slices, n, k) != 0; }

// The loop of kmeans_slices_fit, on flags[0, slices), which it leaves on the device.
void fit_slices(torch::Tensor x, c10::optional<torch::Tensor> keep, torch::Tensor centers, const std::string& metric, int64_t rule,
                double tol, double growth, int64_t max_iter, int64_t check_every, torch::Tensor& flags) {
  x = dev_contig(x, "x");
  TORCH_CHECK(x.dim() == 3 && x.scalar_type() == torch::kFloat32, "x must be float32 [slices, m, k]");
  TORCH_CHECK(centers.is_cuda() && centers.is_contiguous() && centers.scalar_type() == torch::kFloat32 && centers.dim() == 3 &&
                  centers.size(0) == x.size(0) && centers.size(2) == x.size(2) && centers.device() == x.device(),
              "centers must be a contiguous float32 tensor [slices, n, k] on the device of x (it is updated in place)");
  const int64_t slices = x.size(0), m = x.size(1), k = x.size(2), n = centers.size(1);
  const uint32_t* bits = nullptr;
  if (keep.has_value()) {
    TORCH_CHECK(keep->device() == x.device() && keep->is_contiguous() && keep->scalar_type() == torch::kInt32 &&
                    keep->dim() == 2 && keep->size(0) == slices && keep->size(1) == (m + 31) / 32,
                "keep must be a contiguous int32 tensor [slices, ceil(m / 32)] on the device of x");
    bits = reinterpret_cast<const uint32_t*>(keep->data_ptr<int32_t>());
  }
  TORCH_CHECK(check_every > 0, "check_every must be positive");
  const int tag = metric_tag(metric);
  c10::DeviceGuard guard(x.device());
  flags = torch::zeros({slices + 2}, torch::TensorOptions().dtype(torch::kInt32).device(x.device()));
  auto ws = torch::empty({f2cgt_kmeans_slices_workspace_bytes(m, slices, n, k)},
                         torch::TensorOptions().dtype(torch::kUInt8).device(x.device()));
  py::gil_scoped_release unlocked;
  for (int64_t it = 0; it < max_iter; ++it) {
    check_rc(f2cgt_kmeans_slices_step(x.data_ptr<float>(), bits, centers.data_ptr<float>(), flags.data_ptr<int32_t>(), (int)rule,
                                      (float)tol, ws.data_ptr(), ws.numel(), m, slices, n, k, tag, current_stream()),
             "kmeans_slices_fit");
    tol *= growth;
    if (it % check_every == check_every - 1 && it + 1 < max_iter) {
      auto seen = flags.cpu();
      const int32_t* f = seen.data_ptr<int32_t>();
      bool all = true;
      for (int64_t s = 0; s < slices; ++s) all = all && f[s] != 0;
      if (all) return;
    }
  }
}

// Lloyd iterations of all slices on x [slices, m, k] from `centers` [slices, n, k] (updated in place), until every slice
// has met `rule` or for max_iter steps; tol grows by `growth` each step.  The flags are read every check_every steps and
// at the end.  -> the stop flags, int32 [slices] on the host: 0 not met, 1 met, 2 the shift became NaN, 3 no rows.
// rescale: the centres are also rescaled to their slice's mean length, and
// the result is (flags int32 [slices + 2] on the host: the stop flags, bad_row's word, 1 where a value is no number;
// codebooks fp32 [slices, n, k]), with one wait for all of it.
py::object kmeans_slices_fit(torch::Tensor x, c10::optional<torch::Tensor> keep, torch::Tensor centers, std::string metric,
                             int64_t rule, double tol, double growth, int64_t max_iter, int64_t check_every,
                             c10::optional<torch::Tensor> bad_row, bool rescale) {
  torch::Tensor flags, books;
  const int32_t* bad = nullptr;
  if (bad_row.has_value()) {
    TORCH_CHECK(bad_row->device() == centers.device() && bad_row->scalar_type() == torch::kInt32 && bad_row->numel() == 1,
                "bad_row must be one int32 word on the device of centers");
    bad = bad_row->data_ptr<int32_t>();
  }
  fit_slices(x, keep, centers, metric, rule, tol, growth, max_iter, check_every, flags);
  const int64_t slices = centers.size(0);
  if (rescale) {
    c10::DeviceGuard guard(centers.device());
    books = torch::empty_like(centers);
    check_rc(f2cgt_kmeans_rescale(centers.data_ptr<float>(), books.data_ptr<float>(), centers.size(1), centers.size(2), slices, bad,
                                  flags.data_ptr<int32_t>(), current_stream()),
             "kmeans_slices_fit");
  } else {
    flags = flags.narrow(0, 0, slices);
  }
  {
    py::gil_scoped_release unlocked;
    flags = flags.cpu();
  }
  if (!rescale) return py::cast(flags);
  return py::make_tuple(flags, books);
}

// Counterpart of the reference's raft-backed KMeans (src/kmeans.h:13-31, src/kmeans.cu).
// predict() is the fused MFMA distance + arg-min kernel.  fit() is Lloyd's algorithm on the device:
// assignment (f2cgt_kmeans_predict) and centre update (f2cgt_kmeans_update) per iteration, stopped by
// raft's rule (sum of squared centre shifts below tol) which the update kernel evaluates itself; the
// host looks at the flag every eighth iteration only.  The centres start from distinct random rows
// (raft: random rows for cosine, k-means++ for L2; its RNG stream is not reproduced, so fit() is not a
// bit-parity target).  raft's batching and restart parameters have no counterpart here: a value other
// than the default draws a warning instead of being dropped silently.
class KMeans {
 public:
  KMeans(int64_t n_cluster, int64_t feat_dim, std::string metric, int max_iter, double tol, int n_init,
         double oversampling_factor, int batch_samples, int batch_centroids, bool inertia_check)
      : metric_(std::move(metric)), max_iter_(max_iter), tol_(tol), n_clusters_(n_cluster) {
    warn_ignored(n_init, oversampling_factor, batch_samples, batch_centroids, inertia_check);
    TORCH_CHECK(n_cluster > 0 && feat_dim > 0, "KMeans: n_cluster and feat_dim must be positive");
    centers_ = torch::zeros({n_cluster, feat_dim},
                            torch::TensorOptions().dtype(torch::kFloat32).device(torch::kCUDA));
  }
  KMeans(torch::Tensor centers, std::string metric, int max_iter, double tol, int n_init,
         double oversampling_factor, int batch_samples, int batch_centroids, bool inertia_check)
      : metric_(std::move(metric)), max_iter_(max_iter), tol_(tol) {
    warn_ignored(n_init, oversampling_factor, batch_samples, batch_centroids, inertia_check);
    TORCH_CHECK(centers.device().is_cuda(), "centers must be a CUDA tensor");
    TORCH_CHECK(centers.dim() == 2 && centers.scalar_type() == torch::kFloat32,
                "centers must be float32 [n_cluster, feat_dim]");
    centers_ = centers.contiguous();
    n_clusters_ = centers.size(0);
  }

  static void warn_ignored(int n_init, double oversampling_factor, int batch_samples, int batch_centroids,
                           bool inertia_check) {
    auto warn = [](const char* text) { py::module_::import("warnings").attr("warn")(std::string(text)); };
    if (n_init != 1) warn("KMeans: n_init is ignored (one run from one random start)");
    if (oversampling_factor != 2.0) warn("KMeans: oversampling_factor is ignored (no k-means|| seeding)");
    if (batch_samples != (1 << 15)) warn("KMeans: batch_samples is ignored (the kernels stream all rows)");
    if (batch_centroids != 0) warn("KMeans: batch_centroids is ignored (all centres are scored together)");
    if (inertia_check) warn("KMeans: inertia_check is ignored (the centre shift alone stops the fit)");
  }

  void fit(torch::Tensor x) {
    TORCH_CHECK(x.device().is_cuda(), "x must be a CUDA tensor");
    x = x.contiguous().to(torch::kFloat32);
    TORCH_CHECK(x.dim() == 2 && x.size(1) == centers_.size(1), "fit: data must be [n, feat_dim]");
    TORCH_CHECK(x.size(0) >= n_clusters_, "fit: fewer samples than clusters");
    c10::DeviceGuard guard(x.device());
    auto pick = torch::randperm(x.size(0), torch::TensorOptions().dtype(torch::kInt64).device(x.device()))
                    .slice(0, 0, n_clusters_);
    centers_.copy_(x.index_select(0, pick));
    auto stop = torch::zeros({1}, torch::TensorOptions().dtype(torch::kInt32).device(x.device()));
    const bool small = n_clusters_ <= 256;
    n_iter_ = 0;
    for (int it = 0; it < max_iter_; ++it) {
      auto labels = kmeans_predict_impl(x, centers_, metric_, small);
      kmeans_update(x, labels, centers_, stop, /*rule=*/1, tol_);
      ++n_iter_;
      if ((it & 7) == 7 && stop.item<int>() != 0) break;   // later steps are no-ops once the flag is up
    }
    // flag 2: the centre shift is not a number (NaN / infinite rows in the data); the centres are garbage
    TORCH_CHECK(stop.item<int>() != 2, "KMeans.fit: the centre shift became NaN (non-finite input rows?)");
  }

  int64_t n_iter() const { return n_iter_; }

  torch::Tensor predict(torch::Tensor x, bool normalize_weights) {
    (void)normalize_weights;  // sample weights only scale raft's inertia, never the labels
    TORCH_CHECK(x.device().is_cuda(), "x must be a CUDA tensor");
    return kmeans_predict_impl(x, centers_, metric_, false);
  }

  torch::Tensor get_centers() { return centers_; }

 private:
  std::string metric_;
  int max_iter_;
  double tol_;
  int64_t n_clusters_;
  int64_t n_iter_ = 0;
  torch::Tensor centers_;
};

// ---- extensions (not in the reference; defined by the benchmark configurations) -------

torch::Tensor affine_params_checked(torch::Tensor params, int64_t feat_dim, const torch::Tensor& data) {
  params = beside(params, data, "params");
  TORCH_CHECK(params.scalar_type() == torch::kFloat32 && params.dim() == 2 && params.size(0) == 2 &&
                  params.size(1) >= feat_dim,
              "affine params must be float32 [2, >= feat_dim] = (min, scale)");
  return params;
}

torch::Tensor sq_affine_decompress(torch::Tensor compress_data, torch::Tensor params, int64_t target_bits,
                                   int64_t feat_dim) {
  compress_data = dev_contig(compress_data, "compress_data");
  TORCH_CHECK(compress_data.dim() == 2 && (compress_data.scalar_type() == torch::kUInt8 ||
                                           compress_data.scalar_type() == torch::kInt8),
              "compress_data must be uint8 [rows, src_dim]");
  params = affine_params_checked(params, feat_dim, compress_data);
  c10::DeviceGuard guard(compress_data.device());
  auto out = empty_f32({compress_data.size(0), feat_dim}, compress_data);
  check_rc(f2cgt_sq_affine_decompress(static_cast<const uint8_t*>(compress_data.data_ptr()),
                                      out.data_ptr<float>(), params.data_ptr<float>(), params.size(1),
                                      compress_data.size(0), compress_data.size(1), feat_dim,
                                      (int)target_bits, current_stream()),
           "sq_affine_decompress");
  return out;
}

torch::Tensor sq_affine_decompress_spmm_csr(torch::Tensor compress_feat, torch::Tensor params,
                                            torch::Tensor indptr, torch::Tensor indices,
                                            int64_t target_bit, int64_t feat_dim) {
  compress_feat = dev_contig(compress_feat, "compress_feat");
  TORCH_CHECK(compress_feat.dim() == 2 && (compress_feat.scalar_type() == torch::kUInt8 ||
                                           compress_feat.scalar_type() == torch::kInt8),
              "compress_feat must be uint8 [rows, src_dim]");
  params = affine_params_checked(params, feat_dim, compress_feat);
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(compress_feat.device());
  auto out = empty_f32({g.rows, feat_dim}, compress_feat);
  check_rc(f2cgt_sq_affine_decompress_spmm_csr(
               static_cast<const uint8_t*>(compress_feat.data_ptr()), params.data_ptr<float>(),
               params.size(1), g.indptr.data_ptr(), g.indices.data_ptr(), g.tag, out.data_ptr<float>(),
               g.rows, g.edges, compress_feat.size(0), compress_feat.size(1), feat_dim, (int)target_bit,
               current_stream()),
           "sq_affine_decompress_spmm_csr");
  return out;
}

torch::Tensor hybrid_decompress_spmm_csr(torch::Tensor row_map, torch::Tensor sq_codes,
                                         torch::Tensor sq_params, torch::Tensor vq_codes,
                                         torch::Tensor vq_codebooks, torch::Tensor indptr,
                                         torch::Tensor indices, int64_t feat_dim) {
  row_map = dev_contig(row_map, "row_map");
  sq_codes = dev_contig(sq_codes, "sq_codes");
  vq_codes = dev_contig(vq_codes, "vq_codes");
  vq_codebooks = beside(vq_codebooks, vq_codes, "vq_codebooks");
  TORCH_CHECK(row_map.dim() == 1 && row_map.scalar_type() == torch::kInt32, "row_map must be int32 [n]");
  TORCH_CHECK(sq_codes.dim() == 2 && sq_codes.scalar_type() == torch::kUInt8 && sq_codes.size(1) == feat_dim,
              "sq_codes must be uint8 [n_sq, feat_dim]");
  TORCH_CHECK(vq_codes.dim() == 2 && vq_codes.scalar_type() == torch::kUInt8, "vq_codes must be uint8 [n_vq, n_codebooks]");
  TORCH_CHECK(vq_codebooks.dim() == 3 && vq_codebooks.scalar_type() == torch::kFloat32 &&
                  vq_codebooks.size(0) == vq_codes.size(1),
              "vq_codebooks must be float32 [n_codebooks, K, width]");
  sq_params = affine_params_checked(sq_params, feat_dim, sq_codes);
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(row_map.device());
  auto out = empty_f32({g.rows, feat_dim}, row_map);
  check_rc(f2cgt_hybrid_decompress_spmm_csr(
               row_map.data_ptr<int32_t>(), static_cast<const uint8_t*>(sq_codes.data_ptr()),
               sq_params.data_ptr<float>(), sq_params.size(1),
               static_cast<const uint8_t*>(vq_codes.data_ptr()), vq_codebooks.data_ptr<float>(),
               g.indptr.data_ptr(), g.indices.data_ptr(), g.tag, out.data_ptr<float>(), g.rows, g.edges,
               row_map.numel(), sq_codes.size(0), vq_codes.size(0), feat_dim, vq_codebooks.size(0),
               vq_codebooks.size(1), vq_codebooks.size(2), current_stream()),
           "hybrid_decompress_spmm_csr");
  return out;
}

void check_hip(hipError_t err, const char* what) {
  TORCH_CHECK(err == hipSuccess, what, ": ", hipGetErrorString(err));
}

// One extra stream (default priority) and its events per device, made on first use and kept for
// the life of the process.  Calls that overlap on one device from several host threads would share
// the events; the module is used from one thread per device like the reference's.
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t inputs_ready = nullptr, agg_done[2] = {nullptr, nullptr}, gemm_done[2] = {nullptr, nullptr};
};

SideStream* side_stream_of(int device) {
  static std::mutex lock;
  static std::map<int, SideStream> made;
  std::lock_guard<std::mutex> hold(lock);
  auto it = made.find(device);
  if (it != made.end()) return &it->second;
  SideStream s;
  check_hip(hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking), "hipStreamCreateWithFlags");
  for (hipEvent_t* ev : {&s.inputs_ready, &s.agg_done[0], &s.agg_done[1], &s.gemm_done[0], &s.gemm_done[1]})
    check_hip(hipEventCreateWithFlags(ev, hipEventDisableTiming), "hipEventCreateWithFlags");
  return &made.emplace(device, s).first->second;
}

// Aggregation followed by the dense layer that consumes it (the first layer of the GraphSAGE model,
// examples/conv.py:68-69, the layer examples/models.py:25-31 stacks, with the mean aggregator: h = fc_neigh(mean over the neighbours)).
// At the reference's widest shape (768 features -> 256 units, 341k destination rows) the fp32 GEMM
// takes 1.75 ms at 86 % of the matrix cores' fp32 peak and the aggregation 0.5 ms, so the multiply
// is not moved into the aggregation kernel: it would slow the part that already dominates.
//   block_rows == 0   one aggregation into a full-size buffer, one GEMM (the fastest form measured)
//   block_rows  > 0   destination rows in blocks of that many: the aggregate exists one block at a
//                     time, which bounds the extra memory to block_rows*feat_dim*4 bytes (1 GB at
//                     the shape above otherwise); ~6 % slower with 65536-row blocks
//   overlap           with blocks: the aggregation of block b+1 runs on a second stream beside the
//                     GEMM of block b, with two staging buffers.  Measured slower than running them
//                     one after the other (the two kernels contend for the same compute units), so
//                     it is off by default and kept for measurement.
// `agg(indptr_ptr, indices_ptr, rows, edges, dst, stream)` enqueues one block on `stream`.  With
// blocks the call reads the edge offsets of the block boundaries on the host, so it cannot be
// captured into a graph.
template <class Agg>
torch::Tensor aggregate_then_linear(const Graph& g, int64_t feat_dim, const torch::Tensor& like,
                                    torch::Tensor weight, const c10::optional<torch::Tensor>& bias,
                                    int64_t block_rows, bool overlap, Agg agg) {
  weight = dev_contig(weight, "weight");
  TORCH_CHECK(weight.dim() == 2 && weight.scalar_type() == torch::kFloat32 && weight.size(1) == feat_dim,
              "weight must be float32 [out_features, feat_dim]");
  torch::Tensor b;
  if (bias.has_value()) {
    b = dev_contig(*bias, "bias");
    TORCH_CHECK(b.dim() == 1 && b.scalar_type() == torch::kFloat32 && b.size(0) == weight.size(0),
                "bias must be float32 [out_features]");
  }
  TORCH_CHECK(block_rows >= 0, "block_rows must be >= 0 (0 = all rows at once)");
  auto out = empty_f32({g.rows, weight.size(0)}, like);
  if (g.rows == 0) return out;
  if (block_rows == 0) block_rows = g.rows;
  block_rows = std::min(block_rows, g.rows);
  const int64_t n_blocks = (g.rows + block_rows - 1) / block_rows;
  auto wt = weight.t();
  auto gemm = [&](torch::Tensor dst, const torch::Tensor& a) {
    if (b.defined())
      at::addmm_out(dst, b, a, wt);
    else
      at::mm_out(dst, a, wt);
  };
  if (n_blocks == 1) {
    auto whole = empty_f32({g.rows, feat_dim}, like);
    agg(g.indptr.data_ptr(), g.indices.data_ptr(), g.rows, g.edges, whole.data_ptr<float>(), current_stream());
    gemm(out, whole);
    return out;
  }
  // edge offsets at the block boundaries: the one host read of the call
  auto at_rows = torch::arange(0, n_blocks + 1, torch::TensorOptions().dtype(torch::kInt64).device(like.device()))
                     .mul_(block_rows).clamp_max_(g.rows);
  auto bounds = g.indptr.index_select(0, at_rows).to(torch::kInt64).cpu();
  const int64_t* e = bounds.data_ptr<int64_t>();
  TORCH_CHECK(e[0] >= 0 && e[n_blocks] <= g.edges, "indptr does not fit indices");
  for (int64_t blk = 0; blk < n_blocks; ++blk)
    TORCH_CHECK(e[blk] <= e[blk + 1], "indptr must be non-decreasing");

  // indptr of every block relative to the block's first edge (so that the kernel choice sees the
  // block's own degree), all blocks in one [n_blocks, block_rows + 1] tensor
  auto opts64 = torch::TensorOptions().dtype(torch::kInt64).device(like.device());
  auto pos = torch::arange(0, n_blocks, opts64).mul_(block_rows).unsqueeze(1) +
             torch::arange(0, block_rows + 1, opts64).unsqueeze(0);
  auto rebased = (g.indptr.index_select(0, pos.clamp_max_(g.rows).reshape({-1})).reshape({n_blocks, block_rows + 1}) -
                  bounds.slice(0, 0, n_blocks).to(like.device()).to(g.indptr.scalar_type()).unsqueeze(1))
                     .contiguous();

  const bool piped = overlap && n_blocks > 1;
  hipStream_t main_stream = static_cast<hipStream_t>(current_stream());
  SideStream* side = piped ? side_stream_of(like.device().index()) : nullptr;
  hipStream_t agg_stream = piped ? side->stream : main_stream;
  torch::Tensor stage[2];
  for (int i = 0; i < (piped ? 2 : 1); ++i) stage[i] = empty_f32({block_rows, feat_dim}, like);
  if (piped) {
    check_hip(hipEventRecord(side->inputs_ready, main_stream), "hipEventRecord");
    check_hip(hipStreamWaitEvent(agg_stream, side->inputs_ready, 0), "hipStreamWaitEvent");
  }
  const int64_t isz = g.indices.element_size(), psz = g.indptr.element_size();
  try {
  for (int64_t blk = 0; blk < n_blocks; ++blk) {
    const int64_t r0 = blk * block_rows, n = std::min(block_rows, g.rows - r0);
    const int slot = piped ? (int)(blk & 1) : 0;
    // the GEMM that last read this staging buffer must be over
    if (piped && blk >= 2) check_hip(hipStreamWaitEvent(agg_stream, side->gemm_done[slot], 0), "hipStreamWaitEvent");
    agg(static_cast<const char*>(rebased.data_ptr()) + blk * (block_rows + 1) * psz,
        static_cast<const char*>(g.indices.data_ptr()) + e[blk] * isz, n, e[blk + 1] - e[blk],
        stage[slot].data_ptr<float>(), static_cast<void*>(agg_stream));
    if (piped) {
      check_hip(hipEventRecord(side->agg_done[slot], agg_stream), "hipEventRecord");
      check_hip(hipStreamWaitEvent(main_stream, side->agg_done[slot], 0), "hipStreamWaitEvent");
    }
    gemm(out.narrow(0, r0, n), stage[slot].narrow(0, 0, n));
    if (piped) check_hip(hipEventRecord(side->gemm_done[slot], main_stream), "hipEventRecord");
  }
  } catch (...) {
    // a refused launch: nothing on the second stream may still use the staging buffers when they
    // are released
    if (piped) (void)hipStreamSynchronize(agg_stream);
    throw;
  }
  // every launch on the second stream is followed by a wait on the caller's stream, so the staging
  // buffers go back to the allocator under the caller's stream as usual
  return out;
}

torch::Tensor vq_decompress_spmm_csr_linear(torch::Tensor compress_feat, torch::Tensor codebooks,
                                            torch::Tensor indptr, torch::Tensor indices, int64_t feat_dim,
                                            torch::Tensor weight, c10::optional<torch::Tensor> bias,
                                            int64_t block_rows, bool overlap) {
  compress_feat = dev_contig(compress_feat, "compress_feat");
  codebooks = beside(codebooks, compress_feat);
  TORCH_CHECK(compress_feat.dim() == 2, "compress_feat must be [rows, n_codebooks]");
  TORCH_CHECK(codebooks.dim() == 3 && codebooks.scalar_type() == torch::kFloat32,
              "VQ codebooks must be float32 [n_codebooks, K, width]");
  TORCH_CHECK(compress_feat.size(1) == codebooks.size(0), "compress_feat has ", compress_feat.size(1),
              " columns but there are ", codebooks.size(0), " codebooks");
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(compress_feat.device());
  const int tag = dtype_tag(compress_feat, "compress_feat");
  return aggregate_then_linear(
      g, feat_dim, compress_feat, weight, bias, block_rows, overlap,
      [&](const void* ip, const void* ix, int64_t rows, int64_t edges, float* dst, void* stream) {
        check_rc(f2cgt_vq_decompress_spmm_csr(compress_feat.data_ptr(), tag, codebooks.data_ptr<float>(), ip, ix,
                                              g.tag, dst, rows, edges, compress_feat.size(0), feat_dim,
                                              codebooks.size(0), codebooks.size(1), codebooks.size(2),
                                              stream),
                 "vq_decompress_spmm_csr_linear");
      });
}

torch::Tensor sq_decompress_spmm_csr_linear(torch::Tensor compress_feat, torch::Tensor codebooks,
                                            torch::Tensor indptr, torch::Tensor indices, int64_t target_bit,
                                            int64_t column_slice, int64_t feat_dim, torch::Tensor weight,
                                            c10::optional<torch::Tensor> bias, int64_t block_rows, bool overlap) {
  compress_feat = dev_contig(compress_feat, "compress_feat");
  TORCH_CHECK(compress_feat.dim() == 2, "compress_feat must be 2-D");
  codebooks = sq_codebooks_checked(codebooks, compress_feat);
  Graph g = graph_of(indptr, indices);
  c10::DeviceGuard guard(compress_feat.device());
  const int tag = dtype_tag(compress_feat, "compress_feat");
  return aggregate_then_linear(
      g, feat_dim, compress_feat, weight, bias, block_rows, overlap,
      [&](const void* ip, const void* ix, int64_t rows, int64_t edges, float* dst, void* stream) {
        check_rc(f2cgt_sq_decompress_spmm_csr(compress_feat.data_ptr(), tag, codebooks.data_ptr<float>(), ip, ix,
                                              g.tag, dst, rows, edges, compress_feat.size(0),
                                              compress_feat.size(1), feat_dim, codebooks.size(0), (int)target_bit,
                                              column_slice, stream),
                 "sq_decompress_spmm_csr_linear");
      });
}

torch::Tensor kmeans_predict(torch::Tensor x, torch::Tensor centers, std::string metric) {
  return kmeans_predict_impl(x, centers, metric, false);
}

// Row fetch of the feature cache (examples/tensor_cache.py:49-58).  `table` is a device tensor
// or a pinned host tensor (mapped into the device address space); `hot` and `slot_map` are the
// device-resident cache of hot rows and the id -> cache slot array (-1 = not cached).
torch::Tensor fetch_rows(torch::Tensor table, torch::Tensor index, c10::optional<torch::Tensor> hot,
                         c10::optional<torch::Tensor> slot_map) {
  TORCH_CHECK(table.defined() && table.dim() == 2 && table.is_contiguous(), "table must be a contiguous 2-D tensor");
  TORCH_CHECK(table.device().is_cuda() || table.is_pinned(),
              "table must be on the GPU or in pinned host memory");
  index = dev_contig(index, "index");
  TORCH_CHECK(index.dim() == 1, "index must be 1-D");
  auto st = index.scalar_type();
  TORCH_CHECK(st == torch::kInt64 || st == torch::kInt32, "index must be int32 or int64");
  TORCH_CHECK(hot.has_value() == slot_map.has_value(), "hot and slot_map come together");
  torch::Tensor hot_t, slot_t;
  int64_t num_hot = 0;
  if (hot.has_value()) {
    hot_t = dev_contig(*hot, "hot");
    slot_t = dev_contig(*slot_map, "slot_map");
    TORCH_CHECK(hot_t.dim() == 2 && hot_t.size(1) == table.size(1) && hot_t.scalar_type() == table.scalar_type(),
                "hot must have the row shape and dtype of table");
    TORCH_CHECK(slot_t.scalar_type() == torch::kInt32 && slot_t.dim() == 1 && slot_t.numel() == table.size(0),
                "slot_map must be int32 with one entry per row of table");
    num_hot = hot_t.size(0);
  }
  TORCH_CHECK(index.numel() == 0 || table.size(0) > 0, "rows requested from an empty table");
  c10::DeviceGuard guard(index.device());
  auto out = torch::empty({index.numel(), table.size(1)}, table.options().device(index.device()).pinned_memory(false));
  const int64_t row_bytes = table.size(1) * (int64_t)table.element_size();
  check_rc(f2cgt_fetch_rows(table.data_ptr(), num_hot ? hot_t.data_ptr() : nullptr,
                            num_hot ? slot_t.data_ptr<int32_t>() : nullptr, index.data_ptr(),
                            st == torch::kInt64 ? F2CGT_DT_I64 : F2CGT_DT_I32, out.data_ptr(), index.numel(),
                            row_bytes, table.size(0), num_hot, current_stream()),
           "fetch_rows");
  return out;
}

// Rows `index` of a code table in device memory, decoded without a copy of their codes; where a shape is not covered,
// fetched and decoded.
torch::Tensor vq_decompress_rows(torch::Tensor table, torch::Tensor index, torch::Tensor codebooks, int64_t feat_dim) {
  const bool plain = table.defined() && index.defined() && codebooks.defined() && table.is_cuda() && index.device() == table.device() &&
                     codebooks.device() == table.device() && table.dim() == 2 && table.is_contiguous() && index.dim() == 1 &&
                     codebooks.dim() == 3 && table.scalar_type() == torch::kUInt8 && codebooks.scalar_type() == torch::kFloat32 &&
                     (index.scalar_type() == torch::kInt64 || index.scalar_type() == torch::kInt32) &&
                     table.size(0) > 0 && table.size(1) == codebooks.size(0) &&
                     index.numel() >= 1024 && feat_dim >= 64 && feat_dim % 2 == 0;   // (others would be refused after an allocation: 1 us)
  if (plain) {
    index = index.contiguous();
    codebooks = codebooks.contiguous();
    c10::DeviceGuard guard(table.device());
    auto out = empty_f32({index.numel(), feat_dim}, table);
    const int rc = f2cgt_vq_decompress_rows(table.data_ptr<uint8_t>(), index.data_ptr(),
                                            index.scalar_type() == torch::kInt64 ? F2CGT_DT_I64 : F2CGT_DT_I32,
                                            codebooks.data_ptr<float>(), out.data_ptr<float>(), index.numel(), table.size(0),
                                            feat_dim, codebooks.size(0), codebooks.size(1), codebooks.size(2), current_stream());
    if (rc >= 0) {
      check_rc(rc, "vq_decompress_rows");
      return out;
    }
  }
  return vq_decompress(fetch_rows(table, index, c10::nullopt, c10::nullopt), codebooks, feat_dim);
}

// The same for scalar codes.  With a slot map the rows are slot_map[index]; check: ids without a row raise KeyError, ids
// outside the map IndexError, behind a wait for the current stream.
torch::Tensor sq_decompress_rows(torch::Tensor table, torch::Tensor index, torch::Tensor codebooks, int64_t target_bits,
                                 int64_t column_slice, int64_t feat_dim, c10::optional<torch::Tensor> slot_map, bool check) {
  const bool plain = table.defined() && index.defined() && table.is_cuda() && index.device() == table.device() && table.dim() == 2 &&
                     table.is_contiguous() && index.dim() == 1 && table.size(0) > 0 &&
                     (table.scalar_type() == torch::kInt8 || table.scalar_type() == torch::kUInt8) &&
                     (index.scalar_type() == torch::kInt64 || index.scalar_type() == torch::kInt32) && feat_dim >= 8 && feat_dim % 2 == 0;
  const bool mapped = slot_map.has_value();
  if (mapped)
    TORCH_CHECK(slot_map->device() == table.device() && slot_map->dim() == 1 && slot_map->is_contiguous() &&
                    slot_map->scalar_type() == torch::kInt32 && slot_map->numel() > 0,
                "slot_map must be a contiguous int32 tensor on the device of table");
  if (plain) {
    index = index.contiguous();
    auto books = sq_codebooks_checked(codebooks, table);
    c10::DeviceGuard guard(table.device());
    auto out = empty_f32({index.numel(), feat_dim}, table);
    torch::Tensor bad;
    int32_t* flag = nullptr;
    if (mapped && check) {
      // one word of pinned memory, which the kernel writes only for a bad id
      bad = torch::empty({1}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
      flag = bad.data_ptr<int32_t>();
      *flag = 0;
    }
    const int rc = f2cgt_sq_decompress_rows(
        table.data_ptr(), dtype_tag(table, "table"), index.data_ptr(),
        index.scalar_type() == torch::kInt64 ? F2CGT_DT_I64 : F2CGT_DT_I32, mapped ? slot_map->data_ptr<int32_t>() : nullptr,
        mapped ? slot_map->numel() : 0, flag, books.data_ptr<float>(), out.data_ptr<float>(), index.numel(), table.size(0),
        table.size(1), feat_dim, books.size(0), (int)target_bits, column_slice, current_stream());
    if (rc >= 0) {
      check_rc(rc, "sq_decompress_rows");
      if (flag != nullptr) {
        {
          py::gil_scoped_release unlocked;
          c10::hip::getCurrentHIPStream().synchronize();
        }
        const int32_t seen = *const_cast<volatile int32_t*>(flag);
        if (seen == 1) throw py::key_error("a requested id is not a seed row");
        if (seen != 0) throw py::index_error("an id lies outside the slot map");
      }
      return out;
    }
  }
  if (mapped) {
    // ids are held to the map, as in the kernel: an index beyond it would end the process
    auto ids = index.to(slot_map->device(), torch::kInt64);
    ids = torch::where(ids.lt(0), ids.add(slot_map->numel()), ids);
    auto held = ids.clamp(0, slot_map->numel() - 1);
    auto slots = slot_map->index({held}).to(torch::kInt64);
    if (check) {
      auto seen = torch::stack({ids.ne(held).any(), slots.lt(0).any()}).cpu();
      if (seen.data_ptr<bool>()[0]) throw py::index_error("an id lies outside the slot map");
      if (seen.data_ptr<bool>()[1]) throw py::key_error("a requested id is not a seed row");
    }
    index = slots;
  } else if (index.scalar_type() != torch::kInt64 && index.scalar_type() != torch::kInt32) {
    index = index.to(torch::kInt64);
  }
  return sq_decompress(fetch_rows(table, index, c10::nullopt, c10::nullopt), codebooks, target_bits, column_slice, feat_dim);
}

// ---- the dense part of a GraphSAGE layer in one kernel each way ---------------------------------------
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

// Whether an operator's call goes straight to the device now: no transform, forward-mode gradient, autocast, dispatch or
// function mode and no tracing is active.
bool plain_calls() {
  using c10::DispatchKey;
  static const c10::DispatchKeySet plain = c10::DispatchKeySet({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView});
  return (c10::impl::tls_local_dispatch_key_set().included_ | plain) == plain && !at::autocast::is_autocast_enabled(at::kCUDA) &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !torch::jit::tracer::isTracing() &&
         torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr;
}

// Whether t is a torch.Tensor or a Parameter in Python: a subclass of them may have operators of its own
// (__torch_function__), which its keys do not tell.  Holds the GIL.
bool own_class(const torch::Tensor& t) {
  const auto object = py::reinterpret_steal<py::object>(THPVariable_Wrap(t));
  return THPVariable_CheckExact(object.ptr());
}

// Whether t is fp32 memory on `device` and nothing else: no wrapper (a batch, a subclass with its own dispatch), no lazily
// negated or zero tensor.
bool plain_tensor(const torch::Tensor& t, const c10::Device& device) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet plain = c10::DispatchKeySet({DispatchKey::CUDA, DispatchKey::AutogradCUDA,
                                                                DispatchKey::ADInplaceOrView, DispatchKey::AutocastCUDA});
  return t.defined() && (t.key_set() | plain) == plain && t.scalar_type() == torch::kFloat32 && t.layout() == torch::kStrided &&
         t.device() == device;
}
bool dense_rows(const torch::Tensor& t, const c10::Device& device, int64_t rows, int64_t cols) {
  return plain_tensor(t, device) && t.dim() == 2 && t.is_contiguous() && t.size(0) == rows && t.size(1) == cols;
}

// act(x0 w0^T + x1 w1^T + bias) by the kernel or by the library's products.  The two have the same bits at the shapes that
// the kernel is taken for: a value next to zero that two orders of summation put on either side of it, one in 10^7, passes
// its whole gradient in one and none in the other (a gradient of 16 000 rows is 5e-4 away for it).
torch::Tensor sage_forward(bool kernel, const torch::Tensor& x0, const torch::Tensor& x1, const torch::Tensor& w0,
                           const torch::Tensor& w1, const c10::optional<torch::Tensor>& bias, bool relu) {
  if (kernel) {
    c10::DeviceGuard guard(x0.device());
    const int64_t m = x0.size(0), n = w0.size(0);
    auto out = torch::empty({m, n}, x0.options());
    check_rc(f2cgt_sage_linear(x0.data_ptr<float>(), w0.data_ptr<float>(), x1.data_ptr<float>(), w1.data_ptr<float>(),
                               bias.has_value() ? bias->data_ptr<float>() : nullptr, out.data_ptr<float>(), m, n, x0.size(1),
                               x1.size(1), relu ? 1 : 0, current_stream()),
             "sage_linear");
    return out;
  }
  at::AutoDispatchBelowADInplaceOrView products;        // (nothing in here is differentiated by itself)
  auto out = bias.has_value() ? at::addmm(*bias, x0, w0.t()) : at::mm(x0, w0.t());
  out.add_(at::mm(x1, w1.t()));
  if (relu) out.relu_();
  return out;
}

// Only w0, w1 and bias are differentiated.
struct SageLinear : public torch::autograd::Function<SageLinear> {
  static Variable forward(AutogradContext* ctx, const Variable& x0, const Variable& x1, const Variable& w0, const Variable& w1,
                          const c10::optional<Variable>& bias, bool relu, bool kernel) {
    torch::Tensor out = sage_forward(kernel, x0, x1, w0, w1, bias, relu);
    ctx->saved_data["relu"] = relu;
    ctx->saved_data["bias"] = bias.has_value();
    if (relu) ctx->save_for_backward({x0, x1, out});
    else ctx->save_for_backward({x0, x1});
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const bool relu = ctx->saved_data["relu"].toBool();
    const Variable& x0 = saved[0];
    const Variable& x1 = saved[1];
    const bool want0 = ctx->needs_input_grad(2), want1 = ctx->needs_input_grad(3), want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(4);
    variable_list result(7);
    Variable g = grads[0];
    if (!g.defined() || !(want0 || want1 || want_b)) return result;
    // The saved tensors went through the caller's hooks, the gradient through operators between: each is looked at again.
    const c10::Device device = x0.device();
    const bool own = !c10::GradMode::is_enabled() && plain_calls() && plain_tensor(g, device) && g.dim() == 2 &&
                     x0.dim() == 2 && x1.dim() == 2 && dense_rows(x0, device, g.size(0), x0.size(1)) &&
                     dense_rows(x1, device, g.size(0), x1.size(1)) && (!relu || dense_rows(saved[2], device, g.size(0), g.size(1)));
    if (!own) {
      // a gradient that is differentiated itself or is a batch of them, a mode: the same sums from operators
      if (relu) g = at::threshold_backward(g, saved[2], 0);
      if (want0) result[2] = g.t().mm(x0);
      if (want1) result[3] = g.t().mm(x1);
      if (want_b) result[4] = g.sum(0);
      return result;
    }
    c10::DeviceGuard guard(device);
    g = g.contiguous();
    const int64_t m = g.size(0), n = g.size(1), k0 = x0.size(1), k1 = x1.size(1);
    if (want0) result[2] = torch::empty({n, k0}, g.options());
    if (want1) result[3] = torch::empty({n, k1}, g.options());
    if (want_b) result[4] = torch::empty({n}, g.options());
    auto ptr = [](const Variable& v) { return v.defined() ? v.data_ptr<float>() : nullptr; };
    torch::Tensor ws;
    const int64_t bytes = f2cgt_sage_linear_grad_workspace_bytes(m, n, k0, k1);
    if (bytes > 0) ws = torch::empty({bytes}, g.options().dtype(torch::kUInt8));
    check_rc(f2cgt_sage_linear_grad(g.data_ptr<float>(), relu ? saved[2].data_ptr<float>() : nullptr, x0.data_ptr<float>(),
                                    x1.data_ptr<float>(), ptr(result[2]), ptr(result[3]), ptr(result[4]),
                                    bytes > 0 ? ws.data_ptr() : nullptr, bytes, m, n, k0, k1, current_stream()),
             "sage_linear_grad");
    return result;
  }
};

// -> the layer's output, or None for the calls that are left to the module's own operators: other types, layouts, devices
// and sizes; inputs that are differentiated; and whenever an operator's call would not go straight to the device
// (subclasses of Tensor, transforms, forward-mode gradients, autocast, dispatch and function modes, tracing).
c10::optional<torch::Tensor> sage_linear(const torch::Tensor& x0, const torch::Tensor& x1, const torch::Tensor& w0,
                                         const torch::Tensor& w1, const c10::optional<torch::Tensor>& bias, bool relu) {
  if (!plain_calls()) return c10::nullopt;
  if (!x0.defined()) return c10::nullopt;
  auto plain = [&](const torch::Tensor& t, int64_t dims) {
    return plain_tensor(t, x0.device()) && t.dim() == dims && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  if (!plain(x0, 2) || !plain(x1, 2) || !plain(w0, 2) || !plain(w1, 2) || (bias.has_value() && !plain(*bias, 1)))
    return c10::nullopt;
  if (!own_class(x0) || !own_class(x1) || !own_class(w0) || !own_class(w1) || (bias.has_value() && !own_class(*bias)))
    return c10::nullopt;
  const int64_t m = x0.size(0), n = w0.size(0), k0 = x0.size(1), k1 = x1.size(1);
  if (x0.requires_grad() || x1.requires_grad() || m < 1 || n < 1 || k0 < 4 || k1 < 4 || k0 % 4 != 0 || k1 % 4 != 0 ||
      x1.size(0) != m || w1.size(0) != n || w0.size(1) != k0 || w1.size(1) != k1 || (bias.has_value() && bias->size(0) != n))
    return c10::nullopt;
  const int take = f2cgt_sage_linear_ahead(m, n, k0, k1);
  py::gil_scoped_release unlocked;         // as the operators do: the library may look for a kernel, other threads go on
  if (c10::GradMode::is_enabled() && (w0.requires_grad() || w1.requires_grad() || (bias.has_value() && bias->requires_grad()))) {
    if (!(take & F2CGT_SAGE_GRAD)) return c10::nullopt;
    return SageLinear::apply(x0, x1, w0, w1, bias, relu, (take & F2CGT_SAGE_STEP) != 0);
  }
  return sage_forward((take & F2CGT_SAGE_FORWARD) != 0, x0, x1, w0, w1, bias, relu);
}

torch::Tensor vq_encode(torch::Tensor x, torch::Tensor centers, std::string metric) {
  return kmeans_predict_impl(x, centers, metric, true);
}

// Codes of all column slices of a table in one launch, into `out` (uint8 [m, slices]).  -> false, with nothing
// written, for the calls that it does not take (the caller then goes slice by slice through KMeans.predict).
bool vq_encode_slices(torch::Tensor x, torch::Tensor codebooks, torch::Tensor out, std::string metric) {
  const bool plain = x.is_cuda() && x.device() == codebooks.device() && x.device() == out.device() && x.dim() == 2 &&
                     codebooks.dim() == 3 && out.dim() == 2 && x.scalar_type() == torch::kFloat32 &&
                     codebooks.scalar_type() == torch::kFloat32 && out.scalar_type() == torch::kUInt8;
  if (!plain || x.size(1) < 1 || x.stride(1) != 1 || x.stride(0) < x.size(1) || out.size(0) != x.size(0) ||
      out.size(1) != codebooks.size(0) || out.stride(1) != 1 || out.stride(0) < out.size(1))
    return false;
  const int64_t slices = codebooks.size(0), n = codebooks.size(1), k = codebooks.size(2);
  if (!f2cgt_vq_encode_slices_covers(n, k) || slices < 1 || slices > 65536 || x.size(1) >= (1 << 22) ||
      (slices - 1) * k >= x.size(1))
    return false;
  codebooks = codebooks.contiguous();
  c10::DeviceGuard guard(x.device());
  check_rc(f2cgt_vq_encode_slices(x.data_ptr<float>(), x.stride(0), x.size(1), codebooks.data_ptr<float>(),
                                  out.data_ptr<uint8_t>(), out.stride(0), x.size(0), slices, n, k, metric_tag(metric),
                                  current_stream()),
           "vq_encode_slices");
  return true;
}

}  // namespace

// Output store policy of the SQ aggregation operators: "auto" (by output size), "stream"
// (non-temporal stores whatever the size) or "cached" (plain stores); returns the previous one.
std::string set_store_mode(const std::string& mode) {
  static const char* names[] = {"auto", "stream", "cached"};
  int want = -1;
  for (int i = 0; i < 3; ++i)
    if (mode == names[i]) want = i;
  TORCH_CHECK(want >= 0, "set_store_mode: mode must be \"auto\", \"stream\" or \"cached\", got \"", mode, "\"");
  const int was = f2cgt_set_store_mode(want);
  TORCH_CHECK(was >= 0, f2cgt_last_error());
  return names[was];
}

PYBIND11_MODULE(F2CGTLib, m) {
  m.doc() = "MI355X-native drop-in for F2CGT's F2CGTLib operator module";
  m.def("packbits", &packbits, py::arg("unpack"), py::arg("target_bits"))
      .def("unpackbits", &unpackbits, py::arg("pack"), py::arg("target_bits"), py::arg("unpack_dim"))
      .def("sq_compress", &sq_compress, py::arg("src"), py::arg("codebooks"), py::arg("target_bits"),
           py::arg("column_slice"))
      .def("sq_decompress", &sq_decompress, py::arg("compress_data"), py::arg("codebooks"),
           py::arg("target_bits"), py::arg("column_slice"), py::arg("feat_dim"))
      .def("vq_decompress", &vq_decompress, py::arg("index_tensor"), py::arg("codebooks"),
           py::arg("feat_dim"))
      .def("pairwise_distance", &pairwise_distance, py::arg("x"), py::arg("y"), py::arg("metric"))
      .def("spmm_csr", &spmm_csr, py::arg("feat"), py::arg("indptr"), py::arg("indices"))
      .def("vq_decompress_spmm_csr", &vq_decompress_spmm_csr, py::arg("compress_feat"),
           py::arg("codebooks"), py::arg("indptr"), py::arg("indices"), py::arg("feat_dim"))
      .def("sq_decompress_spmm_csr", &sq_decompress_spmm_csr, py::arg("compress_feat"),
           py::arg("codebooks"), py::arg("indptr"), py::arg("indices"), py::arg("target_bit"),
           py::arg("column_slice"), py::arg("feat_dim"));
  // extensions
  m.def("sq_affine_decompress", &sq_affine_decompress, py::arg("compress_data"), py::arg("params"),
        py::arg("target_bits"), py::arg("feat_dim"))
      .def("sq_affine_decompress_spmm_csr", &sq_affine_decompress_spmm_csr, py::arg("compress_feat"),
           py::arg("params"), py::arg("indptr"), py::arg("indices"), py::arg("target_bit"),
           py::arg("feat_dim"))
      .def("hybrid_decompress_spmm_csr", &hybrid_decompress_spmm_csr, py::arg("row_map"),
           py::arg("sq_codes"), py::arg("sq_params"), py::arg("vq_codes"), py::arg("vq_codebooks"),
           py::arg("indptr"), py::arg("indices"), py::arg("feat_dim"))
      .def("vq_decompress_spmm_csr_linear", &vq_decompress_spmm_csr_linear, py::arg("compress_feat"),
           py::arg("codebooks"), py::arg("indptr"), py::arg("indices"), py::arg("feat_dim"),
           py::arg("weight"), py::arg("bias") = py::none(), py::arg("block_rows") = 0, py::arg("overlap") = false)
      .def("sq_decompress_spmm_csr_linear", &sq_decompress_spmm_csr_linear, py::arg("compress_feat"),
           py::arg("codebooks"), py::arg("indptr"), py::arg("indices"), py::arg("target_bit"),
           py::arg("column_slice"), py::arg("feat_dim"), py::arg("weight"), py::arg("bias") = py::none(),
           py::arg("block_rows") = 0, py::arg("overlap") = false)
      .def("sq_encode", &sq_encode, py::arg("src"), py::arg("codebooks"), py::arg("target_bits"),
           py::arg("column_slice"), py::arg("out") = py::none())
      .def("abs_order_stats", &abs_order_stats, py::arg("x"), py::arg("rows"), py::arg("column_slice"), py::arg("ranks"))
      .def("sq_codebooks", &sq_codebooks, py::arg("x"), py::arg("rows"), py::arg("column_slice"), py::arg("ranks"),
           py::arg("weights"))
      .def("kmeans_predict", &kmeans_predict, py::arg("x"), py::arg("centers"), py::arg("metric"))
      .def("vq_encode", &vq_encode, py::arg("x"), py::arg("centers"), py::arg("metric"))
      .def("vq_encode_slices", &vq_encode_slices, py::arg("x"), py::arg("codebooks"), py::arg("out"), py::arg("metric"))
      .def("vq_decompress_rows", &vq_decompress_rows, py::arg("table"), py::arg("index"), py::arg("codebooks"),
           py::arg("feat_dim"))
      .def("sq_decompress_rows", &sq_decompress_rows, py::arg("table"), py::arg("index"), py::arg("codebooks"),
           py::arg("target_bits"), py::arg("column_slice"), py::arg("feat_dim"), py::arg("slot_map") = py::none(),
           py::arg("check") = false)
      .def("sage_linear", &sage_linear, py::arg("h_self"), py::arg("h_neigh"), py::arg("w_self"), py::arg("w_neigh"),
           py::arg("bias"), py::arg("relu"))
      .def("fetch_rows", &fetch_rows, py::arg("table"), py::arg("index"), py::arg("hot") = py::none(),
           py::arg("slot_map") = py::none())
      .def("kmeans_update", &kmeans_update, py::arg("data"), py::arg("labels"), py::arg("centers"),
           py::arg("stop") = py::none(), py::arg("rule") = 0, py::arg("tol") = 0.0)
      .def("slice_rows", &slice_rows, py::arg("x"), py::arg("rows"), py::arg("column_slice"))
      .def("keep_rows", &keep_rows, py::arg("norms"), py::arg("stats"), py::arg("weight"), py::arg("weight_last"))
      .def("kmeans_slices_covers", &kmeans_slices_covers, py::arg("slices"), py::arg("n"), py::arg("k"))
      .def("kmeans_slices_fit", &kmeans_slices_fit, py::arg("x"), py::arg("keep"), py::arg("centers"), py::arg("metric"),
           py::arg("rule"), py::arg("tol"), py::arg("growth"), py::arg("max_iter"), py::arg("check_every"),
           py::arg("bad_row") = py::none(), py::arg("rescale") = false)
      .def("set_store_mode", &set_store_mode, py::arg("mode"));
  py::class_<PendingFlag, std::shared_ptr<PendingFlag>>(m, "PendingFlag").def("wait", &PendingFlag::wait);
  py::class_<KMeans>(m, "KMeans")
      .def(py::init<int64_t, int64_t, std::string, int, double, int, double, int, int, bool>(),
           py::arg("n_cluster"), py::arg("feat_dim"), py::arg("metric"), py::arg("max_iter") = 300,
           py::arg("tol") = 1e-4, py::arg("n_init") = 1, py::arg("oversampling_factor") = 2.0,
           py::arg("batch_samples") = 1 << 15, py::arg("batch_centroids") = 0,
           py::arg("inertia_check") = false)
      .def(py::init<torch::Tensor, std::string, int, double, int, double, int, int, bool>(),
           py::arg("centers"), py::arg("metric"), py::arg("max_iter") = 300, py::arg("tol") = 1e-4,
           py::arg("n_init") = 1, py::arg("oversampling_factor") = 2.0,
           py::arg("batch_samples") = 1 << 15, py::arg("batch_centroids") = 0,
           py::arg("inertia_check") = false)
      .def("fit", &KMeans::fit, py::arg("data"))
      .def("predict", &KMeans::predict, py::arg("data"), py::arg("normalize_weights") = true)
      .def("get_centers", &KMeans::get_centers)
      .def_property_readonly("n_iter", &KMeans::n_iter);   // extension: update steps issued by the last fit()
}
