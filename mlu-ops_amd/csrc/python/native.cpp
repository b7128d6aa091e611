// The host side of the Python package in native code: tensors in, tensors out, one call per
// operator.  A call sets its descriptors, asks for the workspace size, allocates outputs and
// workspace from torch's caching allocator and enqueues the operator through the C API; the
// sparse layers' autograd node lives here as well, so that neither direction of a layer runs
// interpreter code.  What bounds a small layer is this path: with ctypes calls, Python
// descriptors and a Python autograd function a training step of one layer took 290-360 us of
// host time around 90-130 us of kernels.
//
// The library is bound at run time (bind) to the very file the ctypes side loaded, so both
// share its handles.
#include <torch/extension.h>

#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>

#include <atomic>
#include <map>
#include <mutex>
#include <optional>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "mlu_op.h"
#include "mlu_op_ext.h"

namespace py = pybind11;

namespace {

// ---- the library ---------------------------------------------------------------------------

#define MLUOP_NATIVE_FUNCTIONS(X)                          \
  X(mluOpCreate)                                           \
  X(mluOpSetQueue)                                         \
  X(mluOpGetQueue)                                         \
  X(mluOpGetErrorString)                                   \
  X(mluOpCreateTensorDescriptor)                           \
  X(mluOpSetTensorDescriptor_v2)                           \
  X(mluOpSetTensorDescriptorOnchipDataType)                \
  X(mluOpDestroyTensorDescriptor)                          \
  X(mluOpCreateSparseConvolutionDescriptor)                \
  X(mluOpSetSparseConvolutionDescriptor)                   \
  X(mluOpGetSparseConvolutionNumActOut)                    \
  X(mluOpDestroySparseConvolutionDescriptor)               \
  X(mluOpGetIndicePairsWorkspaceSize)                      \
  X(mluOpGetIndicePairs)                                   \
  X(mluOpGetIndiceConvolutionForwardWorkspaceSize)         \
  X(mluOpIndiceConvolutionForward)                         \
  X(mluOpGetIndiceConvolutionBackwardDataWorkspaceSize)    \
  X(mluOpIndiceConvolutionBackwardData)                    \
  X(mluOpGetIndiceConvolutionBackwardFilterWorkspaceSize)  \
  X(mluOpIndiceConvolutionBackwardFilter)                  \
  X(mluOpGetVoxelizationWorkspaceSize)                     \
  X(mluOpVoxelization)                                     \
  X(mluOpGetDynamicPointToVoxelForwardWorkspaceSize)       \
  X(mluOpDynamicPointToVoxelForward)                       \
  X(mluOpGetDynamicPointToVoxelBackwardWorkspaceSize)      \
  X(mluOpDynamicPointToVoxelBackward)                      \
  X(mluOpExtSetSparseConvExtendedModes)                    \
  X(mluOpExtSetDistinctPairsPromise)                       \
  X(mluOpExtSetSinglePairsPromise)                         \
  X(mluOpExtGetSinglePairsPromise)                         \
  X(mluOpExtSetPairTails)                                  \
  X(mluOpExtGetPairTails)                                  \
  X(mluOpExtSetForwardRelu)                                \
  X(mluOpExtGetForwardRelu)                                \
  X(mluOpExtGetOrderVoxelsWorkspaceSize)                   \
  X(mluOpExtOrderVoxels)                                   \
  X(mluOpExtMeanVoxelPoints)                               \
  X(mluOpExtGetIndicePairsHostCounts)                      \
  X(mluOpExtGetVoxelizationHostCount)                      \
  X(mluOpExtGetRowMapSize)                                 \
  X(mluOpExtBuildRowMap)                                   \
  X(mluOpExtUseRowMap)                                     \
  X(mluOpExtForgetRowMap)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
  MLUOP_NATIVE_FUNCTIONS(X)
#undef X
};
Library api;

void bind(const std::string &path) {
  void *so = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (so == nullptr) throw std::runtime_error(std::string("cannot load ") + path + ": " + dlerror());
#define X(name)                                                                         \
  api.name = reinterpret_cast<decltype(&::name)>(dlsym(so, #name));                     \
  if (api.name == nullptr) throw std::runtime_error(path + " does not export " #name);
  MLUOP_NATIVE_FUNCTIONS(X)
#undef X
}

// A status other than success; Python sees it as mluop_hip.MluOpError.
struct StatusError : std::runtime_error {
  StatusError(int status, const char *what)
      : std::runtime_error(std::string(what) + " returned " +
                           api.mluOpGetErrorString(static_cast<mluOpStatus_t>(status))),
        status(status), call(what) {}
  int status;
  std::string call;
};

inline void check(mluOpStatus_t status, const char *what) {
  if (status != MLUOP_STATUS_SUCCESS) throw StatusError(status, what);
}

class TensorDesc {
 public:
  TensorDesc(mluOpTensorLayout_t layout, mluOpDataType_t dtype, at::IntArrayRef dims) {
    check(api.mluOpCreateTensorDescriptor(&d_), "mluOpCreateTensorDescriptor");
    const mluOpStatus_t st =
        api.mluOpSetTensorDescriptor_v2(d_, layout, dtype, static_cast<int>(dims.size()), dims.data());
    if (st != MLUOP_STATUS_SUCCESS) {
      api.mluOpDestroyTensorDescriptor(d_);
      check(st, "mluOpSetTensorDescriptor_v2");
    }
  }
  ~TensorDesc() { api.mluOpDestroyTensorDescriptor(d_); }
  TensorDesc(const TensorDesc &) = delete;
  TensorDesc &operator=(const TensorDesc &) = delete;
  operator mluOpTensorDescriptor_t() const { return d_; }

 private:
  mluOpTensorDescriptor_t d_ = nullptr;
};

mluOpDataType_t dtypeCode(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return MLUOP_DTYPE_HALF;
    case at::kFloat: return MLUOP_DTYPE_FLOAT;
    case at::kBFloat16: return MLUOP_DTYPE_BFLOAT16;
    case at::kInt: return MLUOP_DTYPE_INT32;
    default: throw py::key_error(std::string(c10::toString(t)));
  }
}

// ---- buffers -------------------------------------------------------------------------------

// Outputs and workspaces of one operator call.  In the package's guard mode (bands of a
// pattern around every buffer, checked after the call) they come from the Python functions
// that keep the bands; otherwise straight from the allocator.  Never used with the GIL held.
class Buffers {
 public:
  Buffers(bool guarded, at::Device device) : guarded_(guarded), device_(device) {}

  at::Tensor output(at::IntArrayRef shape, at::ScalarType dtype, const char *what,
                    std::optional<int> fill = std::nullopt) const {
    if (guarded_) {
      py::gil_scoped_acquire gil;
      py::tuple dims(shape.size());
      for (size_t i = 0; i < shape.size(); ++i) dims[i] = shape[i];
      py::object filled = py::none();
      if (fill) filled = py::int_(*fill);
      return package().attr("_output")(dims, py::cast(dtype), py::cast(device_), what, filled).cast<at::Tensor>();
    }
    const auto options = at::TensorOptions().dtype(dtype).device(device_);
    return fill ? at::full(shape, *fill, options) : at::empty(shape, options);
  }
  at::Tensor workspace(size_t bytes) const {
    if (guarded_) {
      py::gil_scoped_acquire gil;
      return package().attr("_workspace")(bytes, py::cast(device_)).cast<at::Tensor>();
    }
    return at::empty({static_cast<int64_t>(bytes > 0 ? bytes : 1)},
                     at::TensorOptions().dtype(at::kByte).device(device_));
  }
  void done(const char *call) const {
    if (!guarded_) return;
    py::gil_scoped_acquire gil;
    package().attr("_guards_intact")(call);
  }

 private:
  static py::module_ package() { return py::module_::import("mluop_hip"); }
  bool guarded_;
  at::Device device_;
};

// ---- operators -----------------------------------------------------------------------------

using Ints = std::vector<int>;
using Counts = std::vector<int64_t>;

struct Rulebook3 {
  at::Tensor pairs, out_indices, indice_num;
  int64_t num_act_out = 0;
  Counts counts;
};

// Sets and destroys the descriptor of one rulebook call.
class ConvDesc {
 public:
  ConvDesc(int batch, const Ints &pad, const Ints &stride, const Ints &dilation, const Ints &input_space,
           const Ints &filter_space, const Ints &output_space, bool sub_m) {
    for (const Ints *v : {&pad, &stride, &dilation, &input_space, &filter_space, &output_space})
      if (v->size() != 3) throw py::value_error("spaces, padding, stride and dilation have three values each");
    check(api.mluOpCreateSparseConvolutionDescriptor(&d_), "mluOpCreateSparseConvolutionDescriptor");
    const mluOpStatus_t st = api.mluOpSetSparseConvolutionDescriptor(
        d_, 5, batch, pad.data(), stride.data(), dilation.data(), input_space.data(), filter_space.data(),
        output_space.data(), sub_m ? 1 : 0, 0, 0);
    if (st != MLUOP_STATUS_SUCCESS) {
      api.mluOpDestroySparseConvolutionDescriptor(d_);
      check(st, "mluOpSetSparseConvolutionDescriptor");
    }
  }
  ~ConvDesc() { api.mluOpDestroySparseConvolutionDescriptor(d_); }
  ConvDesc(const ConvDesc &) = delete;
  ConvDesc &operator=(const ConvDesc &) = delete;
  operator mluOpSparseConvolutionDescriptor_t() const { return d_; }

 private:
  mluOpSparseConvolutionDescriptor_t d_ = nullptr;
};

// A setting of a handle has this value while this is there, and the caller's again afterwards.
class Setting {
 public:
  using Get = mluOpStatus_t (*)(mluOpHandle_t, int *);
  using Set = mluOpStatus_t (*)(mluOpHandle_t, int);
  Setting(mluOpHandle_t handle, Get get, Set set, int value, const char *what) : handle_(handle), set_(set) {
    check(get(handle, &before_), what);
    check(set(handle, value), what);
  }
  ~Setting() { (void)set_(handle_, before_); }
  Setting(const Setting &) = delete;
  Setting &operator=(const Setting &) = delete;

 private:
  mluOpHandle_t handle_;
  Set set_;
  int before_ = 0;
};

// The pair counts of a rulebook built on `handle`, as soon as they are there; false: not on file.
bool hostCounts(mluOpHandle_t handle, const at::Tensor &pairs, Counts *counts) {
  counts->assign(pairs.size(0), 0);
  return pairs.numel() == 0 ||
         api.mluOpExtGetIndicePairsHostCounts(handle, pairs.data_ptr(), static_cast<int>(pairs.size(0)),
                                              counts->data()) == MLUOP_STATUS_SUCCESS;
}

// `for_layer`: out_indices is cut to the active rows (and its tail left as allocated), and with
// `wait_counts` the counts come back on the host.
Rulebook3 indicePairs(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &indices, int batch,
                      const Ints &input_space, const Ints &filter_space, const Ints &output_space, const Ints &pad,
                      const Ints &stride, const Ints &dilation, bool sub_m, std::optional<int64_t> out_rows,
                      std::optional<at::Tensor> out_indices, bool for_layer, bool tails, bool wait_counts) {
  const int64_t L = indices.size(0);
  int64_t K = 1;
  for (int k : filter_space) K *= k;
  if (!out_rows) {
    int64_t volume = batch;
    for (int o : output_space) volume *= o;
    out_rows = sub_m ? L : std::min(volume, K * L);
  }
  Rulebook3 r;
  r.pairs = buffers.output({K, 2, L}, at::kInt, "indice_pairs");
  if (out_indices) {
    r.out_indices = *out_indices;
    out_rows = out_indices->size(0);
  } else {
    // the operator writes the first num_act_out rows only; the rest keep this initial -1
    r.out_indices = buffers.output({*out_rows, 4}, at::kInt, "out_indices",
                                   for_layer ? std::nullopt : std::optional<int>(-1));
  }
  r.indice_num = buffers.output({K}, at::kInt, "indice_num");
  const ConvDesc conv(batch, pad, stride, dilation, input_space, filter_space, output_space, sub_m);
  const TensorDesc d_in(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, {L, 4});
  const TensorDesc d_pairs(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, {K, 2, L});
  const TensorDesc d_out(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, {*out_rows, 4});
  const TensorDesc d_num(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, {K});
  size_t bytes = 0;
  check(api.mluOpGetIndicePairsWorkspaceSize(handle, conv, d_in, d_pairs, d_out, d_num, &bytes),
        "mluOpGetIndicePairsWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  {
    std::optional<Setting> without;
    if (!tails) without.emplace(handle, api.mluOpExtGetPairTails, api.mluOpExtSetPairTails, 0, "mluOpExtSetPairTails");
    check(api.mluOpGetIndicePairs(handle, conv, d_in, indices.data_ptr(), ws.data_ptr(), bytes, d_pairs,
                                  r.pairs.data_ptr(), d_out, r.out_indices.data_ptr(), d_num,
                                  r.indice_num.data_ptr()),
          "mluOpGetIndicePairs");
  }
  r.num_act_out = L;
  if (!sub_m) {
    int n = 0;
    check(api.mluOpGetSparseConvolutionNumActOut(conv, &n), "mluOpGetSparseConvolutionNumActOut");
    r.num_act_out = n;
  }
  if (for_layer) {
    const bool empty = L == 0 || K == 0 || *out_rows == 0;
    if (empty) {
      r.counts.assign(K, 0);
    } else if (wait_counts && !hostCounts(handle, r.pairs, &r.counts)) {
      const at::Tensor host = r.indice_num.cpu();
      const int32_t *n = host.data_ptr<int32_t>();
      r.counts.assign(n, n + K);
    }
    r.out_indices = r.out_indices.narrow(0, 0, r.num_act_out);
  }
  buffers.done("mluOpGetIndicePairs");
  return r;
}

// `counts_of`: the pair counts; it may wait for them, and is asked once all that needs none of them is done.
template <typename COUNTS_OF>
at::Tensor convForward(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &features,
                       const at::Tensor &filters, mluOpTensorLayout_t layout, const at::Tensor &pairs,
                       COUNTS_OF &&counts_of, int64_t num_act_out, bool sub_m, int64_t inverse,
                       const void *row_map) {
  const mluOpDataType_t code = dtypeCode(features.scalar_type());
  const int64_t co = filters.size(layout == MLUOP_LAYOUT_ARRAY ? 4 : 0);
  at::Tensor out = buffers.output({num_act_out, co}, features.scalar_type(), "features_out");
  const TensorDesc d_x(MLUOP_LAYOUT_ARRAY, code, features.sizes());
  const TensorDesc d_w(layout, code, filters.sizes());
  const TensorDesc d_pairs(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, pairs.sizes());
  const TensorDesc d_out(MLUOP_LAYOUT_ARRAY, code, out.sizes());
  size_t bytes = 0;
  // (the workspace is as large for one number of pairs as for another)
  check(api.mluOpGetIndiceConvolutionForwardWorkspaceSize(handle, d_x, d_w, d_pairs, d_out, Counts(pairs.size(0)).data(),
                                                          num_act_out, inverse, sub_m, &bytes),
        "mluOpGetIndiceConvolutionForwardWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  const Counts &counts = counts_of();
  if (row_map != nullptr) check(api.mluOpExtUseRowMap(handle, row_map), "mluOpExtUseRowMap");
  check(api.mluOpIndiceConvolutionForward(handle, d_x, features.data_ptr(), d_w, filters.data_ptr(), d_pairs,
                                          pairs.data_ptr(), counts.data(), num_act_out, inverse, sub_m,
                                          ws.data_ptr(), bytes, d_out, out.data_ptr()),
        "mluOpIndiceConvolutionForward");
  buffers.done("mluOpIndiceConvolutionForward");
  return out;
}

at::Tensor convBackwardData(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &output_grad,
                            const at::Tensor &filters, mluOpTensorLayout_t layout, const at::Tensor &pairs,
                            const Counts &counts, bool sub_m, int64_t ci, int64_t inverse, int64_t rows,
                            const void *row_map) {
  const mluOpDataType_t code = dtypeCode(output_grad.scalar_type());
  at::Tensor dx = buffers.output({rows, ci}, output_grad.scalar_type(), "input_grad");
  const TensorDesc d_dy(MLUOP_LAYOUT_ARRAY, code, output_grad.sizes());
  const TensorDesc d_w(layout, code, filters.sizes());
  const TensorDesc d_pairs(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, pairs.sizes());
  const TensorDesc d_dx(MLUOP_LAYOUT_ARRAY, code, dx.sizes());
  size_t bytes = 0;
  check(api.mluOpGetIndiceConvolutionBackwardDataWorkspaceSize(handle, d_dy, d_w, d_pairs, d_dx, counts.data(),
                                                               inverse, &bytes),
        "mluOpGetIndiceConvolutionBackwardDataWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  if (row_map != nullptr) check(api.mluOpExtUseRowMap(handle, row_map), "mluOpExtUseRowMap");
  check(api.mluOpIndiceConvolutionBackwardData(handle, d_dy, output_grad.data_ptr(), d_w, filters.data_ptr(),
                                               d_pairs, pairs.data_ptr(), counts.data(), inverse, sub_m,
                                               ws.data_ptr(), bytes, d_dx, dx.data_ptr()),
        "mluOpIndiceConvolutionBackwardData");
  buffers.done("mluOpIndiceConvolutionBackwardData");
  return dx;
}

at::Tensor convBackwardFilter(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &features,
                              const at::Tensor &output_grad, const at::Tensor &pairs, const Counts &counts,
                              const Counts &filter_space, bool sub_m, int64_t inverse, bool onchip_float,
                              mluOpTensorLayout_t layout) {
  const mluOpDataType_t code = dtypeCode(features.scalar_type());
  const int64_t ci = features.size(1), co = output_grad.size(1);
  Counts shape;
  if (layout == MLUOP_LAYOUT_NDHWC || layout == MLUOP_LAYOUT_NHWC) {
    shape.push_back(co);
    shape.insert(shape.end(), filter_space.begin(), filter_space.end());
    shape.push_back(ci);
  } else if (layout == MLUOP_LAYOUT_NCDHW || layout == MLUOP_LAYOUT_NCHW) {
    shape = {co, ci};
    shape.insert(shape.end(), filter_space.begin(), filter_space.end());
  } else {
    shape = filter_space;
    shape.push_back(ci);
    shape.push_back(co);
  }
  at::Tensor dw = buffers.output(shape, features.scalar_type(), "filters_grad");
  const TensorDesc d_x(MLUOP_LAYOUT_ARRAY, code, features.sizes());
  const TensorDesc d_dy(MLUOP_LAYOUT_ARRAY, code, output_grad.sizes());
  const TensorDesc d_pairs(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, pairs.sizes());
  const TensorDesc d_dw(layout, code, dw.sizes());
  if (onchip_float)
    check(api.mluOpSetTensorDescriptorOnchipDataType(d_dw, MLUOP_DTYPE_FLOAT),
          "mluOpSetTensorDescriptorOnchipDataType");
  size_t bytes = 0;
  check(api.mluOpGetIndiceConvolutionBackwardFilterWorkspaceSize(handle, d_x, d_dy, d_pairs, d_dw, counts.data(),
                                                                 inverse, sub_m, &bytes),
        "mluOpGetIndiceConvolutionBackwardFilterWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  check(api.mluOpIndiceConvolutionBackwardFilter(handle, d_x, features.data_ptr(), d_dy, output_grad.data_ptr(),
                                                 d_pairs, pairs.data_ptr(), counts.data(), inverse, sub_m,
                                                 ws.data_ptr(), bytes, d_dw, dw.data_ptr()),
        "mluOpIndiceConvolutionBackwardFilter");
  buffers.done("mluOpIndiceConvolutionBackwardFilter");
  return dw;
}

// ---- handles of the layers -----------------------------------------------------------------

// One library handle per (device, stream), made on first use and kept for the life of the
// process.  Several threads may use one stream and so one handle: every operator below that is
// called on it holds its mutex (OperatorLock) from its first look at the handle to the last word
// it waits for, since the calls in between share the handle's stamps, pinned words and settings.
// (A handle that a caller made is the caller's to use from one thread at a time.)
struct StreamHandle {
  mluOpHandle_t handle = nullptr;
  std::mutex mutex;

  // A row map's buffer is about to be freed: from any thread, whatever it holds.  The handle drops
  // its record before the next map is built or used on it.
  void forgetRowMap(const void *map) {
    const std::lock_guard<std::mutex> lock(forget_mutex_);
    forget_.push_back(map);
  }
  // (with `mutex` held)
  void dropForgottenRowMaps() {
    const std::lock_guard<std::mutex> lock(forget_mutex_);
    for (const void *map : forget_) (void)api.mluOpExtForgetRowMap(handle, map);
    forget_.clear();
  }

 private:
  std::mutex forget_mutex_;
  std::vector<const void *> forget_;
};

struct StreamHandles {
  std::mutex mutex;
  std::map<std::pair<int, hipStream_t>, StreamHandle> by_stream;  // (entries stay where they are)
  std::map<mluOpHandle_t, StreamHandle *> by_handle;
};
StreamHandles &streamHandles() {
  static auto *all = new StreamHandles();
  return *all;
}

// That of the current device and stream.
StreamHandle &streamHandle() {
  const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream();
  StreamHandles &all = streamHandles();
  const std::lock_guard<std::mutex> lock(all.mutex);
  StreamHandle &h = all.by_stream[{static_cast<int>(stream.device_index()), stream.stream()}];
  if (h.handle == nullptr) {
    mluOpHandle_t made = nullptr;
    check(api.mluOpCreate(&made), "mluOpCreate");
    check(api.mluOpSetQueue(made, reinterpret_cast<mluOpQueue_t>(stream.stream())), "mluOpSetQueue");
    // SparseInverseConv3d runs the operators with inverse = 1
    check(api.mluOpExtSetSparseConvExtendedModes(made, 1), "mluOpExtSetSparseConvExtendedModes");
    all.by_handle[made] = &h;
    h.handle = made;
  }
  return h;
}

bool isStreamHandle(mluOpHandle_t handle) {
  StreamHandles &all = streamHandles();
  const std::lock_guard<std::mutex> lock(all.mutex);
  return all.by_handle.count(handle) > 0;
}

// Held for one operator on `handle`, without the GIL (a buffer in guard mode takes it).
class OperatorLock {
 public:
  explicit OperatorLock(StreamHandle &h) : lock_(h.mutex) {}
  explicit OperatorLock(mluOpHandle_t handle) {
    StreamHandles &all = streamHandles();
    std::unique_lock<std::mutex> look(all.mutex);
    const auto found = all.by_handle.find(handle);
    if (found == all.by_handle.end()) return;
    look.unlock();
    lock_ = std::unique_lock<std::mutex>(found->second->mutex);
  }

 private:
  std::unique_lock<std::mutex> lock_;
};

// The pair counts of a rulebook built on `handle` (held by the caller), in `indice_num` on the device: as soon as they
// are there, or, where they are no longer on file (the handle keeps 32 rulebooks) or too many, behind what the
// rulebook's own stream holds.  (A handle of the caller's own may have been given another stream since.)
Counts takeHostCounts(mluOpHandle_t handle, const at::Tensor &pairs, const at::Tensor &indice_num) {
  Counts counts;
  if (hostCounts(handle, pairs, &counts)) return counts;
  mluOpQueue_t queue = nullptr;
  check(api.mluOpGetQueue(handle, &queue), "mluOpGetQueue");
  const c10::hip::HIPStreamGuard own(
      c10::hip::getStreamFromExternal(reinterpret_cast<hipStream_t>(queue), pairs.device().index()));
  if (!isStreamHandle(handle) && hipDeviceSynchronize() != hipSuccess)
    throw std::runtime_error("waiting for a rulebook's pair counts failed");
  const at::Tensor host = indice_num.cpu();
  const int32_t *n = host.data_ptr<int32_t>();
  counts.assign(n, n + host.numel());
  return counts;
}

// ---- the layers' autograd node -------------------------------------------------------------

// What the three convolution operators need of a rulebook, with the row maps its calls share.  A
// library handle knows only the maps that were built on it, so there is one for each handle the
// rulebook is used on (one per stream) and pair column that names result rows (1: the layer's
// outputs, 0: its inputs).  They live as long as this object, which a pending backward pass holds.
struct LayerRulebook : torch::CustomClassHolder {
  at::Tensor pairs;
  Counts filter_space;
  int64_t num_act_out = 0;
  bool sub_m = false, distinct = false;
  bool single = false;  // every input row is in one pair at most

  void setCounts(Counts counts) { counts_ = std::move(counts); }
  // They are on the device yet, in `indice_num`, and with the handle that built the rulebook.
  void setCountsPending(const at::Tensor &indice_num, mluOpHandle_t built_on) {
    indice_num_ = indice_num;
    built_on_ = built_on;
    pending_ = true;
  }

  // The pair counts, waited for on first use: a layer's output, workspace and descriptors are made while the device
  // builds its rulebook.  `held` is locked; where the rulebook was built on another handle, takeCountsFrom has
  // been called before that.  (No two handles are ever locked together, and counts_mutex_ only inside one's lock.)
  const Counts &counts(mluOpHandle_t held) {
    if (pending_.load(std::memory_order_acquire)) takeCounts(held);
    return counts_;
  }
  void takeCountsFromOther(mluOpHandle_t own) {
    if (!pending_.load(std::memory_order_acquire) || built_on_ == own) return;
    const OperatorLock lock(built_on_);
    takeCounts(built_on_);
  }

  // The same for a caller who holds no lock.
  const Counts &takenCounts() {
    if (pending_.load(std::memory_order_acquire)) {
      const OperatorLock lock(built_on_);
      takeCounts(built_on_);
    }
    return counts_;
  }

  ~LayerRulebook() override {
    for (const auto &[key, map] : row_maps_)
      if (map.defined()) key.first->forgetRowMap(map.data_ptr());
  }

  // The map for a call on `h` (whose mutex is held), built on first use; null: the operator builds
  // its own, since the coordinates may repeat or there is nothing to map.  The handle carries the
  // promise of distinct pairs, so the build need not count lost ones and wait for the stream.
  const void *rowMap(StreamHandle &h, const Buffers &buffers, int column) {
    if (!distinct) return nullptr;
    h.dropForgottenRowMaps();
    const Key key{&h, column};
    {
      const std::lock_guard<std::mutex> lock(maps_mutex_);
      const auto found = row_maps_.find(key);
      // (a handle keeps so many records: the oldest are gone when there were more)
      if (found != row_maps_.end() && api.mluOpExtUseRowMap(h.handle, found->second.data_ptr()) == MLUOP_STATUS_SUCCESS) {
        check(api.mluOpExtUseRowMap(h.handle, nullptr), "mluOpExtUseRowMap");
        return found->second.data_ptr();
      }
    }
    const int64_t L = pairs.size(2);
    const int64_t rows = column == 1 ? num_act_out : L, source_rows = column == 1 ? L : num_act_out;
    if (rows == 0 || source_rows == 0 || pairs.size(0) == 0) return nullptr;
    const TensorDesc d_pairs(MLUOP_LAYOUT_ARRAY, MLUOP_DTYPE_INT32, pairs.sizes());
    size_t bytes = 0;
    check(api.mluOpExtGetRowMapSize(d_pairs, rows, &bytes), "mluOpExtGetRowMapSize");
    const at::Tensor map = buffers.output({static_cast<int64_t>(bytes)}, at::kByte, "row map");
    check(api.mluOpExtBuildRowMap(h.handle, d_pairs, pairs.data_ptr(), counts(h.handle).data(), rows, source_rows, column,
                                  map.data_ptr(), bytes, nullptr),
          "mluOpExtBuildRowMap");
    buffers.done("mluOpExtBuildRowMap");
    const std::lock_guard<std::mutex> lock(maps_mutex_);
    row_maps_[key] = map;
    return map.data_ptr();
  }

  // (handle, column) of the maps there are
  std::vector<std::pair<uintptr_t, int>> rowMaps() {
    const std::lock_guard<std::mutex> lock(maps_mutex_);
    std::vector<std::pair<uintptr_t, int>> keys;
    for (const auto &[key, map] : row_maps_) keys.emplace_back(reinterpret_cast<uintptr_t>(key.first->handle), key.second);
    return keys;
  }

 private:
  void takeCounts(mluOpHandle_t built_on) {
    const std::lock_guard<std::mutex> lock(counts_mutex_);
    if (!pending_.load(std::memory_order_relaxed)) return;
    counts_ = takeHostCounts(built_on, pairs, indice_num_);
    pending_.store(false, std::memory_order_release);
  }

  Counts counts_;
  at::Tensor indice_num_;
  mluOpHandle_t built_on_ = nullptr;
  std::atomic<bool> pending_{false};
  std::mutex counts_mutex_;
  using Key = std::pair<StreamHandle *, int>;
  std::mutex maps_mutex_;  // never held while anything else is waited for
  std::map<Key, at::Tensor> row_maps_;
};
using LayerRulebookPtr = c10::intrusive_ptr<LayerRulebook>;

struct IndiceConv : torch::autograd::Function<IndiceConv> {
  static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &features,
                            const at::Tensor &weight, const LayerRulebookPtr &rb, bool inverse, bool share_row_maps,
                            bool guarded, bool relu) {
    const at::Tensor x = features.contiguous(), w = weight.contiguous();
    ctx->saved_data["rulebook"] = c10::IValue::make_capsule(rb);
    ctx->saved_data["inverse"] = inverse;
    ctx->saved_data["share_row_maps"] = share_row_maps;
    ctx->saved_data["guarded"] = guarded;
    ctx->saved_data["relu"] = relu;
    StreamHandle &h = streamHandle();
    rb->takeCountsFromOther(h.handle);
    const OperatorLock lock(h);
    check(api.mluOpExtSetDistinctPairsPromise(h.handle, rb->distinct), "mluOpExtSetDistinctPairsPromise");
    const Buffers buffers(guarded, x.device());
    const auto counts_of = [&]() -> const Counts & { return rb->counts(h.handle); };
    const void *map = share_row_maps ? rb->rowMap(h, buffers, inverse ? 0 : 1) : nullptr;
    // an inverse layer runs the partner layer's rulebook backwards: one output row per input
    // row of the partner
    const Setting single(h.handle, api.mluOpExtGetSinglePairsPromise, api.mluOpExtSetSinglePairsPromise, rb->single ? 0 : -1,
                         "mluOpExtSetSinglePairsPromise");
    const Setting stored(h.handle, api.mluOpExtGetForwardRelu, api.mluOpExtSetForwardRelu, relu, "mluOpExtSetForwardRelu");
    const at::Tensor out = inverse ? convForward(h.handle, buffers, x, w, MLUOP_LAYOUT_ARRAY, rb->pairs, counts_of,
                                                 rb->pairs.size(2), false, 1, map)
                                   : convForward(h.handle, buffers, x, w, MLUOP_LAYOUT_ARRAY, rb->pairs, counts_of,
                                                 rb->num_act_out, rb->sub_m, 0, map);
    if (relu)
      ctx->save_for_backward({x, w, out});
    else
      ctx->save_for_backward({x, w});
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &x = saved[0], &w = saved[1];
    const auto rb = c10::static_intrusive_pointer_cast<LayerRulebook>(ctx->saved_data["rulebook"].toCapsule());
    const bool inverse = ctx->saved_data["inverse"].toBool();
    torch::autograd::variable_list out(7);
    if (!grads[0].defined()) return out;
    // behind a ReLU in the store: the gradient that the ReLU would have passed on
    const bool relu = ctx->saved_data["relu"].toBool();
    const at::Tensor dy = (relu ? at::threshold_backward(grads[0], saved[2], 0) : grads[0]).contiguous();
    StreamHandle &h = streamHandle();
    rb->takeCountsFromOther(h.handle);
    const OperatorLock lock(h);
    check(api.mluOpExtSetDistinctPairsPromise(h.handle, rb->distinct), "mluOpExtSetDistinctPairsPromise");
    const Buffers buffers(ctx->saved_data["guarded"].toBool(), x.device());
    const bool sub_m = !inverse && rb->sub_m;
    const Setting single(h.handle, api.mluOpExtGetSinglePairsPromise, api.mluOpExtSetSinglePairsPromise, rb->single ? 0 : -1,
                         "mluOpExtSetSinglePairsPromise");
    if (ctx->needs_input_grad(0)) {
      const void *map =
          ctx->saved_data["share_row_maps"].toBool() ? rb->rowMap(h, buffers, inverse ? 1 : 0) : nullptr;
      out[0] = convBackwardData(h.handle, buffers, dy, w, MLUOP_LAYOUT_ARRAY, rb->pairs, rb->counts(h.handle), sub_m,
                                x.size(1), inverse, x.size(0), map);
    }
    if (ctx->needs_input_grad(1))
      out[1] = convBackwardFilter(h.handle, buffers, x, dy, rb->pairs, rb->counts(h.handle), rb->filter_space, sub_m,
                                  inverse, true, MLUOP_LAYOUT_ARRAY);
    return out;
  }
};

// ---- point operators -----------------------------------------------------------------------

std::vector<at::Tensor> voxelization(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &points,
                                     const at::Tensor &voxel_size, const at::Tensor &coors_range, int64_t max_points,
                                     int64_t max_voxels, bool deterministic) {
  const at::Tensor voxels = buffers.output({max_voxels, max_points, points.size(1)}, at::kFloat, "voxels");
  const at::Tensor coors = buffers.output({max_voxels, 3}, at::kInt, "coors");
  const at::Tensor npv = buffers.output({max_voxels}, at::kInt, "num_points_per_voxel");
  // (a call that keeps nothing enqueues nothing)
  const at::Tensor num = max_points == 0 || max_voxels == 0
                             ? at::zeros({1}, points.options().dtype(at::kInt))
                             : at::empty({1}, points.options().dtype(at::kInt));
  const mluOpTensorLayout_t array = MLUOP_LAYOUT_ARRAY;
  const TensorDesc d_points(array, MLUOP_DTYPE_FLOAT, points.sizes());
  const TensorDesc d_vs(array, MLUOP_DTYPE_FLOAT, {3});
  const TensorDesc d_cr(array, MLUOP_DTYPE_FLOAT, {6});
  const TensorDesc d_voxels(array, MLUOP_DTYPE_FLOAT, voxels.sizes());
  const TensorDesc d_coors(array, MLUOP_DTYPE_INT32, coors.sizes());
  const TensorDesc d_npv(array, MLUOP_DTYPE_INT32, npv.sizes());
  const TensorDesc d_num(array, MLUOP_DTYPE_INT32, {1});
  size_t bytes = 0;
  check(api.mluOpGetVoxelizationWorkspaceSize(handle, d_points, d_vs, d_cr, static_cast<int32_t>(max_points),
                                              static_cast<int32_t>(max_voxels), 3, deterministic, d_voxels, d_coors,
                                              d_npv, d_num, &bytes),
        "mluOpGetVoxelizationWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  check(api.mluOpVoxelization(handle, d_points, points.data_ptr(), d_vs, voxel_size.data_ptr(), d_cr,
                              coors_range.data_ptr(), static_cast<int32_t>(max_points),
                              static_cast<int32_t>(max_voxels), 3, deterministic, ws.data_ptr(), bytes, d_voxels,
                              voxels.data_ptr(), d_coors, coors.data_ptr(), d_npv, npv.data_ptr(), d_num,
                              num.data_ptr()),
        "mluOpVoxelization");
  buffers.done("mluOpVoxelization");
  return {voxels, coors, npv, num};
}

// The same for a layer: cut to the voxels found, whose number the host takes from pinned memory.
std::vector<at::Tensor> voxelizationCut(bool guarded, const at::Tensor &points, const at::Tensor &voxel_size,
                                        const at::Tensor &coors_range, int64_t max_points, int64_t max_voxels) {
  StreamHandle &h = streamHandle();
  const OperatorLock lock(h);
  std::vector<at::Tensor> r = voxelization(h.handle, Buffers(guarded, points.device()), points, voxel_size,
                                           coors_range, max_points, max_voxels, true);
  int32_t found = 0;
  if (max_points == 0 || max_voxels == 0 ||
      api.mluOpExtGetVoxelizationHostCount(h.handle, r[3].data_ptr(), &found) != MLUOP_STATUS_SUCCESS)
    found = r[3].item<int32_t>();
  r.pop_back();
  for (at::Tensor &t : r) t = t.narrow(0, 0, found);
  return r;
}

// Voxels in the order of their cells: (the voxel at each place, its (batch, z, y, x)).
std::vector<at::Tensor> orderVoxels(bool guarded, const at::Tensor &coors, const Counts &space, int64_t batch_index) {
  StreamHandle &h = streamHandle();
  const OperatorLock lock(h);
  const Buffers buffers(guarded, coors.device());
  const int64_t n = coors.size(0);
  const at::Tensor order = buffers.output({n}, at::kLong, "order");
  const at::Tensor indices = buffers.output({n, 4}, at::kInt, "indices");
  size_t bytes = 0;
  check(api.mluOpExtGetOrderVoxelsWorkspaceSize(n, space.data(), &bytes), "mluOpExtGetOrderVoxelsWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  check(api.mluOpExtOrderVoxels(h.handle, coors.data_ptr(), n, space.data(), static_cast<int32_t>(batch_index),
                                ws.data_ptr(), bytes, order.data_ptr(), indices.data_ptr()),
        "mluOpExtOrderVoxels");
  buffers.done("mluOpExtOrderVoxels");
  return {order, indices};
}

// Mean of every voxel's points: [V, max_points, F] fp32 -> [V, F].
at::Tensor meanVoxelPoints(bool guarded, const at::Tensor &voxels, const at::Tensor &counts) {
  StreamHandle &h = streamHandle();
  const OperatorLock lock(h);
  const Buffers buffers(guarded, voxels.device());
  const at::Tensor mean = buffers.output({voxels.size(0), voxels.size(2)}, at::kFloat, "mean");
  check(api.mluOpExtMeanVoxelPoints(h.handle, voxels.data_ptr(), counts.data_ptr(), voxels.size(0),
                                    static_cast<int32_t>(voxels.size(1)), static_cast<int32_t>(voxels.size(2)),
                                    mean.data_ptr()),
        "mluOpExtMeanVoxelPoints");
  buffers.done("mluOpExtMeanVoxelPoints");
  return mean;
}

std::vector<at::Tensor> scatterForward(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &feats,
                                       const at::Tensor &coors, mluOpReduceMode_t mode, int64_t rows) {
  const int64_t n = feats.size(0), c = feats.size(1);
  const at::Tensor voxel_feats = buffers.output({rows, c}, at::kFloat, "voxel_feats");
  const at::Tensor voxel_coors = buffers.output({rows, 3}, at::kInt, "voxel_coors");
  const at::Tensor p2v = buffers.output({n}, at::kInt, "point2voxel_map");
  const at::Tensor count = buffers.output({rows}, at::kInt, "voxel_points_count");
  // (a call on nothing enqueues nothing)
  const at::Tensor num = n == 0 || c == 0 ? at::zeros({1}, coors.options()) : at::empty({1}, coors.options());
  const mluOpTensorLayout_t array = MLUOP_LAYOUT_ARRAY;
  const TensorDesc d_feats(array, MLUOP_DTYPE_FLOAT, feats.sizes());
  const TensorDesc d_coors(array, MLUOP_DTYPE_INT32, coors.sizes());
  const TensorDesc d_vf(array, MLUOP_DTYPE_FLOAT, voxel_feats.sizes());
  const TensorDesc d_vc(array, MLUOP_DTYPE_INT32, voxel_coors.sizes());
  const TensorDesc d_p2v(array, MLUOP_DTYPE_INT32, p2v.sizes());
  const TensorDesc d_count(array, MLUOP_DTYPE_INT32, count.sizes());
  const TensorDesc d_num(array, MLUOP_DTYPE_INT32, {1});
  size_t bytes = 0;
  check(api.mluOpGetDynamicPointToVoxelForwardWorkspaceSize(handle, d_feats, d_coors, &bytes),
        "mluOpGetDynamicPointToVoxelForwardWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  check(api.mluOpDynamicPointToVoxelForward(handle, mode, d_feats, feats.data_ptr(), d_coors, coors.data_ptr(),
                                            ws.data_ptr(), bytes, d_vf, voxel_feats.data_ptr(), d_vc,
                                            voxel_coors.data_ptr(), d_p2v, p2v.data_ptr(), d_count, count.data_ptr(),
                                            d_num, num.data_ptr()),
        "mluOpDynamicPointToVoxelForward");
  buffers.done("mluOpDynamicPointToVoxelForward");
  return {voxel_feats, voxel_coors, p2v, count, num};
}

at::Tensor scatterBackward(mluOpHandle_t handle, const Buffers &buffers, const at::Tensor &grad,
                           const at::Tensor &feats, const at::Tensor &voxel_feats, const at::Tensor &p2v,
                           const at::Tensor &count, const at::Tensor &num, mluOpReduceMode_t mode) {
  const int64_t n = feats.size(0), c = feats.size(1), m = grad.size(0);
  const at::Tensor grad_feats = buffers.output({n, c}, at::kFloat, "grad_feats");
  const mluOpTensorLayout_t array = MLUOP_LAYOUT_ARRAY;
  const TensorDesc d_grad(array, MLUOP_DTYPE_FLOAT, {m, c});
  const TensorDesc d_feats(array, MLUOP_DTYPE_FLOAT, {n, c});
  const TensorDesc d_vf(array, MLUOP_DTYPE_FLOAT, {m, c});
  const TensorDesc d_p2v(array, MLUOP_DTYPE_INT32, {n});
  const TensorDesc d_count(array, MLUOP_DTYPE_INT32, {m});
  const TensorDesc d_num(array, MLUOP_DTYPE_INT32, {1});
  size_t bytes = 0;
  check(api.mluOpGetDynamicPointToVoxelBackwardWorkspaceSize(handle, mode, d_grad, d_feats, d_vf, d_p2v, d_count,
                                                             d_num, &bytes),
        "mluOpGetDynamicPointToVoxelBackwardWorkspaceSize");
  const at::Tensor ws = buffers.workspace(bytes);
  check(api.mluOpDynamicPointToVoxelBackward(handle, mode, d_grad, grad.data_ptr(), d_feats, feats.data_ptr(), d_vf,
                                             voxel_feats.data_ptr(), d_p2v, p2v.data_ptr(), d_count,
                                             count.data_ptr(), d_num, num.data_ptr(), ws.data_ptr(), bytes, d_feats,
                                             grad_feats.data_ptr()),
        "mluOpDynamicPointToVoxelBackward");
  buffers.done("mluOpDynamicPointToVoxelBackward");
  return grad_feats;
}

inline mluOpHandle_t asHandle(uintptr_t h) { return reinterpret_cast<mluOpHandle_t>(h); }

}  // namespace

PYBIND11_MODULE(_native, m) {
  using NoGil = py::gil_scoped_release;
  m.doc() = "Native host path of mluop_hip: operators and the sparse layers' autograd node over the C API.";

  static py::exception<StatusError> unused(m, "StatusError", PyExc_RuntimeError);
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const StatusError &e) {
      const py::object type = py::module_::import("mluop_hip").attr("MluOpError");
      const py::object error = type(e.status, e.call);
      PyErr_SetObject(type.ptr(), error.ptr());
    }
  });

  m.def("bind", &bind, "Binds the C API to the library at this path.");
  m.def("stream_handle", [] { return reinterpret_cast<uintptr_t>(streamHandle().handle); },
        "The library handle of the current device and stream.");

  m.def("get_indice_pairs",
        [](uintptr_t handle, bool guarded, const at::Tensor &indices, int batch, const Ints &input_space,
           const Ints &filter_space, const Ints &output_space, const Ints &pad, const Ints &stride,
           const Ints &dilation, bool sub_m, std::optional<int64_t> out_rows, std::optional<at::Tensor> out_indices,
           bool for_layer, bool tails, bool wait_counts) {
          Rulebook3 r;
          {
            NoGil released;
            const OperatorLock lock(asHandle(handle));
            r = indicePairs(asHandle(handle), Buffers(guarded, indices.device()), indices, batch, input_space,
                            filter_space, output_space, pad, stride, dilation, sub_m, out_rows, std::move(out_indices),
                            for_layer, tails, wait_counts);
          }
          const bool counted = for_layer && r.counts.size() == static_cast<size_t>(r.pairs.size(0));
          py::object num = counted ? py::cast(r.counts) : py::cast(r.indice_num);
          return py::make_tuple(r.pairs, r.out_indices, num, r.num_act_out);
        });
  m.def("rulebook_counts", [](uintptr_t handle, const at::Tensor &pairs, const at::Tensor &indice_num) {
    NoGil released;
    const OperatorLock lock(asHandle(handle));
    return takeHostCounts(asHandle(handle), pairs, indice_num);
  });
  m.def("indice_conv_forward",
        [](uintptr_t handle, bool guarded, const at::Tensor &features, const at::Tensor &filters, int layout,
           const at::Tensor &pairs, const Counts &counts, int64_t num_act_out, bool sub_m, int64_t inverse,
           uintptr_t row_map) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return convForward(asHandle(handle), Buffers(guarded, features.device()), features, filters,
                             static_cast<mluOpTensorLayout_t>(layout), pairs,
                             [&]() -> const Counts & { return counts; }, num_act_out, sub_m, inverse,
                             reinterpret_cast<const void *>(row_map));
        });
  m.def("indice_conv_backward_data",
        [](uintptr_t handle, bool guarded, const at::Tensor &output_grad, const at::Tensor &filters, int layout,
           const at::Tensor &pairs, const Counts &counts, bool sub_m, int64_t ci, int64_t inverse, int64_t rows,
           uintptr_t row_map) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return convBackwardData(asHandle(handle), Buffers(guarded, output_grad.device()), output_grad, filters,
                                  static_cast<mluOpTensorLayout_t>(layout), pairs, counts, sub_m, ci, inverse, rows,
                                  reinterpret_cast<const void *>(row_map));
        });
  m.def("indice_conv_backward_filter",
        [](uintptr_t handle, bool guarded, const at::Tensor &features, const at::Tensor &output_grad,
           const at::Tensor &pairs, const Counts &counts, const Counts &filter_space, bool sub_m, int64_t inverse,
           bool onchip_float, int layout) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return convBackwardFilter(asHandle(handle), Buffers(guarded, features.device()), features, output_grad,
                                    pairs, counts, filter_space, sub_m, inverse, onchip_float,
                                    static_cast<mluOpTensorLayout_t>(layout));
        });
  m.def("voxelization",
        [](uintptr_t handle, bool guarded, const at::Tensor &points, const at::Tensor &voxel_size,
           const at::Tensor &coors_range, int64_t max_points, int64_t max_voxels, bool deterministic) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return voxelization(asHandle(handle), Buffers(guarded, points.device()), points, voxel_size, coors_range,
                              max_points, max_voxels, deterministic);
        });
  m.def("voxelization_cut",
        [](bool guarded, const at::Tensor &points, const at::Tensor &voxel_size, const at::Tensor &coors_range,
           int64_t max_points, int64_t max_voxels) {
          std::vector<at::Tensor> r;
          {
            NoGil released;
            r = voxelizationCut(guarded, points, voxel_size, coors_range, max_points, max_voxels);
          }
          return py::make_tuple(r[0], r[1], r[2]);
        });
  m.def("order_voxels", [](bool guarded, const at::Tensor &coors, const Counts &space, int64_t batch_index) {
    std::vector<at::Tensor> r;
    {
      NoGil released;
      r = orderVoxels(guarded, coors, space, batch_index);
    }
    return py::make_tuple(r[0], r[1]);
  });
  m.def("mean_voxel_points", [](bool guarded, const at::Tensor &voxels, const at::Tensor &counts) {
    NoGil released;
    return meanVoxelPoints(guarded, voxels, counts);
  });
  m.def("dynamic_point_to_voxel_forward",
        [](uintptr_t handle, bool guarded, const at::Tensor &feats, const at::Tensor &coors, int mode, int64_t rows) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return scatterForward(asHandle(handle), Buffers(guarded, feats.device()), feats, coors,
                                static_cast<mluOpReduceMode_t>(mode), rows);
        });
  m.def("dynamic_point_to_voxel_backward",
        [](uintptr_t handle, bool guarded, const at::Tensor &grad, const at::Tensor &feats,
           const at::Tensor &voxel_feats, const at::Tensor &p2v, const at::Tensor &count, const at::Tensor &num,
           int mode) {
          NoGil released;
          const OperatorLock lock(asHandle(handle));
          return scatterBackward(asHandle(handle), Buffers(guarded, feats.device()), grad, feats, voxel_feats, p2v,
                                 count, num, static_cast<mluOpReduceMode_t>(mode));
        });

  py::class_<LayerRulebook, LayerRulebookPtr>(m, "LayerRulebook")
      .def(py::init([](const at::Tensor &pairs, std::optional<Counts> counts, int64_t num_act_out, Counts filter_space,
                       bool sub_m, bool distinct, bool single, std::optional<at::Tensor> indice_num, uintptr_t built_on) {
        auto rb = c10::make_intrusive<LayerRulebook>();
        rb->pairs = pairs;
        if (counts)
          rb->setCounts(std::move(*counts));
        else
          rb->setCountsPending(indice_num.value(), asHandle(built_on));
        rb->num_act_out = num_act_out;
        rb->filter_space = std::move(filter_space);
        rb->sub_m = sub_m;
        rb->distinct = distinct;
        rb->single = single;
        return rb;
      }),
           py::arg("pairs"), py::arg("counts"), py::arg("num_act_out"), py::arg("filter_space"), py::arg("sub_m"),
           py::arg("distinct"), py::arg("single") = false, py::arg("indice_num") = std::nullopt, py::arg("built_on") = 0,
           "With counts None, `indice_num` holds them on the device and the handle at `built_on` has built the rulebook.")
      .def("counts", [](const LayerRulebookPtr &rulebook) {
        NoGil released;
        return rulebook->takenCounts();
      }, "The pair counts, waited for unless a call has taken them.")
      .def("row_maps", &LayerRulebook::rowMaps, "(handle, pair column) of the row maps its calls have built.");
  m.def("indice_conv", [](const at::Tensor &features, const at::Tensor &weight, const LayerRulebookPtr &rulebook,
                          bool inverse, bool share_row_maps, bool guarded, bool relu) {
    NoGil released;
    return IndiceConv::apply(features, weight, rulebook, inverse, share_row_maps, guarded, relu);
  });
}
