// The host side of a layer call: argument checks, allocations and library calls of the kernel-map
// builder, the strided coordinates, the contraction and its gradients, in one native call each.
//
// A layer over a small map runs its kernels in 15-40 us; made of Python statements and ctypes calls,
// the same layer's host side took 80 us (31 us of it in the contraction's wrapper, 90 us more where a
// kernel map was built), so that a network over one scan left the GPU idle for two thirds of the
// time.  Everything here is what those Python functions did, on the same library entries.
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <array>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <optional>
#include <string>
#include <vector>

#include "../../include/wcn_hip.h"

namespace {

using at::Tensor;
using Int3 = std::array<int32_t, 3>;

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// A failed call becomes the package's own exception, also on a thread of the autograd engine, which hands it to the thread
// that called backward().
void check(int status, const char* where) {
  if (status == WCN_OK) return;
  const bool python_thread = PyGILState_Check();
  py::gil_scoped_acquire locked;
  try {
    py::module_::import("warpconvnet_amd._lib").attr("check")(status, where);
  } catch (py::error_already_set& e) {
    if (python_thread) throw;
    e.restore();
    python_error error;
    error.persist();
    throw error;
  }
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return WCN_DTYPE_F32;
    case at::kHalf: return WCN_DTYPE_F16;
    case at::kBFloat16: return WCN_DTYPE_BF16;
    default: return -1;
  }
}

Tensor bytes_on(size_t n, const Tensor& like) {
  return at::empty({static_cast<int64_t>(n < 256 ? 256 : n)}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}

/* Where a piece of device data that outlives its call was made, and the event behind the kernels that made it.  A call on
 * another stream waits for them, and the allocator learns of that stream, so that memory given back by the object is not
 * handed out again while that stream still reads it.  What is made inside a capture is kept by nobody: its
 * kernels run when the graph is replayed, not now. */
struct MadeOn {
  void* stream;
  hipEvent_t event = nullptr;
  int32_t lent = -1;  // the device of an event that goes back to the map builder's
  MadeOn(void* s, void* recorded, int32_t device) : stream(s), event(static_cast<hipEvent_t>(recorded)), lent(device) {}
  explicit MadeOn(void* s) : stream(s) {
    if (hipEventCreateWithFlags(&event, hipEventDisableTiming) != hipSuccess ||
        hipEventRecord(event, static_cast<hipStream_t>(s)) != hipSuccess) {
      if (event) (void)hipEventDestroy(event);
      throw std::runtime_error("an event behind kept device data could not be recorded");
    }
  }
  MadeOn(const MadeOn&) = delete;
  ~MadeOn() {
    if (lent >= 0) wcn_kmap_return_event(event, lent);
    else if (event) (void)hipEventDestroy(event);
  }

  static bool capturing(void* s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(static_cast<hipStream_t>(s), &status) == hipSuccess && status != hipStreamCaptureStatusNone;
  }

  // `data` is about to be read by work on the current stream of its device
  void before_use(std::initializer_list<const Tensor*> data) const {
    const Tensor& first = **data.begin();
    void* s = stream_of(first);
    if (s == stream) return;
    if (!capturing(s)) {
      if (hipStreamWaitEvent(static_cast<hipStream_t>(s), event, 0) != hipSuccess)
        throw std::runtime_error("hipStreamWaitEvent failed");
    } else {  // a graph cannot wait for work outside it: the host does
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      (void)hipThreadExchangeStreamCaptureMode(&mode);
      const hipError_t waited = hipEventSynchronize(event);
      (void)hipThreadExchangeStreamCaptureMode(&mode);
      if (waited != hipSuccess) throw std::runtime_error("hipEventSynchronize failed");
    }
    const c10::Stream reader = c10::impl::VirtualGuardImpl(first.device().type()).getStream(first.device());
    for (const Tensor* t : data)
      if (t->defined()) t->record_stream(reader);
  }
};

std::string shape_text(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

// ------------------------------------------------------------------------------------------------
// Batch column, coordinate table, strided coordinates, kernel map
// ------------------------------------------------------------------------------------------------

/* (n, dims + 1) rows [batch, ...] of int32 coordinates on the device; the offsets (host, int32 or
 * int64) begin at 0 and end at n and describe at most WCN_VOXEL_MAX_BATCH items: the caller checks. */
Tensor batch_rows(const Tensor& coords, const std::vector<int64_t>& offsets) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor c = coords.contiguous();
  const int64_t n = c.size(0), dims = c.size(1);
  Tensor rows = at::empty({n, dims + 1}, c.options());
  check(wcn_batch_indexed_rows(c.const_data_ptr<int32_t>(), n, static_cast<int32_t>(dims), offsets.data(),
                               static_cast<int32_t>(offsets.size() - 1), rows.mutable_data_ptr<int32_t>(), stream_of(c)),
        "wcn_batch_indexed_rows");
  return rows;
}

/* (table workspace, slot count) of the coordinate table over (n, 4) rows; enqueued, not waited for. */
std::pair<Tensor, int64_t> table_build(const Tensor& keys4, int64_t slots) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const int64_t n = keys4.size(0);
  if (slots <= 0) slots = wcn_table_default_capacity(n);
  Tensor table = bytes_on(wcn_table_bytes(n, slots), keys4);
  check(wcn_table_build(keys4.const_data_ptr<int32_t>(), n, table.mutable_data_ptr(), slots, stream_of(keys4)),
        "wcn_table_build");
  return {table, slots};
}

/* (rows, table workspace, slot count): batch_rows and table_build of (n, 3) coordinates in one. */
py::tuple batch_rows_table(const Tensor& coords, const std::vector<int64_t>& offsets) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor c = coords.contiguous();
  const int64_t n = c.size(0), slots = wcn_table_default_capacity(n);
  Tensor rows = at::empty({n, 4}, c.options());
  Tensor table = bytes_on(wcn_table_bytes(n, slots), c);
  check(wcn_table_build_items(c.const_data_ptr<int32_t>(), n, offsets.data(), static_cast<int32_t>(offsets.size() - 1),
                              rows.mutable_data_ptr<int32_t>(), table.mutable_data_ptr(), slots, stream_of(c)),
        "wcn_table_build_items");
  return py::make_tuple(rows, table, slots);
}

struct TableRef {  // what the builder reads of a TorchHashTable object
  Tensor raw, keys;
  int64_t slots;
  explicit TableRef(const py::object& t)
      : raw(t.attr("_table").cast<Tensor>()), keys(t.attr("_keys4").cast<Tensor>()), slots(t.attr("_slots").cast<int64_t>()) {}
};

/* Distinct coarse rows of a table's keys for strides of 1, 2 or 4 (wcn_stride_unique_cells): the
 * (count, 4) rows, and, where the batch items' first rows were asked for and are at most 1024, the
 * (B + 1) batch offsets as int64 and int32 host tensors (undefined otherwise). */
py::tuple stride_cells(const py::object& table, const Int3& stride, bool want_bounds) {
  at::AutoDispatchBelowADInplaceOrView guard;
  constexpr int kBounds = 1025;
  int64_t bounds[kBounds];
  while (true) {
    TableRef t(table);
    const int64_t n = t.keys.size(0);
    void* stream = stream_of(t.keys);
    Tensor out = at::empty({n, 4}, t.keys.options());
    Tensor first = at::empty({n}, t.keys.options());
    Tensor ws = bytes_on(wcn_stride_unique_cells_workspace_bytes(n), t.keys);
    check(wcn_stride_unique_cells(t.raw.const_data_ptr(), n, t.slots, t.keys.const_data_ptr<int32_t>(), stride.data(),
                                  ws.mutable_data_ptr(), out.mutable_data_ptr<int32_t>(), first.mutable_data_ptr<int32_t>(),
                                  stream),
          "wcn_stride_unique_cells");
    int64_t count = 0;
    int status;
    {
      py::gil_scoped_release unlocked;
      status = want_bounds ? wcn_stride_unique_read_bounds(ws.const_data_ptr(), n, t.slots, &count, bounds, stream)
                           : wcn_stride_unique_read_count(ws.const_data_ptr(), n, t.slots, &count, stream);
    }
    if (status == WCN_ERR_TABLE_OVERFLOW) {
      table.attr("_grow")();
      continue;
    }
    check(status, "wcn_stride_unique_cells");
    table.attr("_checked") = true;
    py::object off64 = py::none(), off32 = py::none();
    if (want_bounds && count > 0) {
      int batches = 0;  // the last batch item with rows, plus one
      while (batches < kBounds && bounds[batches] < count) ++batches;
      if (batches < kBounds) {
        Tensor a = at::empty({batches + 1}, at::kLong), b = at::empty({batches + 1}, at::kInt);
        for (int i = 0; i <= batches; ++i) {
          const int64_t v = i < batches ? bounds[i] : count;
          a.mutable_data_ptr<int64_t>()[i] = v;
          b.mutable_data_ptr<int32_t>()[i] = static_cast<int32_t>(v);
        }
        off64 = py::cast(a);
        off32 = py::cast(b);
      }
    }
    return py::make_tuple(out.narrow(0, 0, count), off64, off32);
  }
}

/* A layer whose map is about to be made (`graph`: one whose gradients will be asked for, as conv_forward's), for kernel_map to run between the map's launches and the wait for its
 * offsets.  `out` stays undefined where the layer is none that can: it is then run behind the map, as any other. */
struct LayerAhead {
  Tensor features;
  py::object weight;
  std::optional<Tensor> bias, residual;
  std::optional<at::ScalarType> compute_dtype;
  bool relu = false, keep_tiles = false, graph = false;
  int64_t identity = -1;
  Tensor out;
  void launch(const Tensor& in_maps, const Tensor& out_maps, int64_t expected, const void* map_result, const int32_t* groups,
              int32_t K, int64_t num_out);
};

/* Kernel map of (m, 4) output rows over a coordinate table: count pass, emit pass into buffers of
 * assumed size (`per_row` pairs a row), one wait for the offsets; with more pairs than assumed the
 * emit pass has written nothing and runs again into exact buffers.  Returns (in_maps, out_maps,
 * offsets int64, offsets int32, group starts (bytes) and their address, offsets in device memory, table
 * flags, where and when the lists were made). */
py::tuple kernel_map(const py::object& table, const Tensor& out4, const Int3& ks, const Int3& st,
                     const std::optional<Int3>& dilation, const std::optional<Int3>& centre, double per_row,
                     int64_t keep_workspace_bytes, LayerAhead* ahead) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const int64_t M = out4.size(0);
  const int32_t K = ks[0] * ks[1] * ks[2];
  const int32_t* rows = out4.const_data_ptr<int32_t>();
  void* stream = stream_of(out4);
  // What stays with the map is the workspace's head: its K + 1 offsets and the group starts.  Up to keep_workspace_bytes the
  // workspace itself is kept; beyond, the head is an allocation of its own and the rest is given back.  (Copied out of the
  // workspace it was a copy and its launch between the map and the layer: 5x5x5 16 -> 16 over 1 M rows 435 us a call, 429 so.)
  const size_t ws_bytes = wcn_kmap_workspace_bytes(M, K), head_bytes = wcn_kmap_head_bytes(M, K);
  Tensor ws, parked;
  // a set mapped onto itself can also be probed block by block (opt-in; same results, a little slower)
  const char* probe = std::getenv("WCN_KMAP_PROBE");
  const bool by_blocks = probe != nullptr && std::strcmp(probe, "blocks") == 0, large = static_cast<int64_t>(ws_bytes) > keep_workspace_bytes;
  if (large && !by_blocks) {
    ws = bytes_on(head_bytes, out4);
    parked = bytes_on(ws_bytes - head_bytes, out4);
  } else {
    ws = bytes_on(ws_bytes, out4);
  }
  void* w = ws.mutable_data_ptr();
  Tensor offsets = at::empty({K + 1}, at::kLong);
  int64_t* host_offsets = offsets.mutable_data_ptr<int64_t>();
  const int64_t assumed =
      std::min<int64_t>(K * M, std::max<int64_t>(static_cast<int64_t>(1.25 * per_row * M) + 4096, int64_t{1} << 16));
  Tensor in_buf = at::empty({assumed}, out4.options()), out_buf = at::empty({assumed}, out4.options());
  Tensor kept;
  // The wait is for the counts: the lists and the group starts may be on their way still, so a call on another stream waits for the
  // event behind the kernels that write them (the one that the counts' mailbox has anyway: no launch more).
  std::shared_ptr<MadeOn> made;
  int64_t begin = 0;
  while (true) {
    TableRef t(table);
    const int64_t n = t.keys.size(0);
    const void* raw = t.raw.const_data_ptr();
    const bool blocks = by_blocks && !dilation && st[0] == 1 && st[1] == 1 &&
                        st[2] == 1 && rows == t.keys.const_data_ptr<int32_t>() && M == n &&
                        wcn_kmap_self_supported(ks.data(), M);
    auto fill = [&](int64_t capacity, const Tensor& ins, const Tensor& outs) {
      int32_t *pi = ins.mutable_data_ptr<int32_t>(), *po = outs.mutable_data_ptr<int32_t>();
      check(blocks ? wcn_kmap_fill_self(M, ks.data(), w, capacity, pi, po, stream)
            : parked.defined() ? wcn_kmap_fill_apart(raw, n, t.slots, rows, M, ks.data(), st.data(), w, parked.const_data_ptr(),
                                                     capacity, pi, po, stream)
                   : wcn_kmap_fill(raw, n, t.slots, rows, M, ks.data(), st.data(), w, capacity, pi, po, stream),
            "wcn_kmap_fill");
    };
    if (blocks) {
      check(wcn_kmap_count_self(raw, n, t.slots, ks.data(), w, stream), "wcn_kmap_count_self");
      fill(assumed, in_buf, out_buf);
    } else if (parked.defined()) {
      check(wcn_kmap_count_fill_apart(raw, n, t.slots, rows, M, ks.data(), st.data(), dilation ? dilation->data() : nullptr,
                                      dilation ? centre->data() : nullptr, w, parked.mutable_data_ptr(), assumed,
                                      in_buf.mutable_data_ptr<int32_t>(), out_buf.mutable_data_ptr<int32_t>(), stream),
            "wcn_kmap_count_fill_apart");
    } else {
      check(wcn_kmap_count_fill(raw, n, t.slots, rows, M, ks.data(), st.data(), dilation ? dilation->data() : nullptr,
                                dilation ? centre->data() : nullptr, w, assumed, in_buf.mutable_data_ptr<int32_t>(),
                                out_buf.mutable_data_ptr<int32_t>(), stream),
            "wcn_kmap_count_fill");
    }
    begin = reinterpret_cast<const char*>(wcn_kmap_group_start(w, M, K)) - static_cast<const char*>(w);
    kept = ws.narrow(0, 0, begin + 4 * int64_t{K} * ((M + 63) / 64 + 1));
    if (large && !parked.defined()) kept = kept.clone();
    // what a layer needs of the map is on its way: with it behind, the GPU has work while the host takes the offsets in
    if (ahead) ahead->launch(in_buf, out_buf, static_cast<int64_t>(per_row * M), w, wcn_kmap_group_start(w, M, K), K, M);
    int status;
    {
      py::gil_scoped_release unlocked;
      status = wcn_kmap_read_result(w, M, K, host_offsets, stream);
    }
    if (status == WCN_ERR_TABLE_OVERFLOW) {
      table.attr("_grow")();
      continue;
    }
    check(status, "wcn_kmap_count");
    table.attr("_checked") = true;
    const int64_t total = host_offsets[K];
    if (total > assumed) {
      if (ahead) ahead->out = Tensor();  // it has found no lists
      in_buf = at::empty({total}, out4.options());
      out_buf = at::empty({total}, out4.options());
      fill(total, in_buf, out_buf);
      made = std::make_shared<MadeOn>(stream);
    } else if (2 * total <= assumed && (assumed - total) * 4 > (int64_t{32} << 20)) {
      // far fewer pairs than assumed, more than 32 MiB of each buffer unused: exact copies, so that the
      // map does not hold the large buffers
      in_buf = in_buf.narrow(0, 0, total).clone();
      out_buf = out_buf.narrow(0, 0, total).clone();
      made = std::make_shared<MadeOn>(stream);
    } else {
      in_buf = in_buf.narrow(0, 0, total);
      out_buf = out_buf.narrow(0, 0, total);
      int32_t device = -1;
      void* const behind = wcn_kmap_take_event(w, &device);
      made = behind ? std::make_shared<MadeOn>(stream, behind, device) : std::make_shared<MadeOn>(stream);
    }
    break;
  }
  Tensor offsets32 = at::empty({K + 1}, at::kInt);
  for (int k = 0; k <= K; ++k) offsets32.mutable_data_ptr<int32_t>()[k] = static_cast<int32_t>(host_offsets[k]);
  Tensor groups = kept.narrow(0, begin, kept.numel() - begin);
  const auto address = reinterpret_cast<uintptr_t>(groups.const_data_ptr());
  return py::make_tuple(in_buf, out_buf, offsets, offsets32, groups, address,
                        kept.narrow(0, 0, 8 * (int64_t{K} + 1)).view(at::kLong), wcn_kmap_last_table_flags(),
                        made);
}

// ------------------------------------------------------------------------------------------------
// Contraction
// ------------------------------------------------------------------------------------------------

/* What the contraction reads of an IntSearchResult object. */
struct MapRef {
  Tensor in_maps, out_maps, offsets;  // the offsets as an int64 host tensor
  int64_t identity = -1;
  int32_t K = 0;
  explicit MapRef(const py::object& km) {
    in_maps = km.attr("in_maps").cast<Tensor>();
    out_maps = km.attr("out_maps").cast<Tensor>();
    py::object off = km.attr("_offsets64");
    if (off.is_none()) {
      Tensor o = km.attr("offsets").cast<Tensor>().to(at::kCPU, at::kLong).contiguous();
      off = py::cast(o);
      km.attr("_offsets64") = off;
    }
    offsets = off.cast<Tensor>();
    K = static_cast<int32_t>(offsets.numel() - 1);
    py::object id = km.attr("identity_map_index");
    if (!id.is_none()) identity = id.cast<int64_t>();
    // A builder's lists, and the workspace's head with offsets and group starts, on another stream than the builder's.
    py::object made = km.attr("_made");
    if (made.is_none()) return;
    const MadeOn& m = *made.cast<const MadeOn*>();
    if (m.stream == stream_of(in_maps)) return;
    py::object head = km.attr("_device_offsets");
    const Tensor h = head.is_none() ? Tensor() : head.cast<Tensor>();
    m.before_use({&in_maps, &out_maps, &h});
  }
  const int64_t* host_offsets() const { return offsets.const_data_ptr<int64_t>(); }
  int64_t pairs() const { return host_offsets()[K]; }
};

const int32_t* group_starts(const py::object& kept, int64_t K, int64_t rows) {  // (tensor, address, (K, rows)) or None
  if (kept.is_none()) return nullptr;
  py::tuple t = kept.cast<py::tuple>(), shape = t[2].cast<py::tuple>();
  if (shape[0].cast<int64_t>() != K || shape[1].cast<int64_t>() != rows) return nullptr;
  return reinterpret_cast<const int32_t*>(t[1].cast<uintptr_t>());
}

bool flag(const py::object& o, const char* name) { return o.attr(name).cast<bool>(); }

/* Identity of a weight whose tiles are kept: they are made again when any of this changes. */
struct PreparedWeight {
  int64_t version = 0, c_in = 0;
  const void* data = nullptr;
  at::ScalarType weight_dtype{}, dtype{};
  std::vector<int64_t> shape;
  Tensor tiles[2];  // by half (wcn_conv_prepared_half), each made when it is first asked for
  std::unique_ptr<MadeOn> made[2];
};

/* One half of the kernels' tiles of a weight, kept on the tensor object as `_wcn_prepared` = (what they were made
 * from and the halves, the first of them).  make_w(): the weight as the contraction would receive it. */
template <typename F>
Tensor prepared_tiles(const py::object& weight_obj, const Tensor& weight, const F& make_w, at::ScalarType dtype,
                      int64_t c_in, int half) {
  const int64_t version = weight._version();
  void* stream = stream_of(weight);
  py::object kept = py::getattr(weight_obj, "_wcn_prepared", py::none());
  std::shared_ptr<PreparedWeight> same;
  if (!kept.is_none()) {
    auto p = kept[py::int_(0)].cast<std::shared_ptr<PreparedWeight>>();
    if (p->version == version && p->data == weight.const_data_ptr() && p->weight_dtype == weight.scalar_type() &&
        p->dtype == dtype && p->c_in == c_in && weight.sizes().equals(p->shape)) {
      if (p->tiles[half].defined()) {
        p->made[half]->before_use({&p->tiles[half]});
        return p->tiles[half];
      }
      same = std::move(p);
    }
  }
  const Tensor w = make_w();
  const int32_t K = static_cast<int32_t>(w.size(0)), ci = static_cast<int32_t>(w.size(1)), co = static_cast<int32_t>(w.size(2));
  const size_t nbytes = wcn_conv_prepared_weight_bytes(K, ci, co, dtype_code(dtype)) / 2;
  const Tensor tiles = at::empty({static_cast<int64_t>(nbytes)}, at::TensorOptions().dtype(at::kByte).device(w.device()));
  check(wcn_conv_prepare_weight_half(w.const_data_ptr(), dtype_code(w.scalar_type()), K, ci, co, dtype_code(dtype), half,
                                     tiles.mutable_data_ptr(), nbytes, stream),
        "wcn_conv_prepare_weight_half");
  if (MadeOn::capturing(stream)) return tiles;
  auto p = same ? same : std::make_shared<PreparedWeight>();
  p->tiles[half] = tiles;
  p->made[half] = std::make_unique<MadeOn>(stream);
  if (same) return tiles;
  p->version = version;
  p->data = weight.const_data_ptr();
  p->weight_dtype = weight.scalar_type();
  p->dtype = dtype;
  p->c_in = c_in;
  p->shape = weight.sizes().vec();
  if (py::hasattr(weight_obj, "__dict__")) weight_obj.attr("_wcn_prepared") = py::make_tuple(p, tiles);
  return tiles;
}

bool kernel_bias(const Tensor& bias, const Tensor& features, int64_t c_out);
bool aligned16(const void* p);
bool plain_rows(const Tensor& t);

void LayerAhead::launch(const Tensor& in_maps, const Tensor& out_maps, int64_t expected, const void* map_result,
                        const int32_t* groups, int32_t K, int64_t num_out) {
  out = Tensor();
  const Tensor w = weight.cast<Tensor>();
  const at::ScalarType dtype = features.scalar_type();
  const int code = dtype_code(dtype);
  // what conv_forward has to convert, copy, pad or refuse is left to it
  if (code < 0 || !features.is_cuda() || features.dim() != 2 || w.dim() != 3 || w.size(0) != K || w.size(1) != features.size(1) ||
      w.device() != features.device() || features.device() != in_maps.device() || !features.is_contiguous() || !w.is_contiguous() ||
      (w.scalar_type() != dtype && w.scalar_type() != at::kFloat) || (compute_dtype && *compute_dtype != dtype) || num_out == 0 ||
      features.size(0) == 0 || features.size(0) * features.element_size() == 0 || w.size(2) > INT32_MAX || w.size(1) > INT32_MAX ||
      (graph && (!plain_rows(features) || !plain_rows(w))))
    return;
  const int32_t c_in = static_cast<int32_t>(w.size(1)), c_out = static_cast<int32_t>(w.size(2));
  const void* const px = features.const_data_ptr();
  if (c_in * features.element_size() % 16 != 0 || !aligned16(px)) return;
  const int half = graph ? wcn_conv_graph_ahead(code, K, c_in, c_out, features.size(0), num_out, in_maps.numel()) - 1
                         : wcn_conv_ahead_half(code, K, c_in, c_out, features.size(0), num_out, in_maps.numel());
  if (half < 0) return;
  const bool has_bias = bias && bias->defined(), has_residual = residual && residual->defined();
  if (has_bias && (!kernel_bias(*bias, features, c_out) || !bias->is_contiguous() ||
                   (bias->scalar_type() != dtype && !(graph && bias->scalar_type() == at::kFloat)) ||
                   !(graph ? plain_rows(*bias) : aligned16(bias->const_data_ptr()))))
    return;
  if (has_residual && (residual->dim() != 2 || residual->size(0) != num_out || residual->size(1) != c_out || !residual->is_cuda() ||
                       residual->device() != features.device() || residual->scalar_type() != dtype || !residual->is_contiguous()))
    return;
  void* stream = stream_of(features);
  if (graph) {
    Tensor rows = at::empty({num_out, c_out}, features.options());
    const Tensor ws = bytes_on(wcn_conv_workspace_bytes(num_out, K, c_in, c_out, code, 0, 1), features);
    check(wcn_sparse_conv_fwd_graph_ahead(px, features.size(0), c_in, code, w.const_data_ptr(), dtype_code(w.scalar_type()), K, c_out,
                                          has_bias ? bias->const_data_ptr() : nullptr,
                                          has_bias ? dtype_code(bias->scalar_type()) : code, in_maps.const_data_ptr<int32_t>(),
                                          out_maps.const_data_ptr<int32_t>(), in_maps.numel(), expected,
                                          static_cast<const int64_t*>(map_result), static_cast<int32_t>(identity), groups,
                                          rows.mutable_data_ptr(), num_out, ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()),
                                          stream),
          "wcn_sparse_conv_fwd_graph_ahead");
    out = rows;
    return;
  }
  Tensor tiles;
  if (keep_tiles) {
    tiles = prepared_tiles(weight, w, [&]() { return w; }, dtype, c_in, half);
  } else {
    const size_t nbytes = wcn_conv_prepared_weight_bytes(K, c_in, c_out, code) / 2;
    tiles = bytes_on(nbytes, features);
    check(wcn_conv_prepare_weight_half(w.const_data_ptr(), dtype_code(w.scalar_type()), K, c_in, c_out, code, half,
                                       tiles.mutable_data_ptr(), static_cast<size_t>(tiles.numel()), stream),
          "wcn_conv_prepare_weight_half");
  }
  Tensor rows = at::empty({num_out, c_out}, features.options());
  check(wcn_sparse_conv_fwd_ahead(px, features.size(0), c_in, code, tiles.const_data_ptr(), K, c_out,
                                  has_bias ? bias->const_data_ptr() : nullptr, in_maps.const_data_ptr<int32_t>(),
                                  out_maps.const_data_ptr<int32_t>(), in_maps.numel(), expected, static_cast<const int64_t*>(map_result),
                                  static_cast<int32_t>(identity), groups, has_residual ? residual->const_data_ptr() : nullptr,
                                  relu ? 1 : 0, rows.mutable_data_ptr(), num_out, stream),
        "wcn_sparse_conv_fwd_ahead");
  out = rows;
}

// Plans up to this size stay with their map (4 bytes per row and offset: three times the lists of a map of a scene's
// surface).  27 offsets of 10 M rows: what one 16-bit activation of 64 channels takes there.
constexpr size_t kKeepPlanBytes = size_t{1} << 30;

/* Tile plan of a builder's map (wcn_tile_plan_build), kept on the map object: the layers over a map share
 * it, on whichever stream they run.  Undefined where another contraction is to be taken, or the map is none the plan can be made from.  Where the plan
 * does not pay for itself in the calls that are known to come it is made for the second layer that would use it; which
 * layers came before must not show in the results, so such a plan is for the products alone that have the same bits
 * without one.  Inside a graph (`graph`) that holds for every plan: a sum that rounds to the other side is nothing by itself, but
 * behind a ReLU it switches a gradient off or on.  A plan of more than kKeepPlanBytes is made by the calls that repay it
 * alone, and goes with them. */
Tensor tile_plan(const py::object& km, const MapRef& map, int64_t n_in, int64_t num_out, int code, int32_t c_in, int32_t c_out,
                 int32_t calls, bool graph) {
  const size_t plan_bytes = wcn_tile_plan_bytes(num_out, map.K);
  const bool keep = plan_bytes <= kKeepPlanBytes;
  const int worth = wcn_conv_tiles_supported(code, map.K, c_in, c_out, num_out, map.host_offsets(),
                                             static_cast<int32_t>(map.identity), keep ? calls : 1);
  if (!worth || (!keep && worth < 3)) return Tensor();
  if ((graph || worth < 3) && !wcn_conv_tiles_same_sums(code, map.K, c_in, c_out, n_in, num_out, map.pairs(),
                                                        static_cast<int32_t>(map.identity), graph ? 1 : 0))
    return Tensor();
  py::object kept = km.attr("_tile_plan");
  if (!kept.is_none()) {
    py::tuple t = kept.cast<py::tuple>();
    if (t[1].cast<int64_t>() == n_in && t[2].cast<int64_t>() == num_out) {
      const Tensor plan = t[0].cast<Tensor>();
      t[3].cast<const MadeOn*>()->before_use({&plan});
      return plan;
    }
  }
  py::object dev = km.attr("_device_offsets");
  if (dev.is_none() || !flag(km, "_out_ascend") || !flag(km, "_from_builder")) return Tensor();
  const int32_t* groups = group_starts(km.attr("_group_start"), map.K, num_out);
  if (!groups) return Tensor();
  if (worth < 3 && !flag(km, "_tiles_wanted")) {
    km.attr("_tiles_wanted") = true;
    return Tensor();
  }
  void* stream = stream_of(map.in_maps);
  const Tensor plan = bytes_on(plan_bytes, map.in_maps);
  const Tensor ws = bytes_on(wcn_tile_plan_workspace_bytes(num_out, map.K, map.pairs()), map.in_maps);
  check(wcn_tile_plan_build(map.in_maps.const_data_ptr<int32_t>(), map.out_maps.const_data_ptr<int32_t>(),
                            dev.cast<Tensor>().const_data_ptr<int64_t>(), groups, map.K, static_cast<int32_t>(map.identity),
                            n_in, num_out, map.pairs(), plan.mutable_data_ptr(), static_cast<size_t>(plan.numel()),
                            ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
        "wcn_tile_plan_build");
  if (keep && !MadeOn::capturing(stream)) km.attr("_tile_plan") = py::make_tuple(plan, n_in, num_out, std::make_shared<MadeOn>(stream));
  return plan;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

void check_weight_device(const Tensor& weight, const Tensor& features) {
  if (weight.device() != features.device())
    throw py::value_error("weight is on " + weight.device().str() + ", the features on " + features.device().str());
}

bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }

// The layers' graph nodes have gradients and no forward-mode derivative: a tangent would be lost without a word.
void refuse_tangents(std::initializer_list<const Tensor*> tensors, const char* layer) {
  for (const Tensor* t : tensors)
    if (has_tangent(*t)) TORCH_CHECK_NOT_IMPLEMENTED(false, layer, " has no forward-mode derivative (jvp)");
}

/* Whether a bias is what the kernels read: (c_out) values on the features' device.  Any other (one value for all channels, a
 * row of its own per output row, a scalar in host memory, a wrong length), and one with a forward-mode tangent, is added, or
 * refused, by torch behind them. */
bool kernel_bias(const Tensor& bias, const Tensor& features, int64_t c_out) {
  return bias.dim() == 1 && bias.size(0) == c_out && bias.device() == features.device() && !has_tangent(bias);
}

/* out = act(sum_k scatter(X[in_k] @ W[k]) + bias + residual), see sparse_conv_forward.  `graph`: the form for
 * a layer whose gradients will be asked for: no residual, no clamp, and the bias, whatever its type, is added to the rounded
 * sums. */
Tensor conv_forward(const Tensor& features, const py::object& weight_obj, const py::object& km, int64_t num_out,
                    const std::optional<Tensor>& bias, const std::optional<at::ScalarType>& compute_dtype,
                    const std::optional<Tensor>& residual, bool relu, bool keep_tiles, const py::object& pairs_sorted,
                    bool graph) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor weight = weight_obj.cast<Tensor>();
  if (!features.is_cuda()) throw py::value_error("in_features must be on a GPU device, got " + features.device().str());
  if (features.dim() != 2 || weight.dim() != 3 || weight.size(1) != features.size(1))
    throw py::value_error("shape mismatch: features " + shape_text(features) + ", weight " + shape_text(weight));
  check_weight_device(weight, features);
  MapRef map(km);
  const int32_t K = static_cast<int32_t>(weight.size(0)), c_out = static_cast<int32_t>(weight.size(2));
  if (map.K != K)
    throw py::value_error("kernel map has " + std::to_string(map.K) + " offsets, weight has " + std::to_string(K));
  Tensor x = compute_dtype && *compute_dtype != features.scalar_type() ? features.to(*compute_dtype) : features;
  const at::ScalarType dtype = x.scalar_type();
  const int code = dtype_code(dtype);
  if (code < 0)
    throw py::type_error(std::string("unsupported feature dtype ") + c10::toString(dtype));
  x = x.contiguous();
  auto as_rows = [&](const std::optional<Tensor>& t) -> Tensor {  // in the features' dtype and contiguous
    if (!t || !t->defined()) return Tensor();
    return (t->scalar_type() == dtype && t->is_contiguous()) ? *t : t->to(dtype).contiguous();
  };
  if (bias && bias->defined() && !kernel_bias(*bias, features, c_out)) {
    if (graph) throw py::value_error("bias has shape " + shape_text(*bias) + ", the output " + std::to_string(c_out) + " channels");
    Tensor out = conv_forward(features, weight_obj, km, num_out, std::nullopt, compute_dtype, std::nullopt, false, keep_tiles,
                              pairs_sorted, false);
    out = out + bias->to(out.scalar_type());
    if (residual) out = out + residual->to(out.scalar_type());
    return relu ? at::relu(out) : out;
  }
  // (graph) an fp32 bias goes to the library as it is, any other in the features' type
  Tensor b = graph && bias && bias->scalar_type() == at::kFloat ? bias->contiguous() : as_rows(bias);
  if (b.defined() && !aligned16(b.const_data_ptr())) b = b.clone();
  const int b_code = b.defined() ? dtype_code(b.scalar_type()) : code;
  // Rows that are not whole 16-byte vectors (the 3-channel input of a network's stem) would take the
  // library's slow general kernel: the channels are zero-padded instead, and the weight's with them.
  const int64_t vec = 16 / x.element_size();
  int64_t pad = 0;
  if (x.size(1) % vec != 0 && x.size(0) > 0) {
    pad = vec - x.size(1) % vec;
    x = at::constant_pad_nd(x, {0, pad});
  }
  auto make_w = [&]() {
    Tensor w = weight;
    if (w.scalar_type() != dtype && w.scalar_type() != at::kFloat) w = w.to(dtype);
    if (pad) w = at::constant_pad_nd(w, {0, 0, 0, pad});
    return w.contiguous();
  };
  const int32_t c_in = static_cast<int32_t>(x.size(1));
  const int64_t n_in = x.size(0);
  Tensor r;
  if (residual) {
    if (residual->dim() != 2 || residual->size(0) != num_out || residual->size(1) != c_out)
      throw py::value_error("residual has shape " + shape_text(*residual) + ", the output (" + std::to_string(num_out) +
                            ", " + std::to_string(c_out) + ")");
    if (!residual->is_cuda()) throw py::value_error("residual must be on a GPU device, got " + residual->device().str());
    r = as_rows(residual);
  }
  void* stream = stream_of(x);
  Tensor out = at::empty({num_out, c_out}, x.options());
  const void *px = x.const_data_ptr(), *pb = b.defined() ? b.const_data_ptr() : nullptr,
             *pr = r.defined() ? r.const_data_ptr() : nullptr;
  void* po = out.mutable_data_ptr();
  auto finish = [&]() { return out.scalar_type() == features.scalar_type() ? out : out.to(features.scalar_type()); };

  if (num_out > 0 && n_in > 0 && (dtype == at::kHalf || dtype == at::kBFloat16) && flag(km, "_single_out") &&
      map.pairs() == num_out && wcn_conv_single_supported(code, c_in, c_out, K)) {
    // one pair per output row: nothing is summed, the lists are taken in the order they have
    Tensor w, ws;
    size_t nbytes = 0;
    if (keep_tiles) {
      w = prepared_tiles(weight_obj, weight, make_w, dtype, c_in, 0);
    } else {
      w = make_w();
      nbytes = wcn_conv_prepared_weight_bytes(K, c_in, c_out, code);
      ws = bytes_on(nbytes, x);
    }
    if (graph) {
      check(wcn_sparse_conv_fwd_single_graph(px, n_in, c_in, code, w.const_data_ptr(), dtype_code(w.scalar_type()), K, c_out, pb,
                                             b_code, map.in_maps.const_data_ptr<int32_t>(),
                                             map.out_maps.const_data_ptr<int32_t>(), map.host_offsets(), po, num_out,
                                             ws.mutable_data_ptr(), nbytes, stream),
            "wcn_sparse_conv_fwd_single_graph");
      return finish();
    }
    check(wcn_sparse_conv_fwd_single(px, n_in, c_in, code, w.const_data_ptr(), keep_tiles ? code : dtype_code(w.scalar_type()),
                                     keep_tiles ? 1 : 0, K, c_out, pb, map.in_maps.const_data_ptr<int32_t>(),
                                     map.out_maps.const_data_ptr<int32_t>(), map.host_offsets(), pr, relu ? 1 : 0, po, num_out,
                                     ws.defined() ? ws.mutable_data_ptr() : nullptr, nbytes, stream),
          "wcn_sparse_conv_fwd_single");
    return finish();
  }
  if (num_out > 0 && n_in > 0 && aligned16(px) && aligned16(po) && aligned16(pr)) {
    if (const Tensor plan = tile_plan(km, map, n_in, num_out, code, c_in, c_out, graph ? 2 : 1, graph); plan.defined()) {
      Tensor w, ws;
      size_t nbytes = 0;
      if (keep_tiles) {
        w = prepared_tiles(weight_obj, weight, make_w, dtype, c_in, 0);
      } else {
        w = make_w();
        nbytes = wcn_conv_prepared_weight_bytes(K, c_in, c_out, code);
        ws = bytes_on(nbytes, x);
      }
      check(wcn_sparse_conv_fwd_tiled(px, n_in, c_in, code, w.const_data_ptr(), keep_tiles ? code : dtype_code(w.scalar_type()),
                                      keep_tiles ? 1 : 0, K, c_out, pb, b_code, graph ? 1 : 0, plan.const_data_ptr(), pr, relu ? 1 : 0, po, num_out,
                                      ws.defined() ? ws.mutable_data_ptr() : nullptr, nbytes, stream),
            "wcn_sparse_conv_fwd_tiled");
      return finish();
    }
  }
  const int32_t* groups = nullptr;
  Tensor groups_held;
  if (!flag(km, "_out_ascend") && num_out > 0) {
    // re-ordered once and kept on the map object (a transposed convolution, lists made by hand)
    py::tuple t = pairs_sorted(km, "out", num_out).cast<py::tuple>();
    map.in_maps = t[0].cast<Tensor>();
    map.out_maps = t[1].cast<Tensor>();
    groups_held = t[2].cast<Tensor>();
    groups = groups_held.const_data_ptr<int32_t>();
  } else {
    groups = group_starts(km.attr("_group_start"), K, num_out);
  }
  const int32_t* in_maps = map.in_maps.const_data_ptr<int32_t>();
  const int32_t* out_maps = map.out_maps.const_data_ptr<int32_t>();
  const int32_t iden = static_cast<int32_t>(map.identity);
  if (keep_tiles && groups != nullptr && num_out > 0) {
    const int half = wcn_conv_prepared_half(code, K, c_in, c_out, num_out, aligned16(px) ? 1 : 0);
    const Tensor tiles = prepared_tiles(weight_obj, weight, make_w, dtype, c_in, half);
    const void* const pt = tiles.const_data_ptr();
    py::object dev = km.attr("_device_offsets");
    if (dev.is_none() || dev.cast<Tensor>().device() != x.device() || dev.cast<Tensor>().numel() != K + 1) {
      dev = py::cast(map.offsets.to(x.device()));
      km.attr("_device_offsets") = dev;
    }
    const Tensor device_offsets = dev.cast<Tensor>();
    const size_t nbytes = wcn_conv_prepared_workspace_bytes(num_out, K, c_in, c_out, code);
    Tensor ws;
    if (nbytes) ws = bytes_on(nbytes, x);
    check(wcn_sparse_conv_fwd_prepared_halves(px, n_in, c_in, code, half == 0 ? pt : nullptr, half == 1 ? pt : nullptr, K,
                                              c_out, pb, in_maps, out_maps, map.host_offsets(),
                                              static_cast<const int64_t*>(device_offsets.const_data_ptr()), iden, groups, pr,
                                              relu ? 1 : 0, po, num_out, nbytes ? ws.mutable_data_ptr() : nullptr, nbytes,
                                              stream),
          "wcn_sparse_conv_fwd_prepared");
    return finish();
  }
  const Tensor w = make_w();
  const Tensor ws = bytes_on(wcn_conv_workspace_bytes(num_out, K, c_in, c_out, code, map.pairs(), 1), x);
  if (graph) {
    check(wcn_sparse_conv_fwd_graph(px, n_in, c_in, code, w.const_data_ptr(), dtype_code(w.scalar_type()), K, c_out, pb, b_code,
                                    in_maps, out_maps, map.host_offsets(), iden, 1, groups, po, num_out,
                                    ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
          "wcn_sparse_conv_fwd_graph");
    return finish();
  }
  check(wcn_sparse_conv_fwd_fused(px, n_in, c_in, code, w.const_data_ptr(), dtype_code(w.scalar_type()), K, c_out, pb,
                                  in_maps, out_maps, map.host_offsets(), iden, 1, groups, pr, relu ? 1 : 0, po, num_out,
                                  ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
        "wcn_sparse_conv_fwd_fused");
  return finish();
}

bool in_graph(std::initializer_list<const Tensor*> tensors);

/* Whether a tensor is plain device memory of this call's: no wrapper of a transform, a mode or a subclass. */
bool plain_rows(const Tensor& t) {
  const c10::DispatchKeySet keys = t.key_set() - c10::autograd_dispatch_keyset_with_ADInplaceOrView - c10::autocast_dispatch_keyset;
  return keys == c10::DispatchKeySet(c10::DispatchKey::CUDA) && t.is_contiguous() && aligned16(t.const_data_ptr()) && !has_tangent(t);
}

/* The layer of one voxel and stride 1, outside any graph: features @ weight[0] + bias, or an undefined tensor where torch is to
 * compute it: a call of another kind, or one that a transform, a trace or a mode has to see. */
Tensor pointwise_forward(const Tensor& features, const Tensor& weight, const std::optional<Tensor>& bias) {
  using c10::DispatchKey;
  if (in_graph({&features, &weight, bias ? &*bias : &features}) || at::autocast::is_autocast_enabled(at::kCUDA)) return Tensor();
  for (const DispatchKey key : {DispatchKey::Tracer, DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::Python,
                                DispatchKey::PythonDispatcher, DispatchKey::Functionalize})
    if (c10::impl::tls_is_dispatch_key_included(key)) return Tensor();
  if (at::impl::torch_function_mode_enabled()) return Tensor();
  const int code = dtype_code(features.scalar_type());
  if (features.dim() != 2 || weight.dim() != 3 || weight.size(0) != 1 || weight.size(1) != features.size(1) ||
      weight.scalar_type() != features.scalar_type() || weight.device() != features.device() || !plain_rows(features) ||
      !plain_rows(weight))
    return Tensor();
  if (weight.size(1) > INT32_MAX || weight.size(2) > INT32_MAX) return Tensor();
  const int32_t c_in = static_cast<int32_t>(weight.size(1)), c_out = static_cast<int32_t>(weight.size(2));
  if (!wcn_pointwise_takes(features.size(0), c_in, c_out, code)) return Tensor();
  const bool has_bias = bias && bias->defined();
  if (has_bias && (!kernel_bias(*bias, features, c_out) || bias->scalar_type() != features.scalar_type() || !plain_rows(*bias)))
    return Tensor();
  const c10::DeviceGuard device(features.device());
  Tensor out = at::empty({features.size(0), c_out}, features.options());
  check(wcn_pointwise_fwd(features.const_data_ptr(), features.size(0), c_in, code, weight.const_data_ptr(), c_out,
                          has_bias ? bias->const_data_ptr() : nullptr, out.mutable_data_ptr(), stream_of(features)),
        "wcn_pointwise_fwd");
  return out;
}

/* Sums over the rows, in fp32: the gradient of a bias. */
Tensor column_sums(const Tensor& rows, at::ScalarType out_dtype) {
  if (dtype_code(out_dtype) < 0 || dtype_code(rows.scalar_type()) < 0) return rows.sum(0, false, out_dtype);
  const Tensor r = rows.contiguous();
  const int32_t c = static_cast<int32_t>(r.size(1));
  Tensor out = at::empty({c}, r.options().dtype(out_dtype));
  const Tensor ws = bytes_on(wcn_column_sums_workspace_bytes(c), r);
  check(wcn_column_sums(r.const_data_ptr(), r.size(0), c, dtype_code(r.scalar_type()), out.mutable_data_ptr(),
                        dtype_code(out_dtype), ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream_of(r)),
        "wcn_column_sums");
  return out;
}

/* Pair lists of one order with the group starts that belong to it. */
struct Ordered {
  Tensor in_maps, out_maps, groups_held;
  const int32_t* groups = nullptr;
};

/* What the gradients need of a map, read while the interpreter is at hand. */
struct GradMap {
  MapRef map;
  bool symmetric, in_ascend, single_in;
  const int32_t *groups, *in_groups;
  Tensor groups_tensor, in_groups_tensor;  // hold the memory behind them
  Tensor device_offsets;                   // undefined where the map has none in device memory
  Tensor plan;                             // tile plan, where the input gradient is taken over one,
  int32_t plan_form = 3;                   // and the form the weight is read in
  GradMap(const py::object& km, int64_t n_in, int64_t n_out, int code, int32_t c_in, int32_t c_out, bool need_x)
      : map(km),
        symmetric(flag(km, "_symmetric") && flag(km, "_out_ascend") && n_in == n_out),
        in_ascend(flag(km, "_in_ascend")),
        single_in(flag(km, "_single_in")) {
    py::object g = km.attr("_group_start"), gi = km.attr("_in_group_start");
    groups = group_starts(g, map.K, n_in);
    in_groups = group_starts(gi, map.K, n_in);
    py::object dev = km.attr("_device_offsets");
    if (!dev.is_none() && dev.cast<Tensor>().device() == map.in_maps.device() && dev.cast<Tensor>().numel() == map.K + 1)
      device_offsets = dev.cast<Tensor>();
    if (groups) groups_tensor = g[py::int_(0)].cast<Tensor>();
    if (in_groups) in_groups_tensor = gi[py::int_(0)].cast<Tensor>();
    // the input gradient walks the rows of a symmetric map itself, with the offsets reversed, or those of the forward map
    // that a transposed convolution's map is the exchange of
    py::object forward = km.attr("_forward_map");
    if (!need_x) return;
    if (symmetric && n_in > 0) {
      plan = tile_plan(km, map, n_in, n_in, code, c_out, c_in, 1, false);
      plan_form = 3;
    } else if (!forward.is_none() && n_in > 0 && n_out > 0) {
      const MapRef f(forward);
      if (f.out_maps.const_data_ptr() == map.in_maps.const_data_ptr() && f.in_maps.const_data_ptr() == map.out_maps.const_data_ptr() &&
          f.identity < 0 && map.identity < 0)
        plan = tile_plan(forward, f, n_out, n_in, code, c_out, c_in, 1, false);
      plan_form = 2;
    }
  }
};

/* (dX or undefined, dW or undefined), see sparse_conv_backward.  sorted(): the lists ascending in
 * input row, asked for only where the map needs re-ordering.  `grad_bias`: filled with the sums of grad_output's rows
 * (which are then of the features' type) beside dW. */
template <typename F>
std::pair<Tensor, Tensor> backward(const Tensor& grad_output, const Tensor& in_features, const Tensor& weight,
                                   const GradMap& g, at::ScalarType dtype, bool need_x, bool need_w, const F& sorted,
                                   Tensor* grad_bias = nullptr) {
  const int code = dtype_code(dtype);
  const int32_t K = g.map.K, c_in = static_cast<int32_t>(weight.size(1)), c_out = static_cast<int32_t>(weight.size(2));
  const Tensor x = in_features.to(dtype).contiguous(), gy = grad_output.to(dtype).contiguous();
  Tensor w = weight;
  if (w.scalar_type() != dtype && w.scalar_type() != at::kFloat) w = w.to(dtype);
  w = w.contiguous();
  const int wcode = dtype_code(w.scalar_type());
  const int64_t n_in = x.size(0), n_out = gy.size(0), pairs = g.map.pairs();
  const int32_t iden = static_cast<int32_t>(g.map.identity);
  void* stream = stream_of(x);
  const void* pgy = gy.const_data_ptr();
  Tensor grad_x, grad_w;
  if (need_x) {
    if (n_in == 0 || n_out == 0) {
      grad_x = at::zeros_like(x);
    } else if (grad_x = at::empty({n_in, c_in}, x.options());
               g.single_in && pairs == n_in && (dtype == at::kHalf || dtype == at::kBFloat16) &&
               wcn_conv_single_supported(code, c_out, c_in, K)) {
      // every input row is in exactly one pair: dX[in] = dY[out] @ W[k]^T, the lists as they are
      const size_t nbytes = wcn_conv_prepared_weight_bytes(K, c_out, c_in, code);
      Tensor ws = bytes_on(nbytes, x);
      check(wcn_sparse_conv_fwd_single(pgy, n_out, c_out, code, w.const_data_ptr(), wcode, 2, K, c_in, nullptr,
                                       g.map.out_maps.const_data_ptr<int32_t>(), g.map.in_maps.const_data_ptr<int32_t>(),
                                       g.map.host_offsets(), nullptr, 0, grad_x.mutable_data_ptr(), n_in,
                                       ws.mutable_data_ptr(), nbytes, stream),
            "wcn_sparse_conv_fwd_single");
    } else if (g.plan.defined() && aligned16(pgy) && aligned16(grad_x.const_data_ptr())) {
      const size_t nbytes = wcn_conv_prepared_weight_bytes(K, c_out, c_in, code);
      Tensor ws = bytes_on(nbytes, x);
      check(wcn_sparse_conv_fwd_tiled(pgy, n_out, c_out, code, w.const_data_ptr(), wcode, g.plan_form, K, c_in, nullptr, code, 0,
                                      g.plan.const_data_ptr(), nullptr, 0, grad_x.mutable_data_ptr(), n_in,
                                      ws.mutable_data_ptr(), nbytes, stream),
            "wcn_sparse_conv_fwd_tiled");
    } else {
      Ordered o{g.map.in_maps, g.map.out_maps, Tensor(), g.symmetric ? g.groups : g.in_groups};
      if (!g.symmetric && !g.in_ascend) o = sorted();
      Tensor ws = bytes_on(wcn_conv_workspace_bytes(n_in, K, c_out, c_in, code, pairs, 1), x);
      check(wcn_sparse_conv_dgrad(pgy, n_out, c_out, code, w.const_data_ptr(), wcode, K, c_in,
                                  o.in_maps.const_data_ptr<int32_t>(), o.out_maps.const_data_ptr<int32_t>(),
                                  g.map.host_offsets(), iden, g.symmetric ? 1 : 0, 1, o.groups, grad_x.mutable_data_ptr(),
                                  n_in, ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
            "wcn_sparse_conv_dgrad");
    }
    grad_x = grad_x.to(in_features.scalar_type());
  }
  if (need_w) {
    grad_w = at::empty({K, c_in, c_out}, w.options());
    const int64_t identity_rows = iden >= 0 ? std::min(n_in, n_out) : 0;
    Tensor ws = bytes_on(wcn_conv_wgrad_workspace_bytes(K, c_in, c_out, pairs, identity_rows), x);
    const int64_t* device_offsets = g.device_offsets.defined() ? g.device_offsets.const_data_ptr<int64_t>() : nullptr;
    const int32_t *in_maps = g.map.in_maps.const_data_ptr<int32_t>(), *out_maps = g.map.out_maps.const_data_ptr<int32_t>();
    const size_t nbytes = static_cast<size_t>(ws.numel());
    if (grad_bias) {
      Tensor sums = bytes_on(wcn_column_sums_workspace_bytes(c_out), x);
      check(wcn_sparse_conv_wgrad_bias(x.const_data_ptr(), n_in, c_in, pgy, n_out, c_out, code, in_maps, out_maps,
                                       g.map.host_offsets(), device_offsets, K, iden, grad_w.mutable_data_ptr(), wcode,
                                       ws.mutable_data_ptr(), nbytes, grad_bias->mutable_data_ptr(),
                                       dtype_code(grad_bias->scalar_type()), sums.mutable_data_ptr(),
                                       static_cast<size_t>(sums.numel()), stream),
            "wcn_sparse_conv_wgrad_bias");
    } else {
      check(wcn_sparse_conv_wgrad_mapped(x.const_data_ptr(), n_in, c_in, pgy, n_out, c_out, code, in_maps, out_maps,
                                         g.map.host_offsets(), device_offsets, K, iden, grad_w.mutable_data_ptr(), wcode,
                                         ws.mutable_data_ptr(), nbytes, stream),
            "wcn_sparse_conv_wgrad");
    }
    grad_w = grad_w.to(weight.scalar_type());
  }
  return {grad_x, grad_w};
}

Ordered sorted_by_in(const py::object& km, const py::object& pairs_sorted, int64_t n_in) {
  py::tuple t = pairs_sorted(km, "in", n_in).cast<py::tuple>();  // (gathered = out side, ascending = in side, groups)
  Ordered o{t[1].cast<Tensor>(), t[0].cast<Tensor>(), t[2].cast<Tensor>()};
  o.groups = o.groups_held.const_data_ptr<int32_t>();
  return o;
}

py::tuple conv_backward(const Tensor& grad_output, const Tensor& in_features, const Tensor& weight, const py::object& km,
                        const std::optional<at::ScalarType>& compute_dtype, bool need_x, bool need_w,
                        const py::object& pairs_sorted) {
  at::AutoDispatchBelowADInplaceOrView guard;
  for (const auto* t : {&grad_output, &in_features})
    if (!t->is_cuda())
      throw py::value_error(std::string(t == &grad_output ? "grad_output" : "in_features") + " must be on a GPU device, got " +
                            t->device().str());
  const at::ScalarType dtype = compute_dtype.value_or(in_features.scalar_type());
  if (dtype_code(dtype) < 0) throw py::type_error(std::string("unsupported feature dtype ") + c10::toString(dtype));
  GradMap g(km, in_features.size(0), grad_output.size(0), dtype_code(dtype), static_cast<int32_t>(in_features.size(1)),
            static_cast<int32_t>(grad_output.size(1)), need_x);
  if (weight.dim() != 3 || g.map.K != weight.size(0) || in_features.size(1) != weight.size(1) ||
      grad_output.size(1) != weight.size(2))
    throw py::value_error("shape mismatch: features " + shape_text(in_features) + ", grad_output " + shape_text(grad_output) +
                          ", weight " + shape_text(weight) + ", " + std::to_string(g.map.K) + " offsets");
  check_weight_device(weight, in_features);
  auto r = backward(grad_output, in_features, weight, g, dtype, need_x, need_w,
                    [&]() { return sorted_by_in(km, pairs_sorted, in_features.size(0)); });
  return py::make_tuple(r.first.defined() ? py::cast(r.first) : py::none(), r.second.defined() ? py::cast(r.second) : py::none());
}

/* A Python object owned by a graph node: the node may go away on a thread without the interpreter. */
struct HeldObject {
  py::object o;
  explicit HeldObject(py::object v) : o(std::move(v)) {}
  ~HeldObject() {
    if (Py_IsInitialized()) {
      py::gil_scoped_acquire locked;
      o = py::object();
    } else {
      o.release();
    }
  }
};

struct ConvBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable x_, w_;
  std::unique_ptr<HeldObject> km_, sorted_;
  std::unique_ptr<GradMap> map_;
  at::ScalarType dtype_{}, bias_dtype_{};
  bool has_bias_ = false;

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    torch::autograd::variable_list out(has_bias_ ? 3 : 2);
    if (!grads[0].defined()) return out;
    TORCH_CHECK(map_ != nullptr, "Trying to backward through the graph a second time (the map was given back after the first)");
    const Tensor x = x_.unpack(shared_from_this()), w = w_.unpack(shared_from_this());
    at::NoGradGuard no_grad;
    const bool need_x = task_should_compute_output(0), need_w = task_should_compute_output(1);
    const bool need_b = has_bias_ && task_should_compute_output(2);
    const bool joined = need_b && need_w && grads[0].scalar_type() == dtype_ && dtype_code(bias_dtype_) >= 0;
    if (joined) out[2] = at::empty({grads[0].size(1)}, grads[0].options().dtype(bias_dtype_));
    if (need_x || need_w) {
      auto r = backward(grads[0], x, w, *map_, dtype_, need_x, need_w, [&]() {
        py::gil_scoped_acquire locked;
        return sorted_by_in(km_->o, sorted_->o, x.size(0));
      }, joined ? &out[2] : nullptr);
      out[0] = r.first;
      out[1] = r.second;
    }
    if (need_b && !joined) out[2] = column_sums(grads[0], bias_dtype_);
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x_.reset_data();
    w_.reset_data();
    map_.reset();
    km_.reset();
    sorted_.reset();
  }
  std::string name() const override { return "SparseConvBackward"; }
};

/* The contraction with its gradients as one graph node.  The bias is added to the rounded product, as
 * a separate addition behind the function would: fusing it into the sums moves values across the zero of
 * a following ReLU, whose gradient then differs.  `ahead`: what a LayerAhead of the same arguments has left. */
Tensor conv_autograd(const Tensor& features, const py::object& weight_obj, const std::optional<Tensor>& bias,
                     const py::object& km, int64_t num_out, const std::optional<at::ScalarType>& compute_dtype,
                     const py::object& pairs_sorted, const std::optional<Tensor>& ahead) {
  const Tensor weight = weight_obj.cast<Tensor>();
  refuse_tangents({&features, &weight}, "the sparse convolution");
  // a product in another type than the features' comes back in theirs before the bias is added
  const bool given = bias && bias->defined(), has_bias = given && kernel_bias(*bias, features, weight.size(-1));
  const bool inside = !compute_dtype || *compute_dtype == features.scalar_type();
  Tensor out = ahead ? *ahead
                     : conv_forward(features, weight_obj, km, num_out, inside && has_bias ? bias : std::nullopt, compute_dtype,
                                    std::nullopt, false, false, pairs_sorted, true);
  if (has_bias && !inside) {
    at::AutoDispatchBelowADInplaceOrView guard;
    out.add_(bias->scalar_type() == out.scalar_type() ? *bias : bias->to(out.scalar_type()));
  }
  auto node = std::shared_ptr<ConvBackward>(new ConvBackward(), torch::autograd::deleteNode);
  node->set_next_edges(has_bias ? torch::autograd::collect_next_edges(features, weight, *bias)
                                : torch::autograd::collect_next_edges(features, weight));
  node->x_ = torch::autograd::SavedVariable(features, false);
  node->w_ = torch::autograd::SavedVariable(weight, false);
  node->dtype_ = compute_dtype.value_or(features.scalar_type());
  node->has_bias_ = has_bias;
  if (has_bias) node->bias_dtype_ = bias->scalar_type();
  node->map_ = std::make_unique<GradMap>(km, features.size(0), num_out, dtype_code(node->dtype_),
                                         static_cast<int32_t>(weight.size(1)), static_cast<int32_t>(weight.size(2)),
                                         features.requires_grad());
  node->km_ = std::make_unique<HeldObject>(km);
  node->sorted_ = std::make_unique<HeldObject>(pairs_sorted);
  torch::autograd::set_history(out, node);
  return given && !has_bias ? out + bias->to(out.scalar_type()) : out;
}

// ------------------------------------------------------------------------------------------------
// Pooling and depthwise convolution over a rows form
// ------------------------------------------------------------------------------------------------

/* The rows form of a map (wcn_map_rows_build) by output row or, with the lists exchanged, by input row.
 * It depends on the map alone and is kept on the map object: the layers and the backward passes that
 * share a map share it, on whichever stream they run.  A builder's map comes with what the one-pass build reads. */
Tensor rows_form(const py::object& km, const MapRef& map, bool by_out, int64_t num_rows) {
  const Tensor &gathered = by_out ? map.in_maps : map.out_maps, &grouping = by_out ? map.out_maps : map.in_maps;
  py::object kept = km.attr("_rows_forms");
  if (kept.is_none()) {
    kept = py::dict();
    km.attr("_rows_forms") = kept;
  }
  py::dict forms = kept.cast<py::dict>();
  const py::tuple key = py::make_tuple(reinterpret_cast<uintptr_t>(grouping.const_data_ptr()),
                                       reinterpret_cast<uintptr_t>(gathered.const_data_ptr()), num_rows);
  if (forms.contains(key)) {
    py::tuple t = forms[key].cast<py::tuple>();
    const Tensor rows = t[0].cast<Tensor>();
    t[1].cast<const MadeOn*>()->before_use({&rows});
    return rows;
  }
  const int64_t pairs = map.pairs();
  void* stream = stream_of(gathered);
  const Tensor ws = bytes_on(wcn_map_rows_workspace_bytes(num_rows, map.K, pairs), gathered);
  const int32_t* groups = nullptr;
  py::object dev = km.attr("_device_offsets");
  if (map.K <= 128 && flag(km, "_from_builder") && flag(km, by_out ? "_out_ascend" : "_in_ascend") && !dev.is_none())
    groups = group_starts(km.attr(by_out ? "_group_start" : "_in_group_start"), map.K, num_rows);
  if (groups)
    check(wcn_map_rows_build_grouped(gathered.const_data_ptr<int32_t>(), grouping.const_data_ptr<int32_t>(),
                                     dev.cast<Tensor>().const_data_ptr<int64_t>(), groups, map.K, num_rows, pairs,
                                     ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
          "wcn_map_rows_build_grouped");
  else
    check(wcn_map_rows_build(gathered.const_data_ptr<int32_t>(), grouping.const_data_ptr<int32_t>(), map.host_offsets(),
                             map.K, num_rows, ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
          "wcn_map_rows_build");
  if (!MadeOn::capturing(stream)) forms[key] = py::make_tuple(ws, std::make_shared<MadeOn>(stream));
  return ws;
}

/* A map as the gradients of these layers read it, with the object itself for the rows form that only
 * some of them need (asked for on a thread that has to take the interpreter first). */
struct RowsMap {
  MapRef map;
  Tensor by_out;
  bool symmetric = false;
  const int32_t* groups = nullptr;
  Tensor groups_tensor, device_offsets;
  std::unique_ptr<HeldObject> km;
  RowsMap(const py::object& k, int64_t n_in, int64_t n_out) : map(k) {
    symmetric = flag(k, "_symmetric") && flag(k, "_out_ascend") && n_in == n_out;
    if (n_in > 0 && n_out > 0) by_out = rows_form(k, map, true, n_out);
    py::object g = k.attr("_group_start"), dev = k.attr("_device_offsets");
    if (flag(k, "_out_ascend") && !dev.is_none() && (groups = group_starts(g, map.K, n_out)) != nullptr) {
      groups_tensor = g[py::int_(0)].cast<Tensor>();
      device_offsets = dev.cast<Tensor>();
    }
    km = std::make_unique<HeldObject>(k);
  }
  Tensor by_in(int64_t n_in) const {
    py::gil_scoped_acquire locked;
    return rows_form(km->o, map, false, n_in);
  }
};

void check_rows_features(const Tensor& t, at::ScalarType dtype, const char* what) {
  if (!t.is_cuda()) throw py::value_error(std::string(what) + " must be on a GPU device, got " + t.device().str());
  if (dtype_code(dtype) < 0) throw py::type_error(std::string("unsupported feature dtype ") + c10::toString(dtype));
}

/* A weight as the kernels read it: in the features' type or fp32. */
Tensor depthwise_weight(const Tensor& weight, at::ScalarType dtype) {
  return (weight.scalar_type() == dtype || weight.scalar_type() == at::kFloat ? weight : weight.to(dtype)).contiguous();
}

Tensor depthwise_rows(const Tensor& x, const Tensor& w, const Tensor& rows, const MapRef& map, int64_t num_rows,
                      bool reverse, const Tensor& bias) {
  const int32_t c = static_cast<int32_t>(x.size(1));
  Tensor out = at::empty({num_rows, c}, x.options());
  check(wcn_sparse_depthwise_fwd_fused(x.const_data_ptr(), x.size(0), c, dtype_code(x.scalar_type()), w.const_data_ptr(),
                                       dtype_code(w.scalar_type()), rows.const_data_ptr(), num_rows, map.K, map.pairs(),
                                       static_cast<int32_t>(map.identity), reverse ? 1 : 0,
                                       bias.defined() ? bias.const_data_ptr() : nullptr, out.mutable_data_ptr(), stream_of(x)),
        "wcn_sparse_depthwise_fwd");
  return out;
}

Tensor depthwise_out(const Tensor& features, const Tensor& weight, const Tensor& bias, const RowsMap& m, int64_t num_out,
                     at::ScalarType dtype) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor x = features.to(dtype).contiguous();
  const bool has_bias = bias.defined(), fuse = has_bias && dtype == features.scalar_type();
  Tensor out;
  if (num_out == 0 || x.size(0) == 0)
    out = at::zeros({num_out, x.size(1)}, x.options());
  else
    out = depthwise_rows(x, depthwise_weight(weight, dtype), m.by_out, m.map, num_out, false,
                         fuse ? bias.to(dtype).contiguous() : Tensor());
  out = out.to(features.scalar_type());
  if (has_bias && (!fuse || num_out == 0 || x.size(0) == 0)) out.add_(bias.to(out.scalar_type()));
  return out;
}

std::pair<Tensor, Tensor> depthwise_grads(const Tensor& grad_output, const Tensor& in_features, const Tensor& weight,
                                          const RowsMap& m, at::ScalarType dtype, bool need_x, bool need_w,
                                          Tensor* grad_bias = nullptr) {
  const Tensor x = in_features.to(dtype).contiguous(), gy = grad_output.to(dtype).contiguous();
  const Tensor w = depthwise_weight(weight, dtype);
  const int64_t n_in = x.size(0), n_out = gy.size(0);
  const int32_t K = m.map.K, c = static_cast<int32_t>(x.size(1)), code = dtype_code(dtype),
                iden = static_cast<int32_t>(m.map.identity);
  Tensor grad_x, grad_w;
  if (need_x) {
    if (n_in == 0 || n_out == 0)
      grad_x = at::zeros_like(x);
    else
      grad_x = depthwise_rows(gy, w, m.symmetric ? m.by_out : m.by_in(n_in), m.map, n_in, m.symmetric, Tensor());
    grad_x = grad_x.to(in_features.scalar_type());
  }
  if (need_w) {
    grad_w = at::empty_like(w);
    const int32_t *in_maps = m.map.in_maps.const_data_ptr<int32_t>(), *out_maps = m.map.out_maps.const_data_ptr<int32_t>();
    void* stream = stream_of(x);
    if (m.groups) {
      const Tensor ws = bytes_on(wcn_depthwise_wgrad_grouped_workspace_bytes(K, c, n_out), x);
      if (grad_bias) {
        const Tensor sums = bytes_on(wcn_column_sums_workspace_bytes(c), x);
        check(wcn_sparse_depthwise_wgrad_grouped_bias(x.const_data_ptr(), n_in, gy.const_data_ptr(), n_out, c, code, in_maps, out_maps,
                                                      m.device_offsets.const_data_ptr<int64_t>(), m.groups, K, iden,
                                                      grad_w.mutable_data_ptr(), dtype_code(w.scalar_type()),
                                                      ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()),
                                                      grad_bias->mutable_data_ptr(), dtype_code(grad_bias->scalar_type()),
                                                      sums.mutable_data_ptr(), static_cast<size_t>(sums.numel()), stream),
              "wcn_sparse_depthwise_wgrad_grouped_bias");
      } else check(wcn_sparse_depthwise_wgrad_grouped(x.const_data_ptr(), n_in, gy.const_data_ptr(), n_out, c, code, in_maps, out_maps,
                                               m.device_offsets.const_data_ptr<int64_t>(), m.groups, K, iden,
                                               grad_w.mutable_data_ptr(), dtype_code(w.scalar_type()), ws.mutable_data_ptr(),
                                               static_cast<size_t>(ws.numel()), stream),
            "wcn_sparse_depthwise_wgrad_grouped");
    } else {
      const int64_t identity_rows = iden >= 0 ? std::min(n_in, n_out) : 0;
      const Tensor ws = bytes_on(wcn_depthwise_wgrad_workspace_bytes(K, c, m.map.pairs(), identity_rows), x);
      check(wcn_sparse_depthwise_wgrad(x.const_data_ptr(), n_in, gy.const_data_ptr(), n_out, c, code, in_maps, out_maps,
                                       m.map.host_offsets(), K, iden, grad_w.mutable_data_ptr(), dtype_code(w.scalar_type()),
                                       ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()), stream),
            "wcn_sparse_depthwise_wgrad");
    }
    grad_w = grad_w.to(weight.scalar_type());
  }
  return {grad_x, grad_w};
}

void check_depthwise(const Tensor& features, const Tensor& weight, const RowsMap& m) {
  if (features.dim() != 2 || weight.dim() != 2 || weight.size(1) != features.size(1) || weight.size(0) != m.map.K)
    throw py::value_error("shape mismatch: features " + shape_text(features) + ", weight " + shape_text(weight) + ", " +
                          std::to_string(m.map.K) + " offsets");
  check_weight_device(weight, features);
}

Tensor depthwise_forward(const Tensor& features, const Tensor& weight, const py::object& km, int64_t num_out,
                         const std::optional<at::ScalarType>& compute_dtype) {
  const at::ScalarType dtype = compute_dtype.value_or(features.scalar_type());
  check_rows_features(features, dtype, "in_features");
  const RowsMap m(km, features.size(0), num_out);
  check_depthwise(features, weight, m);
  return depthwise_out(features, weight, Tensor(), m, num_out, dtype);
}

py::tuple depthwise_backward(const Tensor& grad_output, const Tensor& in_features, const Tensor& weight, const py::object& km,
                             const std::optional<at::ScalarType>& compute_dtype, bool need_x, bool need_w) {
  at::AutoDispatchBelowADInplaceOrView guard;
  const RowsMap m(km, in_features.size(0), grad_output.size(0));
  auto r = depthwise_grads(grad_output, in_features, weight, m, compute_dtype.value_or(in_features.scalar_type()), need_x, need_w);
  return py::make_tuple(r.first.defined() ? py::cast(r.first) : py::none(), r.second.defined() ? py::cast(r.second) : py::none());
}

struct DepthwiseBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable x_, w_;
  std::unique_ptr<RowsMap> map_;
  at::ScalarType dtype_{}, bias_dtype_{};
  bool has_bias_ = false;

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    torch::autograd::variable_list out(has_bias_ ? 3 : 2);
    if (!grads[0].defined()) return out;
    TORCH_CHECK(map_ != nullptr, "Trying to backward through the graph a second time (the map was given back after the first)");
    const Tensor x = x_.unpack(shared_from_this()), w = w_.unpack(shared_from_this());
    at::NoGradGuard no_grad;
    const bool need_w = task_should_compute_output(1), need_b = has_bias_ && task_should_compute_output(2);
    const bool joined = need_b && need_w && map_->groups && grads[0].scalar_type() == dtype_ && dtype_code(bias_dtype_) >= 0;
    if (joined) out[2] = at::empty({grads[0].size(1)}, grads[0].options().dtype(bias_dtype_));
    auto r = depthwise_grads(grads[0], x, w, *map_, dtype_, task_should_compute_output(0), need_w, joined ? &out[2] : nullptr);
    out[0] = r.first;
    out[1] = r.second;
    if (need_b && !joined) out[2] = column_sums(grads[0], bias_dtype_);
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x_.reset_data();
    w_.reset_data();
    map_.reset();
  }
  std::string name() const override { return "SparseDepthwiseConvBackward"; }
};

bool in_graph(std::initializer_list<const Tensor*> tensors) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : tensors)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

/* The depthwise convolution, with its gradients as one graph node. */
Tensor depthwise_autograd(const Tensor& features, const Tensor& weight, const std::optional<Tensor>& bias,
                          const py::object& km, int64_t num_out, const std::optional<at::ScalarType>& compute_dtype) {
  const at::ScalarType dtype = compute_dtype.value_or(features.scalar_type());
  check_rows_features(features, dtype, "in_features");
  refuse_tangents({&features, &weight}, "the sparse depthwise convolution");
  auto m = std::make_unique<RowsMap>(km, features.size(0), num_out);
  check_depthwise(features, weight, *m);
  const bool given = bias && bias->defined(), has_bias = given && kernel_bias(*bias, features, weight.size(1));
  const Tensor b = has_bias ? *bias : Tensor();
  Tensor out = depthwise_out(features, weight, b, *m, num_out, dtype);
  auto with_bias = [&]() { return given && !has_bias ? out + bias->to(out.scalar_type()) : out; };
  if (!in_graph({&features, &weight, &b})) return with_bias();
  auto node = std::shared_ptr<DepthwiseBackward>(new DepthwiseBackward(), torch::autograd::deleteNode);
  node->set_next_edges(b.defined() ? torch::autograd::collect_next_edges(features, weight, b)
                                   : torch::autograd::collect_next_edges(features, weight));
  node->x_ = torch::autograd::SavedVariable(features, false);
  node->w_ = torch::autograd::SavedVariable(weight, false);
  node->dtype_ = dtype;
  node->has_bias_ = b.defined();
  if (b.defined()) node->bias_dtype_ = b.scalar_type();
  node->map_ = std::move(m);
  torch::autograd::set_history(out, node);
  return with_bias();
}

struct PoolBackward : public torch::autograd::Node {
  std::unique_ptr<RowsMap> map_;
  Tensor arg_;
  int64_t n_in_ = 0;
  int32_t mode_ = 0;
  bool single_in_ = false;  // every input row is in exactly one pair

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    torch::autograd::variable_list out(1);
    if (!grads[0].defined()) return out;
    TORCH_CHECK(map_ != nullptr, "Trying to backward through the graph a second time (the map was given back after the first)");
    at::NoGradGuard no_grad;
    const Tensor gy = grads[0].contiguous();
    const int32_t c = static_cast<int32_t>(gy.size(1));
    const MapRef& map = map_->map;
    if (n_in_ == 0 || gy.size(0) == 0) {
      out[0] = at::zeros({n_in_, c}, gy.options());
      return out;
    }
    const bool spread = single_in_ && map.pairs() == n_in_;
    const Tensor by_in = spread ? Tensor() : map_->by_in(n_in_);
    Tensor gx = at::empty({n_in_, c}, gy.options());
    check(wcn_sparse_pool_bwd_offsets(gy.const_data_ptr(), gy.size(0), c, dtype_code(gy.scalar_type()),
                                      spread ? nullptr : by_in.const_data_ptr(), map_->by_out.const_data_ptr(), n_in_, map.K,
                                      map.pairs(), mode_, arg_.defined() ? arg_.const_data_ptr() : nullptr,
                                      gx.mutable_data_ptr(), stream_of(gy)),
          "wcn_sparse_pool_bwd");
    out[0] = gx;
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    map_.reset();
    arg_ = Tensor();
  }
  std::string name() const override { return "SparsePoolBackward"; }
};

/* Pooling over a map (mode as in wcn_sparse_pool_fwd), with its gradient as one graph node. */
Tensor pool_autograd(const Tensor& features, const py::object& km, int64_t num_out, int32_t mode, bool single_in) {
  check_rows_features(features, features.scalar_type(), "features");
  refuse_tangents({&features}, "sparse pooling");
  auto m = std::make_unique<RowsMap>(km, features.size(0), num_out);
  const bool graph = in_graph({&features});
  const int32_t c = static_cast<int32_t>(features.size(1));
  Tensor out, arg;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    const Tensor x = features.contiguous();
    if (num_out == 0 || x.size(0) == 0) {
      out = at::zeros({num_out, c}, x.options());
    } else {
      out = at::empty({num_out, c}, x.options());
      if (graph && mode >= 2) arg = bytes_on(static_cast<size_t>(num_out) * c * wcn_pool_offset_bytes(m->map.K), x);
      check(wcn_sparse_pool_fwd_offsets(x.const_data_ptr(), x.size(0), c, dtype_code(x.scalar_type()),
                                        m->by_out.const_data_ptr(), num_out, m->map.K, m->map.pairs(), mode,
                                        out.mutable_data_ptr(), arg.defined() ? arg.mutable_data_ptr() : nullptr, stream_of(x)),
            "wcn_sparse_pool_fwd");
    }
  }
  if (!graph) return out;
  auto node = std::shared_ptr<PoolBackward>(new PoolBackward(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(features));
  node->arg_ = arg;
  node->n_in_ = features.size(0);
  node->mode_ = mode;
  node->single_in_ = single_in;
  node->map_ = std::move(m);
  torch::autograd::set_history(out, node);
  return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::class_<MadeOn, std::shared_ptr<MadeOn>>(m, "MadeOn")
      .def("before_use", [](const MadeOn& made, const Tensor& a, const Tensor& b, const Tensor& c) { made.before_use({&a, &b, &c}); });
  // behind what the current stream of a tensor's device has been given; None inside a capture
  m.def("made_now", [](const Tensor& t) {
    void* stream = stream_of(t);
    return MadeOn::capturing(stream) ? nullptr : std::make_shared<MadeOn>(stream);
  });
  py::class_<PreparedWeight, std::shared_ptr<PreparedWeight>>(m, "PreparedWeight");
  m.def("batch_rows", &batch_rows);
  m.def("batch_rows_table", &batch_rows_table);
  m.def("table_build", &table_build);
  m.def("stride_cells", &stride_cells);
  py::class_<LayerAhead>(m, "LayerAhead")
      .def(py::init([](const Tensor& features, const py::object& weight, const std::optional<Tensor>& bias,
                       const std::optional<at::ScalarType>& compute_dtype, const std::optional<Tensor>& residual, bool relu,
                       bool keep_tiles, bool graph) {
        return LayerAhead{features, weight, bias, residual, compute_dtype, relu, keep_tiles, graph, -1, Tensor()};
      }), py::arg("features"), py::arg("weight"), py::arg("bias"), py::arg("compute_dtype"), py::arg("residual"), py::arg("relu"),
           py::arg("keep_tiles"), py::arg("graph") = false)
      .def_property("identity", [](const LayerAhead& a) { return a.identity; },
                    [](LayerAhead& a, std::optional<int64_t> k) { a.identity = k.value_or(-1); })
      .def_property_readonly("out", [](const LayerAhead& a) { return a.out.defined() ? py::cast(a.out) : py::none(); });
  m.def("kernel_map", &kernel_map, py::arg("table"), py::arg("rows"), py::arg("kernel_size"), py::arg("stride"), py::arg("dilation"),
        py::arg("centre"), py::arg("per_row"), py::arg("keep_workspace_bytes"), py::arg("ahead") = py::none());
  m.def("conv_forward", [](const Tensor& features, const py::object& weight, const py::object& km, int64_t num_out,
                           const std::optional<Tensor>& bias, const std::optional<at::ScalarType>& compute_dtype,
                           const std::optional<Tensor>& residual, bool relu, bool keep_tiles, const py::object& pairs_sorted) {
    return conv_forward(features, weight, km, num_out, bias, compute_dtype, residual, relu, keep_tiles, pairs_sorted, false);
  });
  m.def("pointwise_forward", [](const Tensor& features, const Tensor& weight, const std::optional<Tensor>& bias) -> py::object {
    const Tensor out = pointwise_forward(features, weight, bias);
    return out.defined() ? py::cast(out) : py::none();
  });
  m.def("conv_backward", &conv_backward);
  m.def("conv_autograd", &conv_autograd, py::arg("features"), py::arg("weight"), py::arg("bias"), py::arg("km"), py::arg("num_out"),
        py::arg("compute_dtype"), py::arg("pairs_sorted"), py::arg("ahead") = py::none());
  m.def("depthwise_forward", &depthwise_forward);
  m.def("depthwise_backward", &depthwise_backward);
  m.def("depthwise_autograd", &depthwise_autograd);
  m.def("pool_autograd", &pool_autograd);
}
