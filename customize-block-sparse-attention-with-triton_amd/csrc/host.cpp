// The host path of the operator: what happens between a call in Python and the C ABI (include/bsattn.h), natively.
// A small call is bound by it: argument checks, result and list allocation, workspace look-up, marshalling and the
// autograd bookkeeping took 12 us per forward and over 100 us per training step in Python and ctypes.
// The library itself is reached through its C ABI only, by the path Python gives to bind().
//
// Mirrors fa2_custom_mask/fa2_custom_mask.py:15-155 of the reference (build_groups_from_block_mask's lists, _attention).
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <dlfcn.h>
#include <algorithm>
#include <climits>
#include <list>
#include <mutex>
#include "bsattn.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

namespace {

// ---- the library ----
struct Library {
  decltype(&::bsattn_strerror) strerror_ = nullptr;
  decltype(&::bsattn_mask_lists_workspace) lists_workspace = nullptr;
  decltype(&::bsattn_block_mask_to_lists) lists = nullptr;
  decltype(&::bsattn_gather_mask_tiles) gather = nullptr;
  decltype(&::bsattn_fwd_workspace) fwd_workspace = nullptr;
  decltype(&::bsattn_fwd_tokens) fwd = nullptr;
  decltype(&::bsattn_fwd_block_mask_workspace) fwd_block_mask_workspace = nullptr;
  decltype(&::bsattn_fwd_block_mask_tokens) fwd_block_mask = nullptr;
  decltype(&::bsattn_fwd_takes_mask) fwd_takes_mask = nullptr;
  decltype(&::bsattn_fwd_mask_copy_tokens) fwd_mask = nullptr;
  decltype(&::bsattn_bwd_workspace) bwd_workspace = nullptr;
  decltype(&::bsattn_bwd_tokens) bwd = nullptr;
  decltype(&::bsattn_reorder_inplace_workspace) reorder_workspace = nullptr;
  decltype(&::bsattn_reorder_inplace) reorder = nullptr;
} lib;

void bind(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h != nullptr, "cannot load ", path, ": ", dlerror());
  auto get = [&](auto& f, const char* name) {
    f = reinterpret_cast<std::decay_t<decltype(f)>>(dlsym(h, name));
    TORCH_CHECK(f != nullptr, path, " has no ", name);
  };
  get(lib.strerror_, "bsattn_strerror");
  get(lib.lists_workspace, "bsattn_mask_lists_workspace");
  get(lib.lists, "bsattn_block_mask_to_lists");
  get(lib.gather, "bsattn_gather_mask_tiles");
  get(lib.fwd_workspace, "bsattn_fwd_workspace");
  get(lib.fwd, "bsattn_fwd_tokens");
  get(lib.fwd_block_mask_workspace, "bsattn_fwd_block_mask_workspace");
  get(lib.fwd_block_mask, "bsattn_fwd_block_mask_tokens");
  get(lib.fwd_takes_mask, "bsattn_fwd_takes_mask");
  get(lib.fwd_mask, "bsattn_fwd_mask_copy_tokens");
  get(lib.bwd_workspace, "bsattn_bwd_workspace");
  get(lib.bwd, "bsattn_bwd_tokens");
  get(lib.reorder_workspace, "bsattn_reorder_inplace_workspace");
  get(lib.reorder, "bsattn_reorder_inplace");
}

void check(int rc, const char* what) {
  if (rc != 0) throw std::runtime_error(std::string(what) + " failed: " + lib.strerror_(rc) + " (code " + std::to_string(rc) + ")");
}

int dtype_code(at::ScalarType t) {
  if (t == at::kHalf) return BSATTN_F16;
  if (t == at::kBFloat16) return BSATTN_BF16;
  if (t == at::kFloat) return BSATTN_F32;
  throw py::type_error(std::string("unsupported dtype ") + toString(t));
}

constexpr int64_t TILE = BSATTN_TILE;
int64_t whole(int64_t n) { return (n + TILE - 1) / TILE * TILE; }

hipStream_t stream_of(const Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

// ---- workspaces ----
// Scratch memory for one call, kept per (device, stream) and reused by the next call on that stream: the kernels need no
// particular contents on entry, and what is enqueued on one stream runs in order.  The lock is held while a call is
// enqueued, so that the launches of two threads on one stream, which share a workspace, do not interleave.  The token
// reorder, whose one launch is not made under the lock, has a workspace of its own: it may land between the launches of
// an attention call.  Bounded: the least recently used workspace goes first, one above WORKSPACE_CACHE_BYTES is not
// kept.  Nothing is kept or taken from the cache while the stream is being captured: memory first allocated under
// capture belongs to the graph's pool.
constexpr size_t WORKSPACE_CACHE_STREAMS = 8, WORKSPACE_CACHE_BYTES = (size_t)256 << 20;
enum class Use { attention, reorder };
struct Kept { int device; hipStream_t stream; Use use; Tensor memory; };
std::mutex workspace_mutex;
// The lock, waited for without the GIL: its holder may need the GIL (backward runs on threads that do not have it).
struct WorkspaceLock {
  std::unique_lock<std::mutex> lock{workspace_mutex, std::try_to_lock};
  WorkspaceLock() {
    if (lock.owns_lock()) return;
    if (PyGILState_Check()) {
      py::gil_scoped_release release;
      lock.lock();
    } else {
      lock.lock();
    }
  }
};
std::list<Kept>& workspaces() {       // most recently used last (never destroyed: tensors must not outlive the runtime)
  static auto* list = new std::list<Kept>;
  return *list;
}

Tensor workspace_locked(size_t bytes, at::Device device, hipStream_t stream, Use use = Use::attention) {
  const auto fresh = [&] {
    return at::empty({(int64_t)std::max<size_t>(bytes, 1)}, at::TensorOptions().dtype(at::kByte).device(device));
  };
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return fresh();
  auto& kept = workspaces();
  for (auto it = kept.begin(); it != kept.end(); ++it) {
    if (it->device != device.index() || it->stream != stream || it->use != use) continue;
    if ((size_t)it->memory.numel() < bytes) { kept.erase(it); break; }
    if (std::next(it) != kept.end()) kept.splice(kept.end(), kept, it);
    return kept.back().memory;
  }
  Tensor t = fresh();
  if (bytes <= WORKSPACE_CACHE_BYTES) {
    kept.push_back({device.index(), stream, use, t});
    while (kept.size() > WORKSPACE_CACHE_STREAMS) kept.pop_front();
  }
  return t;
}

void clear_workspaces() {
  const WorkspaceLock lock;
  workspaces().clear();
}

// ---- kept-tile lists ----
// Of a block mask [Bm, Hm, nb, nb] (fixed shapes, no host synchronisation): row_ptr int32 [Bm*Hm*nb+1], col_idx int32
// [Bm*Hm*nb*nb] (first T entries valid), counts int32 [2] = (G, T), groups int32 [Bm*Hm*nb, 5] (first G rows valid) or
// none, all in one int32 buffer (workspace | row_ptr | counts | col_idx | groups).  Elementwise masks: per kept tile the
// "partly set" flag and its packed 64 x 64 bits.
struct TileLists : torch::CustomClassHolder {
  int64_t Bm, Hm, nb, ws_bytes, off_ptr, off_counts, off_cols, off_groups;
  bool has_groups;
  Tensor buf, partial, bits;

  TileLists(int64_t Bm_, int64_t Hm_, int64_t nb_, at::Device device, bool want_groups)
      : Bm(Bm_), Hm(Hm_), nb(nb_), has_groups(want_groups) {
    size_t bytes = 0;
    check(lib.lists_workspace((int)Bm, (int)Hm, (int)nb, &bytes), "bsattn_mask_lists_workspace");
    const int64_t rows = Bm * Hm * nb;
    ws_bytes = (int64_t)bytes;
    off_ptr = (ws_bytes + 3) / 4;
    off_counts = off_ptr + rows + 1;
    off_cols = off_counts + 2;
    off_groups = off_cols + rows * nb;
    buf = at::empty({off_groups + (want_groups ? rows * 5 : 0)}, at::TensorOptions().dtype(at::kInt).device(device));
  }
  int32_t* at_(int64_t off) const { return buf.data_ptr<int32_t>() + off; }
  int32_t* row_ptr() const { return at_(off_ptr); }
  int32_t* counts() const { return at_(off_counts); }
  int32_t* col_idx() const { return at_(off_cols); }
  int32_t* groups() const { return has_groups ? at_(off_groups) : nullptr; }
  Tensor view(int64_t from, int64_t to) const { return buf.narrow(0, from, to - from); }
};
using ListsPtr = c10::intrusive_ptr<TileLists>;

ListsPtr block_mask_to_lists(const Tensor& block, bool transpose, bool want_groups) {
  c10::DeviceGuard guard(block.device());
  auto lists = c10::make_intrusive<TileLists>(block.size(0), block.size(1), block.size(2), block.device(), want_groups);
  const int64_t sm = block.stride(transpose ? 3 : 2), sn = block.stride(transpose ? 2 : 3);
  check(lib.lists((const uint8_t*)block.const_data_ptr(), (int)lists->Bm, (int)lists->Hm, (int)lists->nb, block.stride(0),
                  block.stride(1), sm, sn, lists->row_ptr(), lists->col_idx(), lists->groups(), lists->counts(),
                  lists->at_(0), (size_t)lists->ws_bytes, stream_of(block)), "bsattn_block_mask_to_lists");
  return lists;
}

// ---- q, k, v ----
void check_qkv(const Tensor& q, const Tensor& k, const Tensor& v) {
  if (!(q.is_cuda() && k.is_cuda() && v.is_cuda())) throw std::runtime_error("q, k, v must be GPU tensors (there is no CPU path)");
  if (q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes())
    throw py::value_error("q, k, v must share one shape [B, H, N, D]");            // :53-57
  const auto t = q.scalar_type();
  if ((t != at::kHalf && t != at::kBFloat16) || k.scalar_type() != t || v.scalar_type() != t)
    throw py::type_error("q, k, v must all be float16 or all bfloat16");
  const int64_t D = q.size(3);
  if (D != 16 && D != 32 && D != 64 && D != 128 && D != 256)                       // :58
    throw py::value_error("head dimension must be 16, 32, 64, 128 or 256");
  if (q.size(2) < 1) throw py::value_error("empty sequence");
}

void check_mask_heads(int64_t Bm, int64_t Hm, const Tensor& q) {
  if ((Bm != 1 && Bm != q.size(0)) || (Hm != 1 && Hm != q.size(1))) throw py::value_error("mask batch/head sizes must be 1 or match q");
}

// The kernels work on head dimensions 64, 128 and 256: smaller ones are embedded in zeros.  Zero columns change neither
// q k^T nor the real columns of the output.
Tensor padded(const Tensor& x) {
  if (x.size(3) >= 64) return x;
  Tensor p = at::zeros({x.size(0), x.size(1), x.size(2), 64}, x.options());
  p.narrow(3, 0, x.size(3)).copy_(x);
  return p;
}
Tensor unpadded(const Tensor& x, int64_t D) { return x.size(3) == D ? x : x.narrow(3, 0, D); }

// Unit stride along the head dimension, 16-byte aligned rows.
bool rows_aligned(const Tensor& x) {
  const int64_t e = x.element_size();
  return x.stride(3) == 1 && (((x.stride(0) | x.stride(1) | x.stride(2)) * e) & 15) == 0 && ((uintptr_t)x.const_data_ptr() & 15) == 0;
}
Tensor prepared(const Tensor& x) { return rows_aligned(x) ? x : x.clone(at::MemoryFormat::Contiguous); }

// A result laid out as the reference's torch.empty_like(x) lays it out (:59, 101-103): the dimension order of x by
// stride, without gaps.  For q, k, v sliced out of one packed [B, N, 3, H, D] tensor that is [B, N, H, D] order behind a
// [B, H, N, D] shape.
Tensor like(const Tensor& x, at::ScalarType dtype) {
  Tensor t = at::empty_like(x, x.options().dtype(dtype));
  return rows_aligned(t) ? t : at::empty(x.sizes(), x.options().dtype(dtype));
}

std::tuple<Tensor, Tensor> forward_core(const Tensor& q_, const Tensor& k_, const Tensor& v_, const TileLists& l, double sm_scale,
                                        at::ScalarType out_dtype, bool want_lse) {
  c10::DeviceGuard guard(q_.device());
  const Tensor q = prepared(q_), k = prepared(k_), v = prepared(v_), o = like(q, out_dtype);
  const int B = (int)q.size(0), H = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3);
  Tensor lse;
  if (want_lse) lse = at::empty({B, H, N}, q.options().dtype(at::kFloat));
  size_t bytes = 0;
  check(lib.fwd_workspace(B, H, (int)whole(N), D, &bytes), "bsattn_fwd_workspace");
  const hipStream_t stream = stream_of(q);
  const WorkspaceLock lock;
  const Tensor ws = workspace_locked(bytes, q.device(), stream);
  const bool words = l.bits.defined();          // elementwise mask: exact inside partly set tiles
  check(lib.fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.data_ptr(), want_lse ? lse.data_ptr<float>() : nullptr,
                l.row_ptr(), l.col_idx(), words ? (const uint8_t*)l.partial.const_data_ptr() : nullptr,
                words ? (const uint64_t*)l.bits.const_data_ptr() : nullptr, (int)l.Bm, (int)l.Hm, B, H, N, D,
                dtype_code(q.scalar_type()), dtype_code(out_dtype), (float)sm_scale, q.strides().data(), k.strides().data(),
                v.strides().data(), o.strides().data(), ws.data_ptr(), bytes, stream), "bsattn_fwd");
  return {o, lse};
}

std::tuple<Tensor, Tensor, Tensor> backward_core(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_,
                                                 const Tensor& do_, const Tensor& lse, const TileLists& l, const TileLists& lt,
                                                 double sm_scale, at::ScalarType out_dtype) {
  c10::DeviceGuard guard(q_.device());
  const Tensor q = prepared(q_), k = prepared(k_), v = prepared(v_), o = prepared(o_), g = prepared(do_);
  const Tensor dq = like(q, out_dtype), dk = like(k, out_dtype), dv = like(v, out_dtype);       // :101-103
  const int B = (int)q.size(0), H = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3);
  size_t bytes = 0;
  check(lib.bwd_workspace(B, H, (int)whole(N), D, &bytes), "bsattn_bwd_workspace");
  const hipStream_t stream = stream_of(q);
  const WorkspaceLock lock;
  const Tensor ws = workspace_locked(bytes, q.device(), stream);
  const bool words = l.bits.defined();
  check(lib.bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.const_data_ptr(), g.const_data_ptr(),
                lse.const_data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), l.row_ptr(), l.col_idx(), lt.row_ptr(),
                lt.col_idx(), words ? (const uint64_t*)l.bits.const_data_ptr() : nullptr,
                words ? (const uint64_t*)lt.bits.const_data_ptr() : nullptr, (int)l.Bm, (int)l.Hm, B, H, N, D,
                dtype_code(q.scalar_type()), dtype_code(out_dtype), (float)sm_scale, q.strides().data(), k.strides().data(),
                v.strides().data(), o.strides().data(), g.strides().data(), dq.strides().data(), dk.strides().data(),
                dv.strides().data(), ws.data_ptr(), bytes, stream), "bsattn_bwd");
  return {dq, dk, dv};
}

at::ScalarType result_type(const Tensor& q, bool out_fp32) { return out_fp32 ? at::kFloat : q.scalar_type(); }

py::object results(const Tensor& o, const Tensor& lse, int64_t D, bool return_lse) {
  if (return_lse) return py::make_tuple(unpadded(o, D), lse);
  return py::cast(unpadded(o, D));
}

// Forward without anything kept for a backward.
py::object forward(const Tensor& q, const Tensor& k, const Tensor& v, const ListsPtr& lists, double sm_scale, bool out_fp32,
                   bool return_lse) {
  check_qkv(q, k, v);
  check_mask_heads(lists->Bm, lists->Hm, q);
  at::NoGradGuard no_grad;
  auto [o, lse] = forward_core(padded(q), padded(k), padded(v), *lists, sm_scale, result_type(q, out_fp32), return_lse);
  return results(o, lse, q.size(3), return_lse);
}

// Lists and forward from one call into the library, for a block mask whose lists are not at hand: (results, lists).
py::tuple forward_block_mask(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& mask, double sm_scale, bool out_fp32,
                             bool return_lse) {
  check_qkv(q_, k_, v_);
  check_mask_heads(mask.size(0), mask.size(1), q_);
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(q_.device());
  const Tensor q = prepared(padded(q_)), k = prepared(padded(k_)), v = prepared(padded(v_));
  const at::ScalarType out_dtype = result_type(q, out_fp32);
  const Tensor o = like(q, out_dtype);
  const int B = (int)q.size(0), H = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3), Bm = (int)mask.size(0), Hm = (int)mask.size(1);
  auto lists = c10::make_intrusive<TileLists>(Bm, Hm, mask.size(2), q.device(), false);
  Tensor lse;
  if (return_lse) lse = at::empty({B, H, N}, q.options().dtype(at::kFloat));
  size_t bytes = 0;
  check(lib.fwd_block_mask_workspace(Bm, Hm, B, H, (int)whole(N), D, &bytes), "bsattn_fwd_block_mask_workspace");
  const hipStream_t stream = stream_of(q);
  {
    const WorkspaceLock lock;
    const Tensor ws = workspace_locked(bytes, q.device(), stream);
    check(lib.fwd_block_mask(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.data_ptr(),
                             return_lse ? lse.data_ptr<float>() : nullptr, (const uint8_t*)mask.const_data_ptr(),
                             mask.strides().data(), Bm, Hm, lists->row_ptr(), lists->col_idx(), lists->counts(), B, H, N, D,
                             dtype_code(q.scalar_type()), dtype_code(out_dtype), (float)sm_scale, q.strides().data(),
                             k.strides().data(), v.strides().data(), o.strides().data(), ws.data_ptr(), bytes, stream),
          "bsattn_fwd_block_mask");
  }
  return py::make_tuple(results(o, lse, q_.size(3), return_lse), lists);
}

// Forward straight from a block mask: (results, the mask as the forward saw it if `keep`, else None).  None where the launch needs
// the mask's lists (or the mask is on another device).
py::object forward_mask(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& mask, double sm_scale, bool out_fp32,
                        bool return_lse, bool keep) {
  check_mask_heads(mask.size(0), mask.size(1), q_);
  const int64_t D_ = q_.size(3) < 64 ? 64 : q_.size(3);
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(q_.device());
  if (mask.device() != q_.device() || lib.fwd_takes_mask((int)q_.size(0), (int)q_.size(1), (int)q_.size(2), (int)D_) == 0) return py::none();
  const Tensor q = prepared(padded(q_)), k = prepared(padded(k_)), v = prepared(padded(v_));
  const at::ScalarType out_dtype = result_type(q, out_fp32);
  const Tensor o = like(q, out_dtype);
  const int B = (int)q.size(0), H = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3);
  Tensor lse, copy;
  if (return_lse) lse = at::empty({B, H, N}, q.options().dtype(at::kFloat));
  if (keep) copy = at::empty(mask.sizes(), mask.options());
  size_t bytes = 0;
  check(lib.fwd_workspace(B, H, (int)whole(N), D, &bytes), "bsattn_fwd_workspace");
  const hipStream_t stream = stream_of(q);
  {
    const WorkspaceLock lock;
    const Tensor ws = workspace_locked(bytes, q.device(), stream);
    check(lib.fwd_mask(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.data_ptr(), return_lse ? lse.data_ptr<float>() : nullptr,
                       (const uint8_t*)mask.const_data_ptr(), mask.strides().data(), keep ? (uint8_t*)copy.data_ptr() : nullptr,
                       (int)mask.size(0), (int)mask.size(1), B, H, N, D, dtype_code(q.scalar_type()), dtype_code(out_dtype),
                       (float)sm_scale, q.strides().data(), k.strides().data(), v.strides().data(), o.strides().data(), ws.data_ptr(),
                       bytes, stream), "bsattn_fwd_mask");
  }
  return py::make_tuple(results(o, lse, q_.size(3), return_lse), keep ? py::cast(copy) : py::none());
}

// ---- autograd ----
// The column lists of an elementwise mask, which only a backward walks and which hold as many words as the row lists, are
// made by the first backward that needs them: a forward may have none.  While the words by grid position are in Python's
// cache (held weakly here) without the GIL and before the cache of lists is told, so that the GPU does not wait for it
// (a training step with a new mask, 8 heads N = 4000: 300 us, through Python 375, made in the forward 284).
struct Grid : torch::CustomClassHolder {       // of an elementwise mask: block mask, "partly set" flags, words
  using Weak = c10::weak_intrusive_ptr<c10::TensorImpl, c10::UndefinedTensorImpl>;
  Weak block, partial, bits;
  Grid(const Tensor& a, const Tensor& b, const Tensor& c) : block(a.getIntrusivePtr()), partial(b.getIntrusivePtr()), bits(c.getIntrusivePtr()) {}
};

struct PythonLists { py::object make, keep; };                     // mask_to_lists of the column lists, their cache
PythonLists* python_lists = nullptr;                               // (set once, never destroyed)

template <typename F>
auto in_python(F&& f) {
  py::gil_scoped_acquire gil;
  TORCH_CHECK(python_lists != nullptr, "the host path has not been given Python's list functions");
  try {
    return f();
  } catch (py::error_already_set& e) {       // as autograd hands Python errors on
    e.restore();
    python_error err;
    err.persist();
    throw std::move(err);
  }
}

// fresh: Python's cache does not know them yet
ListsPtr column_lists(const Tensor& mask, int64_t N, const c10::intrusive_ptr<Grid>& grid, bool& fresh) {
  if (grid) {
    const auto block = grid->block.lock(), partial = grid->partial.lock(), bits = grid->bits.lock();
    if (block.defined() && partial.defined() && bits.defined()) {
      const Tensor grid_block{block}, grid_partial{partial}, grid_bits{bits};
      ListsPtr lists = block_mask_to_lists(grid_block, true, false);
      lists->partial = at::empty_like(grid_partial);
      lists->bits = at::empty_like(grid_bits);
      check(lib.gather((const uint8_t*)grid_partial.const_data_ptr(), (const uint64_t*)grid_bits.const_data_ptr(), (int)lists->Bm, (int)lists->Hm,
                       (int)lists->nb, 1, lists->row_ptr(), lists->col_idx(), (uint8_t*)lists->partial.data_ptr(),
                       (uint64_t*)lists->bits.data_ptr(), stream_of(mask)), "bsattn_gather_mask_tiles");
      fresh = true;
      return lists;
    }
  }
  return in_python([&] { return py::cast<ListsPtr>(python_lists->make(mask, N)); });
}

// forward(q, k, v, mask, sm_scale) and backward of the reference's _attention (:43-155) for a mask given by its row lists
// (and its column lists, where they are at hand);
// two further arguments select an fp32 output and the LSE as second result.  Autograd hands gradients back in the type
// of q, k, v.
struct Attention : torch::autograd::Function<Attention> {
  static variable_list forward(AutogradContext* ctx, const Variable& q_, const Variable& k_, const Variable& v_, const Variable& mask,
                               const ListsPtr& lists, const ListsPtr& lists_t, const c10::intrusive_ptr<Grid>& grid, double sm_scale,
                               bool out_fp32, bool return_lse) {
    const Tensor q = padded(q_), k = padded(k_), v = padded(v_);
    auto [o, lse] = forward_core(q, k, v, *lists, sm_scale, result_type(q, out_fp32), true);
    const Tensor out = unpadded(o, q_.size(3));
    ctx->save_for_backward({q, k, v, out, lse, mask});                   // :89 (a mask written to before the backward is refused)
    ctx->saved_data["lists"] = c10::IValue::make_capsule(lists);
    if (lists_t) ctx->saved_data["lists_t"] = c10::IValue::make_capsule(lists_t);
    else if (grid) ctx->saved_data["grid"] = c10::IValue::make_capsule(grid);
    ctx->saved_data["sm_scale"] = sm_scale;
    if (!return_lse) return {out};                                       // :94
    ctx->mark_non_differentiable({lse});
    return {out, lse};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    at::NoGradGuard no_grad;
    const int64_t D = out.size(3);
    const auto t = q.scalar_type();
    const Tensor o = padded(out.scalar_type() == t ? out : out.to(t));
    const Tensor g = grads[0].defined() ? padded(grads[0].scalar_type() == t ? grads[0] : grads[0].to(t)) : at::zeros_like(o);
    const auto lists = c10::static_intrusive_pointer_cast<TileLists>(ctx->saved_data["lists"].toCapsule());
    const Tensor& mask = saved[5];
    ListsPtr lists_t;
    bool fresh = false;
    if (const auto at_hand = ctx->saved_data.find("lists_t"); at_hand != ctx->saved_data.end()) {
      lists_t = c10::static_intrusive_pointer_cast<TileLists>(at_hand->second.toCapsule());
    } else {
      const auto grid = ctx->saved_data.find("grid");
      lists_t = column_lists(mask, q.size(2), grid == ctx->saved_data.end() ? nullptr : c10::static_intrusive_pointer_cast<Grid>(grid->second.toCapsule()), fresh);
    }
    auto [dq, dk, dv] = backward_core(q, k, v, o, g, lse, *lists, *lists_t, ctx->saved_data["sm_scale"].toDouble(), t);
    if (fresh) in_python([&] { python_lists->keep(mask, q.size(2), true, lists_t); });
    return {unpadded(dq, D), unpadded(dk, D), unpadded(dv, D), Variable(), Variable(), Variable(), Variable(), Variable(), Variable(), Variable()};   // :155
  }
};

py::object attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, const ListsPtr& lists,
                     const ListsPtr& lists_t, const std::optional<std::tuple<Tensor, Tensor, Tensor>>& grid, double sm_scale, bool out_fp32,
                     bool return_lse) {
  check_qkv(q, k, v);
  check_mask_heads(lists->Bm, lists->Hm, q);
  c10::intrusive_ptr<Grid> weak;
  if (grid) weak = c10::make_intrusive<Grid>(std::get<0>(*grid), std::get<1>(*grid), std::get<2>(*grid));
  variable_list r = Attention::apply(q, k, v, mask, lists, lists_t, weak, sm_scale, out_fp32, return_lse);
  if (return_lse) return py::make_tuple(r[0], r[1]);
  return py::cast(r[0]);
}

// (o, lse, dq, dk, dv) in one call, in the result type
py::tuple forward_backward(const Tensor& q_, const Tensor& k_, const Tensor& v_, const ListsPtr& lists, const ListsPtr& lists_t,
                           double sm_scale, const Tensor& do_, bool out_fp32) {
  check_qkv(q_, k_, v_);
  check_mask_heads(lists->Bm, lists->Hm, q_);
  at::NoGradGuard no_grad;
  const auto t = q_.scalar_type(), out_dtype = result_type(q_, out_fp32);
  const int64_t D = q_.size(3);
  const Tensor q = padded(q_), k = padded(k_), v = padded(v_);
  auto [o, lse] = forward_core(q, k, v, *lists, sm_scale, out_dtype, true);
  const Tensor g = padded(do_.scalar_type() == t ? do_ : do_.to(t));
  auto [dq, dk, dv] = backward_core(q, k, v, o.scalar_type() == t ? o : o.to(t), g, lse, *lists, *lists_t, sm_scale, out_dtype);
  return py::make_tuple(unpadded(o, D), lse, unpadded(dq, D), unpadded(dk, D), unpadded(dv, D));
}

// ---- token reorder in place ----
// Dimensions (stride, size) around stretches of `need` elements of which no two share an element.
bool nested(std::vector<std::pair<int64_t, int64_t>> dims, int64_t need) {
  std::sort(dims.begin(), dims.end());
  for (const auto& [stride, size] : dims)
    if (size > 1) {
      if (stride < need) return false;
      need += stride * (size - 1);
    }
  return true;
}

// The image tokens (behind n_text others) of every tensor moved where they are, head by head, by the permutation numbers [heads].
// Returns the library's code, or none where it does not take the call: numbers that are not a tensor it can read, layouts, tensors
// that autograd watches, sizes that do not fit (functional.py moves those out of place, or says what is wrong).  (In Python the views,
// checks and marshalling took 15 us a call, two calls a layer: 23 heads of 2 807 tokens 33 us a pass, 19 here; 5 heads of 906 33 and 10.)
std::optional<int> reorder_inplace(const std::vector<Tensor>& tensors, const Tensor& numbers, bool inverse, int64_t F, int64_t H, int64_t W,
                                   int64_t n_text) {
  constexpr size_t MOST = 4;
  if (tensors.empty() || tensors.size() > MOST) return std::nullopt;
  const Tensor& x = tensors[0];
  if (!x.is_cuda() || x.dim() != 4 || F < 1 || H < 1 || W < 1 || F > INT_MAX || H > INT_MAX || W > INT_MAX) return std::nullopt;
  const int64_t BS = x.size(0), NH = x.size(1), T = x.size(2) - n_text, D = x.size(3), e = x.element_size();
  if (n_text < 0 || T < 1 || T > INT_MAX || F * H > T || F * H * W != T || BS < 1 || NH < 1 || D < 1) return std::nullopt;
  if (!numbers.is_cuda() || numbers.device() != x.device() || (numbers.scalar_type() != at::kLong && numbers.scalar_type() != at::kInt) ||
      numbers.dim() != 1 || numbers.size(0) != NH || !numbers.is_contiguous()) return std::nullopt;
  const bool grad = at::GradMode::is_enabled();
  std::vector<std::pair<int64_t, int64_t>> dims[MOST];
  void* ptrs[MOST];
  int64_t strides[3 * MOST];
  for (size_t i = 0; i < tensors.size(); ++i) {
    const Tensor& t = tensors[i];
    if (!t.is_cuda() || t.device() != x.device() || t.sizes() != x.sizes() || t.scalar_type() != x.scalar_type() || (grad && t.requires_grad()) ||
        t.stride(3) != 1) return std::nullopt;
    ptrs[i] = (char*)t.data_ptr() + n_text * t.stride(2) * e;
    if (((uintptr_t)ptrs[i] & 15) != 0) return std::nullopt;
    for (int d = 0; d < 3; ++d) {
      if (((t.stride(d) * e) & 15) != 0) return std::nullopt;
      strides[3 * i + d] = t.stride(d);
      dims[i].emplace_back(t.stride(d), d == 2 ? T : t.size(d));
    }
    if (!nested(dims[i], D)) return std::nullopt;
    // no row shares memory with another tensor's (those cut from one storage: the q, k, v of a packed projection)
    for (size_t j = 0; j < i; ++j) {
      if (tensors[j].storage().data() != t.storage().data()) continue;
      const int64_t apart = std::abs(t.storage_offset() - tensors[j].storage_offset());
      auto both = dims[i];
      both.emplace_back(apart, 2);
      if (t.strides() != tensors[j].strides() || apart == 0 || !nested(both, D)) return std::nullopt;
    }
  }
  const int n = (int)tensors.size();
  size_t bytes = 0;
  c10::DeviceGuard guard(x.device());
  if (BS > INT_MAX || NH > INT_MAX || D > INT_MAX || lib.reorder_workspace(n, (int)BS, (int)NH, (int)F, (int)H, (int)W, (int)D, (int)e, &bytes) != 0) return std::nullopt;
  const hipStream_t stream = stream_of(x);
  Tensor ws;
  {
    const WorkspaceLock lock;
    ws = workspace_locked(bytes, x.device(), stream, Use::reorder);
  }
  const int rc = lib.reorder(ptrs, strides, n, (int)BS, (int)NH, (int)F, (int)H, (int)W, (int)D, (int)e, numbers.const_data_ptr(),
                             (int)numbers.element_size(), inverse ? 1 : 0, ws.data_ptr(), bytes, stream);
  if (rc == 0)
    for (const Tensor& t : tensors)
      if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
  return rc;
}

std::optional<Tensor> defined_or_none(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("bind", &bind);
  m.def("check_qkv", [](const Tensor& q, const Tensor& k, const Tensor& v) { check_qkv(q, k, v); return q.size(2); });
  m.def("clear_workspaces", &clear_workspaces);
  m.def("reorder_workspace", [](size_t bytes, const Tensor& like) {
    const WorkspaceLock lock;
    // (a view: the kept tensor itself never has a Python object, so it can be dropped without the GIL)
    return workspace_locked(bytes, like.device(), stream_of(like), Use::reorder).view({-1});
  });
  m.def("reorder_inplace", &reorder_inplace);
  m.def("block_mask_to_lists", &block_mask_to_lists);
  m.def("forward", &forward);
  m.def("forward_block_mask", &forward_block_mask);
  m.def("forward_mask", &forward_mask);
  m.def("attention", &attention, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("mask"), py::arg("lists"),
        py::arg("lists_t").none(true), py::arg("grid"), py::arg("sm_scale"), py::arg("out_fp32"), py::arg("return_lse"));
  m.def("set_python_lists", [](py::object make, py::object keep) { python_lists = new PythonLists{std::move(make), std::move(keep)}; });
  m.def("forward_backward", &forward_backward);
  py::class_<TileLists, ListsPtr>(m, "TileLists")
      .def(py::init([](int64_t Bm, int64_t Hm, int64_t nb, py::object device, bool want_groups) {
             return c10::make_intrusive<TileLists>(Bm, Hm, nb, at::Device(py::cast<std::string>(py::str(device))), want_groups);
           }), py::arg("Bm"), py::arg("Hm"), py::arg("nb"), py::arg("device"), py::arg("want_groups") = false)
      .def_readonly("Bm", &TileLists::Bm)
      .def_readonly("Hm", &TileLists::Hm)
      .def_readonly("nb", &TileLists::nb)
      .def_readonly("buf", &TileLists::buf)
      .def_readonly("has_groups", &TileLists::has_groups)
      .def_property("partial", [](const TileLists& l) { return defined_or_none(l.partial); },
                    [](TileLists& l, const std::optional<Tensor>& t) { l.partial = t ? *t : Tensor(); })
      .def_property("bits", [](const TileLists& l) { return defined_or_none(l.bits); },
                    [](TileLists& l, const std::optional<Tensor>& t) { l.bits = t ? *t : Tensor(); })
      .def_property_readonly("row_ptr", [](const TileLists& l) { return l.view(l.off_ptr, l.off_counts); })
      .def_property_readonly("counts", [](const TileLists& l) { return l.view(l.off_counts, l.off_cols); })
      .def_property_readonly("col_idx", [](const TileLists& l) { return l.view(l.off_cols, l.off_groups); })
      .def_property_readonly("groups", [](const TileLists& l) {
        return l.has_groups ? std::optional<Tensor>(l.view(l.off_groups, l.buf.size(0)).view({-1, 5})) : std::nullopt;
      })
      .def_property_readonly("row_ptr_ptr", [](const TileLists& l) { return (uintptr_t)l.row_ptr(); })
      .def_property_readonly("col_idx_ptr", [](const TileLists& l) { return (uintptr_t)l.col_idx(); });
}
