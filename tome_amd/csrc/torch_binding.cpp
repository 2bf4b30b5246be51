// Host side of the operators on torch tensors: argument checks, output and workspace allocation and the C-ABI call in
// native code.  The launches of a decode-sized call take 5-10 us on the GPU; in Python the same work (a dozen torch calls, two
// ctypes calls) took 15-21 us a call and was what such a call cost (8 x 151936 fp32: 21.6 us a call, the kernels 7.5).
// Nothing is kept between calls.  The stream is torch's current one, passed by the caller as a raw handle; no HIP headers
// are needed here.
// The operators run without the GIL: a mask, lengths or uniforms in host memory are copied to the GPU in the call, and such a
// copy waits for all work queued on the stream before it.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/utils/pybind.h>

#include <cstring>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/tome_logprob.h"

namespace py = pybind11;
using at::Tensor;
typedef std::optional<Tensor> MaybeTensor;

namespace {

std::string str(const c10::Device& d) { return d.str(); }

void require_gpu(const Tensor& t) {
  if (!t.is_cuda())
    throw std::runtime_error("tome_amd operators run on a ROCm GPU only (there is no CPU fallback); got a tensor on " + str(t.device()));
}
void require_same(const Tensor& t, const c10::Device& dev) {
  require_gpu(t);
  if (t.device() != dev) throw py::value_error("all tensors must be on the same device");
}

int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return TOME_F32;
  if (t.scalar_type() == at::kBFloat16) return TOME_BF16;
  throw py::type_error(std::string("logits must be float32 or bfloat16, got ") + c10::toString(t.scalar_type()));
}

// Status codes become the exceptions of tome_amd._lib.check.
void check(int code) {
  if (code == TOME_OK) return;
  py::gil_scoped_acquire gil;
  py::module_::import("tome_amd._lib").attr("check")(code);
}

// [..., V] -> [rows, V] with unit stride along V, copying only when no such view exists.
Tensor rows_view(const Tensor& x) {
  if (x.dim() == 0) throw py::value_error("expected a tensor with a vocabulary axis");
  const int64_t V = x.size(-1);
  Tensor y = x.stride(-1) != 1 && V > 1 ? x.contiguous() : x;
  if (y.dim() == 2) return y;
  if (y.dim() == 1) return y.unsqueeze(0);
  int64_t rows = 1;
  for (int64_t d = 0; d + 1 < y.dim(); ++d) rows *= y.size(d);
  return y.reshape({rows, V});
}

// Outputs of `n` rows take the leading shape of the input; `v` is already of that shape for [rows, V] inputs.
Tensor shaped(const Tensor& v, const Tensor& like) {
  if (like.dim() == 2) return v;
  return v.view(like.sizes().slice(0, like.dim() - 1));
}
MaybeTensor shaped(const MaybeTensor& v, const Tensor& like) { return v ? MaybeTensor(shaped(*v, like)) : v; }

// Integer ids of `n` entries on `dev`, int32 or int64 as they are, other integer types as int32.
Tensor ids_of(const Tensor& t, int64_t n, const c10::Device& dev, const char* what) {
  if (t.device() != dev) throw py::value_error(std::string(what) + " must be on " + str(dev));
  if (t.numel() != n)
    throw py::value_error(std::string(what) + " has " + std::to_string(t.numel()) + " entries, expected " + std::to_string(n));
  const auto st = t.scalar_type();
  if (!at::isIntegralType(st, /*includeBool=*/false)) throw py::type_error(std::string(what) + " must be an integer tensor");
  if (st == at::kInt || st == at::kLong) return t.contiguous();
  return t.to(at::kInt).contiguous();
}

// TomeRowSel and the tensors it points into.
struct Sel {
  TomeRowSel c{};
  Tensor targets, mask;

  Sel(const MaybeTensor& tg, const MaybeTensor& lengths, const MaybeTensor& row_valid, const Tensor& like, int64_t n,
      const c10::Device& dev) {
    if (lengths && row_valid) throw py::value_error("pass lengths or row_valid, not both");
    if (tg) {
      targets = ids_of(*tg, n, dev, "targets");
      c.targets = targets.data_ptr();
      c.target_bytes = (int32_t)targets.element_size();
    }
    if (row_valid) {
      if (row_valid->numel() != n)
        throw py::value_error("row_valid has " + std::to_string(row_valid->numel()) + " entries, expected " + std::to_string(n));
      const auto st = row_valid->scalar_type();
      const bool as_is = st == at::kBool || st == at::kByte || st == at::kChar || st == at::kInt || st == at::kLong;
      mask = row_valid->device() == dev && as_is ? row_valid->contiguous() : row_valid->to(dev, at::kInt).contiguous();
      c.row_valid = mask.data_ptr();
      c.valid_bytes = (int32_t)mask.element_size();
    } else if (lengths) {
      if (like.dim() != 3) throw py::value_error("lengths needs inputs shaped [batch, seq, ...]");
      if (lengths->numel() != like.size(0))
        throw py::value_error("lengths has " + std::to_string(lengths->numel()) + " entries, expected " + std::to_string(like.size(0)));
      const auto st = lengths->scalar_type();
      mask = lengths->device() == dev && (st == at::kInt || st == at::kLong) ? lengths->contiguous()
                                                                             : lengths->to(dev, at::kLong).contiguous();
      c.lengths = mask.data_ptr();
      c.length_bytes = (int32_t)mask.element_size();
      c.seq_len = like.size(1) > 0 ? like.size(1) : 1;
    }
  }
};

Tensor workspace(size_t bytes, const at::TensorOptions& o) {
  return bytes > 0 ? at::empty({(int64_t)bytes}, o.dtype(at::kByte)) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
template <typename T>
T* ptr(const MaybeTensor& t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }
MaybeTensor maybe_empty(bool want, int64_t n, const at::TensorOptions& o) {
  return want ? MaybeTensor(at::empty({n}, o)) : MaybeTensor();
}
void* stream_ptr(uintptr_t s) { return reinterpret_cast<void*>(s); }

typedef std::tuple<Tensor, MaybeTensor, MaybeTensor, MaybeTensor> RowOutputs;  // lp, lse, entropy, argmax

RowOutputs token_logprobs(const Tensor& logits, const Tensor& targets, double temperature, const MaybeTensor& lengths,
                          const MaybeTensor& row_valid, bool want_lse, bool want_entropy, bool want_argmax, uintptr_t stream) {
  require_gpu(logits);
  const c10::Device dev = logits.device();
  const int dtype = dtype_code(logits);
  const Tensor x = rows_view(logits);
  const int64_t rows = x.size(0), V = x.size(1);
  c10::DeviceGuard guard(dev);
  const Sel sel(targets, lengths, row_valid, logits, rows, dev);
  const at::TensorOptions f32 = at::TensorOptions().dtype(at::kFloat).device(dev), i32 = f32.dtype(at::kInt);
  Tensor lp = at::empty({rows}, f32);
  MaybeTensor lse = maybe_empty(want_lse, rows, f32), ent = maybe_empty(want_entropy, rows, f32), amax = maybe_empty(want_argmax, rows, i32);
  const size_t bytes = tome_row_logprob_workspace(rows, V);
  const Tensor ws = workspace(bytes, f32);
  check(tome_row_logprob_sel(x.data_ptr(), dtype, rows, V, rows > 1 ? x.stride(0) : V, &sel.c, (float)temperature,
                             lp.data_ptr<float>(), ptr<float>(lse), ptr<float>(ent), ptr<int32_t>(amax), ptr(ws), bytes,
                             stream_ptr(stream)));
  return {shaped(lp, logits), shaped(lse, logits), shaped(ent, logits), shaped(amax, logits)};
}

RowOutputs token_logprobs_rows(const Tensor& logits, const Tensor& row_index, const Tensor& targets, double temperature,
                               bool want_lse, bool want_entropy, bool want_argmax, uintptr_t stream) {
  require_gpu(logits);
  const c10::Device dev = logits.device();
  const int dtype = dtype_code(logits);
  const Tensor x = rows_view(logits);
  const int64_t rows = x.size(0), V = x.size(1), n = row_index.numel();
  c10::DeviceGuard guard(dev);
  const Tensor idx = ids_of(row_index, n, dev, "row_index").to(at::kInt), tg = ids_of(targets, n, dev, "targets").to(at::kInt);
  const at::TensorOptions f32 = at::TensorOptions().dtype(at::kFloat).device(dev), i32 = f32.dtype(at::kInt);
  Tensor lp = at::empty({n}, f32);
  MaybeTensor lse = maybe_empty(want_lse, n, f32), ent = maybe_empty(want_entropy, n, f32), amax = maybe_empty(want_argmax, n, i32);
  const size_t bytes = tome_row_logprob_workspace(n, V);
  const Tensor ws = workspace(bytes, f32);
  check(tome_row_logprob_rows(x.data_ptr(), dtype, rows, V, rows > 1 ? x.stride(0) : V, idx.data_ptr<int32_t>(), n,
                              tg.data_ptr<int32_t>(), (float)temperature, lp.data_ptr<float>(), ptr<float>(lse), ptr<float>(ent),
                              ptr<int32_t>(amax), ptr(ws), bytes, stream_ptr(stream)));
  return {lp, lse, ent, amax};
}

// token, lp, argmax (rows of one allocation, in this order), candidate ids and logits; `mask` int32
std::tuple<Tensor, Tensor, Tensor, MaybeTensor, MaybeTensor> sample_tokens(const Tensor& logits, double temperature, int64_t top_k,
                                                                           const MaybeTensor& uniforms, const MaybeTensor& mask,
                                                                           bool want_topk, uintptr_t stream) {
  require_gpu(logits);
  const c10::Device dev = logits.device();
  const int dtype = dtype_code(logits);
  const Tensor x = rows_view(logits);
  const int64_t rows = x.size(0), V = x.size(1);
  if (top_k < 1 || top_k > 32) throw py::value_error("top_k must be in 1..32");
  c10::DeviceGuard guard(dev);
  if (mask) require_same(*mask, dev);
  Tensor u;
  if (uniforms) {
    u = uniforms->to(dev, at::kFloat).contiguous();
    if (u.numel() != rows)
      throw py::value_error("uniforms must have one value per row (" + std::to_string(rows) + "), got " + std::to_string(u.numel()));
  }
  const at::TensorOptions i32 = at::TensorOptions().dtype(at::kInt).device(dev);
  const Tensor packed = at::empty({3, rows}, i32);
  const Tensor tok = packed.select(0, 0), lp = packed.select(0, 1).view(at::kFloat), amax = packed.select(0, 2);
  MaybeTensor tki, tkl;
  if (want_topk) {
    tki = at::empty({rows, top_k}, i32);
    tkl = at::empty({rows, top_k}, i32.dtype(at::kFloat));
  }
  const size_t bytes = tome_row_sample_workspace(dtype, rows, V, (int)top_k);
  const Tensor ws = workspace(bytes, i32);
  int32_t* out = packed.data_ptr<int32_t>();
  check(tome_row_sample(x.data_ptr(), dtype, rows, V, rows > 1 ? x.stride(0) : V, u.defined() ? u.data_ptr<float>() : nullptr,
                        ptr<const int32_t>(mask), (float)temperature, (int)top_k, out,
                        reinterpret_cast<float*>(out + rows), nullptr, out + 2 * rows, ptr<int32_t>(tki), ptr<float>(tkl), ptr(ws),
                        bytes, stream_ptr(stream)));
  if (want_topk && logits.dim() != 2) {
    std::vector<int64_t> shape(logits.sizes().begin(), logits.sizes().end());
    shape.back() = top_k;
    tki = tki->view(shape);
    tkl = tkl->view(shape);
  }
  return {shaped(tok, logits), shaped(lp, logits), shaped(amax, logits), tki, tkl};
}

// One step of a decode loop: `active` int32 [rows] on the GPU (updated), `host` int32 [2, rows] in page-locked memory or on the GPU
// (receives tokens and log-probs once the stream is synchronised); both dense: the kernel is given their addresses.  `pinned`: the
// caller has allocated `host` page-locked itself (asking the runtime costs 0.2 us a call).  Returns the next step's int64 input ids.
Tensor sample_step(const Tensor& logits, double temperature, int64_t top_k, const MaybeTensor& uniforms, const Tensor& active,
                   const Tensor& host, int64_t stop_token, int64_t idle_token, bool pinned, uintptr_t stream) {
  require_gpu(logits);
  const c10::Device dev = logits.device();
  const int dtype = dtype_code(logits);
  const Tensor x = rows_view(logits);
  const int64_t rows = x.size(0), V = x.size(1);
  if (top_k < 1 || top_k > 32) throw py::value_error("top_k must be in 1..32");
  c10::DeviceGuard guard(dev);
  require_same(active, dev);
  if (active.scalar_type() != at::kInt || host.scalar_type() != at::kInt) throw py::type_error("active and host must be int32 tensors");
  if (active.numel() != rows)
    throw py::value_error("logits must have one row per sequence (" + std::to_string(active.numel()) + "), got " + std::to_string(rows));
  if (host.numel() != 2 * rows)
    throw py::value_error("host must hold two values per sequence (" + std::to_string(2 * rows) + "), got " + std::to_string(host.numel()));
  if (!active.is_contiguous() || !host.is_contiguous()) throw py::value_error("active and host must be contiguous");
  if (rows > 0 && host.device() != dev && !(host.is_cpu() && (pinned || host.is_pinned())))
    throw py::value_error("host must be page-locked memory or on " + str(dev) + ": the GPU writes to it");
  Tensor u;
  if (uniforms) {
    u = uniforms->to(dev, at::kFloat).contiguous();
    if (u.numel() != rows)
      throw py::value_error("uniforms must have one value per row (" + std::to_string(rows) + "), got " + std::to_string(u.numel()));
  }
  const Tensor next = at::empty({rows}, active.options().dtype(at::kLong));
  const size_t bytes = tome_row_sample_workspace(dtype, rows, V, (int)top_k);
  const Tensor ws = workspace(bytes, active.options());
  int32_t* out = host.data_ptr<int32_t>();
  const int32_t stop = stop_token >= 0 && stop_token <= INT32_MAX ? (int32_t)stop_token : -2;
  check(tome_row_sample_step(x.data_ptr(), dtype, rows, V, rows > 1 ? x.stride(0) : V, u.defined() ? u.data_ptr<float>() : nullptr,
                             active.data_ptr<int32_t>(), (float)temperature, (int)top_k, stop, idle_token, out,
                             reinterpret_cast<float*>(out + rows), next.data_ptr<int64_t>(), ptr(ws), bytes, stream_ptr(stream)));
  return next;
}

Tensor fused_log_softmax(const Tensor& logits, double temperature, uintptr_t stream) {
  require_gpu(logits);
  const c10::Device dev = logits.device();
  const int dtype = dtype_code(logits);
  const Tensor x = rows_view(logits);
  const int64_t rows = x.size(0), V = x.size(1);
  c10::DeviceGuard guard(dev);
  const at::TensorOptions f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
  const Tensor out = at::empty(logits.sizes(), f32.dtype(logits.scalar_type()));
  // the rows' lse, and behind it the workspace
  const size_t lse_bytes = ((size_t)rows * 4 + 255) & ~(size_t)255, bytes = tome_row_logprob_workspace(rows, V);
  const Tensor ws = at::empty({(int64_t)(lse_bytes + bytes)}, f32.dtype(at::kByte));
  char* base = static_cast<char*>(ws.data_ptr());
  check(tome_full_log_softmax(x.data_ptr(), out.data_ptr(), dtype, rows, V, rows > 1 ? x.stride(0) : V, V, (float)temperature,
                              reinterpret_cast<float*>(base), bytes > 0 ? base + lse_bytes : nullptr, bytes, stream_ptr(stream)));
  return out;
}

void check_bf16(const Tensor& hidden, const Tensor& weight) {
  if (hidden.scalar_type() != at::kBFloat16 || weight.scalar_type() != at::kBFloat16)
    throw py::type_error("hidden and lm_head weights must be bfloat16 (the reference loads bf16 weights, mlx-impl/load_weights.py:20-22)");
}
void check_weight(const Tensor& w, int64_t H) {
  if (w.dim() != 2 || w.size(1) != H)
    throw py::value_error("weight must be [V, " + std::to_string(H) + "] (rows = vocabulary, as embed_tokens.weight)");
}
Tensor unit_columns(const Tensor& w) { return w.stride(1) == 1 ? w : w.contiguous(); }
Tensor check_norm(const MaybeTensor& norm, int64_t H, const c10::Device& dev) {
  if (!norm) return Tensor();
  if (norm->scalar_type() != at::kBFloat16 || norm->dim() != 1 || norm->size(0) != H || norm->device() != dev)
    throw py::value_error("norm_weight must be a bfloat16 [" + std::to_string(H) + "] tensor on " + str(dev));
  return norm->contiguous();
}

// hidden_rows: a list of rows of the flattened hidden states; targets and outputs are then packed in list order.
RowOutputs lmhead_logprobs(const Tensor& hidden, const Tensor& weight, const Tensor& targets, double temperature,
                           const MaybeTensor& lengths, const MaybeTensor& row_valid, bool want_lse, bool want_entropy,
                           bool want_argmax, const MaybeTensor& norm_weight, double norm_eps, const MaybeTensor& hidden_rows,
                           uintptr_t stream) {
  require_gpu(hidden);
  const c10::Device dev = hidden.device();
  require_same(weight, dev);
  check_bf16(hidden, weight);
  const int64_t H = hidden.size(-1);
  check_weight(weight, H);
  const Tensor h = rows_view(hidden), w = unit_columns(weight);
  const int64_t n_rows = h.size(0), V = w.size(0), n = hidden_rows ? hidden_rows->numel() : n_rows;
  c10::DeviceGuard guard(dev);
  const Sel sel(targets, lengths, row_valid, hidden, n, dev);
  const Tensor list = hidden_rows ? ids_of(*hidden_rows, n, dev, "hidden_rows").to(at::kInt) : Tensor();
  const Tensor nw = check_norm(norm_weight, H, dev);
  const at::TensorOptions f32 = at::TensorOptions().dtype(at::kFloat).device(dev), i32 = f32.dtype(at::kInt);
  Tensor lp = at::empty({n}, f32);
  MaybeTensor lse = maybe_empty(want_lse, n, f32), ent = maybe_empty(want_entropy, n, f32), amax = maybe_empty(want_argmax, n, i32);
  const size_t bytes = nw.defined() ? tome_norm_lmhead_logprob_workspace(n, H, V) : tome_fused_lmhead_logprob_workspace(n, H, V);
  const Tensor ws = workspace(bytes, f32);
  check(tome_lmhead_logprob_sel(h.data_ptr(), static_cast<const int32_t*>(ptr(list)), n_rows, ptr(nw), (float)norm_eps, w.data_ptr(),
                                n, H, V, n_rows > 1 ? h.stride(0) : H, w.stride(0), &sel.c, (float)temperature,
                                lp.data_ptr<float>(), ptr<float>(lse), ptr<float>(ent), ptr<int32_t>(amax), ptr(ws), bytes,
                                stream_ptr(stream)));
  if (hidden_rows) return {lp, lse, ent, amax};
  return {shaped(lp, hidden), shaped(lse, hidden), shaped(ent, hidden), shaped(amax, hidden)};
}

// policy log-prob, reference log-prob, k3, policy entropy
std::tuple<Tensor, Tensor, Tensor, Tensor> grpo_pair(const Tensor& hidden_policy, const MaybeTensor& hidden_ref, const Tensor& w_policy,
                                                     const MaybeTensor& w_ref, const Tensor& targets, double temperature,
                                                     const MaybeTensor& lengths, const MaybeTensor& row_valid,
                                                     const MaybeTensor& norm_weight, double norm_eps, uintptr_t stream) {
  require_gpu(hidden_policy);
  const c10::Device dev = hidden_policy.device();
  require_same(w_policy, dev);
  check_bf16(hidden_policy, w_policy);
  const int64_t H = hidden_policy.size(-1);
  check_weight(w_policy, H);
  if (w_ref) {
    require_same(*w_ref, dev);
    check_bf16(hidden_policy, *w_ref);
    check_weight(*w_ref, H);
    if (w_ref->sizes() != w_policy.sizes()) throw py::value_error("policy and reference weights must have the same shape");
  }
  Tensor h = rows_view(hidden_policy), r = h;
  if (hidden_ref) {
    require_same(*hidden_ref, dev);
    if (hidden_ref->scalar_type() != at::kBFloat16 || hidden_ref->sizes() != hidden_policy.sizes())
      throw py::value_error("hidden_ref must be bfloat16 with hidden_policy's shape");
    r = rows_view(*hidden_ref);
  }
  Tensor wp = unit_columns(w_policy), wr = w_ref ? unit_columns(*w_ref) : wp;
  c10::DeviceGuard guard(dev);
  if (wp.stride(0) != wr.stride(0)) {
    wp = wp.contiguous();
    wr = wr.contiguous();
  }
  const int64_t n = h.size(0), V = wp.size(0);
  if (n > 1 && h.stride(0) != r.stride(0)) {
    h = h.contiguous();
    r = r.contiguous();
  }
  const Sel sel(targets, lengths, row_valid, hidden_policy, n, dev);
  const Tensor nw = check_norm(norm_weight, H, dev);
  const at::TensorOptions f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
  const Tensor lp = at::empty({n}, f32), ref_lp = at::empty({n}, f32), k3 = at::empty({n}, f32), ent = at::empty({n}, f32);
  const size_t bytes = tome_grpo_pair_workspace(n, H, V, nw.defined() ? 1 : 0);
  const Tensor ws = workspace(bytes, f32);
  check(tome_grpo_pair_sel(h.data_ptr(), r.data_ptr(), ptr(nw), (float)norm_eps, wp.data_ptr(), wr.data_ptr(), n, H, V,
                           n > 1 ? h.stride(0) : H, wp.stride(0), &sel.c, (float)temperature, lp.data_ptr<float>(),
                           ref_lp.data_ptr<float>(), k3.data_ptr<float>(), ent.data_ptr<float>(), ptr(ws), bytes, stream_ptr(stream)));
  return {shaped(lp, hidden_policy), shaped(ref_lp, hidden_policy), shaped(k3, hidden_policy), shaped(ent, hidden_policy)};
}

// ---- LoRA adapters and merge jobs --------------------------------------------------------------
// The bytes of a Python object that has some, held until the end of the scope (with the GIL).
struct ByteView {
  Py_buffer b{};
  bool held = false;
  explicit ByteView(py::handle o) {
    if (PyObject_GetBuffer(o.ptr(), &b, PyBUF_SIMPLE) != 0) throw py::error_already_set();
    held = true;
  }
  ByteView(ByteView&& o) noexcept : b(o.b), held(o.held) { o.held = false; }
  ByteView(const ByteView&) = delete;
  ~ByteView() {
    if (held) PyBuffer_Release(&b);
  }
};

// `n` elements as the two-dimensional `shape`, of which one extent may be -1 (numpy's reshape).
std::pair<int64_t, int64_t> matrix_shape(int64_t n, std::vector<int64_t> shape) {
  int64_t known = 1, open = -1;
  for (size_t i = 0; i < shape.size(); ++i) {
    if (shape[i] == -1 && open < 0) open = (int64_t)i;
    else if (shape[i] < 0 || (shape[i] > 0 && known > INT64_MAX / shape[i])) throw py::value_error("bad adapter shape");
    else known *= shape[i];
  }
  if (open >= 0) {
    if (known == 0 || n % known != 0) throw py::value_error("adapter bytes do not fill the stated shape");
    shape[open] = n / known;
    known = n;
  }
  if (known != n) throw py::value_error("adapter bytes do not fill the stated shape");
  if (shape.size() != 2) throw py::value_error("lora_A and lora_B do not form a rank decomposition");
  return {shape[0], shape[1]};
}

struct Staged {  // one matrix: source, and its place (zero-padded to out_rows x out_cols) in the staging buffer
  const uint16_t* src;
  int64_t rows, cols, out_rows, out_cols, off;
  int64_t size() const { return out_rows * out_cols; }
  void copy_to(uint16_t* stage) const {
    uint16_t* dst = stage + off;
    if (cols == out_cols) {
      std::memcpy(dst, src, (size_t)(rows * cols) * 2);
      std::memset(dst + rows * cols, 0, (size_t)((out_rows - rows) * cols) * 2);
      return;
    }
    for (int64_t r = 0; r < rows; ++r) {
      std::memcpy(dst + r * out_cols, src + r * cols, (size_t)cols * 2);
      std::memset(dst + r * out_cols + cols, 0, (size_t)(out_cols - cols) * 2);
    }
  }
};

// Adapters as they came over the wire - (lora_A bytes, its shape, lora_B bytes, its shape), raw bf16 - to `dev`: one buffer, every
// matrix on a 16-byte boundary, the rank zero-padded to a multiple of 8 (extra terms of the product are exact zeros).
// Returns (lora_A [rank, in], lora_B [out, rank]) per entry, views of the buffer.  The bytes go through page-locked memory (torch's
// pool, which holds a block until the copies that read it are done), a megabyte's copy under way while the next is filled.
// (Four threads filled 7 MB in 340 us where this takes 310, but in 1000 to 4600 whenever the request's other work had left the
// process's CPUs busy.)
constexpr int64_t kStagePart = 1 << 19;  // elements
std::vector<std::pair<Tensor, Tensor>> stage_adapters(const py::list& entries, const std::string& device) {
  const c10::Device dev(device);
  std::vector<ByteView> views;
  std::vector<Staged> parts;
  views.reserve(2 * entries.size());
  int64_t total = 0;
  for (const py::handle& h : entries) {
    const py::tuple e = py::cast<py::tuple>(h);
    std::pair<int64_t, int64_t> shape[2];
    for (int i = 0; i < 2; ++i) {
      views.emplace_back(e[2 * i]);
      if (views.back().b.len % 2 != 0) throw py::value_error("adapter bytes are not whole bf16 values");
      shape[i] = matrix_shape(views.back().b.len / 2, py::cast<std::vector<int64_t>>(e[2 * i + 1]));
    }
    const int64_t rank = shape[0].first;
    if (shape[1].second != rank) throw py::value_error("lora_A and lora_B do not form a rank decomposition");
    const int64_t padded = (rank + 7) / 8 * 8;
    for (int i = 0; i < 2; ++i) {
      const auto& v = views[views.size() - 2 + i];
      parts.push_back(Staged{static_cast<const uint16_t*>(v.b.buf), shape[i].first, shape[i].second,
                             i == 0 ? padded : shape[i].first, i == 0 ? shape[i].second : padded, total});
      total += (parts.back().size() + 7) / 8 * 8;
    }
  }
  Tensor buf;
  {
    py::gil_scoped_release nogil;
    c10::OptionalDeviceGuard guard;
    if (dev.is_cuda()) guard.reset_device(dev);
    const Tensor host = at::empty({total}, at::TensorOptions().dtype(at::kShort).pinned_memory(dev.is_cuda()));
    buf = dev.is_cuda() ? at::empty({total}, at::TensorOptions().dtype(at::kShort).device(dev)) : host;
    uint16_t* stage = reinterpret_cast<uint16_t*>(host.data_ptr<int16_t>());
    size_t begin = 0;
    for (size_t i = 0; i < parts.size(); ++i) {
      parts[i].copy_to(stage);
      const int64_t lo = parts[begin].off, hi = i + 1 < parts.size() ? parts[i + 1].off : total;
      if (hi - lo < kStagePart && i + 1 < parts.size()) continue;
      if (dev.is_cuda()) buf.slice(0, lo, hi).copy_(host.slice(0, lo, hi), /*non_blocking=*/true);
      begin = i + 1;
    }
  }
  const Tensor bf = buf.view(at::kBFloat16);
  std::vector<std::pair<Tensor, Tensor>> out;
  out.reserve(parts.size() / 2);
  for (size_t i = 0; i + 1 < parts.size(); i += 2)
    out.emplace_back(bf.narrow(0, parts[i].off, parts[i].size()).view({parts[i].out_rows, parts[i].out_cols}),
                     bf.narrow(0, parts[i + 1].off, parts[i + 1].size()).view({parts[i + 1].out_rows, parts[i + 1].out_cols}));
  return out;
}

// jobs: (base, out, lora_A or None, lora_B or None, scale)
void lora_merge(const py::list& jobs, uintptr_t stream) {
  std::vector<TomeLoraJob> table;
  std::vector<Tensor> keep;
  table.reserve(jobs.size());
  c10::Device dev(c10::kCPU);
  for (const py::handle& h : jobs) {
    const py::tuple e = py::cast<py::tuple>(h);
    if (e.size() != 5) throw py::value_error("a merge job is (base, out, lora_A, lora_B, scale)");
    const Tensor base = py::cast<Tensor>(e[0]), out = py::cast<Tensor>(e[1]);
    if (table.empty()) dev = base.device();
    MaybeTensor a, b;
    if (!e[2].is_none()) a = py::cast<Tensor>(e[2]);
    if (!e[3].is_none()) b = py::cast<Tensor>(e[3]);
    auto check_tensor = [&](const Tensor& t) {
      require_gpu(t);
      if (t.device() != dev) throw py::value_error("all tensors of a merge must be on the same device");
      if (t.scalar_type() != at::kBFloat16 || t.dim() != 2) throw py::type_error("LoRA merges work on 2-D bfloat16 tensors (inference.proto:71-72)");
    };
    check_tensor(base);
    check_tensor(out);
    if (a) check_tensor(*a);
    if (b) check_tensor(*b);
    if (out.sizes() != base.sizes() || base.stride(1) != 1 || out.stride(1) != 1)
      throw py::value_error("base and out must have the same shape and unit stride along the input dimension");
    const int64_t rows = base.size(0), cols = base.size(1);
    int64_t rank = 0;
    if (a.has_value() != b.has_value()) throw py::value_error("lora_A and lora_B come together");
    if (a) {
      rank = a->size(0);
      if (a->size(1) != cols || b->size(0) != rows || b->size(1) != rank)
        throw py::value_error("lora_A must be [rank, " + std::to_string(cols) + "] and lora_B [" + std::to_string(rows) + ", rank]; rank is " +
                              std::to_string(rank));
      a = a->contiguous();
      b = b->contiguous();
      if (rank % 8 != 0) {  // zero-pad the rank: extra terms of the product are exact zeros
        const int64_t pad = 8 - rank % 8;
        a = at::cat({*a, at::zeros({pad, cols}, a->options())}, 0);
        b = at::cat({*b, at::zeros({rows, pad}, b->options())}, 1).contiguous();
        rank += pad;
      }
      keep.push_back(*a);  // stream-ordered: torch frees on the same stream
      keep.push_back(*b);
    }
    TomeLoraJob j{};
    j.base = base.data_ptr();
    j.out = out.data_ptr();
    j.lora_a = a ? a->data_ptr() : nullptr;
    j.lora_b = b ? b->data_ptr() : nullptr;
    j.rows = rows;
    j.cols = cols;
    j.rank = rank;
    j.base_stride = rows > 1 ? base.stride(0) : cols;
    j.out_stride = rows > 1 ? out.stride(0) : cols;
    j.scale = (float)py::cast<double>(e[4]);
    table.push_back(j);
  }
  if (table.empty()) return;
  py::gil_scoped_release nogil;
  c10::DeviceGuard guard(dev);
  const size_t bytes = tome_lora_merge_workspace(table.data(), (int64_t)table.size());
  const Tensor ws = workspace(bytes, at::TensorOptions().dtype(at::kByte).device(dev));
  check(tome_lora_merge(table.data(), (int64_t)table.size(), ptr(ws), bytes, stream_ptr(stream)));
}

}  // namespace

PYBIND11_MODULE(_torch_ops, m) {
  m.doc() = "Native host side of tome_amd's operators (argument checks, allocation, C-ABI calls)";
  typedef py::call_guard<py::gil_scoped_release> NoGil;
  m.def("rows_view", &rows_view, NoGil());
  m.def("token_logprobs", &token_logprobs, NoGil());
  m.def("token_logprobs_rows", &token_logprobs_rows, NoGil());
  m.def("sample_tokens", &sample_tokens, NoGil());
  m.def("sample_step", &sample_step, NoGil());
  m.def("fused_log_softmax", &fused_log_softmax, NoGil());
  m.def("lmhead_logprobs", &lmhead_logprobs, NoGil());
  m.def("grpo_pair", &grpo_pair, NoGil());
  m.def("stage_adapters", &stage_adapters);
  m.def("lora_merge", &lora_merge);
}
