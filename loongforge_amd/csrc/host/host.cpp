// Native host layer of the tensor-level entry points (loongforge_amd/ops.py): argument checks, output and workspace
// allocation and the call into the C-ABI library, one C++ call per operation.  In Python the same steps cost 13 - 20 us
// per operation and the custom-op dispatcher another 8 - 10, more than most kernels of a decode step run; here 4 - 6 us
// in all (one decode step, six operations: 150 us of host time before).
//
// Every function returns None, without having done anything, when a tensor is not a plain one (a subclass, a fake or
// functional tensor, a traced or transformed call, or one whose gradient is being recorded): the caller then goes
// through the registered custom op, whose implementation calls back here with force = true.
#include <torch/extension.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <hip/hip_runtime_api.h>

#include "../../../include/dsa_hip.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

// ---- plain tensors --------------------------------------------------------------------------------
bool plain_call() {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
  constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::Tracer,
                                     c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchVmapMode,
                                     c10::DispatchKey::VmapMode});
  return !c10::impl::tls_local_dispatch_key_set().included_.has_any(odd);
}
bool plain_tensor(const Tensor& t, bool grad) {
  constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched,
                                     c10::DispatchKey::Batched,
                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return !t.key_set().has_any(odd) && !(grad && t.requires_grad()) && !t._fw_grad(0).defined();
}
bool plain_tensor(const OptTensor& t, bool grad) { return !t || plain_tensor(*t, grad); }
template <class... T>
bool plain(const T&... t) {
  if (!plain_call()) return false;
  const bool grad = at::GradMode::is_enabled();
  return (plain_tensor(t, grad) && ...);
}
bool ordinary(const std::vector<OptTensor>& tensors) {
  if (!plain_call()) return false;
  for (const OptTensor& t : tensors)
    if (!plain_tensor(t, false)) return false;
  return true;
}
#define PLAIN_OR_NONE(...) do { if (!force && !plain(__VA_ARGS__)) return py::none(); } while (0)

// ---- checks ---------------------------------------------------------------------------------------
const Tensor* present(const Tensor& t) { return &t; }
const Tensor* present(const OptTensor& t) { return t ? &*t : nullptr; }
// All tensors that a kernel is given: with memory, on one device.
template <class... T>
void need_gpus(const T&... t) {
  const Tensor* const all[] = {present(t)...};
  const Tensor* first = nullptr;
  for (const Tensor* p : all) {
    if (!p) continue;
    TORCH_CHECK(p->is_cuda(), "DSA kernels need tensors on a HIP device; got a ", c10::DeviceTypeName(p->device().type(), true), " tensor");
    if (!first) first = p;
    TORCH_CHECK(p->device() == first->device(), "DSA kernels need tensors on one device; got ", first->device(), " and ", p->device());
  }
  // (fake tensors and wrappers of transforms have a device but no memory)
  for (const Tensor* p : all)
    TORCH_CHECK(!p || p->numel() == 0 || (p->has_storage() && p->storage().data() != nullptr), "DSA kernels need tensors with memory of their own");
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = dsa_last_error();
  if (rc == DSA_ERR_BAD_ARG) throw py::value_error(std::string(what) + ": " + msg);
  PyErr_SetString(py::module_::import("loongforge_amd._lib").attr("DsaError").ptr(),
                  (std::string(what) + " failed (status " + std::to_string(rc) + "): " + msg).c_str());
  throw py::error_already_set();
}
// One call into the library, without the interpreter lock (a launch blocks while the queue is full).
template <class F, class... A>
void run(const char* what, F f, A... a) {
  RECORD_FUNCTION(what, c10::ArrayRef<const c10::IValue>{});     // shows as a range in torch's profiler
  int rc;
  {
    py::gil_scoped_release unlocked;
    rc = f(a...);
  }
  check(rc, what);
}
#define REQUIRE(cond, ...) do { if (!(cond)) throw py::value_error(c10::str(__VA_ARGS__)); } while (0)

// The device of a call: current for its duration, with its current stream.
struct Call {
  c10::DeviceGuard guard;
  void* stream;
  explicit Call(const Tensor& t) : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

Tensor f32(const Tensor& t) { return t.to(at::kFloat).contiguous(); }
Tensor i32(const Tensor& t) { return t.to(at::kInt).contiguous(); }
// (past the dispatcher: 0.5 us and not 0.8 a tensor, of which a training pass of a layer makes fifty)
Tensor make(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  if (!like.is_cuda()) return at::empty(shape, like.options().dtype(type));
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}
at::ScalarType payload_type(bool raw) { return raw ? at::kByte : at::kFloat8_e4m3fn; }
const void* ptr(const OptTensor& t) { return t && t->numel() ? t->const_data_ptr() : nullptr; }
template <class P> P* out_ptr(const Tensor& t) { return t.numel() ? (P*)t.data_ptr() : nullptr; }

Tensor as_u8(const Tensor& t) {
  REQUIRE(t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte, "expected an fp8-e4m3 (or raw uint8) tensor, got ",
          t.scalar_type());
  return t.contiguous();
}

// ---- quantisers -------------------------------------------------------------------------------------
py::object quant_rowwise(const Tensor& x_, double eps, bool pow2, bool force) {
  PLAIN_OR_NONE(x_);
  need_gpus(x_);
  REQUIRE(x_.scalar_type() == at::kBFloat16, "quant_rowwise_e4m3 expects bf16 input, got ", x_.scalar_type());
  const Tensor x = x_.contiguous();
  const int64_t cols = x.size(-1), rows = x.numel() / std::max<int64_t>(cols, 1);
  Call call(x);
  Tensor x8 = make(x.sizes(), payload_type(force), x), scale_inv = make(x.sizes().slice(0, x.dim() - 1), at::kFloat, x);
  run("dsa_quant_rowwise_e4m3", dsa_quant_rowwise_e4m3, x.const_data_ptr(), rows, (int)cols, x8.data_ptr(), (float*)scale_inv.data_ptr(), (float)eps, pow2, call.stream);
  return py::make_tuple(x8, scale_inv);
}

py::object rotate_quant(const Tensor& x_, double eps, bool pow2, bool want_payload, bool want_rotated, bool force) {
  PLAIN_OR_NONE(x_);
  need_gpus(x_);
  REQUIRE(x_.scalar_type() == at::kBFloat16, "rotate_quant_e4m3 expects bf16 input, got ", x_.scalar_type());
  REQUIRE(x_.size(-1) == 128, "rotate_quant_e4m3 rotates rows of 128 elements, got ", x_.size(-1));
  REQUIRE(want_payload || want_rotated, "rotate_quant_e4m3: no output requested");
  const Tensor x = x_.contiguous();
  Call call(x);
  const auto lead = x.sizes().slice(0, x.dim() - 1);
  Tensor x8 = want_payload ? make(x.sizes(), payload_type(force), x) : make({0}, payload_type(force), x);
  Tensor scale_inv = want_payload ? make(lead, at::kFloat, x) : make({0}, at::kFloat, x);
  Tensor y = want_rotated ? make(x.sizes(), at::kBFloat16, x) : make({0}, at::kBFloat16, x);
  run("dsa_rotate_quant_e4m3", dsa_rotate_quant_e4m3, x.const_data_ptr(), x.numel() / 128, 128, want_payload ? x8.data_ptr() : nullptr, want_payload ? (float*)scale_inv.data_ptr() : nullptr, want_rotated ? y.data_ptr() : nullptr, (float)eps, pow2, call.stream);
  return py::make_tuple(x8, scale_inv, y);
}

py::object quant_weights(const Tensor& x_, const Tensor& weights_, double factor, bool rotate, double eps, bool pow2, bool force) {
  PLAIN_OR_NONE(x_, weights_);
  need_gpus(x_, weights_);
  REQUIRE(x_.scalar_type() == at::kBFloat16 && x_.size(-1) == 128, "quant_rowwise_e4m3_weights expects bf16 rows of 128 elements");
  const auto lead = x_.sizes().slice(0, x_.dim() - 1);
  REQUIRE(weights_.sizes() == lead, "quant_rowwise_e4m3_weights: one weight per row expected, got ", weights_.sizes(), " for rows ", lead);
  const Tensor x = x_.contiguous(), weights = f32(weights_);
  Call call(x);
  Tensor x8 = make(x.sizes(), payload_type(force), x), scale_inv = make(lead, at::kFloat, x), scaled = make(lead, at::kFloat, x);
  run("dsa_quant_rowwise_e4m3_weights", dsa_quant_rowwise_e4m3_weights, x.const_data_ptr(), x.numel() / 128, 128, x8.data_ptr(), (float*)scale_inv.data_ptr(), (float)eps, pow2, rotate, (const float*)weights.const_data_ptr(), (float)factor, (float*)scaled.data_ptr(), call.stream);
  return py::make_tuple(x8, scale_inv, scaled);
}

struct FrontTables { Tensor cos, sin; OptTensor positions; };
FrontTables front_tables(const OptTensor& cos, const OptTensor& sin, const OptTensor& positions, int64_t batch, int64_t tokens,
                         const char* what = "indexer_front_e4m3") {
  REQUIRE(batch > 0, what, ": batch must be positive, got ", batch);       // (divided by below)
  REQUIRE(cos && sin && cos->scalar_type() == sin->scalar_type() &&
          (cos->scalar_type() == at::kFloat || cos->scalar_type() == at::kBFloat16),
          what, ": cos / sin must both be fp32 or bf16 tables");
  REQUIRE(cos->size(-1) == 64 && sin->size(-1) == 64 && cos->numel() == sin->numel(),
          what, ": cos / sin rows must have 64 entries");
  FrontTables t{cos->contiguous(), sin->contiguous(), {}};
  if (positions) {
    t.positions = i32(*positions);
    REQUIRE(t.positions->numel() == tokens, what, ": one position per token expected");
  } else {
    REQUIRE((tokens + batch - 1) / batch <= t.cos.numel() / 64, what, ": cos / sin tables are shorter than the sequence");
  }
  return t;
}
std::pair<Tensor, Tensor> front_norm(const Tensor& weight, const Tensor& bias) {
  REQUIRE(weight.numel() == 128 && bias.numel() == 128, "indexer_front_e4m3: LayerNorm weight and bias must have 128 entries");
  return {f32(weight), f32(bias)};
}

py::object indexer_front(const Tensor& x_, int64_t rows_per_token, const OptTensor& ln_weight_, const OptTensor& ln_bias_, double ln_eps,
                         const OptTensor& cos_, const OptTensor& sin_, int64_t pairing, const OptTensor& positions_, int64_t batch,
                         bool rotate, const OptTensor& weights_, double factor, bool want_payload, bool want_rows, double eps, bool pow2,
                         bool force) {
  PLAIN_OR_NONE(x_, ln_weight_, ln_bias_, cos_, sin_, positions_, weights_);
  REQUIRE(batch > 0, "indexer_front_e4m3: batch must be positive, got ", batch);       // (divided by below)
  need_gpus(x_, ln_weight_, ln_bias_, cos_, sin_, positions_, weights_);
  REQUIRE(x_.scalar_type() == at::kBFloat16 && x_.size(-1) == 128, "indexer_front_e4m3 expects bf16 rows of 128 elements");
  const Tensor x = x_.contiguous();
  const int64_t rows = x.numel() / 128;
  REQUIRE(rows_per_token > 0 && rows % rows_per_token == 0, "indexer_front_e4m3: ", rows, " rows are not a multiple of ", rows_per_token,
          " rows per token");
  REQUIRE(ln_weight_.has_value() == ln_bias_.has_value(), "indexer_front_e4m3: LayerNorm needs weight and bias");
  const int64_t tokens = rows / rows_per_token;
  int tables_f32 = 0;
  OptTensor cos, sin, positions, ln_weight, ln_bias, weights;
  if (pairing >= 0) {
    FrontTables t = front_tables(cos_, sin_, positions_, batch, tokens);
    tables_f32 = t.cos.scalar_type() == at::kFloat;
    cos = t.cos; sin = t.sin; positions = t.positions;
  }
  if (ln_weight_) std::tie(ln_weight, ln_bias) = front_norm(*ln_weight_, *ln_bias_);
  if (weights_) {
    REQUIRE(want_payload && weights_->numel() == rows, "indexer_front_e4m3: one weight per row expected, together with the payload");
    weights = f32(*weights_);
  }
  Call call(x);
  const auto lead = x.sizes().slice(0, x.dim() - 1);
  Tensor x8 = want_payload ? make(x.sizes(), payload_type(force), x) : make({0}, payload_type(force), x);
  Tensor scale_inv = want_payload ? make(lead, at::kFloat, x) : make({0}, at::kFloat, x);
  Tensor y = want_rows ? make(x.sizes(), at::kBFloat16, x) : make({0}, at::kBFloat16, x);
  Tensor scaled = weights ? make(lead, at::kFloat, x) : make({0}, at::kFloat, x);
  run("dsa_indexer_front_e4m3", dsa_indexer_front_e4m3, x.const_data_ptr(), rows, 128, (int)rows_per_token, (const float*)ptr(ln_weight), (const float*)ptr(ln_bias), (float)ln_eps, ptr(cos), ptr(sin), tables_f32, (int)pairing, (const int32_t*)ptr(positions), (int)batch, rotate, out_ptr<void>(x8), out_ptr<float>(scale_inv), out_ptr<void>(y), (float)eps, pow2, (const float*)ptr(weights), (float)factor, out_ptr<float>(scaled), call.stream);
  return py::make_tuple(x8, scale_inv, y, scaled);
}

py::tuple quant_padded(const Tensor& x_, int64_t heads_out, const OptTensor& weights_, double factor) {
  need_gpus(x_, weights_);
  REQUIRE(x_.dim() == 3, "quant_padded expects [tokens, heads, dim]");
  const Tensor x = x_.to(at::kBFloat16).contiguous();
  OptTensor weights;
  if (weights_) {
    REQUIRE(weights_->numel() == x.size(0) * x.size(1), "quant_padded: one weight per row expected");
    weights = weights_->scalar_type() == at::kBFloat16 ? weights_->contiguous() : f32(*weights_);
  }
  Call call(x);
  const int64_t T = x.size(0);
  Tensor x8 = make({T, heads_out, 128}, at::kFloat8_e4m3fn, x), scale_inv = make({T, heads_out}, at::kFloat, x), scaled;
  if (weights) scaled = make({T, heads_out}, at::kFloat, x);
  run("dsa_quant_padded_e4m3", dsa_quant_padded_e4m3, x.const_data_ptr(), T, (int)x.size(1), (int)x.size(2), (int)heads_out, x8.data_ptr(),
      (float*)scale_inv.data_ptr(), 1e-12f, 1, ptr(weights), weights && weights->scalar_type() == at::kBFloat16, (float)factor,
      weights ? (float*)scaled.data_ptr() : nullptr, call.stream);
  return py::make_tuple(x8, scale_inv, weights ? py::cast(scaled) : py::none());
}

// ---- separate operations of the indexer's front end ---------------------------------------------------
bool frequencies(const Tensor& t) {
  return t.is_cuda() && plain(t) && t.scalar_type() == at::kFloat && t.dim() == 1 && t.numel() > 0 && t.is_contiguous();
}

py::object rotary_angles(const Tensor& inv_freq, int64_t n, double offset) {
  if (!frequencies(inv_freq)) return py::none();
  Call call(inv_freq);
  Tensor a = make({n, 1, 1, 2 * inv_freq.numel()}, at::kFloat, inv_freq);
  run("dsa_rotary_tables", dsa_rotary_tables, (const float*)inv_freq.const_data_ptr(), (int)inv_freq.numel(), (int)n, (float)offset, 0,
      out_ptr<void>(a), (void*)nullptr, call.stream);
  return py::cast(a);
}

py::object rotary_cos_sin(const Tensor& inv_freq, int64_t n, double offset, at::ScalarType type) {
  if (!frequencies(inv_freq) || (type != at::kFloat && type != at::kBFloat16)) return py::none();
  Call call(inv_freq);
  Tensor c = make({n, 1, 1, 2 * inv_freq.numel()}, type, inv_freq), s = at::empty_like(c);
  run("dsa_rotary_tables", dsa_rotary_tables, (const float*)inv_freq.const_data_ptr(), (int)inv_freq.numel(), (int)n, (float)offset,
      type == at::kFloat ? 1 : 2, out_ptr<void>(c), out_ptr<void>(s), call.stream);
  return py::make_tuple(c, s);
}

// t [s, (b,) h, d] as rows [s * b, h][d] of unit stride with one token pitch, copied if it does not lie like that.  Where s or b
// is 1 its stride says nothing, and contiguous() keeps it: [s, 1, h, d] out of a batch-first tensor has the whole sequence there.
std::pair<Tensor, int64_t> token_rows(const Tensor& t) {
  REQUIRE(t.dim() == 3 || t.dim() == 4, "expected [s, h, d] or [s, b, h, d], got ", t.sizes());
  const bool one_pitch = t.dim() == 3 || t.size(0) == 1 || t.size(1) == 1 || t.stride(0) == t.size(1) * t.stride(1);
  const Tensor x = t.stride(-1) == 1 && one_pitch ? t : t.contiguous();
  return {x, x.dim() == 3 || x.size(1) == 1 ? x.stride(0) : x.stride(1)};
}

// -> contiguous result of t's shape
Tensor rope_steps(const Tensor& t, const Tensor& angles, double mscale, bool interleaved, bool transpose) {
  const auto [x, pitch] = token_rows(t);
  need_gpus(x, angles);
  const int64_t batch = x.dim() == 4 ? x.size(1) : 1, rows = x.size(0) * batch, d = x.size(-1), heads = x.size(-2);
  REQUIRE(x.scalar_type() == at::kBFloat16 && angles.scalar_type() == at::kFloat && angles.is_contiguous() && angles.size(-1) == d &&
          angles.size(0) >= x.size(0) && angles.numel() == angles.size(0) * d, "rope_steps: inconsistent arguments");
  Call call(x);
  Tensor y = make(x.sizes(), at::kBFloat16, x);
  if (x.numel() == 0) return y;
  run("dsa_rope_steps", dsa_rope_steps, x.const_data_ptr(), pitch, x.stride(-2), out_ptr<void>(y), heads * d, d,
      (const float*)angles.const_data_ptr(), (float)mscale, (int)interleaved, (int)batch, rows, (int)heads, (int)d, (int)transpose, call.stream);
  return y;
}

Tensor hadamard(const Tensor& x_) {
  need_gpus(x_);
  REQUIRE(x_.scalar_type() == at::kBFloat16, "hadamard expects bf16 rows");
  Tensor x = x_.contiguous();
  if ((uintptr_t)x.const_data_ptr() % 16) x = x.clone();        // a view that starts inside a 16-byte piece
  Call call(x);
  Tensor y = at::empty_like(x);
  run("dsa_hadamard", dsa_hadamard, x.const_data_ptr(), out_ptr<void>(y), x.numel() / std::max<int64_t>(x.size(-1), 1), (int)x.size(-1), call.stream);
  return y;
}

// ---- indexer ----------------------------------------------------------------------------------------
struct IndexerShape { int S, Hi, Sk; };
IndexerShape indexer_shape(const Tensor& q8, const Tensor& q_w, const Tensor& k8, const Tensor& k_scale, const Tensor& ks, const Tensor& ke) {
  need_gpus(q8, q_w, k8, k_scale, ks, ke);
  REQUIRE(q8.dim() == 3 && k8.dim() == 2 && q_w.dim() == 2, "indexer expects q8 [S,H,128], k8 [Sk,128], q_w [S,H]");
  REQUIRE(q8.size(2) == 128 && k8.size(1) == 128, "Only support dim with size 128.");
  const int64_t S = q8.size(0), Hi = q8.size(1), Sk = k8.size(0);
  REQUIRE(q_w.size(0) == S && q_w.size(1) == Hi && k_scale.dim() == 1 && k_scale.size(0) == Sk && ks.dim() == 1 && ks.size(0) == S &&
          ke.dim() == 1 && ke.size(0) == S, "indexer: inconsistent shapes");
  return {(int)S, (int)Hi, (int)Sk};
}

py::object indexer_topk(const Tensor& q8_, const Tensor& q_w_, const Tensor& k8_, const Tensor& k_scale_, const Tensor& ks_, const Tensor& ke_,
                        int64_t K, bool sort, bool force) {
  PLAIN_OR_NONE(q8_, q_w_, k8_, k_scale_, ks_, ke_);
  const auto [S, Hi, Sk] = indexer_shape(q8_, q_w_, k8_, k_scale_, ks_, ke_);
  const Tensor q8 = as_u8(q8_), k8 = as_u8(k8_), q_w = f32(q_w_), k_scale = f32(k_scale_), ks = i32(ks_), ke = i32(ke_);
  Call call(q8);
  Tensor scores = make({S, K}, at::kFloat, q8), ids = make({S, K}, at::kInt, q8);
  const size_t nbytes = dsa_indexer_topk_workspace_bytes(S, Sk, (int)K);
  Tensor ws = make({(int64_t)std::max<size_t>(nbytes, 1)}, at::kByte, q8);
  run("dsa_indexer_topk_fwd", dsa_indexer_topk_fwd, q8.const_data_ptr(), (const float*)q_w.const_data_ptr(), k8.const_data_ptr(), (const float*)k_scale.const_data_ptr(), (const int32_t*)ks.const_data_ptr(), (const int32_t*)ke.const_data_ptr(), S, Hi, Sk, (int)K, sort, (float*)scores.data_ptr(), (int32_t*)ids.data_ptr(), ws.data_ptr(), nbytes, call.stream);
  return py::make_tuple(scores, ids);
}

py::object topk(const Tensor& logits_, int64_t K, const OptTensor& row_begin, const OptTensor& row_end, const OptTensor& id_base, bool sort,
                bool force) {
  PLAIN_OR_NONE(logits_, row_begin, row_end, id_base);
  need_gpus(logits_, row_begin, row_end, id_base);
  REQUIRE(logits_.dim() == 2 && logits_.scalar_type() == at::kFloat, "topk expects a 2-D fp32 tensor");
  const Tensor logits = logits_.stride(1) == 1 ? logits_ : logits_.contiguous();
  const int64_t S = logits.size(0), width = logits.size(1);
  OptTensor rb, re, ib;
  if (row_begin) rb = i32(*row_begin);
  if (row_end) re = i32(*row_end);
  if (id_base) ib = i32(*id_base);
  Call call(logits);
  Tensor scores = make({S, K}, at::kFloat, logits), ids = make({S, K}, at::kInt, logits);
  run("dsa_topk", dsa_topk, (const float*)logits.const_data_ptr(), (int)S, S > 0 ? logits.stride(0) : width, (const int32_t*)ptr(rb), (const int32_t*)ptr(re), (int)width, (const int32_t*)ptr(ib), (int)K, sort, (float*)scores.data_ptr(), (int32_t*)ids.data_ptr(), call.stream);
  return py::make_tuple(scores, ids);
}

// Slots are processed 128 at a time: gradients and ids padded with empty slots to a multiple of that.
std::pair<Tensor, Tensor> padded_slots(const Tensor& g_, const Tensor& ids_) {
  Tensor g = f32(g_), ids = i32(ids_);
  const int64_t pad = (128 - ids.size(1) % 128) % 128;
  if (pad) { g = at::constant_pad_nd(g, {0, pad}, 0.0); ids = at::constant_pad_nd(ids, {0, pad}, -1); }
  return {g, ids};
}

py::object indexer_bwd(const Tensor& g_, const Tensor& q8_, const Tensor& k8_, const Tensor& k_scale_, const Tensor& q_w_, const Tensor& ids_,
                       bool force) {
  PLAIN_OR_NONE(g_, q8_, k8_, k_scale_, q_w_, ids_);
  need_gpus(g_, q8_, k8_, k_scale_, q_w_, ids_);
  const int64_t S = q8_.size(0), Hi = q8_.size(1), Sk = k8_.size(0);
  REQUIRE(ids_.dim() == 2 && g_.sizes() == ids_.sizes() && ids_.size(0) == S, "indexer_bwd: grad and ids must both be [S, K]");
  const auto [g, ids] = padded_slots(g_, ids_);
  const Tensor q8 = as_u8(q8_), k8 = as_u8(k8_), q_w = f32(q_w_), k_scale = f32(k_scale_);
  Call call(q8);
  Tensor d_q8 = make(q8.sizes(), at::kFloat, q8), d_k8 = make(k8.sizes(), at::kFloat, q8), d_qw = make({S, Hi}, at::kFloat, q8);
  const size_t nbytes = dsa_indexer_bwd_workspace_bytes((int)S, (int)Hi, (int)Sk, (int)ids.size(1));
  Tensor ws = make({(int64_t)std::max<size_t>(nbytes, 256)}, at::kByte, q8);
  run("dsa_indexer_bwd", dsa_indexer_bwd, (const float*)g.const_data_ptr(), q8.const_data_ptr(), k8.const_data_ptr(),
      (const float*)k_scale.const_data_ptr(), (const float*)q_w.const_data_ptr(), (const int32_t*)ids.const_data_ptr(), (int)S, (int)Hi, (int)Sk,
      (int)ids.size(1), (float*)d_q8.data_ptr(), (float*)d_k8.data_ptr(), (float*)d_qw.data_ptr(), ws.data_ptr(), nbytes, call.stream);
  return py::make_tuple(d_q8, d_k8, d_qw);
}

py::tuple indexer_grads(const Tensor& g_, const Tensor& q8_, const Tensor& k8_, const Tensor& k_scale_, const Tensor& q_w_, const Tensor& ids_,
                        const Tensor& q_scale_, double w_scale, int64_t rotate, const OptTensor& cos_, const OptTensor& sin_, int64_t pairing,
                        const OptTensor& positions_q, const OptTensor& positions_k, int64_t batch, const OptTensor& k_in, const OptTensor& ln_w_,
                        double ln_eps, int64_t heads, int64_t dim, int64_t span, at::ScalarType q_type, at::ScalarType k_type, at::ScalarType w_type) {
  need_gpus(g_, q8_, k8_, k_scale_, q_w_, ids_, q_scale_, cos_, sin_, positions_q, positions_k, k_in, ln_w_);
  const int64_t S = q8_.size(0), Hi = q8_.size(1), Sk = k8_.size(0);
  REQUIRE(ids_.dim() == 2 && g_.sizes() == ids_.sizes() && ids_.size(0) == S && q_scale_.numel() == S * Hi,
          "indexer_grads: grad and ids must both be [S, K], q_scale [S, H]");
  const auto [g, ids] = padded_slots(g_, ids_);
  const Tensor q8 = as_u8(q8_), k8 = as_u8(k8_), q_w = f32(q_w_), k_scale = f32(k_scale_), q_scale = f32(q_scale_);
  OptTensor cos, sin, pos_q, pos_k, ln_w;
  if (pairing >= 0) {
    const FrontTables tq = front_tables(cos_, sin_, positions_q, batch, S, "indexer_grads"), tk = front_tables(cos_, sin_, positions_k, batch, Sk, "indexer_grads");
    cos = tq.cos; sin = tq.sin; pos_q = tq.positions; pos_k = tk.positions;
  }
  Tensor d_ln_w, d_ln_b;
  if (k_in) {
    REQUIRE(k_in->scalar_type() == at::kBFloat16 && k_in->is_contiguous() && k_in->numel() == Sk * 128 && ln_w_ && ln_w_->numel() == 128,
            "indexer_grads: the LayerNorm's input must be bf16 [Sk, 128], its weight [128]");
    ln_w = f32(*ln_w_);
    d_ln_w = make({128}, at::kFloat, q8);
    d_ln_b = make({128}, at::kFloat, q8);
  }
  Call call(q8);
  auto out_type = [](at::ScalarType t) { return t == at::kBFloat16 ? t : at::kFloat; };
  Tensor d_q = make({S, heads, dim}, out_type(q_type), q8), d_k = make({Sk, dim}, out_type(k_type), q8), d_w = make({S, heads}, out_type(w_type), q8);
  const size_t nbytes = dsa_indexer_grads_span_workspace_bytes((int)S, (int)Hi, (int)Sk, (int)ids.size(1), (int)span);
  Tensor ws = make({(int64_t)std::max<size_t>(nbytes, 256)}, at::kByte, q8);
  auto is_f32 = [](const Tensor& t) { return (int)(t.scalar_type() == at::kFloat); };
  run("dsa_indexer_grads", dsa_indexer_grads_span, (const float*)g.const_data_ptr(), q8.const_data_ptr(), k8.const_data_ptr(),
      (const float*)k_scale.const_data_ptr(), (const float*)q_w.const_data_ptr(), (const int32_t*)ids.const_data_ptr(), (int)S, (int)Hi, (int)Sk,
      (int)ids.size(1), (int)span, (const float*)q_scale.const_data_ptr(), (float)w_scale, (int)rotate, ptr(cos), ptr(sin), cos ? is_f32(*cos) : 0,
      (int)pairing, (const int32_t*)ptr(pos_q), (const int32_t*)ptr(pos_k), (int)batch, ptr(k_in), (const float*)ptr(ln_w), (float)ln_eps,
      (int)heads, (int)dim, d_q.data_ptr(), is_f32(d_q), d_k.data_ptr(), is_f32(d_k), d_w.data_ptr(), is_f32(d_w),
      k_in ? (float*)d_ln_w.data_ptr() : nullptr, k_in ? (float*)d_ln_b.data_ptr() : nullptr, ws.data_ptr(), nbytes, call.stream);
  return py::make_tuple(d_q.to(q_type), d_k.to(k_type), d_w.to(w_type), k_in ? py::cast(d_ln_w) : py::none(), k_in ? py::cast(d_ln_b) : py::none());
}

// ---- windows of packed sequences ------------------------------------------------------------------------
// Whether the sequences cover the queries is only known on the device; the kernel leaves their length in pinned memory
// and wait() looks at it, called after the kernels that use the window were launched: the device has work while the
// host waits.  Under graph capture nothing can be checked: queries that no sequence holds then have empty windows.
struct WindowCheck {
  Tensor total;
  int64_t need = 0;
  hipEvent_t done = nullptr;
  WindowCheck() = default;
  WindowCheck(const WindowCheck&) = delete;
  int32_t* pinned() const { return need ? (int32_t*)total.data_ptr() : nullptr; }
  void launched(const Call& call) {
    if (need && (hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess || hipEventRecord(done, (hipStream_t)call.stream) != hipSuccess))
      throw std::runtime_error("indexer window: no event");
  }
  ~WindowCheck() { if (done) { (void)hipEventSynchronize(done); (void)hipEventDestroy(done); } }
  void wait() {
    if (!done) return;
    hipError_t rc;
    {
      py::gil_scoped_release unlocked;
      rc = hipEventSynchronize(done);
    }
    TORCH_CHECK(rc == hipSuccess, "indexer window: ", hipGetErrorString(rc));
    REQUIRE(*total.const_data_ptr<int>() >= 0, "indexer: the cumulative lengths of the packed sequences decrease");
    REQUIRE(*total.const_data_ptr<int>() >= need, "indexer: inconsistent shapes (the packed sequences hold ", *total.const_data_ptr<int>(),
            " tokens, the queries end at ", need, ")");
  }
};

Tensor seqlens(const Tensor& cu, const c10::Device& device) {
  Tensor t = cu.to(device);
  if (t.scalar_type() != at::kInt && t.scalar_type() != at::kLong) t = t.to(at::kLong);
  return t.contiguous();
}

struct Window { Tensor bounds; std::unique_ptr<WindowCheck> check; };      // [2, S]: first key, key behind the last

// The tensors that a kernel fills with the windows; check->pinned() goes to it, check->launched() comes behind it.
Window pending_window(const OptTensor& cu, int64_t S, int64_t chunk_offset, const Tensor& like, const Call& call) {
  Window w{make({2, S}, at::kInt, like), std::make_unique<WindowCheck>()};
  if (cu && S > 0) {
    hipStreamCaptureStatus capturing;
    if (hipStreamIsCapturing((hipStream_t)call.stream, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone) {
      w.check->total = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
      w.check->need = chunk_offset + S;
    }
  }
  return w;
}

Window key_windows(const OptTensor& cu_, int64_t S, int64_t chunk_offset, const Tensor& like) {
  need_gpus(like);
  OptTensor cu;
  if (cu_) cu = seqlens(*cu_, like.device());
  REQUIRE(!cu || S == 0 || cu->numel() > 1, "indexer: inconsistent shapes (no packed sequence)");
  Call call(like);
  Window w = pending_window(cu, S, chunk_offset, like, call);
  run("dsa_indexer_window", dsa_indexer_window, cu ? ptr(cu) : nullptr, cu && cu->scalar_type() == at::kLong, cu ? (int)cu->numel() : 0, (int)S,
      (int)chunk_offset, out_ptr<int32_t>(w.bounds), out_ptr<int32_t>(w.bounds) + S, w.check->pinned(), call.stream);
  w.check->launched(call);
  return w;
}

py::tuple indexer_window(const OptTensor& cu, int64_t S, int64_t chunk_offset, const Tensor& like) {
  Window w = key_windows(cu, S, chunk_offset, like);
  return py::make_tuple(w.bounds.select(0, 0), w.bounds.select(0, 1), std::move(w.check));
}

// The indexer's forward in one call: quantisers (behind the front end if there are rotary tables, else behind the rotation if
// asked for), key windows, logits and top-k.  Five calls from Python cost 35 - 40 us of host time, more than the kernels of a few
// queries take.  ratio > 0: the windows are those over compressed keys.  None for shapes and types that need padding or conversion
// first.  -> (scores, ids, q8, q_scale, scaled weights, k8, k_scale, check or None): check.wait() belongs behind it, as with
// indexer_window.
py::object indexer_forward(const Tensor& q, const Tensor& k, const Tensor& weights, bool rotate, double factor, const OptTensor& cu,
                           int64_t chunk_offset, int64_t K, bool sort, const OptTensor& cos, const OptTensor& sin, int64_t pairing,
                           const OptTensor& positions_q, const OptTensor& positions_k, int64_t batch, const OptTensor& ln_weight,
                           const OptTensor& ln_bias, double ln_eps, int64_t ratio, double weights_scale) {
  if (!plain(q, k, weights, cu, cos, sin, positions_q, positions_k, ln_weight, ln_bias)) return py::none();
  if (!q.is_cuda() || q.dim() != 3 || k.dim() != 2 || q.size(2) != 128 || k.size(1) != 128 || (q.size(1) != 32 && q.size(1) != 64) ||
      q.scalar_type() != at::kBFloat16 || k.scalar_type() != at::kBFloat16 || weights.sizes() != q.sizes().slice(0, 2)) return py::none();
  if (cos ? !ln_weight || !ln_bias || pairing < 0 : weights_scale != 1.0) return py::none();
  Tensor q8, q_scale, scaled, k8, k_scale;
  Window w;
  if (cos) {
    need_gpus(q, k, weights, cos, sin, positions_q, positions_k, ln_weight, ln_bias);
    const int64_t S = q.size(0), Sk = k.size(0);
    REQUIRE(S > 0 && Sk > 0, "indexer_front_e4m3: no rows");
    const Tensor qc = q.contiguous(), kc = k.contiguous();
    const Tensor wc = weights.scalar_type() == at::kBFloat16 ? weights.contiguous() : f32(weights);
    const FrontTables tq = front_tables(cos, sin, positions_q, batch, S), tk = front_tables(cos, sin, positions_k, batch, Sk);
    const auto [lw, lb] = front_norm(*ln_weight, *ln_bias);
    OptTensor lens;
    if (cu) lens = seqlens(*cu, q.device());
    REQUIRE(!lens || lens->numel() > 1, "indexer: inconsistent shapes (no packed sequence)");
    Call call(qc);
    q8 = make(qc.sizes(), at::kFloat8_e4m3fn, qc); q_scale = make(weights.sizes(), at::kFloat, qc); scaled = make(weights.sizes(), at::kFloat, qc);
    k8 = make(kc.sizes(), at::kFloat8_e4m3fn, kc); k_scale = make({Sk}, at::kFloat, kc);
    w = pending_window(lens, S, chunk_offset, qc, call);
    run("dsa_indexer_fronts_e4m3", dsa_indexer_fronts_e4m3, qc.const_data_ptr(), (int)S, (int)q.size(1), kc.const_data_ptr(), (int)Sk,
        (const float*)lw.const_data_ptr(), (const float*)lb.const_data_ptr(), (float)ln_eps, tq.cos.const_data_ptr(), tq.sin.const_data_ptr(),
        (int)(tq.cos.scalar_type() == at::kFloat), (int)pairing, (const int32_t*)ptr(tq.positions), (const int32_t*)ptr(tk.positions), (int)batch, (int)rotate,
        out_ptr<void>(q8), out_ptr<float>(q_scale), out_ptr<void>(k8), out_ptr<float>(k_scale), wc.const_data_ptr(),
        (int)(wc.scalar_type() == at::kBFloat16), (float)weights_scale, (float)factor, out_ptr<float>(scaled), lens ? ptr(lens) : nullptr,
        (int)(lens && lens->scalar_type() == at::kLong), lens ? (int)lens->numel() : 0, (int)chunk_offset, out_ptr<int32_t>(w.bounds),
        out_ptr<int32_t>(w.bounds) + S, w.check->pinned(), call.stream);
    w.check->launched(call);
  } else {
    need_gpus(q, k, weights);
    const Tensor qc = q.contiguous(), kc = k.contiguous();
    const Tensor wc = weights.scalar_type() == at::kBFloat16 ? weights.contiguous() : f32(weights);
    const int64_t S = q.size(0);
    Call call(qc);
    q8 = make(qc.sizes(), at::kFloat8_e4m3fn, qc); q_scale = make(weights.sizes(), at::kFloat, qc); scaled = make(weights.sizes(), at::kFloat, qc);
    k8 = make(kc.sizes(), at::kFloat8_e4m3fn, kc); k_scale = make({kc.size(0)}, at::kFloat, kc);
    w.bounds = make({2, S}, at::kInt, qc);
    run("dsa_indexer_inputs_e4m3", dsa_indexer_inputs_e4m3, qc.const_data_ptr(), qc.numel() / 128, kc.const_data_ptr(), kc.size(0), rotate,
        out_ptr<void>(q8), out_ptr<float>(q_scale), out_ptr<void>(k8), out_ptr<float>(k_scale), 1e-12f, 1, wc.const_data_ptr(),
        wc.scalar_type() == at::kBFloat16, (float)factor, out_ptr<float>(scaled), cu ? 0 : (int)S, chunk_offset, (int)ratio, (int)kc.size(0),
        out_ptr<int32_t>(w.bounds), out_ptr<int32_t>(w.bounds) + S, call.stream);
  }
  if (cu && !cos) w = key_windows(cu, q.size(0), chunk_offset, q8);
  const auto [scores, ids] = py::cast<std::pair<Tensor, Tensor>>(
      indexer_topk(q8, scaled, k8, k_scale, w.bounds.select(0, 0), w.bounds.select(0, 1), K, sort, false));
  return py::make_tuple(scores, ids, q8, q_scale, scaled, k8, k_scale, w.check && w.check->done ? py::cast(std::move(w.check)) : py::none());
}

// indexer_forward for heads of 64 rotary channels behind their projections (q [S, heads, 64], k [Sk, 64] behind its norm; cos, sin bf16
// [positions, 64]), padded on the way to 32 or 64 heads of 128 channels, one sequence.  -> (scores, ids, q8, q_scale, scaled
// weights, k8, k_scale); None for other arguments.
py::object indexer_forward_narrow(const Tensor& q, const Tensor& k, const Tensor& weights, const Tensor& cos, const Tensor& sin,
                                  double weights_scale, double factor, int64_t chunk_offset, int64_t K, bool sort) {
  if (!plain(q, k, weights, cos, sin) || !q.is_cuda() || q.dim() != 3 || k.dim() != 2 || q.size(2) != 64 || k.size(1) != 64 || q.size(1) < 1 ||
      q.size(1) > 64 || q.scalar_type() != at::kBFloat16 || k.scalar_type() != at::kBFloat16 || weights.sizes() != q.sizes().slice(0, 2) ||
      cos.scalar_type() != at::kBFloat16 || sin.scalar_type() != at::kBFloat16 || cos.numel() != sin.numel() || cos.numel() % 64) return py::none();
  need_gpus(q, k, weights, cos, sin);
  const int64_t S = q.size(0), heads = q.size(1), heads_out = heads <= 32 ? 32 : 64, Sk = k.size(0), positions = cos.numel() / 64;
  if (positions < std::max(S, Sk)) return py::none();
  auto lined = [](const Tensor& t) {           // a view may start inside a 16-byte piece
    const Tensor x = t.contiguous();
    return (uintptr_t)x.const_data_ptr() % 16 ? x.clone() : x;
  };
  const Tensor qc = lined(q), kc = lined(k), c = lined(cos), s = lined(sin);
  const Tensor wc = weights.scalar_type() == at::kBFloat16 ? weights.contiguous() : f32(weights);
  Call call(qc);
  Tensor q8 = make({S, heads_out, 128}, at::kFloat8_e4m3fn, qc), q_scale = make({S, heads_out}, at::kFloat, qc), scaled = at::empty_like(q_scale);
  Tensor k8 = make({Sk, 128}, at::kFloat8_e4m3fn, qc), k_scale = make({Sk}, at::kFloat, qc), bounds = make({2, S}, at::kInt, qc);
  run("dsa_indexer_narrow_e4m3", dsa_indexer_narrow_e4m3, qc.const_data_ptr(), (int)S, (int)heads, (int)heads_out, kc.const_data_ptr(), (int)Sk,
      c.const_data_ptr(), s.const_data_ptr(), (int)positions, out_ptr<void>(q8), out_ptr<float>(q_scale), out_ptr<void>(k8), out_ptr<float>(k_scale),
      wc.const_data_ptr(), wc.scalar_type() == at::kBFloat16, (float)weights_scale, (float)factor, out_ptr<float>(scaled), chunk_offset, out_ptr<int32_t>(bounds),
      out_ptr<int32_t>(bounds) + S, call.stream);
  const auto [scores, ids] = py::cast<std::pair<Tensor, Tensor>>(
      indexer_topk(q8, scaled, k8, k_scale, bounds.select(0, 0), bounds.select(0, 1), K, sort, false));
  return py::make_tuple(scores, ids, q8, q_scale, scaled, k8, k_scale);
}

py::object thd_positions(const Tensor& cu_, int64_t tokens, int64_t offset) {
  if (!cu_.is_cuda() || !plain(cu_) || cu_.numel() < 2) return py::none();
  const Tensor cu = seqlens(cu_, cu_.device());
  Call call(cu);
  Tensor pos = make({tokens}, at::kInt, cu);
  run("dsa_thd_positions", dsa_thd_positions, cu.const_data_ptr(), cu.scalar_type() == at::kLong, (int)cu.numel(), (int)tokens, offset,
      out_ptr<int32_t>(pos), call.stream);
  return py::cast(pos);
}

// ---- sparse MLA ---------------------------------------------------------------------------------------
void mla_shape(const Tensor& q, const Tensor& kv, const Tensor& ids) {
  need_gpus(q, kv, ids);
  REQUIRE(q.dim() == 3 && kv.dim() == 2 && ids.dim() == 2, "sparse MLA expects q [S,H,576], kv [Skv,576], ids [S,K]");
  REQUIRE(q.scalar_type() == at::kBFloat16 && kv.scalar_type() == at::kBFloat16, "sparse MLA expects bf16 q and kv");
  REQUIRE(q.size(2) == 576 && kv.size(1) == 576, "you should assign dim otherwise: d_qk must be 576 (512 latent + 64 rope)");
  REQUIRE(ids.size(0) == q.size(0), "ids and q disagree on the number of queries");
  REQUIRE(ids.size(1) % 64 == 0, "top-k must be padded to a multiple of 64 (pad ids with -1)");
}

py::object mla_fwd(const Tensor& q_, const Tensor& kv_, const Tensor& ids_, int64_t q_start, double sm_scale, int64_t d_v, int64_t p_out_mode,
                   const OptTensor& attn_sink, int64_t p_out_skip, bool force) {
  PLAIN_OR_NONE(q_, kv_, ids_, attn_sink);
  mla_shape(q_, kv_, ids_);
  const Tensor q = q_.contiguous(), kv = kv_.contiguous(), ids = i32(ids_);
  const int64_t S = q.size(0), H = q.size(1), K = ids.size(1), Skv = kv.size(0);
  OptTensor sink;
  if (attn_sink) {
    need_gpus(q, attn_sink);
    REQUIRE(attn_sink->numel() == H, "attn_sink must hold one logit per head (", H, "), got ", attn_sink->numel());
    sink = f32(attn_sink->reshape({H}));
  }
  REQUIRE(p_out_mode == 0 || (p_out_skip >= 0 && p_out_skip < K && p_out_skip % 32 == 0),
          "p_out_skip must be a multiple of 32 in [0, top-k), got ", p_out_skip);
  Call call(q);
  Tensor out = make({S, H, d_v}, at::kBFloat16, q), lse = make({S, H}, at::kFloat, q);
  Tensor p_out = p_out_mode == 0 ? make({0}, at::kBFloat16, q)
                                 : make({S, H, K - p_out_skip}, p_out_mode == 2 ? at::kFloat : at::kBFloat16, q);
  const size_t nbytes = dsa_sparse_mla_fwd_workspace_bytes((int)S, (int)H, (int)Skv, (int)K);
  Tensor ws;
  if (nbytes) ws = make({(int64_t)nbytes}, at::kByte, q);
  run("dsa_sparse_mla_fwd", dsa_sparse_mla_fwd_ws, q.const_data_ptr(), kv.const_data_ptr(), (const int32_t*)ids.const_data_ptr(), (int)S, (int)H, (int)Skv, (int)K, (int)q_start, (float)sm_scale, (int)d_v, out.data_ptr(), (float*)lse.data_ptr(), p_out_mode ? p_out.data_ptr() : nullptr, p_out_mode == 2, (const float*)ptr(sink), (int)p_out_skip, nbytes ? ws.data_ptr() : nullptr, nbytes, call.stream);
  return py::make_tuple(out, lse, p_out);
}

// The forward with the head-averaged distribution, `block` queries' logits at a time
py::object mla_fwd_dist(const Tensor& q_, const Tensor& kv_, const Tensor& ids_, int64_t q_start, double sm_scale, int64_t d_v, int64_t dist_heads,
                        int64_t block, const OptTensor& attn_sink, bool force) {
  PLAIN_OR_NONE(q_, kv_, ids_, attn_sink);
  mla_shape(q_, kv_, ids_);
  const Tensor q = q_.contiguous(), kv = kv_.contiguous(), ids = i32(ids_);
  const int64_t S = q.size(0), H = q.size(1), K = ids.size(1), Skv = kv.size(0);
  OptTensor sink;
  if (attn_sink) {
    need_gpus(q, attn_sink);
    REQUIRE(attn_sink->numel() == H, "attn_sink must hold one logit per head (", H, "), got ", attn_sink->numel());
    sink = f32(attn_sink->reshape({H}));
  }
  Call call(q);
  Tensor out = make({S, H, d_v}, at::kBFloat16, q), lse = make({S, H}, at::kFloat, q), dist = make({S, K}, at::kFloat, q);
  block = std::max<int64_t>(1, std::min(block, S));
  Tensor logits = make({block, H, K}, at::kBFloat16, q);
  const size_t nbytes = dsa_sparse_mla_fwd_block_workspace_bytes((int)S, (int)block, (int)H, (int)Skv, (int)K);
  Tensor ws;
  if (nbytes) ws = make({(int64_t)nbytes}, at::kByte, q);
  for (int64_t s0 = 0; s0 < S; s0 += block)
    run("dsa_sparse_mla_fwd_dist", dsa_sparse_mla_fwd_dist, (const char*)q.const_data_ptr() + s0 * H * 576 * 2, kv.const_data_ptr(),
        (const int32_t*)ids.const_data_ptr() + s0 * K, (int)S, (int)std::min(block, S - s0), (int)H, (int)Skv, (int)K, (int)(q_start + s0),
        (float)sm_scale, (int)d_v, (char*)out.data_ptr() + s0 * H * d_v * 2, (float*)lse.data_ptr() + s0 * H, (const float*)ptr(sink),
        (int)dist_heads, (float*)dist.data_ptr() + s0 * K, logits.data_ptr(), nbytes ? ws.data_ptr() : nullptr, nbytes, call.stream);
  return py::make_tuple(out, lse, dist);
}

// bf16 [S, h, width] -> [S, heads, width] with zeros behind
Tensor with_zero_heads(const Tensor& x_, int64_t heads) {
  Tensor x = x_.contiguous();
  if ((uintptr_t)x.const_data_ptr() % 16) x = x.clone();        // a view that starts inside a 16-byte piece
  Call call(x);
  Tensor y = make({x.size(0), heads, x.size(2)}, at::kBFloat16, x);
  run("dsa_pad_heads", dsa_pad_heads, x.const_data_ptr(), (int)x.size(0), (int)x.size(1), (int)heads, (int)x.size(2) * 2, out_ptr<void>(y), call.stream);
  return y;
}
py::object pad_heads(const Tensor& x, int64_t heads) {
  if (!plain(x) || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.dim() != 3 || x.size(2) % 8 || x.size(2) > 32768 || x.size(1) < 1 ||
      x.size(1) > heads || heads > 1024 || x.size(2) < 1) return py::none();
  need_gpus(x);
  return py::cast(with_zero_heads(x, heads));
}

py::object mla_bwd(const Tensor& q_, const Tensor& kv_, const Tensor& out_, const Tensor& dout_, const Tensor& ids_, const Tensor& lse_,
                   int64_t q_start, double sm_scale, int64_t d_v, int64_t heads, const py::function& workspace, bool force) {
  PLAIN_OR_NONE(q_, kv_, out_, dout_, ids_, lse_);
  mla_shape(q_, kv_, ids_);
  need_gpus(q_, out_, dout_, lse_);
  const Tensor q = q_.contiguous(), kv = kv_.contiguous(), ids = i32(ids_), out = out_.contiguous(), lse = f32(lse_);
  const int64_t S = q.size(0), H = q.size(1), K = ids.size(1), Skv = kv.size(0);
  const bool some = heads > 0 && heads < H;          // only the first heads are real: dout has theirs, and dq
  REQUIRE(!some || dout_.sizes() == at::IntArrayRef({S, heads, d_v}), "sparse_mla_bwd: dout must be [S,heads,d_v]");
  Tensor dout = dout_.to(at::kBFloat16).contiguous();
  if (some) dout = with_zero_heads(dout, H);
  REQUIRE(out.sizes() == at::IntArrayRef({S, H, d_v}) && dout.sizes() == out.sizes() && lse.sizes() == at::IntArrayRef({S, H}),
          "sparse_mla_bwd: out/dout must be [S,H,d_v] and lse [S,H]");
  Tensor dq = some ? make({S, heads, 576}, at::kBFloat16, q) : at::empty_like(q), dkv = at::empty_like(kv);
  const size_t full = dsa_sparse_mla_bwd_workspace_bytes((int)S, (int)H, (int)Skv, (int)K);
  Call call(q);
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)call.stream, &status) != hipSuccess) status = hipStreamCaptureStatusActive;
  const auto [ws, nbytes] = py::cast<std::pair<Tensor, size_t>>(workspace(full, q.device(), (size_t)call.stream, status != hipStreamCaptureStatusNone));
  run("dsa_sparse_mla_bwd", dsa_sparse_mla_bwd_heads, q.const_data_ptr(), kv.const_data_ptr(), out.const_data_ptr(), dout.const_data_ptr(),
      (const int32_t*)ids.const_data_ptr(), (const float*)lse.const_data_ptr(), (int)S, (int)H, (int)(some ? heads : H), (int)Skv, (int)K, (int)q_start, (float)sm_scale,
      (int)d_v, dq.data_ptr(), dkv.data_ptr(), ws.data_ptr(), nbytes, call.stream);
  return py::make_tuple(dq, dkv);
}

// `as_input`: in the logits' type, rounded by the kernel
Tensor attn_dist_of(const Tensor& p_, double sm_scale, bool as_input) {
  need_gpus(p_);
  REQUIRE(p_.dim() == 3 && (p_.scalar_type() == at::kBFloat16 || p_.scalar_type() == at::kFloat), "attn_dist expects p_out [S,H,K] in bf16 or fp32");
  const Tensor p = p_.stride(2) == 1 ? p_ : p_.contiguous();
  const int64_t S = p.size(0), H = p.size(1), K = p.size(2);
  Call call(p);
  const auto type = as_input ? p.scalar_type() : at::kFloat;
  Tensor target = make({S, K}, type, p);
  run("dsa_attn_dist", dsa_attn_dist_as, p.const_data_ptr(), p.scalar_type() == at::kFloat, (int)S, (int)H, (int)K, S > 0 ? p.stride(0) : H * K, p.stride(1), (float)sm_scale, target.data_ptr(), type == at::kBFloat16, call.stream);
  return target;
}

py::object attn_dist(const Tensor& p, double sm_scale, bool force) {
  PLAIN_OR_NONE(p);
  return py::cast(attn_dist_of(p, sm_scale, false));
}
py::object attn_dist_as_input(const Tensor& p, double sm_scale, bool force) {
  PLAIN_OR_NONE(p);
  return py::cast(attn_dist_of(p, sm_scale, true));
}

std::pair<Tensor, Tensor> kl_rows(const Tensor& scores_, const Tensor& target_, double eps) {
  need_gpus(scores_, target_);
  REQUIRE(scores_.dim() == 2 && target_.sizes() == scores_.sizes(), "indexer_kl_loss expects scores and target of one shape [S, K]");
  const int64_t S = scores_.size(0), K = scores_.size(1);
  // bf16 targets are read as they are, but for rows that overlap (one row for all of them): those become fp32 rows of their own
  const bool as_is = target_.scalar_type() == at::kBFloat16 && (S < 2 || target_.stride(0) >= K);
  Tensor scores = scores_.to(at::kFloat), target = as_is ? target_ : target_.to(at::kFloat);
  if (scores.stride(1) != 1) scores = scores.contiguous();
  if (target.stride(1) != 1) target = target.contiguous();
  Call call(scores);
  Tensor row_loss = make({S}, at::kFloat, scores), grad = make({S, K}, at::kFloat, scores);
  run("dsa_indexer_kl_loss", dsa_indexer_kl_loss_scaled, (const float*)scores.const_data_ptr(), S > 1 ? scores.stride(0) : K, target.const_data_ptr(), target.scalar_type() == at::kBFloat16, S > 1 ? target.stride(0) : K, (int)S, (int)K, (float)eps, 1.0f, (float*)row_loss.data_ptr(), (float*)grad.data_ptr(), call.stream);
  return {row_loss, grad};
}

py::object kl_loss(const Tensor& scores, const Tensor& target, double eps, bool force) {
  PLAIN_OR_NONE(scores, target);
  const auto [row_loss, grad] = kl_rows(scores, target, eps);
  return py::make_tuple(row_loss, grad);
}

// The loss of all rows times factor, and its gradient behind kl_loss: grad * g * factor.  None for what the kernels do not take.
Tensor rows_total(const Tensor& row_loss, double factor) {
  Call call(row_loss);
  Tensor total = make({}, at::kFloat, row_loss);
  run("dsa_indexer_kl_total", dsa_indexer_kl_total, (const float*)ptr(row_loss), (int)row_loss.numel(), (float)factor, (float*)total.data_ptr(), call.stream);
  return total;
}
py::object kl_total(const Tensor& row_loss, double factor) {
  if (!plain(row_loss) || !row_loss.is_cuda() || row_loss.scalar_type() != at::kFloat || row_loss.dim() != 1 || !row_loss.is_contiguous()) return py::none();
  return py::cast(rows_total(row_loss, factor));
}
// Both: (loss of all rows times factor, gradient of the loss without it).
py::object kl_loss_total(const Tensor& scores, const Tensor& target, double eps, double factor) {
  const auto [row_loss, grad] = kl_rows(scores, target, eps);
  return py::make_tuple(rows_total(row_loss, factor), grad);
}

py::object kl_scale(const Tensor& grad, const Tensor& g, double factor) {
  if (!plain(grad, g) || !grad.is_cuda() || !g.is_cuda() || g.device() != grad.device() || grad.scalar_type() != at::kFloat || g.scalar_type() != at::kFloat || g.numel() != 1 ||
      !grad.is_contiguous() || (uintptr_t)grad.const_data_ptr() % 16) return py::none();
  Call call(grad);
  Tensor y = at::empty_like(grad);
  run("dsa_indexer_kl_scale", dsa_indexer_kl_scale, (const float*)ptr(grad), (const float*)ptr(g), (float)factor, out_ptr<float>(y), grad.numel(), call.stream);
  return py::cast(y);
}

// ---- absorption and rotary kernels (write into their arguments) ---------------------------------------
void need_bf16(const Tensor& a, const Tensor& b, const Tensor& c) {
  REQUIRE(a.scalar_type() == at::kBFloat16 && b.scalar_type() == at::kBFloat16 && c.scalar_type() == at::kBFloat16,
          "mla_absorb expects bf16 tensors");
}

void absorb_into(const Tensor& a, const Tensor& w_, const Tensor& c) {
  need_gpus(a, w_, c);
  need_bf16(a, w_, c);
  REQUIRE(a.dim() == 3 && c.dim() == 3 && w_.dim() == 3 && a.size(0) == c.size(0) && a.size(1) == c.size(1) && w_.size(0) == a.size(1) &&
          w_.size(1) == c.size(2) && w_.size(2) == a.size(2),
          "mla_absorb: shapes a ", a.sizes(), ", w ", w_.sizes(), ", c ", c.sizes(), " do not fit c[s,h,:] = a[s,h,:] @ w[h].T");
  REQUIRE(a.stride(2) == 1 && c.stride(2) == 1, "mla_absorb: rows must be contiguous");
  const Tensor w = w_.contiguous();
  Call call(a);
  run("dsa_mla_absorb", dsa_mla_absorb, a.const_data_ptr(), a.stride(0), a.stride(1), w.const_data_ptr(), c.data_ptr(), c.stride(0), c.stride(1), (int)a.size(0), (int)a.size(1), (int)a.size(2), (int)c.size(2), call.stream);
}

// cos / sin as contiguous [positions, emb] tables of one type
// rows of the tables in a type that the kernels read; where a token's row is its number / batch, that many are there
std::pair<Tensor, Tensor> tables(const Tensor& cos_, const Tensor& sin_, int64_t emb, bool positions, int64_t batch, int64_t tokens) {
  Tensor cos = cos_.reshape({-1, emb}), sin = sin_.reshape({-1, emb});
  REQUIRE(positions || batch <= 0 || (tokens + batch - 1) / batch <= std::min(cos.size(0), sin.size(0)), "cos / sin tables are shorter than the sequence");
  if (cos.scalar_type() != at::kFloat && cos.scalar_type() != at::kBFloat16) { cos = cos.to(at::kFloat); sin = sin.to(at::kFloat); }
  if (sin.scalar_type() != cos.scalar_type()) sin = sin.to(cos.scalar_type());
  return {cos.contiguous(), sin.contiguous()};
}

void absorb_rope_query_into(const Tensor& q_up, const Tensor& w_, const Tensor& query, const Tensor& cos_, const Tensor& sin_, int64_t out_pairing,
                            const OptTensor& positions_, int64_t batch) {
  need_gpus(q_up, w_, query, cos_, sin_, positions_);
  need_bf16(q_up, w_, query);
  const int64_t S = q_up.size(0), H = q_up.dim() > 1 ? q_up.size(1) : 0;
  REQUIRE(q_up.dim() == 3 && q_up.size(2) == 192 && query.sizes() == at::IntArrayRef({S, H, 576}) && w_.sizes() == at::IntArrayRef({H, 512, 128}),
          "absorb_rope_query: shapes q_up ", q_up.sizes(), ", w ", w_.sizes(), ", query ", query.sizes(), " do not fit");
  REQUIRE(q_up.stride(2) == 1 && query.stride(2) == 1, "mla_absorb: rows must be contiguous");
  const Tensor w = w_.contiguous();
  const auto [cos, sin] = tables(cos_, sin_, 64, positions_.has_value(), batch, S);
  OptTensor positions;
  if (positions_) {
    positions = i32(*positions_);
    REQUIRE(positions->numel() == S, "positions must hold one entry per token");
  }
  Call call(q_up);
  run("dsa_absorb_rope_query", dsa_absorb_rope_query, q_up.const_data_ptr(), q_up.stride(0), q_up.stride(1), w.const_data_ptr(), query.data_ptr(), query.stride(0), query.stride(1), cos.const_data_ptr(), sin.const_data_ptr(), cos.scalar_type() == at::kFloat, (const int32_t*)ptr(positions), (int)batch, (int)S, (int)H, (int)out_pairing, call.stream);
}

// The two projections around the attention without autograd: output allocation and kernel in one call.  (The query side's kernel
// has one shape; the other pair of widths that the projection takes goes through the two kernels.)
py::object absorbed_query(const Tensor& q_up, const Tensor& w, const Tensor& cos, const Tensor& sin, const OptTensor& positions,
                          int64_t out_pairing) {
  if (!plain(q_up, w, cos, sin, positions) || q_up.dim() < 3 || w.dim() != 3 || w.size(1) != 512 || w.size(2) != 128 ||
      q_up.size(-1) != 192) return py::none();
  std::vector<int64_t> shape = q_up.sizes().vec();
  const int64_t batch = q_up.dim() == 4 ? q_up.size(1) : 1;
  const Tensor q3 = q_up.dim() == 3 ? q_up : q_up.reshape({-1, q_up.size(-2), q_up.size(-1)});
  Tensor query = make({q3.size(0), q3.size(1), w.size(1) + 64}, q_up.scalar_type(), q_up);
  absorb_rope_query_into(q3, w, query, cos, sin, out_pairing, positions, batch);
  shape.back() = query.size(2);
  return py::cast(q_up.dim() == 3 ? query : query.view(shape));
}

void rope_rows(const OptTensor& pe_src, const OptTensor& pe_dst, const OptTensor& cos_, const OptTensor& sin_, int64_t in_pairing,
               int64_t out_pairing, bool inverse, const OptTensor& positions_, int64_t batch, const OptTensor& main_src, const OptTensor& main_dst);

// kv [s, b, h, d] (packed: [t, h, d]) and the rotated k_pe that the heads share, side by side in new rows
py::object absorbed_key(const Tensor& kv, const Tensor& k_pe, const Tensor& cos, const Tensor& sin, const OptTensor& positions, int64_t emb,
                        bool packed, int64_t out_pairing) {
  if (!plain(kv, k_pe, cos, sin, positions) || kv.dim() != (packed ? 3 : 4) || !kv.is_contiguous() || !k_pe.is_contiguous() ||
      !cos.is_contiguous() || !sin.is_contiguous() || emb % 4) return py::none();
  const int64_t heads = kv.size(-2), d = kv.size(-1), T = packed ? kv.size(0) : kv.size(0) * kv.size(1);
  if (k_pe.numel() != T * emb) return py::none();
  Tensor key = make({T, heads, d + emb}, kv.scalar_type(), kv);
  rope_rows(k_pe.view({T, 1, emb}).expand({T, heads, emb}), key.narrow(2, d, emb), cos, sin, 0, out_pairing, false, positions,
            packed ? 1 : kv.size(1), kv.view({T, heads, d}), key.narrow(2, 0, d));
  return py::cast(packed ? key : key.view({kv.size(0), kv.size(1), heads, d + emb}));
}

py::object absorb(const Tensor& a, const Tensor& w, bool flat) {
  if (!plain(a, w) || a.dim() < 3 || w.dim() != 3) return py::none();
  const Tensor a3 = a.dim() == 3 ? a : a.reshape({-1, a.size(-2), a.size(-1)});
  Tensor out = make({a3.size(0), a3.size(1), w.size(1)}, a.scalar_type(), a);
  absorb_into(a3, w, out);
  if (!flat) return py::cast(out);
  std::vector<int64_t> shape = a.sizes().slice(0, a.dim() - 1).vec();
  shape.back() *= w.size(1);
  return py::cast(out.view(shape));
}

struct Rows { void* p; int64_t tok, head; };
Rows rows_view(const Tensor& t, const char* what) {
  REQUIRE(t.scalar_type() == at::kBFloat16 && t.dim() == 3 && (t.size(2) <= 1 || t.stride(2) == 1), what,
          " must be a bf16 [tokens, heads, width] view with unit inner stride");
  return {t.data_ptr(), t.stride(0), t.stride(1)};
}

void rope_rows(const OptTensor& pe_src, const OptTensor& pe_dst, const OptTensor& cos_, const OptTensor& sin_, int64_t in_pairing,
               int64_t out_pairing, bool inverse, const OptTensor& positions_, int64_t batch, const OptTensor& main_src, const OptTensor& main_dst) {
  REQUIRE(pe_dst || main_dst, "rope_rows: nothing to do");
  const Tensor& ref = pe_dst ? *pe_dst : *main_dst;
  need_gpus(pe_src, pe_dst, cos_, sin_, positions_, main_src, main_dst);
  const int64_t tokens = ref.size(0), heads = ref.size(1);
  int64_t emb = 0, d_main = 0;
  Rows ps{nullptr, 0, 0}, pd{nullptr, 0, 0}, ms{nullptr, 0, 0}, md{nullptr, 0, 0};
  Tensor cos, sin;
  OptTensor positions;
  if (pe_dst) {
    emb = pe_dst->size(2);
    REQUIRE(pe_src && pe_src->sizes() == pe_dst->sizes(), "pe_src and pe_dst differ in shape: ", pe_src ? c10::str(pe_src->sizes()) : "none", " vs ",
            pe_dst->sizes());
    REQUIRE(cos_ && sin_, "rope_rows: rotary part without cos / sin");
    ps = rows_view(*pe_src, "pe_src");
    pd = rows_view(*pe_dst, "pe_dst");
    std::tie(cos, sin) = tables(*cos_, *sin_, emb, positions_.has_value(), batch, tokens);
    if (positions_) {
      positions = i32(*positions_);
      REQUIRE(positions->numel() == tokens, "positions must hold one entry per token");
    }
  }
  if (main_dst) {
    REQUIRE(main_src && main_src->sizes() == main_dst->sizes() && main_dst->size(0) == tokens && main_dst->size(1) == heads,
            "main_src / main_dst shapes do not match the pe rows");
    d_main = main_dst->size(2);
    ms = rows_view(*main_src, "main_src");
    md = rows_view(*main_dst, "main_dst");
  }
  Call call(ref);
  run("dsa_rope_rows", dsa_rope_rows, ms.p, ms.tok, ms.head, md.p, md.tok, md.head, (int)d_main, ps.p, ps.tok, ps.head, pd.p, pd.tok, pd.head, (int)emb, emb ? cos.const_data_ptr() : nullptr, emb ? sin.const_data_ptr() : nullptr, emb && cos.scalar_type() == at::kFloat, emb ? (const int32_t*)ptr(positions) : nullptr, (int)batch, (int)tokens, (int)heads, (int)in_pairing, (int)out_pairing, inverse, call.stream);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("ordinary", &ordinary);
  m.doc() = "Native host layer of loongforge_amd.ops";
  py::class_<WindowCheck>(m, "WindowCheck").def("wait", &WindowCheck::wait);
#define DEF(name) m.def(#name, torch::wrap_pybind_function(name))
  DEF(quant_rowwise);
  DEF(rotate_quant);
  DEF(quant_weights);
  DEF(indexer_front);
  DEF(quant_padded);
  DEF(rotary_angles);
  DEF(rotary_cos_sin);
  DEF(token_rows);
  DEF(rope_steps);
  DEF(hadamard);
  DEF(indexer_topk);
  DEF(topk);
  DEF(indexer_bwd);
  DEF(indexer_grads);
  DEF(mla_fwd);
  DEF(mla_fwd_dist);
  DEF(pad_heads);
  DEF(mla_bwd);
  DEF(attn_dist);
  DEF(attn_dist_as_input);
  DEF(kl_loss);
  DEF(kl_total);
  DEF(kl_loss_total);
  DEF(kl_scale);
  DEF(indexer_window);
  DEF(indexer_forward);
  DEF(indexer_forward_narrow);
  DEF(thd_positions);
  DEF(absorb_into);
  DEF(absorb);
  DEF(absorb_rope_query_into);
  DEF(absorbed_query);
  DEF(absorbed_key);
  DEF(rope_rows);
#undef DEF
}
