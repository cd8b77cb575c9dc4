// PyTorch PrivateUse1 device `applegpu` on the MI355X backend.
//
// The reference registers aten kernels for PrivateUse1 that call its eager
// C ABI (backend_cpp/applegpu_backend.cpp:1055-1100: allocator, 39 kernels,
// a boxed CPU fallback, DeviceGuard, hooks, init at load).  This shim keeps
// that registration surface and the C ABI calls, with three changes the
// discrete-HBM device needs or the hot path gains from:
//   - a torch tensor maps to a typed eager view of its storage (dtype, byte
//     offset, strides: applegpu_eager_view_typed), created per call and freed
//     when the kernel returns;
//   - no host dereference of device pointers: copies, fill_, zero_ and _cat
//     run on the device (applegpu_eager_copy_*, _fill, concat);
//   - Linear (addmm) is one GEMM with the bias in its epilogue and the weight
//     read transposed in place; mse_loss and its backward are one kernel each.
// Every kernel computes on the device; ops without a kernel here go through
// the boxed CPU fallback (logged with APPLEGPU_LOG_FALLBACK=1, as in the
// reference, applegpu_backend.cpp:753-764).
#include <ATen/EmptyTensor.h>
#include <ATen/InferSize.h>
#include <ATen/core/op_registration/adaption.h>
#include <ATen/detail/PrivateUse1HooksInterface.h>
#include <ATen/native/CPUFallback.h>
#include <ATen/native/transformers/attention.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <torch/library.h>
#include <torch/torch.h>

#include <algorithm>
#include <cmath>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "applegpu_ffi.h"

namespace {

const c10::Device kDev(c10::DeviceType::PrivateUse1, 0);

[[noreturn]] void fail_last(const char* what) {
  const char* e = applegpu_eager_last_error();
  TORCH_CHECK(false, "applegpu ", what, " failed: ", e ? e : "unknown error");
}

// ── runtime init (lazy, so the library loads without a GPU) ─────────────────
bool g_ready = false;
std::string g_init_error;

void ensure_init() {
  if (g_ready) return;
  if (!applegpu_eager_init()) {
    const char* e = applegpu_eager_last_error();
    g_init_error = e ? e : "unknown error";
    TORCH_CHECK(false, "applegpu backend init failed: ", g_init_error);
  }
  (void)applegpu_ffi_init();
  g_ready = true;
}

// ── dtypes (wire codes of crates/core/src/tensor.rs:59-90) ──────────────────
int8_t wire_of(at::ScalarType st) {
  switch (st) {
    case at::kFloat: return 0;
    case at::kHalf: return 1;
    case at::kDouble: return 2;
    case at::kChar: return 3;
    case at::kShort: return 4;
    case at::kInt: return 5;
    case at::kLong: return 6;
    case at::kByte: return 7;
    case at::kBool: return 9;
    case at::kBFloat16: return 10;
    default: TORCH_CHECK(false, "applegpu: unsupported dtype ", c10::toString(st));
  }
}

at::ScalarType st_of(int8_t w) {
  switch (w) {
    case 0: return at::kFloat;
    case 1: return at::kHalf;
    case 2: return at::kDouble;
    case 3: return at::kChar;
    case 4: return at::kShort;
    case 5: return at::kInt;
    case 6: return at::kLong;
    case 7: return at::kByte;
    case 9: return at::kBool;
    case 10: return at::kBFloat16;
    default: TORCH_CHECK(false, "applegpu: unsupported wire dtype ", (int)w);
  }
}

// ── storage ─────────────────────────────────────────────────────────────────
struct Ctx {
  uint64_t id;
};

void free_ctx(void* p) {
  auto* c = static_cast<Ctx*>(p);
  applegpu_eager_free(c->id);
  delete c;
}

c10::DataPtr data_ptr_for(void* ptr, uint64_t id) {
  return c10::DataPtr(ptr, new Ctx{id}, &free_ctx, kDev);
}

struct ApplegpuAllocator final : public c10::Allocator {
  // Raw storage: a 1-D uint8 eager tensor of the byte count (zero bytes get
  // the runtime's minimum allocation, so every storage has an id).
  c10::DataPtr allocate(size_t nbytes) override {
    ensure_init();
    uint64_t n = nbytes, id = 0;
    void* p = applegpu_eager_alloc(&n, 1, 7, &id);
    if (!p) fail_last("alloc");
    return data_ptr_for(p, id);
  }
  c10::DeleterFnPtr raw_deleter() const override { return nullptr; }
  // Device-to-device copy between two allocations of this allocator.
  void copy_data(void* dest, const void* src, std::size_t count) const override {
    if (count == 0) return;
    const uint64_t did = applegpu_eager_find_by_data_ptr((const uint8_t*)dest);
    const uint64_t sid = applegpu_eager_find_by_data_ptr((const uint8_t*)src);
    TORCH_CHECK(did && sid, "applegpu: copy_data on pointers it did not allocate");
    uint64_t n = count, st = 1, dv = 0, sv = 0;
    if (!applegpu_eager_view_typed(did, &n, &st, 1, 0, 7, &dv)) fail_last("copy_data");
    if (!applegpu_eager_view_typed(sid, &n, &st, 1, 0, 7, &sv)) {
      applegpu_eager_free(dv);
      fail_last("copy_data");
    }
    const int32_t rc = applegpu_eager_copy_(dv, sv);
    applegpu_eager_free(dv);
    applegpu_eager_free(sv);
    if (rc != 0) fail_last("copy_data");
  }
};

ApplegpuAllocator g_allocator;

at::Tensor make_tensor(c10::Storage storage, at::ScalarType st, c10::IntArrayRef size, c10::IntArrayRef stride,
                       int64_t offset = 0) {
  auto t = at::detail::make_tensor<c10::TensorImpl>(std::move(storage), c10::DispatchKeySet(c10::DispatchKey::PrivateUse1),
                                                    c10::scalarTypeToTypeMeta(st));
  t.unsafeGetTensorImpl()->set_sizes_and_strides(size, stride, offset);
  return t;
}

// Wraps an eager output id (a contiguous tensor the runtime allocated).
at::Tensor wrap(uint64_t id) {
  uint64_t dims[8];
  uint32_t nd = 0;
  if (applegpu_eager_shape(id, dims, &nd) != 0) fail_last("shape");
  const int8_t w = applegpu_eager_dtype(id);
  void* p = applegpu_eager_data_ptr(id);
  if (!p) fail_last("data_ptr");
  std::vector<int64_t> sizes(dims, dims + nd);
  const auto st = st_of(w);
  int64_t numel = 1;
  for (auto d : sizes) numel *= d;
  c10::Storage storage(c10::Storage::use_byte_size_t(), numel * c10::elementSize(st), data_ptr_for(p, id),
                       &g_allocator, false);
  return make_tensor(std::move(storage), st, sizes, c10::contiguous_strides(sizes));
}

// Wraps any eager id, a strided view included, as a tensor that owns the id
// (freed with the storage).  The storage starts at the id's first element
// and spans the bytes its strides reach.  torch.compile graph outputs come
// back this way without a copy.
at::Tensor wrap_eager(int64_t id) {
  ensure_init();
  uint64_t dims[8];
  int64_t strides[8];
  uint32_t nd = 0, nd2 = 0;
  if (applegpu_eager_shape((uint64_t)id, dims, &nd) != 0) fail_last("shape");
  if (applegpu_eager_strides((uint64_t)id, strides, &nd2) != 0 || nd2 != nd) fail_last("strides");
  const auto st = st_of(applegpu_eager_dtype((uint64_t)id));
  std::vector<int64_t> sizes(dims, dims + nd), str(strides, strides + nd);
  int64_t numel = 1, last = 0;
  for (uint32_t i = 0; i < nd; ++i) {
    numel *= sizes[i];
    last += (sizes[i] - 1) * str[i];
  }
  void* p = applegpu_eager_data_ptr((uint64_t)id);
  if (!p && numel > 0) fail_last("data_ptr");
  const size_t bytes = numel > 0 ? (size_t)(last + 1) * c10::elementSize(st) : 0;
  c10::Storage storage(c10::Storage::use_byte_size_t(), bytes, data_ptr_for(p, (uint64_t)id), &g_allocator, false);
  return make_tensor(std::move(storage), st, sizes, str);
}

// Wraps an output as `like`'s shape when the runtime returned a [1] scalar.
at::Tensor wrap_as(uint64_t id, c10::IntArrayRef sizes) {
  at::Tensor t = wrap(id);
  if (t.sizes() != sizes) t = t.view(sizes);
  return t;
}

// Typed eager views of torch tensors, freed when the kernel returns.
struct Views {
  std::vector<uint64_t> ids;
  Views() = default;
  Views(const Views&) = delete;
  ~Views() {
    for (uint64_t id : ids) applegpu_eager_free(id);
  }
  uint64_t of(const at::Tensor& t) {
    TORCH_CHECK(t.device().type() == c10::DeviceType::PrivateUse1, "applegpu: expected an applegpu tensor, got ",
                t.device());
    auto* ctx = static_cast<Ctx*>(t.storage().data_ptr().get_context());
    TORCH_CHECK(ctx, "applegpu: tensor has no applegpu storage");
    const int64_t nd = std::max<int64_t>(t.dim(), 1);
    std::vector<uint64_t> shape(nd, 1), strides(nd, 1);
    for (int64_t i = 0; i < t.dim(); ++i) {
      shape[i] = (uint64_t)t.size(i);
      strides[i] = (uint64_t)t.stride(i);
    }
    uint64_t id = 0;
    if (!applegpu_eager_view_typed(ctx->id, shape.data(), strides.data(), (uint32_t)nd,
                                   (uint64_t)(t.storage_offset() * t.element_size()), wire_of(t.scalar_type()), &id) &&
        !id)
      fail_last("view");
    ids.push_back(id);
    return id;
  }
};

// One generic eager op (applegpu_eager_op) -> its single output id.
uint64_t run(const char* op, std::initializer_list<uint64_t> in, std::vector<double> f = {},
             std::vector<int64_t> iv = {}) {
  std::vector<uint64_t> ids(in);
  uint64_t out = 0;
  const int32_t n = applegpu_eager_op(op, ids.data(), (uint32_t)ids.size(), f.empty() ? nullptr : f.data(),
                                      (uint32_t)f.size(), iv.empty() ? nullptr : iv.data(), (uint32_t)iv.size(), &out, 1);
  if (n != 1) fail_last(op);
  return out;
}

at::Tensor run_t(const char* op, std::initializer_list<at::Tensor> in, std::vector<double> f = {},
                 std::vector<int64_t> iv = {}) {
  Views v;
  std::vector<uint64_t> ids;
  for (const auto& t : in) ids.push_back(v.of(t));
  uint64_t out = 0;
  const int32_t n = applegpu_eager_op(op, ids.data(), (uint32_t)ids.size(), f.empty() ? nullptr : f.data(),
                                      (uint32_t)f.size(), iv.empty() ? nullptr : iv.data(), (uint32_t)iv.size(), &out, 1);
  if (n != 1) fail_last(op);
  return wrap(out);
}

bool on_dev(const at::Tensor& t) { return t.device().type() == c10::DeviceType::PrivateUse1; }

// A CPU "wrapped number" (a Python scalar in a binary op) or any CPU tensor
// moved to the device in the other operand's dtype.
at::Tensor to_dev(const at::Tensor& t, at::ScalarType st) {
  if (on_dev(t)) return t.scalar_type() == st ? t : t.to(st);
  return t.to(st).to(kDev);
}

// ── tensor creation and copies ──────────────────────────────────────────────
at::Tensor ag_empty_strided(c10::IntArrayRef size, c10::IntArrayRef stride, std::optional<at::ScalarType> dtype,
                         std::optional<at::Layout>, std::optional<at::Device>, std::optional<bool>) {
  const auto st = dtype.value_or(at::kFloat);
  const int64_t nbytes = at::detail::computeStorageNbytes(size, stride, c10::elementSize(st));
  c10::Storage storage(c10::Storage::use_byte_size_t(), nbytes, g_allocator.allocate(nbytes), &g_allocator, true);
  return make_tensor(std::move(storage), st, size, stride);
}

at::Tensor ag_empty_memory_format(c10::IntArrayRef size, std::optional<at::ScalarType> dtype,
                               std::optional<at::Layout> layout, std::optional<at::Device> device,
                               std::optional<bool> pin, std::optional<at::MemoryFormat>) {
  return ag_empty_strided(size, c10::contiguous_strides(size), dtype, layout, device, pin);
}

// dst = src for any pair of devices with at least one on applegpu.
void copy_any(const at::Tensor& dst, const at::Tensor& src) {
  if (dst.numel() == 0) return;
  TORCH_CHECK(dst.numel() == src.numel() || src.numel() == 1, "applegpu copy: size mismatch ", dst.sizes(), " vs ",
              src.sizes());
  if (on_dev(dst) && on_dev(src)) {
    Views v;
    at::Tensor s = src.numel() == dst.numel() ? src : src.expand(dst.sizes());
    if (s.numel() != dst.numel() || s.sizes() != dst.sizes()) s = s.reshape(dst.sizes());
    if (applegpu_eager_copy_(v.of(dst), v.of(s)) != 0) fail_last("copy_");
    return;
  }
  if (on_dev(dst)) {  // host -> device
    at::Tensor h = src.to(dst.scalar_type()).expand(dst.sizes()).contiguous();
    Views v;
    if (applegpu_eager_copy_from_host(v.of(dst), h.data_ptr(), h.nbytes()) != 0) fail_last("copy from host");
    return;
  }
  // device -> host
  at::Tensor c = src.contiguous();
  at::Tensor h = at::empty(c.sizes(), c.options().device(c10::kCPU));
  {
    Views v;
    if (applegpu_eager_copy_to_host(v.of(c), h.data_ptr(), h.nbytes()) != 0) fail_last("copy to host");
  }
  dst.copy_(h);
}

at::Tensor& ag_copy_(at::Tensor& self, const at::Tensor& src, bool) {
  copy_any(self, src);
  return self;
}

at::Tensor ag_copy_from(const at::Tensor& self, const at::Tensor& dst, bool) {
  copy_any(dst, self);
  return dst;
}

at::Tensor ag_copy_from_and_resize(const at::Tensor& self, const at::Tensor& dst) {
  dst.resize_(self.sizes());
  copy_any(dst, self);
  return dst;
}

const at::Tensor& ag_resize_(const at::Tensor& self, c10::IntArrayRef size, std::optional<at::MemoryFormat>) {
  auto* impl = self.unsafeGetTensorImpl();
  const auto strides = c10::contiguous_strides(size);
  const int64_t need = at::detail::computeStorageNbytes(size, strides, self.element_size()) +
                       self.storage_offset() * self.element_size();
  if (need > (int64_t)self.storage().nbytes()) {
    c10::Storage fresh(c10::Storage::use_byte_size_t(), need, g_allocator.allocate(need), &g_allocator, true);
    const int64_t keep = (int64_t)self.storage().nbytes();
    if (keep > 0) g_allocator.copy_data(fresh.mutable_data(), self.storage().data(), keep);
    impl->set_storage_keep_dtype(fresh);
  }
  impl->set_sizes_and_strides(size, strides, self.storage_offset());
  return self;
}

// ── views (metadata only; storage shared) ───────────────────────────────────
at::Tensor alias(const at::Tensor& self, c10::IntArrayRef size, c10::IntArrayRef stride, int64_t offset) {
  return make_tensor(self.storage(), self.scalar_type(), size, stride, offset);
}

at::Tensor ag_view(const at::Tensor& self, c10::SymIntArrayRef size_sym) {
  auto size = C10_AS_INTARRAYREF_SLOW(size_sym);
  auto inferred = at::infer_size_dv(size, self.numel());
  auto stride = at::detail::computeStride(self.sizes(), self.strides(), inferred);
  TORCH_CHECK(stride.has_value(), "applegpu view: size is not compatible with the input's strides; use reshape");
  return alias(self, inferred, *stride, self.storage_offset());
}

at::Tensor ag_reshape_alias(const at::Tensor& self, c10::SymIntArrayRef size, c10::SymIntArrayRef stride) {
  return alias(self, C10_AS_INTARRAYREF_SLOW(size), C10_AS_INTARRAYREF_SLOW(stride), self.storage_offset());
}

at::Tensor ag_as_strided(const at::Tensor& self, c10::SymIntArrayRef size, c10::SymIntArrayRef stride,
                      std::optional<c10::SymInt> offset) {
  const int64_t off = offset.has_value() ? offset->expect_int() : self.storage_offset();
  return alias(self, C10_AS_INTARRAYREF_SLOW(size), C10_AS_INTARRAYREF_SLOW(stride), off);
}

// ── elementwise ─────────────────────────────────────────────────────────────
at::ScalarType promoted(const at::Tensor& a, const at::Tensor& b) { return at::result_type(a, b); }

at::Tensor binary(const char* op, const at::Tensor& a, const at::Tensor& b) {
  const auto st = promoted(a, b);
  return run_t(op, {to_dev(a, st), to_dev(b, st)});
}

at::Tensor scaled(const at::Tensor& t, double s) { return s == 1.0 ? t : run_t("scalar_mul", {t}, {s}); }

at::Tensor ag_add(const at::Tensor& a, const at::Tensor& b, const at::Scalar& alpha) {
  const double al = alpha.toDouble();
  const auto st = promoted(a, b);
  return run_t("add", {to_dev(a, st), scaled(to_dev(b, st), al)});
}
at::Tensor ag_sub(const at::Tensor& a, const at::Tensor& b, const at::Scalar& alpha) {
  const double al = alpha.toDouble();
  const auto st = promoted(a, b);
  return run_t("sub", {to_dev(a, st), scaled(to_dev(b, st), al)});
}
at::Tensor ag_mul(const at::Tensor& a, const at::Tensor& b) {
  if (!on_dev(b) && b.dim() == 0 && at::isFloatingType(a.scalar_type())) return run_t("scalar_mul", {a}, {b.item<double>()});
  return binary("mul", a, b);
}
at::Tensor ag_div(const at::Tensor& a, const at::Tensor& b) {
  if (!on_dev(b) && b.dim() == 0 && at::isFloatingType(a.scalar_type()))
    return run_t("scalar_mul", {a}, {1.0 / b.item<double>()});
  return binary("div", a, b);
}
at::Tensor ag_mul_scalar(const at::Tensor& a, const at::Scalar& s) { return run_t("scalar_mul", {a}, {s.toDouble()}); }
at::Tensor ag_div_scalar(const at::Tensor& a, const at::Scalar& s) {
  return run_t("scalar_mul", {a}, {1.0 / s.toDouble()});
}

// In-place: self += alpha * other (the reference's add_scaled_inplace,
// crates/core/src/eager.rs:1084-1096); other layouts compute out of place.
at::Tensor& ag_add_(at::Tensor& self, const at::Tensor& other, const at::Scalar& alpha) {
  const at::Tensor o = to_dev(other, self.scalar_type());
  if (self.is_contiguous()) {
    Views v;
    if (applegpu_eager_add_scaled_inplace(v.of(self), v.of(o), (float)alpha.toDouble()) == 0) return self;
  }
  copy_any(self, ag_add(self, o, alpha));
  return self;
}
at::Tensor& ag_mul_(at::Tensor& self, const at::Tensor& other) {
  copy_any(self, ag_mul(self, other));
  return self;
}
at::Tensor& ag_mul_scalar_(at::Tensor& self, const at::Scalar& s) {
  copy_any(self, ag_mul_scalar(self, s));
  return self;
}
at::Tensor& ag_fill_(at::Tensor& self, const at::Scalar& value) {
  if (self.numel() == 0) return self;
  Views v;
  if (applegpu_eager_fill(v.of(self), value.toDouble()) != 0) fail_last("fill_");
  return self;
}
at::Tensor& ag_zero_(at::Tensor& self) { return ag_fill_(self, 0); }

at::Tensor ag_relu(const at::Tensor& x) { return run_t("relu", {x}); }
at::Tensor ag_neg(const at::Tensor& x) { return run_t("neg", {x}); }
at::Tensor ag_tanh_(const at::Tensor& x) { return run_t("tanh", {x}); }
at::Tensor ag_exp_(const at::Tensor& x) { return run_t("exp", {x}); }
at::Tensor ag_sigmoid_(const at::Tensor& x) { return run_t("sigmoid", {x}); }
at::Tensor ag_gelu(const at::Tensor& x, c10::string_view approximate) {
  return run_t(approximate == "tanh" ? "gelu" : "gelu_exact", {x});
}
at::Tensor ag_threshold_backward(const at::Tensor& grad, const at::Tensor& self, const at::Scalar& thr) {
  return run_t("threshold_backward", {grad, self}, {thr.toDouble()});
}

// ── GEMM ────────────────────────────────────────────────────────────────────
at::Tensor ag_mm(const at::Tensor& a, const at::Tensor& b) { return run_t("matmul", {a, b}); }
at::Tensor ag_bmm(const at::Tensor& a, const at::Tensor& b) { return run_t("matmul", {a, b}); }

// ag_addmm(bias, x, W^T) = x W^T + bias: Linear in one GEMM, bias in the
// epilogue, the weight read through its transpose in place (the reference
// copies W^T and adds the bias in a second kernel, applegpu_backend.cpp:584-620).
at::Tensor ag_addmm(const at::Tensor& bias, const at::Tensor& m1, const at::Tensor& m2, const at::Scalar& beta,
                 const at::Scalar& alpha) {
  const double be = beta.toDouble(), al = alpha.toDouble();
  if (be == 1.0 && al == 1.0 && bias.dim() == 1 && bias.size(0) == m2.size(1) && m2.dim() == 2) {
    // W [N, K] as a view of m2 [K, N]: swap sizes and strides.
    at::Tensor w = alias(m2, {m2.size(1), m2.size(0)}, {m2.stride(1), m2.stride(0)}, m2.storage_offset());
    Views v;
    uint64_t out = 0;
    if (!applegpu_eager_linear(v.of(m1), v.of(w), v.of(bias.contiguous()), 0, &out)) fail_last("addmm");
    return wrap(out);
  }
  at::Tensor prod = scaled(ag_mm(m1, m2), al);
  if (be == 0.0) return prod;
  return ag_add(prod, bias, be);
}

// ── losses and reductions ───────────────────────────────────────────────────
at::Tensor ag_mse_loss(const at::Tensor& self, const at::Tensor& target, int64_t reduction) {
  if (reduction == at::Reduction::None) {
    at::Tensor d = run_t("sub", {self, target});
    return run_t("mul", {d, d});
  }
  Views v;
  uint64_t out = 0;
  if (!applegpu_eager_mse_loss(v.of(self), v.of(target), &out)) fail_last("mse_loss");
  at::Tensor m = wrap_as(out, {});
  return reduction == at::Reduction::Sum ? ag_mul_scalar(m, (double)self.numel()) : m;
}

at::Tensor ag_mse_loss_backward(const at::Tensor& grad, const at::Tensor& self, const at::Tensor& target,
                             int64_t reduction) {
  if (reduction == at::Reduction::None) {
    at::Tensor d = run_t("sub", {self, target});
    return run_t("mul", {scaled(d, 2.0), to_dev(grad, self.scalar_type())});
  }
  Views v;
  uint64_t out = 0;
  const at::Tensor g = grad.reshape({1});
  if (!applegpu_eager_mse_loss_backward(v.of(g), v.of(self), v.of(target), &out)) fail_last("mse_loss_backward");
  at::Tensor r = wrap(out);
  return reduction == at::Reduction::Sum ? ag_mul_scalar(r, (double)self.numel()) : r;
}

at::Tensor ag_sum_dim(const at::Tensor& self, at::OptionalIntArrayRef dims, bool keepdim, std::optional<at::ScalarType> dtype) {
  at::Tensor x = dtype.has_value() && *dtype != self.scalar_type() ? self.to(*dtype) : self;
  std::vector<int64_t> ds;
  if (dims.has_value() && !dims->empty()) {
    for (int64_t d : *dims) ds.push_back(c10::maybe_wrap_dim(d, x.dim()));
  } else {
    for (int64_t d = 0; d < x.dim(); ++d) ds.push_back(d);
  }
  std::sort(ds.rbegin(), ds.rend());
  if (x.dim() == 0) return x.clone();
  for (int64_t d : ds) x = run_t("sum_dim", {x}, {}, {d, 1});
  if (!keepdim) {
    std::vector<int64_t> out;
    for (int64_t d = 0; d < x.dim(); ++d)
      if (std::find(ds.begin(), ds.end(), d) == ds.end()) out.push_back(x.size(d));
    x = x.reshape(out);
  }
  return x;
}

at::Tensor ag_sum(const at::Tensor& self, std::optional<at::ScalarType> dtype) {
  return ag_sum_dim(self, at::OptionalIntArrayRef(), false, dtype);
}

// ── GPT-2 ops ───────────────────────────────────────────────────────────────
at::Tensor ag_embedding(const at::Tensor& weight, const at::Tensor& indices, int64_t, bool, bool) {
  at::Tensor flat = run_t("embedding", {weight, indices.reshape({-1})});
  std::vector<int64_t> shape(indices.sizes().begin(), indices.sizes().end());
  shape.push_back(weight.size(1));
  return flat.view(shape);
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> ag_native_layer_norm(const at::Tensor& input, c10::SymIntArrayRef nshape,
                                                                 const std::optional<at::Tensor>& weight,
                                                                 const std::optional<at::Tensor>& bias, double eps) {
  const int64_t cols = input.size(-1);
  TORCH_CHECK(nshape.size() == 1, "applegpu native_layer_norm: normalized over the last dim only");
  at::Tensor g = weight.has_value() && weight->defined() ? *weight : at::ones({cols}, input.options());
  at::Tensor b = bias.has_value() && bias->defined() ? *bias : at::zeros({cols}, input.options());
  std::vector<int64_t> sshape(input.sizes().begin(), input.sizes().end());
  sshape.back() = 1;
  // Row statistics for autograd, mean and 1/sqrt(var + eps) as [..., 1]: from
  // the launch that normalises.  As ops of their own (mean, var, three fills,
  // add, sqrt, div) they were eight launches after it: a training step of a
  // transformer block, 2048 tokens of 768, takes 943 us instead of 1000.
  if (cols > 0) {
    Views v;
    uint64_t ins[3] = {v.of(input), v.of(g), v.of(b)};
    uint64_t out[3] = {0, 0, 0};
    if (applegpu_eager_op("layer_norm_stats", ins, 3, &eps, 1, nullptr, 0, out, 3) != 3) fail_last("layer_norm_stats");
    at::Tensor y = wrap(out[0]), mean = wrap(out[1]), rstd = wrap(out[2]);
    return {y, mean.view(sshape), rstd.view(sshape)};
  }
  // rows of no columns: what the reductions make of them
  at::Tensor y = run_t("layer_norm", {input, g, b}, {eps});
  at::Tensor mean = run_t("mean", {input}).view(sshape);
  at::Tensor var = run_t("var", {input}, {}, {0});
  at::Tensor eps_t = at::full({1}, eps, input.options());
  at::Tensor rstd = run_t("div", {at::ones({1}, input.options()), run_t("sqrt", {run_t("add", {var, eps_t})})}).view(sshape);
  return {y, mean, rstd};
}

// dx (and dgamma, dbeta) from the forward's saved mean and rstd, so the
// forward's eps carries over; the reference recomputes with eps = 1e-5 and
// forms dgamma/dbeta on the CPU (python/applegpu_runtime/torch_backend.py:1652-1692).
std::tuple<at::Tensor, at::Tensor, at::Tensor> ag_native_layer_norm_backward(
    const at::Tensor& grad_out, const at::Tensor& input, c10::SymIntArrayRef nshape, const at::Tensor& mean,
    const at::Tensor& rstd, const std::optional<at::Tensor>& weight, const std::optional<at::Tensor>& bias,
    std::array<bool, 3> mask) {
  TORCH_CHECK(nshape.size() == 1, "applegpu native_layer_norm_backward: normalized over the last dim only");
  const int64_t cols = input.size(-1);
  const bool has_w = weight.has_value() && weight->defined();
  at::Tensor g = has_w ? *weight : at::ones({cols}, input.options());
  Views v;
  uint64_t ins[5] = {v.of(grad_out), v.of(input), v.of(g), v.of(mean.to(input.scalar_type())),
                     v.of(rstd.to(input.scalar_type()))};
  uint64_t out[3] = {0, 0, 0};
  const double eps = 1e-5;  // unused: the saved statistics are used
  if (applegpu_eager_op("layer_norm_grads", ins, 5, &eps, 1, nullptr, 0, out, 3) != 3) fail_last("layer_norm_grads");
  at::Tensor dx = wrap(out[0]), dg = wrap(out[1]), db = wrap(out[2]);
  return {mask[0] ? dx.view(input.sizes()) : at::Tensor(), mask[1] && has_w ? dg : at::Tensor(),
          mask[2] && bias.has_value() && bias->defined() ? db : at::Tensor()};
}

at::Tensor ag_gelu_backward(const at::Tensor& grad, const at::Tensor& self, c10::string_view approximate) {
  return run_t(approximate == "tanh" ? "gelu_backward" : "gelu_exact_backward", {grad, self});
}

// Rows summed in token order on the device (deterministic); padding_idx's
// row stays zero as torch defines it.
at::Tensor ag_embedding_dense_backward(const at::Tensor& grad, const at::Tensor& indices, c10::SymInt num_weights,
                                       c10::SymInt padding_idx, bool scale_grad_by_freq) {
  TORCH_CHECK(!scale_grad_by_freq, "applegpu embedding backward: scale_grad_by_freq is not supported");
  const int64_t nw = num_weights.expect_int(), pad = padding_idx.expect_int();
  at::Tensor idx = indices.reshape({-1});
  at::Tensor g = grad.reshape({idx.numel(), grad.size(-1)});
  at::Tensor dw = run_t("embedding_backward", {g, idx}, {}, {nw});
  if (pad >= 0 && pad < nw) dw.select(0, pad).zero_();
  return dw;
}

at::Tensor ag_softmax_backward_data(const at::Tensor& grad, const at::Tensor& out, int64_t dim,
                                    at::ScalarType input_dtype) {
  TORCH_CHECK(input_dtype == grad.scalar_type(), "applegpu _softmax_backward_data: mixed dtypes are not supported");
  const int64_t d = c10::maybe_wrap_dim(dim, grad.dim());
  if (d == grad.dim() - 1) return run_t("softmax_backward", {grad, out});
  return run_t("softmax_backward", {grad.transpose(d, -1), out.transpose(d, -1)}).transpose(d, -1);
}

// ── masks ───────────────────────────────────────────────────────────────────
at::Tensor ag_masked_fill(const at::Tensor& self, const at::Tensor& mask, const at::Scalar& value) {
  return run_t("masked_fill", {self, to_dev(mask, at::kBool)}, {value.toDouble()});
}
at::Tensor& ag_masked_fill_(at::Tensor& self, const at::Tensor& mask, const at::Scalar& value) {
  self.copy_(ag_masked_fill(self, mask, value));
  return self;
}
at::Tensor ag_where(const at::Tensor& cond, const at::Tensor& self, const at::Tensor& other) {
  const auto st = at::result_type(self, other);
  return run_t("where", {to_dev(cond, at::kBool), to_dev(self, st), to_dev(other, st)});
}
at::Tensor ag_triu(const at::Tensor& self, int64_t diagonal) { return run_t("triu", {self}, {}, {diagonal}); }
at::Tensor ag_tril(const at::Tensor& self, int64_t diagonal) { return run_t("tril", {self}, {}, {diagonal}); }

// ── scaled_dot_product_attention ────────────────────────────────────────────
// torch asks _fused_sdp_choice which backend serves SDPA on this device.
// Calls without a mask, dropout or grouped K/V go to the fused attention
// kernel through the overrideable backend; anything else takes torch's math
// path, whose ops are device kernels too.  The reference registers neither
// and runs SDPA through its CPU fallback.
int64_t ag_fused_sdp_choice(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                            const std::optional<at::Tensor>& mask, double dropout, bool, std::optional<double>,
                            bool enable_gqa) {
  const bool fused = !(mask.has_value() && mask->defined()) && dropout == 0.0 && !enable_gqa && q.dim() >= 2 &&
                     q.dim() <= 4 && k.dim() == q.dim() && v.dim() == q.dim() && q.size(-1) == k.size(-1) &&
                     v.size(-1) == q.size(-1) && k.size(-2) == v.size(-2) && q.scalar_type() == k.scalar_type() &&
                     q.scalar_type() == v.scalar_type() && at::isFloatingType(q.scalar_type()) &&
                     q.scalar_type() != at::kDouble;
  bool same_lead = fused;
  for (int64_t i = 0; same_lead && i < q.dim() - 2; ++i) same_lead = k.size(i) == q.size(i) && v.size(i) == q.size(i);
  return same_lead ? 4 /* SDPBackend::overrideable */ : 0 /* SDPBackend::math */;
}

double sdp_scale(const at::Tensor& q, std::optional<double> scale) {
  return scale.has_value() ? *scale : 1.0 / std::sqrt((double)q.size(-1));
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, c10::SymInt, c10::SymInt, at::Tensor, at::Tensor, at::Tensor>
ag_sdpa_overrideable(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                     const std::optional<at::Tensor>& bias, double dropout, bool is_causal, bool,
                     std::optional<double> scale) {
  TORCH_CHECK(!(bias.has_value() && bias->defined()) && dropout == 0.0,
              "applegpu fused attention: no attention bias or dropout");
  at::Tensor out = run_t(is_causal ? "attention_causal" : "attention", {q, k, v}, {sdp_scale(q, scale)});
  // logsumexp is not formed (the backward recomputes the probabilities); an
  // empty [..., Tq] float tensor stands in for it
  std::vector<int64_t> ls(q.sizes().begin(), q.sizes().end() - 1);
  at::Tensor lse = at::empty(ls, q.options().dtype(at::kFloat));
  return {out, lse, at::Tensor(), at::Tensor(), c10::SymInt(q.size(-2)), c10::SymInt(k.size(-2)), at::Tensor(),
          at::Tensor(), at::Tensor()};
}

// One op (fp32: the fused backward kernel; else P recomputed and the products
// on the device GEMM).
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> ag_sdpa_overrideable_backward(
    const at::Tensor& go, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor&,
    std::array<bool, 4> mask, const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&,
    c10::SymInt, c10::SymInt, double dropout, bool is_causal, const at::Tensor&, const at::Tensor&,
    std::optional<double> scale) {
  TORCH_CHECK(dropout == 0.0, "applegpu fused attention backward: no dropout");
  const double s = sdp_scale(q, scale);
  Views vw;
  uint64_t ins[4] = {vw.of(go), vw.of(q), vw.of(k), vw.of(v)}, outs[3] = {0, 0, 0};
  const int64_t iv[4] = {is_causal, mask[0], mask[1], mask[2]};
  if (applegpu_eager_op("attention_backward", ins, 4, &s, 1, iv, 4, outs, 3) != 3) fail_last("attention_backward");
  at::Tensor g[3];
  for (int i = 0; i < 3; ++i) {
    at::Tensor t = wrap(outs[i]);
    if (mask[i]) g[i] = t;
  }
  return {g[0], g[1], g[2], at::Tensor()};
}

at::Tensor ag_softmax(const at::Tensor& self, int64_t dim, bool half_to_float) {
  TORCH_CHECK(!half_to_float, "applegpu _softmax: half_to_float is not supported");
  const int64_t d = c10::maybe_wrap_dim(dim, self.dim());
  if (d == self.dim() - 1) return run_t("softmax", {self});
  return run_t("softmax", {self.transpose(d, -1)}).transpose(d, -1);
}
at::Tensor ag_log_softmax(const at::Tensor& self, int64_t dim, bool half_to_float) {
  TORCH_CHECK(!half_to_float, "applegpu _log_softmax: half_to_float is not supported");
  const int64_t d = c10::maybe_wrap_dim(dim, self.dim());
  if (d == self.dim() - 1) return run_t("log_softmax", {self});
  return run_t("log_softmax", {self.transpose(d, -1)}).transpose(d, -1);
}

at::Tensor ag_cat(const at::ITensorListRef& tensors, int64_t dim) {
  std::vector<at::Tensor> ts;
  for (const auto& t : tensors)
    if (t.numel() > 0 || t.dim() > 1) ts.push_back(t);
  TORCH_CHECK(!ts.empty(), "applegpu cat: no tensors");
  const int64_t d = c10::maybe_wrap_dim(dim, ts[0].dim());
  at::Tensor acc = ts[0];
  for (size_t i = 1; i < ts.size(); ++i) acc = run_t("concat", {acc, ts[i]}, {}, {d});
  return ts.size() == 1 ? acc.clone() : acc;
}

at::Tensor ag_clone(const at::Tensor& self, std::optional<at::MemoryFormat>) {
  at::Tensor out = ag_empty_strided(self.sizes(), c10::contiguous_strides(self.sizes()), self.scalar_type(), {}, {}, {});
  copy_any(out, self);
  return out;
}

// .item(): one element read back to the host.
at::Scalar ag_local_scalar_dense(const at::Tensor& self) {
  at::Tensor h = at::empty({}, self.options().device(c10::kCPU));
  copy_any(h, self);
  return h.item();
}

// ── CPU fallback for everything else ────────────────────────────────────────
std::atomic<uint64_t> g_fallbacks{0};

void cpu_fallback(const c10::OperatorHandle& op, torch::jit::Stack* stack) {
  g_fallbacks.fetch_add(1, std::memory_order_relaxed);
  static const bool log = [] {
    const char* v = std::getenv("APPLEGPU_LOG_FALLBACK");
    return v && *v && *v != '0';
  }();
  if (log) fprintf(stderr, "[applegpu] CPU fallback: %s\n", op.schema().operator_name().name.c_str());
  at::native::cpu_fallback(op, stack);
}

}  // namespace

TORCH_LIBRARY_IMPL(aten, PrivateUse1, m) {
  m.impl("empty.memory_format", ag_empty_memory_format);
  m.impl("empty_strided", ag_empty_strided);
  m.impl("copy_", ag_copy_);
  m.impl("_copy_from", ag_copy_from);
  m.impl("_copy_from_and_resize", ag_copy_from_and_resize);
  m.impl("resize_", ag_resize_);
  m.impl("clone", ag_clone);
  m.impl("view", ag_view);
  m.impl("_reshape_alias", ag_reshape_alias);
  m.impl("as_strided", ag_as_strided);
  m.impl("add.Tensor", ag_add);
  m.impl("sub.Tensor", ag_sub);
  m.impl("mul.Tensor", ag_mul);
  m.impl("div.Tensor", ag_div);
  m.impl("mul.Scalar", ag_mul_scalar);
  m.impl("div.Scalar", ag_div_scalar);
  m.impl("add_.Tensor", ag_add_);
  m.impl("mul_.Tensor", ag_mul_);
  m.impl("mul_.Scalar", ag_mul_scalar_);
  m.impl("fill_.Scalar", ag_fill_);
  m.impl("zero_", ag_zero_);
  m.impl("relu", ag_relu);
  m.impl("neg", ag_neg);
  m.impl("tanh", ag_tanh_);
  m.impl("exp", ag_exp_);
  m.impl("sigmoid", ag_sigmoid_);
  m.impl("gelu", ag_gelu);
  m.impl("threshold_backward", ag_threshold_backward);
  m.impl("mm", ag_mm);
  m.impl("bmm", ag_bmm);
  m.impl("addmm", ag_addmm);
  m.impl("mse_loss", ag_mse_loss);
  m.impl("mse_loss_backward", ag_mse_loss_backward);
  m.impl("sum.dim_IntList", ag_sum_dim);
  m.impl("sum", ag_sum);
  m.impl("embedding", ag_embedding);
  m.impl("native_layer_norm", ag_native_layer_norm);
  m.impl("native_layer_norm_backward", ag_native_layer_norm_backward);
  m.impl("gelu_backward", ag_gelu_backward);
  m.impl("embedding_dense_backward", ag_embedding_dense_backward);
  m.impl("_softmax_backward_data", ag_softmax_backward_data);
  m.impl("masked_fill.Scalar", ag_masked_fill);
  m.impl("masked_fill_.Scalar", ag_masked_fill_);
  m.impl("where.self", ag_where);
  m.impl("triu", ag_triu);
  m.impl("tril", ag_tril);
  m.impl("_fused_sdp_choice", ag_fused_sdp_choice);
  m.impl("_scaled_dot_product_fused_attention_overrideable", ag_sdpa_overrideable);
  m.impl("_scaled_dot_product_fused_attention_overrideable_backward", ag_sdpa_overrideable_backward);
  m.impl("_softmax", ag_softmax);
  m.impl("_log_softmax", ag_log_softmax);
  m.impl("cat", ag_cat);
  m.impl("_local_scalar_dense", ag_local_scalar_dense);
}

// torch.ops.applegpu.wrap_eager(id): see wrap_eager above.
TORCH_LIBRARY(applegpu, m) { m.def("wrap_eager(int id) -> Tensor", &wrap_eager); }

TORCH_LIBRARY_IMPL(_, PrivateUse1, m) { m.fallback(torch::CppFunction::makeFromBoxedFunction<&cpu_fallback>()); }

// scaled_dot_product_attention reads its backend choice from this stub
// (the _fused_sdp_choice op above answers the same question when called).
namespace at::native {
REGISTER_PRIVATEUSE1_DISPATCH(_fused_sdp_choice_stub, &ag_fused_sdp_choice);
}

// ── DeviceGuard, hooks, allocator registration ──────────────────────────────
namespace {

struct GuardImpl final : public c10::impl::DeviceGuardImplInterface {
  c10::DeviceType type() const override { return c10::DeviceType::PrivateUse1; }
  c10::Device exchangeDevice(c10::Device) const override { return kDev; }
  c10::Device getDevice() const override { return kDev; }
  void setDevice(c10::Device) const override {}
  void uncheckedSetDevice(c10::Device) const noexcept override {}
  c10::Stream getStream(c10::Device) const noexcept override { return c10::Stream(c10::Stream::DEFAULT, kDev); }
  c10::Stream getDefaultStream(c10::Device) const override { return c10::Stream(c10::Stream::DEFAULT, kDev); }
  c10::Stream exchangeStream(c10::Stream) const noexcept override { return c10::Stream(c10::Stream::DEFAULT, kDev); }
  c10::DeviceIndex deviceCount() const noexcept override { return 1; }
};

struct Hooks : public at::PrivateUse1HooksInterface {
  bool hasPrimaryContext(c10::DeviceIndex) const override { return true; }
};

}  // namespace

C10_REGISTER_GUARD_IMPL(PrivateUse1, GuardImpl);

namespace {
const bool g_registered = [] {
  at::RegisterPrivateUse1HooksInterface(new Hooks());
  c10::SetAllocator(c10::DeviceType::PrivateUse1, &g_allocator);
  return true;
}();
}  // namespace

// Ops that ran through the CPU fallback since load (tests assert none on the
// hot path).
extern "C" uint64_t applegpu_backend_fallback_count(void) { return g_fallbacks.load(); }

// The loader calls this after load_library to surface a missing GPU early.
extern "C" int32_t applegpu_backend_ready(void) {
  try {
    ensure_init();
    return 1;
  } catch (...) {
    return 0;
  }
}
