// PyTorch operators over the C ABI of librglru_hip.so: argument checks, allocation and autograd in C++.
//
// Why native: a training step of a small layer is a handful of launches of 3-10 us, and the same glue in Python
// (autograd.Function, one torch.empty per buffer, ctypes calls of twenty arguments) kept the host busy for 190 us of
// a 50 us step and 790 us of a 560 us block step.  Here an operator costs its allocations and launches.
// Scratch buffers that live and die together are parts of one allocation.
//
// Errors follow the reference's operator module (griffin/triton_scan.py:213-224): RuntimeError for a missing GPU,
// ValueError for shapes, TypeError for types.
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/rglru_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
using MaybeTensor = std::optional<Tensor>;

// Whether a decode step of `rows` rows, so many multiply-adds in its three projections, takes the library's own kernels.  A call
// of the BLAS library costs the host 17 to 25 us, so a block's step through it takes 90 us however few rows it has, in a stack
// of blocks too (nothing waits between them); its kernels are the faster ones beyond about 16 rows of a 768 x 1024 block.  The
// line lies where our kernels take the 60 us that are left next to the step's other launches, at the rate they reach: with up to 64
// rows (one tile of rows: every weight is used once) 31e6 multiply-adds a us in bf16 and 13e6 in fp32, with more 50e6 and 24e6.
// Per layer in a stack of eight, alone / with an MLP of three products behind each block, us own : BLAS
// (profiles/block_products_own_vs_blas_in_stacks.txt): bf16 2560 -> 2560 64 rows 64 : 91 / 134 : 200, 128 rows 77 : 89 / 173 : 184, 256 rows 107 : 89 /
// 221 : 185; fp32 768 -> 1024 512 rows 70 : 100 / 150 : 172, 2560 32 rows 87 : 89 / 170 : 185, 64 rows 120 : 89 / 227 : 184, 128 rows 142 : 115 /
// 351 : 323.  Inside a captured graph, where host time is nothing, it lies where the kernels themselves are no slower.
bool own_projections_captured(double macs) { return macs < 1e8; }
bool own_projections(int64_t rows, double macs, at::ScalarType dtype) {
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return own_projections_captured(macs);
  return macs < (dtype == at::kBFloat16 ? (rows > 64 ? 3e9 : 1.9e9) : (rows > 64 ? 1.45e9 : 8e8));
}

// ---- small helpers ---------------------------------------------------------------------------------------------

Tensor opt(const MaybeTensor& t) { return t.has_value() ? *t : Tensor(); }
MaybeTensor maybe(const Tensor& t) { return t.defined() ? MaybeTensor(t) : MaybeTensor(); }

void check(int code, const char* what) {
  if (code == RGLRU_OK) return;
  const char* why = rglru_hip_last_error();
  if (code == RGLRU_E_ARG || code == RGLRU_E_UNSUPPORTED) TORCH_CHECK_VALUE(false, what, " failed: ", why);
  TORCH_CHECK(false, what, " failed: ", why);
}

bool known(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }

int code_of(at::ScalarType t) {
  TORCH_CHECK_TYPE(known(t), "hip RG-LRU supports float32 and bfloat16 activations, got ", t);
  return t == at::kBFloat16 ? RGLRU_BF16 : RGLRU_F32;
}

// Forward-mode tangents: none of the operators carries one on, so a dual tensor is refused (also where no gradient is asked
// for and no autograd function would notice it).  A tangent lives only inside an entered level, which is one question.
bool dual_level() { return torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr; }
bool is_dual(const Tensor& t) { return t.defined() && t._fw_grad(0).defined(); }
void refuse_tangent(const char* name, const Tensor& t) {
  TORCH_CHECK_NOT_IMPLEMENTED(!is_dual(t), name, " has no forward-mode derivative; it takes no dual tensors");
}
template <typename Tensors>
void refuse_tangents(const char* name, const Tensors& tensors) {
  if (!dual_level()) return;
  for (const Tensor& t : tensors) refuse_tangent(name, t);
}

void require_gpu(const char* name, std::initializer_list<const Tensor*> tensors) {
  for (const Tensor* t : tensors)
    TORCH_CHECK(!t->defined() || t->is_cuda(), name, " requires CUDA/HIP tensors, got a ", t->device().type(), " tensor");
  if (!dual_level()) return;
  for (const Tensor* t : tensors) refuse_tangent(name, *t);
}

// The kernels take addresses: an operand on another GPU than x's is an error, as it is for PyTorch's own operators.
bool on_device_of(const Tensor& x, const Tensor& t) { return !t.defined() || t.device() == x.device(); }
void require_device_of(const char* name, const Tensor& x, std::initializer_list<const Tensor*> tensors) {
  for (const Tensor* t : tensors)
    TORCH_CHECK(on_device_of(x, *t), name, " expects all tensors on the same device, found ", x.device(), " and ", t->device());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }
const int64_t* iptr(const Tensor& t) { return t.defined() ? static_cast<const int64_t*>(t.data_ptr()) : nullptr; }
const uint8_t* bptr(const Tensor& t) { return t.defined() ? static_cast<const uint8_t*>(t.data_ptr()) : nullptr; }

const uint8_t* flags_ptr(const Tensor& flags, bool first_reset) {
  return first_reset ? RGLRU_FLAGS_FIRST_RESET : bptr(flags);
}

Tensor fresh(at::IntArrayRef size, at::ScalarType dtype, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}
Tensor fresh_like(const Tensor& t) { return fresh(t.sizes(), t.scalar_type(), t); }
Tensor bytes(size_t n, const Tensor& like) { return fresh({static_cast<int64_t>(n)}, at::kByte, like); }

size_t round_up(size_t n) { return (n + 255) & ~size_t(255); }

// A contiguous tensor over part of a buffer's storage, `at` bytes in.  An allocation (and its release) costs the host a
// microsecond and more; a tensor over memory that is there, a fraction of one.
Tensor part(const Tensor& buffer, size_t at, at::IntArrayRef size, at::ScalarType dtype) {
  Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(buffer.storage()), c10::DispatchKeySet(c10::DispatchKey::CUDA),
                                                      c10::scalarTypeToTypeMeta(dtype));
  t.unsafeGetTensorImpl()->set_storage_offset(static_cast<int64_t>(at / c10::elementSize(dtype)));
  t.unsafeGetTensorImpl()->set_sizes_contiguous(size);
  return t;
}

// Scratch areas that live as long as each other, as parts of one allocation: first their sizes, then the memory, then the
// addresses in the same order.  What a caller gets to keep is not such a part: keeping or saving one would keep or save all.
// Carried state is tensors of their own; gradients share memory with their like at most (see take_gates).
struct Parts {
  std::vector<size_t> offsets;
  size_t total = 0, next = 0;
  Tensor buffer;
  void add(size_t n) { offsets.push_back(total), total += round_up(n); }
  void allocate(const Tensor& like) { buffer = bytes(total, like); }
  char* raw() { return static_cast<char*>(buffer.data_ptr()) + offsets[next++]; }
};

// Contiguous and on a 16-byte boundary (what every fresh allocation is): a view at an odd offset costs one copy
// instead of sending the whole call to the portable kernels, which are several times slower.
Tensor aligned(const Tensor& t) {
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone(at::MemoryFormat::Contiguous);
}
bool is_aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

Tensor as(const Tensor& t, at::ScalarType dtype) {
  if (!t.defined()) return t;
  return t.scalar_type() == dtype ? t.contiguous() : t.to(dtype).contiguous();
}

// A parameter as the library reads it: its own type when that is fp32 or bf16, else converted.
Tensor operand(const Tensor& t, at::ScalarType like) {
  if (!t.defined()) return t;
  return as(t, known(t.scalar_type()) ? t.scalar_type() : like);
}

bool wants_grad(std::initializer_list<const Tensor*> tensors) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : tensors)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// The gradients of a first-order operator: a second differentiation meets an error instead of a wrong number.
variable_list once(variable_list grads) {
  if (!at::GradMode::is_enabled()) return grads;
  variable_list marked;
  marked.reserve(grads.size());
  for (auto& g : grads) marked.push_back(g.defined() ? g.detach().set_requires_grad(true) : Tensor());
  auto error = std::make_shared<torch::autograd::DelayedError>(
      "trying to differentiate twice a function that was marked with @once_differentiable", marked.size());
  return error->apply(std::move(marked));
}

// ---- RG-LRU ----------------------------------------------------------------------------------------------------

// The five parameters as the library reads them: gate weights in the storage type; biases and Lambda in their own
// type when the three agree on one the library knows, so the usual cases launch no conversion kernels.
struct Operands {
  Tensor w_a, b_a, w_x, b_x, lam;
  int vec;
  Operands(const Tensor& wa, const Tensor& ba, const Tensor& wx, const Tensor& bx, const Tensor& l, at::ScalarType dtype) {
    auto v = ba.scalar_type();
    if (bx.scalar_type() != v || l.scalar_type() != v || !known(v)) v = at::kFloat;
    w_a = as(wa, dtype), b_a = as(ba, v), w_x = as(wx, dtype), b_x = as(bx, v), lam = as(l, v);
    vec = v == at::kBFloat16 ? RGLRU_BF16 : RGLRU_F32;
  }
};

size_t prep_bytes(int64_t W, int64_t nb, int code) {
  const size_t n = rglru_hip_prep_bytes(W, nb, code);
  if (n == 0) check(RGLRU_E_UNSUPPORTED, "rglru_hip_prep_bytes");
  return n;
}

int64_t kernel_path(int64_t B, int64_t T, int64_t W, int64_t nb, at::ScalarType dtype, bool on_boundary) {
  const int path = rglru_hip_backward_path(B, T, W, nb, code_of(dtype), on_boundary ? 1 : 0);
  if (path < 0) check(RGLRU_E_UNSUPPORTED, "rglru_hip_backward_path");
  return path;
}

// The kernels read as many elements as the first gate's weights say: the other four parameters have to have them.
void check_gates(const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x, const Tensor& lam) {
  TORCH_CHECK_VALUE(w_a.dim() == 3 && w_a.size(1) == w_a.size(2) && w_x.sizes() == w_a.sizes(), "gate weights must both have shape [blocks, width, width], got ",
                    w_a.sizes(), " and ", w_x.sizes());
  const int64_t W = w_a.size(0) * w_a.size(1);
  TORCH_CHECK_VALUE(b_a.numel() == W && b_x.numel() == W && lam.numel() == W, "gate biases and Lambda must have ", W, " elements, got ", b_a.numel(),
                    ", ", b_x.numel(), " and ", lam.numel());
}

Tensor prepare(const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x, const Tensor& lam, double c,
               at::ScalarType dtype) {
  check_gates(w_a, b_a, w_x, b_x, lam);
  require_device_of("hip RG-LRU", w_a, {&b_a, &w_x, &b_x, &lam});
  const int64_t nb = w_a.size(0), W = nb * w_a.size(1);
  const int code = code_of(dtype);
  refuse_tangents("hip RG-LRU", std::array<Tensor, 5>{w_a, b_a, w_x, b_x, lam});
  c10::DeviceGuard guard(w_a.device());
  at::NoGradGuard no_grad;
  Operands p(w_a, b_a, w_x, b_x, lam, dtype);
  Tensor image = bytes(prep_bytes(W, nb, code), w_a);
  check(rglru_hip_prepare(ptr(p.w_a), ptr(p.b_a), ptr(p.w_x), ptr(p.b_x), ptr(p.lam), static_cast<float>(c), W, nb, code,
                          p.vec, ptr(image), stream_of(w_a)), "rglru_hip_prepare");
  return image;
}

void check_fused(const Tensor& x, const Tensor& w_a, const Tensor& h0, const Tensor& flags) {
  TORCH_CHECK_VALUE(x.dim() == 3, "hip RG-LRU expects [batch, sequence, width], got ", x.sizes());
  const int64_t B = x.size(0), T = x.size(1), W = x.size(2);
  TORCH_CHECK_VALUE(w_a.dim() == 3 && w_a.size(1) == w_a.size(2) && w_a.size(0) * w_a.size(1) == W, "gate weights ",
                    w_a.sizes(), " do not match width ", W);
  TORCH_CHECK_VALUE(!h0.defined() || (h0.dim() == 2 && h0.size(0) == B && h0.size(1) == W), "initial state must have shape (",
                    B, ", ", W, ")");
  TORCH_CHECK_VALUE(!flags.defined() || (flags.dim() == 2 && flags.size(0) == B && flags.size(1) == T),
                    "token flags must have shape (", B, ", ", T, ")");
  TORCH_CHECK_VALUE(T > 0 && B > 0, "hip RG-LRU does not accept empty batches or sequences");
  code_of(x.scalar_type());
}

// What a forward pass keeps for its backward: the parameter image and the workspace in one allocation.
struct Kept {
  Tensor buffer;
  void *image = nullptr, *ws = nullptr;
  Kept(const Tensor& held, int64_t W, int64_t nb, int code) : buffer(held) {
    image = held.data_ptr();
    ws = static_cast<char*>(image) + round_up(prep_bytes(W, nb, code));
  }
  Kept(const Tensor& like, int64_t B, int64_t T, int64_t W, int64_t nb, int code)
      : Kept(bytes(round_up(prep_bytes(W, nb, code)) + rglru_hip_workspace_bytes(B, T, W, nb), like), W, nb, code) {}
};

struct ForwardResult {
  Tensor x, h0, y, h_last, kept;
};

ForwardResult rglru_forward(const Tensor& x_in, const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x,
                            const Tensor& lam, const Tensor& h0_in, const Tensor& flags, bool first_reset, double c, int64_t path,
                            bool clear_backward = false) {
  ForwardResult r;
  c10::DeviceGuard guard(x_in.device());
  r.x = aligned(x_in);
  const int64_t B = r.x.size(0), T = r.x.size(1), W = r.x.size(2), nb = w_a.size(0);
  const int code = code_of(r.x.scalar_type());
  Operands p(w_a, b_a, w_x, b_x, lam, r.x.scalar_type());
  r.h0 = as(h0_in, at::kFloat);
  r.y = fresh_like(r.x);
  r.h_last = fresh({B, W}, at::kFloat, r.x);
  Kept kept(r.x, B, T, W, nb, code);
  r.kept = kept.buffer;
  void* stream = stream_of(r.x);
  const uint8_t* fl = flags_ptr(flags, first_reset);
  if (path == RGLRU_PATH_PRE) {
    Tensor pre = fresh({nb, B * T, 2 * (W / nb)}, r.x.scalar_type(), r.x);  // scratch of the call
    check(rglru_hip_prepare(ptr(p.w_a), ptr(p.b_a), ptr(p.w_x), ptr(p.b_x), ptr(p.lam), static_cast<float>(c), W, nb, code,
                            p.vec, kept.image, stream), "rglru_hip_prepare");
    check(rglru_hip_fwd_pre(ptr(r.x), ptr(pre), kept.image, fptr(r.h0), fl, ptr(r.y), fptr(r.h_last), kept.ws, B, T, W, nb,
                            code, stream), "rglru_hip_fwd_pre");
  } else {
    // parameter conversion, workspace clearing and the forward kernel: two launches, or one where the forward kernel
    // does all three (batch-rich shapes)
    check(rglru_hip_prepare_fwd(ptr(p.w_a), ptr(p.b_a), ptr(p.w_x), ptr(p.b_x), ptr(p.lam), static_cast<float>(c), p.vec,
                                kept.image, ptr(r.x), fptr(r.h0), fl, ptr(r.y), fptr(r.h_last), kept.ws, B, T, W, nb,
                                code | (clear_backward ? RGLRU_BACKWARD_CLEAR : 0), stream), "rglru_hip_prepare_fwd");
  }
  return r;
}

struct ParamGrads {
  Tensor dx, dw_a, db_a, dw_x, db_x, dlam, dh0;
};

// The gates' gradients, the two weights in one allocation and the three vectors in another: memory that the backward's thread
// allocates and the caller's frees costs the host 2 to 3 us (layer B2 T256 W256 fp32: 91 us a step with all five in one, 94 so,
// 103 with five allocations).
void take_gates(int64_t nb, int64_t bw, at::ScalarType dtype, const Tensor& like, Tensor& dw_a, Tensor& db_a, Tensor& dw_x, Tensor& db_x,
                Tensor& dlam) {
  const int64_t W = nb * bw;
  const size_t es = c10::elementSize(dtype), weight = round_up(W * bw * es), vector = round_up(W * es);
  Tensor weights = bytes(2 * weight, like), vectors = bytes(3 * vector, like);
  dw_a = part(weights, 0, {nb, bw, bw}, dtype), dw_x = part(weights, weight, {nb, bw, bw}, dtype);
  db_a = part(vectors, 0, {nb, bw}, dtype), db_x = part(vectors, vector, {nb, bw}, dtype), dlam = part(vectors, 2 * vector, {W}, dtype);
}

// Backward pass of the RG-LRU on what its forward kept; the parameter gradients come back in the parameters' types
// (w_a, b_a, w_x, b_x, lam).
ParamGrads rglru_backward(const Tensor& x, const Tensor& y, int64_t nb, const Tensor& h0, const Tensor& flags, bool first_reset,
                          const Tensor& held, const Tensor& dy_in, const Tensor& dh_last_in,
                          const std::array<at::ScalarType, 5>& types, bool need_dh0, bool ws_clear) {
  ParamGrads g;
  c10::DeviceGuard guard(x.device());
  const int64_t B = x.size(0), T = x.size(1), W = x.size(2), bw = W / nb;
  const auto dtype = x.scalar_type();
  const int code = code_of(dtype);
  Kept kept(held, W, nb, code);
  Tensor dy = dy_in.defined() ? aligned(dy_in.to(dtype)) : at::zeros_like(x);
  Tensor dh_last = as(dh_last_in, at::kFloat);
  // one type for all five gradients where the parameters share one that the library writes; else fp32, converted below
  auto gt = types[0];
  for (auto t : types)
    if (t != gt) gt = at::kFloat;
  if (!known(gt)) gt = at::kFloat;
  const int gcode = code_of(gt) | (ws_clear ? RGLRU_BACKWARD_CLEAR : 0);
  g.dx = fresh_like(x);
  take_gates(nb, bw, gt, x, g.dw_a, g.db_a, g.dw_x, g.db_x, g.dlam);
  if (need_dh0) g.dh0 = fresh({B, W}, at::kFloat, x);
  void* stream = stream_of(x);
  const uint8_t* fl = flags_ptr(flags, first_reset);
  const int64_t path = kernel_path(B, T, W, nb, dtype, is_aligned(x) && is_aligned(y) && is_aligned(dy));
  const size_t scratch_bytes = round_up(rglru_hip_bwd_scratch_bytes(B, T, W, nb, code));
  const size_t tensor_bytes = round_up(x.numel() * x.element_size());
  // scratch of this call, the operand tensors of the paths that keep some in memory behind it
  const int extra = path == RGLRU_PATH_PRE ? 4 : path == RGLRU_PATH_PORTABLE ? 2 : 0;
  Tensor scratch = bytes(scratch_bytes + extra * tensor_bytes, x);
  char* sp = static_cast<char*>(scratch.data_ptr());
  char* more = sp + scratch_bytes;
  if (path == RGLRU_PATH_FAST_CHAIN || path == RGLRU_PATH_FAST_TILED) {
    check(rglru_hip_bwd_full(ptr(x), ptr(y), kept.image, fptr(h0), fl, ptr(dy), fptr(dh_last), kept.ws, sp, ptr(g.dx),
                             ptr(g.dw_a), ptr(g.dw_x), ptr(g.db_a), ptr(g.db_x), ptr(g.dlam), fptr(g.dh0), B, T, W, nb, code,
                             gcode, stream), "rglru_hip_bwd_full");
  } else if (path == RGLRU_PATH_WIDE) {
    check(rglru_hip_bwd_wide(ptr(x), kept.image, fptr(h0), fl, ptr(dy), fptr(dh_last), kept.ws, sp, ptr(g.dx), ptr(g.dw_a),
                             ptr(g.dw_x), ptr(g.db_a), ptr(g.db_x), ptr(g.dlam), fptr(g.dh0), B, T, W, nb, code, gcode,
                             stream), "rglru_hip_bwd_wide");
  } else if (path == RGLRU_PATH_PRE) {
    check(rglru_hip_bwd_pre(ptr(x), more, kept.image, fptr(h0), fl, ptr(dy), fptr(dh_last), kept.ws, sp, ptr(g.dx),
                            more + 2 * tensor_bytes, ptr(g.dw_a), ptr(g.dw_x), ptr(g.db_a), ptr(g.db_x), ptr(g.dlam),
                            fptr(g.dh0), B, T, W, nb, code, code_of(gt), stream), "rglru_hip_bwd_pre");
  } else {
    check(rglru_hip_bwd(ptr(x), kept.image, fptr(h0), fl, ptr(dy), fptr(dh_last), kept.ws, sp, ptr(g.dx), more,
                        more + tensor_bytes, ptr(g.dw_a), ptr(g.dw_x), ptr(g.db_a), ptr(g.db_x), ptr(g.dlam), fptr(g.dh0), B,
                        T, W, nb, code, gcode, stream), "rglru_hip_bwd");
  }
  Tensor* out[5] = {&g.dw_a, &g.db_a, &g.dw_x, &g.db_x, &g.dlam};
  for (int i = 0; i < 5; ++i)
    if (types[i] != gt) *out[i] = out[i]->to(types[i]);
  return g;
}

std::array<at::ScalarType, 5> types_of(const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x,
                                       const Tensor& lam) {
  return {w_a.scalar_type(), b_a.scalar_type(), w_x.scalar_type(), b_x.scalar_type(), lam.scalar_type()};
}

void pack(AutogradContext* ctx, std::initializer_list<int64_t> values) {
  ctx->saved_data["meta"] = c10::List<int64_t>(values);
}
std::vector<int64_t> unpack(AutogradContext* ctx) { return ctx->saved_data["meta"].toIntVector(); }
at::ScalarType type_at(const std::vector<int64_t>& m, size_t i) { return static_cast<at::ScalarType>(m[i]); }
constexpr int64_t kNone = -1;

// The capture that the current stream of t's device records into (0: none), or kNone where the runtime does not say.
int64_t capture_of(const Tensor& t) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream_of(t)), &status, &id) != hipSuccess) {
    (void)hipGetLastError();
    return kNone;
  }
  return status == hipStreamCaptureStatusNone ? 0 : status == hipStreamCaptureStatusActive ? static_cast<int64_t>(id) + 1 : kNone;
}

// The forward's clearing launch covers what the first backward pass over it needs clear (a repeated pass clears that itself).
// That holds where both run, or both are recorded, together: a graph that holds the backward alone is replayed without
// the forward, and one that holds the forward alone does its clearing at another time than the backward.
void note_cleared(AutogradContext* ctx, const Tensor& t) { ctx->saved_data["clear"] = capture_of(t); }
bool take_cleared(AutogradContext* ctx, const Tensor& t) {
  auto noted = ctx->saved_data.find("clear");
  if (noted == ctx->saved_data.end()) return false;
  const int64_t capture = noted->second.toInt();
  ctx->saved_data.erase(noted);
  return capture != kNone && capture == capture_of(t);
}

// Whether the gradient of tensor argument i of a Function's forward is asked for.  The node has an edge only for the
// arguments that were there, so an optional argument in front shifts the ones behind it: forward notes which were.
void note_arguments(AutogradContext* ctx, std::initializer_list<bool> present) {
  c10::List<int64_t> edges;
  int64_t next = 0;
  for (bool p : present) edges.push_back(p ? next++ : kNone);
  ctx->saved_data["edges"] = edges;
}
struct Needs {
  AutogradContext* ctx;
  std::vector<int64_t> edges;
  explicit Needs(AutogradContext* c) : ctx(c), edges(c->saved_data["edges"].toIntVector()) {}
  bool operator()(size_t i) const { return edges[i] != kNone && ctx->needs_input_grad(edges[i]); }
};

int64_t type_or_none(const Tensor& t) { return t.defined() ? static_cast<int64_t>(t.scalar_type()) : kNone; }

struct RGLRU : torch::autograd::Function<RGLRU> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w_a, const Tensor& b_a, const Tensor& w_x,
                               const Tensor& b_x, const Tensor& lam, const MaybeTensor& h0_, const MaybeTensor& flags_, bool first_reset,
                               double c, int64_t path) {
    Tensor h0 = opt(h0_), flags = opt(flags_);
    note_arguments(ctx, {true, true, true, true, true, true, h0.defined()});
    const bool clears = path != RGLRU_PATH_FAST_CHAIN && path != RGLRU_PATH_PRE;   // the kernels that use records
    ForwardResult r = rglru_forward(x, w_a, b_a, w_x, b_x, lam, h0, flags, first_reset, c, path, clears);
    if (clears) note_cleared(ctx, r.x);
    ctx->save_for_backward({r.x, r.h0, flags, r.kept, r.y});
    auto t = types_of(w_a, b_a, w_x, b_x, lam);
    pack(ctx, {first_reset, w_a.size(0), type_or_none(h0), (int64_t)t[0], (int64_t)t[1], (int64_t)t[2], (int64_t)t[3], (int64_t)t[4]});
    ctx->set_materialize_grads(false);  // an unused output arrives undefined, not as a tensor of zeros
    return {r.y, r.h_last};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto saved = ctx->get_saved_variables();
    auto m = unpack(ctx);
    ParamGrads g;
    {
      at::NoGradGuard no_grad;
      g = rglru_backward(saved[0], saved[4], m[1], saved[1], saved[2], m[0], saved[3], grads[0], grads[1],
                         {type_at(m, 3), type_at(m, 4), type_at(m, 5), type_at(m, 6), type_at(m, 7)},
                         Needs(ctx)(6), take_cleared(ctx, saved[0]));
      if (g.dh0.defined() && type_at(m, 2) != at::kFloat) g.dh0 = g.dh0.to(type_at(m, 2));
    }
    return once({g.dx, g.dw_a, g.db_a, g.dw_x, g.db_x, g.dlam, g.dh0, Tensor(), Tensor(), Tensor(), Tensor()});
  }
};

std::tuple<Tensor, Tensor> rglru(const Tensor& x, const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x,
                                 const Tensor& lam, const MaybeTensor& h0_, const MaybeTensor& flags_, bool first_reset,
                                 double c, int64_t path) {
  Tensor h0 = opt(h0_), flags = opt(flags_);
  require_gpu("hip RG-LRU", {&x, &w_a, &b_a, &w_x, &b_x, &lam, &h0, &flags});
  require_device_of("hip RG-LRU", x, {&w_a, &b_a, &w_x, &b_x, &lam, &h0, &flags});
  check_fused(x, w_a, h0, flags);
  check_gates(w_a, b_a, w_x, b_x, lam);
  if (wants_grad({&x, &w_a, &b_a, &w_x, &b_x, &lam, &h0})) {
    auto out = RGLRU::apply(x, w_a, b_a, w_x, b_x, lam, maybe(h0), maybe(flags), first_reset, c, path);
    return {out[0], out[1]};
  }
  at::NoGradGuard no_grad;
  ForwardResult r = rglru_forward(x, w_a, b_a, w_x, b_x, lam, h0, flags, first_reset, c, path);
  return {r.y, r.h_last};
}

// Storage addresses and version counters of some tensors, one after the other: unchanged while nobody replaced one or
// wrote to it through PyTorch.
py::tuple fingerprint(const std::vector<Tensor>& tensors) {
  refuse_tangents("the recurrent block", tensors);            // what is kept under a fingerprint carries none
  py::tuple out(2 * tensors.size());
  for (size_t i = 0; i < tensors.size(); ++i) {
    out[2 * i] = reinterpret_cast<uintptr_t>(tensors[i].data_ptr());
    out[2 * i + 1] = tensors[i]._version();
  }
  return out;
}

// What a prepared parameter image was made from, compared on this side: a decode loop asks every step.
struct Stamp {
  std::vector<std::pair<const void*, int64_t>> seen;
  Tensor image;
  int64_t blocks = 0;
  double c = 0.0;
  at::ScalarType dtype = at::kFloat;
  Stamp() = default;
  Stamp(const std::vector<Tensor>& tensors, const Tensor& img, int64_t nb, double decay, at::ScalarType type)
      : image(img), blocks(nb), c(decay), dtype(type) {
    for (const Tensor& t : tensors) seen.emplace_back(t.data_ptr(), static_cast<int64_t>(t._version()));
  }
  template <typename Tensors>
  bool holds(const Tensors& tensors, size_t n, double decay, at::ScalarType type) const {
    if (n != seen.size() || c != decay || dtype != type || dual_level()) return false;   // a dual tensor shares its primal's memory
    for (size_t i = 0; i < n; ++i)
      if (tensors[i].data_ptr() != seen[i].first || static_cast<int64_t>(tensors[i]._version()) != seen[i].second) return false;
    return true;
  }
  bool matches(const std::vector<Tensor>& tensors, double decay, at::ScalarType type, c10::Device device) const {
    return image.defined() && image.device() == device && holds(tensors, tensors.size(), decay, type);
  }
};

// ---- decode steps ----------------------------------------------------------------------------------------------

// The ends of the autograd graph at a module's parameters, held between training steps.  A leaf keeps its accumulation node only
// by a weak reference, so the node dies with every graph and is made again by the next forward: with the five parameters of the
// RG-LRU 9 us of the 114 us that the host takes for a training step (width 256; the device needs 30).  A node made under
// another stream or for another shape of the parameter is not kept: a new one is made as if none had been there.
struct Leaves {
  typedef std::shared_ptr<torch::autograd::Node> NodePtr;
  std::vector<NodePtr> nodes;
  std::optional<c10::Stream> stream;
  static bool ends(const Tensor& t) { return t.defined() && t.requires_grad() && t.is_leaf(); }
  static bool current(const NodePtr& node, const Tensor& t) {
    if (!ends(t)) return node == nullptr;
    return node != nullptr && node == torch::autograd::impl::try_get_grad_accumulator(t) && node->input_metadata(0).is_same_shape(t);
  }
  // under the interpreter's lock; every change of `nodes` is one step, so another thread may come in where a node's end lets it
  void hold(const std::vector<Tensor>& tensors) {
    const c10::Stream now = c10::hip::getCurrentHIPStream(tensors[0].device().index()).unwrap();
    bool same = nodes.size() == tensors.size() && stream == now;
    for (size_t i = 0; same && i < tensors.size(); ++i) same = current(nodes[i], tensors[i]);
    if (same) return;
    std::vector<NodePtr>().swap(nodes);
    std::vector<NodePtr> fresh;
    for (const Tensor& t : tensors) fresh.push_back(ends(t) ? torch::autograd::impl::grad_accumulator(t) : nullptr);
    stream = now;
    nodes.swap(fresh);
  }
};

// Hold the leaves `tensors` of a module in its instance dictionary.
void hold_leaves(const py::dict& members, const std::vector<Tensor>& tensors) {
  if (!at::GradMode::is_enabled() || tensors.empty() || !tensors[0].is_cuda()) return;
  PyObject* held = PyDict_GetItemString(members.ptr(), "_leaves");
  if (held == nullptr || !py::isinstance<Leaves>(held)) {
    py::object made = py::cast(new Leaves(), py::return_value_policy::take_ownership);
    members["_leaves"] = made;
    made.cast<Leaves*>()->hold(tensors);
  } else {
    py::handle(held).cast<Leaves*>()->hold(tensors);
  }
}

// One flag byte for each of so many tokens, as the kernels read them.
Tensor token_bytes(const Tensor& flags, int64_t tokens) {
  if (!flags.defined()) return flags;
  TORCH_CHECK_VALUE(flags.numel() == tokens && flags.element_size() == 1, "expected one byte for each of ", tokens, " tokens, got ", flags.sizes());
  return flags.contiguous();
}

Tensor rglru_step(const Tensor& x_in, const Tensor& image, int64_t blocks, const Tensor& state, const MaybeTensor& flags_) {
  Tensor flags = opt(flags_);
  require_gpu("hip RG-LRU step", {&x_in, &state, &flags});
  require_device_of("hip RG-LRU step", x_in, {&image, &state, &flags});
  TORCH_CHECK_VALUE(state.sizes() == x_in.sizes() && state.scalar_type() == at::kFloat && state.is_contiguous(),
                    "step expects a contiguous fp32 state of the same shape as x");
  flags = token_bytes(flags, x_in.size(0));
  c10::DeviceGuard guard(x_in.device());
  Tensor x = x_in.contiguous();
  Tensor y = fresh_like(x);
  check(rglru_hip_step(ptr(x), ptr(image), fptr(state), bptr(flags), ptr(y), x.size(0), x.size(1), blocks,
                       code_of(x.scalar_type()), stream_of(x)), "rglru_hip_step");
  return y;
}

Tensor rglru_steps(const Tensor& xs_in, const Tensor& image, int64_t blocks, const Tensor& state, const MaybeTensor& flags_) {
  Tensor flags = opt(flags_);
  require_gpu("hip RG-LRU steps", {&xs_in, &state, &flags});
  require_device_of("hip RG-LRU steps", xs_in, {&image, &state, &flags});
  c10::DeviceGuard guard(xs_in.device());
  Tensor xs = xs_in.contiguous();
  Tensor ys = fresh_like(xs);
  Tensor fl = flags.defined() ? flags.contiguous() : flags;
  if (xs.size(0) > 0 && xs.size(1) > 0)
    check(rglru_hip_steps(ptr(xs), ptr(image), fptr(state), bptr(fl), ptr(ys), xs.size(0), xs.size(1), xs.size(2), blocks,
                          code_of(xs.scalar_type()), stream_of(xs)), "rglru_hip_steps");
  return ys;
}

// One token per row of the bare layer: y and the new state, the old one untouched (x [B, 1, W]).
std::tuple<Tensor, Tensor> rglru_module_step(const Tensor& x_in, const Tensor& image, int64_t blocks, const MaybeTensor& state,
                                             const MaybeTensor& flags_) {
  Tensor flags = opt(flags_), carried = opt(state);
  require_gpu("hip RG-LRU step", {&x_in, &flags, &carried});
  require_device_of("hip RG-LRU step", x_in, {&image, &flags, &carried});
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(x_in.device());
  const int64_t B = x_in.size(0), W = x_in.size(2);
  flags = token_bytes(flags, B);
  TORCH_CHECK_VALUE(!state.has_value() || (state->dim() == 2 && state->size(0) == B && state->size(1) == W), "the state must have shape (", B, ", ", W, ")");
  Tensor x = x_in.contiguous();
  Tensor h = state.has_value() ? as(*state, at::kFloat) : at::zeros({B, W}, x.options().dtype(at::kFloat));
  Tensor h_new = fresh({B, W}, at::kFloat, x);
  Tensor y = fresh({B, 1, W}, x.scalar_type(), x);
  check(rglru_hip_step_gated(ptr(x), ptr(image), fptr(h), fptr(h_new), bptr(flags), nullptr, 0, ptr(y), B, W, blocks,
                             code_of(x.scalar_type()), stream_of(x)), "rglru_hip_step_gated");
  return {y, h_new};
}

// ---- scan-only operator: h_t = a_t h_{t-1} + z_t (griffin/triton_scan.py:207-276) --------------------------------

Tensor scan_forward(const Tensor& a, const Tensor& z, const Tensor& h0, Tensor* ws_out) {
  Tensor out = fresh_like(z);
  if (out.numel() == 0) return out;
  const int64_t B = a.size(0), T = a.size(1), W = a.size(2);
  Tensor ws = bytes(rglru_hip_scan_workspace_bytes(B, T, W), a);
  check(rglru_hip_scan_fwd(fptr(a), fptr(z), fptr(h0), fptr(out), ptr(ws), B, T, W, stream_of(a)), "rglru_hip_scan_fwd");
  if (ws_out != nullptr) *ws_out = ws;
  return out;
}

struct Scan : torch::autograd::Function<Scan> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a_in, const Tensor& z, const Tensor& h0_in) {
    c10::DeviceGuard guard(a_in.device());
    Tensor a = a_in.contiguous(), h0 = h0_in.contiguous(), ws;
    Tensor out = scan_forward(a, z.contiguous(), h0, &ws);
    ctx->save_for_backward({a, h0, out});
    if (ws.defined()) ctx->saved_data["ws"] = ws, note_cleared(ctx, a);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto saved = ctx->get_saved_variables();
    const Tensor &a = saved[0], &h0 = saved[1], &out = saved[2];
    Tensor da, dz, dh0;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(a.device());
      Tensor dh = grads[0].contiguous();
      const int64_t B = a.size(0), T = a.size(1), W = a.size(2);
      da = fresh_like(a), dz = fresh_like(a), dh0 = fresh_like(h0);
      if (a.numel() == 0) {
        dh0.zero_();
      } else {
        const bool clear = take_cleared(ctx, a);
        Tensor ws = clear ? ctx->saved_data["ws"].toTensor() : bytes(rglru_hip_scan_workspace_bytes(B, T, W), a);
        ctx->saved_data.erase("ws");
        check(rglru_hip_scan_bwd(fptr(a), fptr(h0), fptr(out), fptr(dh), fptr(da), fptr(dz), fptr(dh0), ptr(ws), clear ? 1 : 0, B,
                                 T, W, stream_of(a)), "rglru_hip_scan_bwd");
      }
    }
    return once({da, dz, dh0});
  }
};

Tensor scan(const Tensor& a, const Tensor& z, const Tensor& h0) {
  require_gpu("hip_rglru_scan", {&a, &z, &h0});
  require_device_of("hip_rglru_scan", a, {&z, &h0});
  TORCH_CHECK_VALUE(a.dim() == 3 && a.sizes() == z.sizes(), "decay and current_input must share shape [batch, sequence, width]");
  TORCH_CHECK_VALUE(h0.dim() == 2 && h0.size(0) == a.size(0) && h0.size(1) == a.size(2), "initial_state must have shape [batch, width]");
  TORCH_CHECK_TYPE(a.scalar_type() == at::kFloat && z.scalar_type() == at::kFloat, "hip_rglru_scan expects fp32 decay and normalized input");
  TORCH_CHECK_TYPE(h0.scalar_type() == at::kFloat, "hip_rglru_scan expects fp32 recurrent state");
  if (wants_grad({&a, &z, &h0})) return Scan::apply(a, z, h0);
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(a.device());
  return scan_forward(a.contiguous(), z.contiguous(), h0.contiguous(), nullptr);
}

// ---- causal depthwise convolution (griffin/griffin.py:474-510) ----------------------------------------------------

// What an activity mask says about every token (rglru_hip_token_facts), and, once the host asks, whether all tokens are
// active and whether the rows are right-padded.  The answer is written to host memory by the kernel: asking waits for that
// kernel alone, not for work queued behind it.
struct TokenFacts {
  Tensor positions, flags, conv_positions, rows, last_position;
  TokenFacts(const Tensor& active_in, const MaybeTensor& segment_pos, const MaybeTensor& prev_pos) : event_(at::kCUDA) {
    require_gpu("token facts", {&active_in});
    at::NoGradGuard no_grad;
    c10::DeviceGuard guard(active_in.device());
    // before anything is launched: a graph that held the kernel would write to the host memory on every replay
    TORCH_CHECK(c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None,
                "an activity mask is answered on the host, which a stream that is being captured does not allow");
    Tensor active = active_in.contiguous();
    TORCH_CHECK_VALUE(active.dim() == 2 && active.element_size() == 1, "active_mask must be a [batch, sequence] mask");
    const int64_t B = active.size(0), T = active.size(1);
    Tensor prev;
    if (segment_pos.has_value()) positions = segment_pos->to(active.device(), at::kLong).contiguous();
    if (prev_pos.has_value()) prev = prev_pos->to(active.device(), at::kLong).contiguous();
    const bool given = positions.defined();
    TORCH_CHECK_VALUE(!given || positions.sizes() == active.sizes(), "segment_pos must have the shape of active_mask");
    TORCH_CHECK_VALUE(!prev.defined() || (prev.dim() == 1 && prev.size(0) == B), "Cached segment positions have an incompatible shape");
    if (!given) positions = fresh({B, T}, at::kLong, active);
    flags = fresh({B, T}, at::kByte, active);
    conv_positions = fresh({B, T}, at::kLong, active);
    rows = fresh({3, B}, at::kInt, active);
    last_position = fresh({B}, at::kLong, active);
    answer_ = at::empty({B}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    check(rglru_hip_token_facts(bptr(active), given ? iptr(positions) : nullptr, iptr(prev),
                                given ? nullptr : static_cast<int64_t*>(positions.data_ptr()), static_cast<uint8_t*>(flags.data_ptr()),
                                static_cast<int64_t*>(conv_positions.data_ptr()), static_cast<int32_t*>(rows.data_ptr()),
                                static_cast<int64_t*>(last_position.data_ptr()), static_cast<uint32_t*>(answer_.data_ptr()), B, T,
                                stream_of(active)), "rglru_hip_token_facts");
    try {
      event_.record(c10::Stream(c10::Stream::UNSAFE, active.device(), c10::hip::getCurrentHIPStream(active.device().index()).id()));
    } catch (...) {
      abandon();
      throw;
    }
  }
  TokenFacts(const TokenFacts&) = delete;
  // the kernel writes into memory that this object gives back, so its end is waited for; where that fails (an error is
  // pending on the device, and resolve() has reported it) the memory is not given back
  ~TokenFacts() {
    try {
      wait();
    } catch (...) {
      abandon();
    }
  }
  std::tuple<bool, bool> resolve() {
    {
      py::gil_scoped_release no_gil;
      wait();
    }
    bool all_active = true, prefix = true;
    const int32_t* a = static_cast<const int32_t*>(answer_.data_ptr());
    active_tokens = 0;
    for (int64_t b = 0; b < answer_.size(0); ++b)
      all_active &= (a[b] & 1) != 0, prefix &= (a[b] & 2) != 0, active_tokens += static_cast<uint32_t>(a[b]) >> 2;
    return {all_active, prefix};
  }
  int64_t active_tokens = 0;                               // of all rows, once resolved

 private:
  void wait() {
    if (!done_) event_.synchronize();
    done_ = true;
  }
  void abandon() { new Tensor(std::move(answer_)); }
  Tensor answer_;
  c10::Event event_;
  bool done_ = false;
};

Tensor pack_flags(const MaybeTensor& reset_, const MaybeTensor& active_) {
  at::NoGradGuard no_grad;
  auto mask = [](const MaybeTensor& m) { return m.has_value() ? m->to(at::kBool).contiguous() : Tensor(); };
  Tensor reset = mask(reset_), active = mask(active_);
  const Tensor& like = reset.defined() ? reset : active;
  require_gpu("hip RG-LRU", {&reset, &active});
  require_device_of("hip RG-LRU", like, {&reset, &active});
  c10::DeviceGuard guard(like.device());
  Tensor flags = fresh(like.sizes(), at::kByte, like);
  if (flags.numel() > 0)
    check(rglru_hip_pack_flags(bptr(reset), bptr(active), static_cast<uint8_t*>(flags.data_ptr()), flags.numel(), stream_of(like)),
          "rglru_hip_pack_flags");
  return flags;
}

struct ConvMeta {  // types of the forward's arguments (kNone: absent)
  int64_t state, weight, bias;
};

// Reverse mode of the dense convolution on contiguous operands.  `du_out`: where to write du instead of a new tensor --
// [B, T, W] with unit stride along W and rows a common distance apart (a column range of a wider matrix).
variable_list conv_backward(const Tensor& u, const Tensor& state, const Tensor& taps, const Tensor& pos, const Tensor& dout_in,
                            ConvMeta meta, bool need_u, bool need_state, bool need_w, bool need_b, const Tensor& du_out,
                            const Tensor& rows = Tensor()) {
  const int64_t B = u.size(0), T = u.size(1), W = u.size(2), K = taps.size(2);
  Tensor dout = as(dout_in, u.scalar_type());
  const auto gt = taps.scalar_type();
  Tensor du = du_out.defined() ? du_out : fresh_like(u);
  Tensor dstate, dtaps, dbias;
  if (need_state && state.defined()) dstate = fresh_like(state);
  if (need_w) dtaps = fresh({W, 1, K}, gt, u);
  if (need_b && meta.bias != kNone) dbias = fresh({W}, gt, u);
  Tensor scratch = bytes(rglru_hip_conv_scratch_bytes(B, T, W, K), u);
  check(rglru_hip_conv_rows_bwd(ptr(u), ptr(state), ptr(taps), iptr(pos), static_cast<const int32_t*>(ptr(rows)), ptr(dout),
                                ptr(scratch), ptr(du), du.stride(1), ptr(dstate), ptr(dtaps), ptr(dbias), B, T, W, K,
                                code_of(u.scalar_type()), code_of(gt), code_of(gt), stream_of(u)), "rglru_hip_conv_rows_bwd");
  if (dtaps.defined()) dtaps = dtaps.to(static_cast<at::ScalarType>(meta.weight));
  if (dbias.defined()) dbias = dbias.to(static_cast<at::ScalarType>(meta.bias));
  if (need_state && meta.state != kNone)
    dstate = (dstate.defined() ? dstate : at::zeros({B, K - 1, W}, u.options())).to(static_cast<at::ScalarType>(meta.state));
  return {need_u ? du : Tensor(), dstate, dtaps, dbias};
}

void check_conv(const char* name, const Tensor& u, const Tensor& state, const Tensor& weight, const Tensor& bias,
                const Tensor& pos) {
  TORCH_CHECK_VALUE(u.dim() == 3, name, " expects [batch, sequence, width], got ", u.sizes());
  const int64_t B = u.size(0), T = u.size(1), W = u.size(2);
  TORCH_CHECK_VALUE(weight.dim() == 3 && weight.size(0) == W && weight.size(1) == 1,
                    "weight must be that of a depthwise Conv1d: [width, 1, kernel_size]");
  TORCH_CHECK_VALUE(!bias.defined() || (bias.dim() == 1 && bias.size(0) == W), "bias must have shape [width]");
  TORCH_CHECK_VALUE(!state.defined() || (state.dim() == 3 && state.size(0) == B && state.size(1) == weight.size(2) - 1 && state.size(2) == W),
                    "state must have shape [batch, kernel_size - 1, width]");
  TORCH_CHECK_VALUE(pos.dim() == 2 && pos.size(0) == B && pos.size(1) == T, "segment_pos must have shape [batch, sequence]");
  code_of(u.scalar_type());
}

struct ConvOperands {
  Tensor u, state, taps, bias, pos;
  ConvOperands(const Tensor& u_in, const Tensor& st, const Tensor& weight, const Tensor& b, const Tensor& segment_pos) {
    u = u_in.contiguous();
    state = weight.size(2) == 1 ? Tensor() : as(st, u.scalar_type());
    taps = operand(weight, u.scalar_type());
    bias = as(b, taps.scalar_type());
    pos = segment_pos.to(u.device(), at::kLong).contiguous();
  }
};

struct CausalConv : torch::autograd::Function<CausalConv> {
  static Tensor forward(AutogradContext* ctx, const Tensor& u, const MaybeTensor& state_, const Tensor& weight,
                        const MaybeTensor& bias_, const Tensor& pos) {
    Tensor state = opt(state_), bias = opt(bias_);
    note_arguments(ctx, {true, state.defined(), true, bias.defined()});
    c10::DeviceGuard guard(u.device());
    ConvOperands o(u, state, weight, bias, pos);
    Tensor out = fresh_like(o.u);
    check(rglru_hip_conv_fwd(ptr(o.u), ptr(o.state), ptr(o.taps), ptr(o.bias), iptr(o.pos), ptr(out), nullptr, u.size(0),
                             u.size(1), u.size(2), weight.size(2), code_of(u.scalar_type()), code_of(o.taps.scalar_type()),
                             stream_of(u)), "rglru_hip_conv_fwd");
    ctx->save_for_backward({o.u, o.state, o.taps, o.pos});
    pack(ctx, {type_or_none(state), type_or_none(weight), type_or_none(bias)});
    ctx->set_materialize_grads(false);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return variable_list(5);
    auto s = ctx->get_saved_variables();
    auto m = unpack(ctx);
    variable_list g;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(s[0].device());
      Needs need(ctx);
      g = conv_backward(s[0], s[1], s[2], s[3], grads[0], {m[0], m[1], m[2]}, need(0), need(1), need(2), need(3), Tensor());
    }
    g.emplace_back();
    return once(std::move(g));
  }
};

Tensor causal_conv(const Tensor& u, const MaybeTensor& state_, const Tensor& weight, const MaybeTensor& bias_, const Tensor& pos) {
  Tensor state = opt(state_), bias = opt(bias_);
  require_gpu("hip_causal_conv", {&u, &state, &weight, &bias, &pos});
  require_device_of("hip_causal_conv", u, {&state, &weight, &bias});
  check_conv("hip_causal_conv", u, state, weight, bias, pos);
  return CausalConv::apply(u, maybe(state), weight, maybe(bias), pos);
}

struct CausalConvPadded : torch::autograd::Function<CausalConvPadded> {
  static variable_list forward(AutogradContext* ctx, const Tensor& u, const MaybeTensor& state_, const Tensor& weight,
                               const MaybeTensor& bias_, const Tensor& pos, const Tensor& active) {
    Tensor state = opt(state_), bias = opt(bias_);
    note_arguments(ctx, {true, state.defined(), true, bias.defined()});
    c10::DeviceGuard guard(u.device());
    ConvOperands o(u, state, weight, bias, pos);
    Tensor live = active.to(u.device(), at::kByte).contiguous();
    const int64_t B = u.size(0), T = u.size(1), W = u.size(2), K = weight.size(2);
    Tensor out = fresh_like(o.u);
    Tensor new_state = fresh({B, K - 1, W}, u.scalar_type(), u);
    Tensor scratch = bytes(rglru_hip_conv_padded_scratch_bytes(B, T), u);
    check(rglru_hip_conv_padded_fwd(ptr(o.u), ptr(o.state), ptr(o.taps), ptr(o.bias), iptr(o.pos), bptr(live), ptr(scratch),
                                    ptr(out), K > 1 ? ptr(new_state) : nullptr, B, T, W, K, code_of(u.scalar_type()),
                                    code_of(o.taps.scalar_type()), stream_of(u)), "rglru_hip_conv_padded_fwd");
    ctx->save_for_backward({o.u, o.state, o.taps, o.pos, live});
    pack(ctx, {type_or_none(state), type_or_none(weight), type_or_none(bias)});
    ctx->mark_non_differentiable({new_state});
    ctx->set_materialize_grads(false);
    return {out, new_state};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    if (!grads[0].defined()) return variable_list(6);
    auto s = ctx->get_saved_variables();
    auto m = unpack(ctx);
    const Tensor &u = s[0], &state = s[1], &taps = s[2], &pos = s[3], &live = s[4];
    Tensor du, dstate, dtaps, dbias;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(u.device());
      const int64_t B = u.size(0), T = u.size(1), W = u.size(2), K = taps.size(2);
      Needs need(ctx);
      const bool need_state = need(1);
      Tensor dout = as(grads[0], u.scalar_type());
      const auto gt = taps.scalar_type();
      du = fresh_like(u);
      if (need_state && K > 1) dstate = fresh({B, K - 1, W}, u.scalar_type(), u);
      if (need(2)) dtaps = fresh({W, 1, K}, gt, u);
      if (need(3) && m[2] != kNone) dbias = fresh({W}, gt, u);
      const size_t index_bytes = round_up(rglru_hip_conv_padded_scratch_bytes(B, T));
      Tensor scratch = bytes(index_bytes + rglru_hip_conv_scratch_bytes(B, T, W, K), u);
      char* sp = static_cast<char*>(scratch.data_ptr());
      check(rglru_hip_conv_padded_bwd(ptr(u), ptr(state), ptr(taps), iptr(pos), bptr(live), ptr(dout), sp, sp + index_bytes,
                                      ptr(du), ptr(dstate), ptr(dtaps), ptr(dbias), B, T, W, K, code_of(u.scalar_type()),
                                      code_of(gt), code_of(gt), stream_of(u)), "rglru_hip_conv_padded_bwd");
      if (dtaps.defined()) dtaps = dtaps.to(type_at(m, 1));
      if (dbias.defined()) dbias = dbias.to(type_at(m, 2));
      if (need_state && m[0] != kNone)
        dstate = (dstate.defined() ? dstate : at::zeros({B, K - 1, W}, u.options())).to(type_at(m, 0));
      else
        dstate = Tensor();
      if (!need(0)) du = Tensor();
    }
    return once({du, dstate, dtaps, dbias, Tensor(), Tensor()});
  }
};

std::tuple<Tensor, Tensor> causal_conv_padded(const Tensor& u, const MaybeTensor& state_, const Tensor& weight,
                                              const MaybeTensor& bias_, const Tensor& pos, const Tensor& active) {
  Tensor state = opt(state_), bias = opt(bias_);
  require_gpu("hip_causal_conv_padded", {&u, &state, &weight, &bias, &pos, &active});
  require_device_of("hip_causal_conv_padded", u, {&state, &weight, &bias});
  check_conv("hip_causal_conv_padded", u, state, weight, bias, pos);
  TORCH_CHECK_VALUE(active.sizes() == pos.sizes(), "segment_pos and active_mask must have shape [batch, sequence]");
  auto out = CausalConvPadded::apply(u, maybe(state), weight, maybe(bias), pos, active);
  return {out[0], out[1]};
}

// ---- output gate h * gelu_tanh(v) (griffin/griffin.py:464, :520) --------------------------------------------------

struct GeluGate : torch::autograd::Function<GeluGate> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h_in, const Tensor& v_in) {
    c10::DeviceGuard guard(h_in.device());
    Tensor h = h_in.contiguous(), v = v_in.contiguous();
    Tensor out = fresh_like(h);
    if (h.numel() > 0)
      check(rglru_hip_gelu_gate_fwd(ptr(h), ptr(v), ptr(out), h.numel(), code_of(h.scalar_type()), stream_of(h)),
            "rglru_hip_gelu_gate_fwd");
    ctx->save_for_backward({h, v});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto s = ctx->get_saved_variables();
    const Tensor &h = s[0], &v = s[1];
    Tensor dh, dv;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(h.device());
      Tensor dout = as(grads[0], h.scalar_type());
      dh = fresh_like(h), dv = fresh_like(v);
      if (h.numel() > 0)
        check(rglru_hip_gelu_gate_bwd(ptr(dout), ptr(h), ptr(v), ptr(dh), ptr(dv), h.numel(), h.size(-1), 0,
                                      code_of(h.scalar_type()), stream_of(h)), "rglru_hip_gelu_gate_bwd");
    }
    return once({dh, dv});
  }
};

Tensor gelu_gate(const Tensor& h, const Tensor& v) {
  require_gpu("hip_gelu_gate", {&h, &v});
  require_device_of("hip_gelu_gate", h, {&v});
  TORCH_CHECK_VALUE(h.sizes() == v.sizes(), "hip_gelu_gate expects equal shapes, got ", h.sizes(), " and ", v.sizes());
  TORCH_CHECK_TYPE(h.scalar_type() == v.scalar_type(), "hip_gelu_gate expects equal dtypes, got ", h.scalar_type(), " and ", v.scalar_type());
  code_of(h.scalar_type());
  return GeluGate::apply(h, v);
}

// ---- convolution, RG-LRU and output gate of the block in one forward launch ---------------------------------------

// [B, T, W] as the library addresses it: channels contiguous, one row stride for all tokens, rows on 16 bytes.
Tensor row_view(const Tensor& t) {
  const int64_t B = t.size(0), T = t.size(1), W = t.size(2);
  if (t.stride(2) == 1 && t.stride(1) >= W && (B == 1 || t.stride(0) == T * t.stride(1)) &&
      (t.stride(1) * t.element_size()) % 16 == 0 && is_aligned(t))
    return t;
  return t.contiguous();
}

Tensor block_flags(const Tensor& segment_pos) {
  require_gpu("hip_block_flags", {&segment_pos});
  c10::DeviceGuard guard(segment_pos.device());
  Tensor pos = segment_pos.to(at::kLong).contiguous();
  Tensor flags = fresh(pos.sizes(), at::kByte, pos);
  if (pos.numel() > 0)
    check(rglru_hip_block_flags(iptr(pos), static_cast<uint8_t*>(flags.data_ptr()), pos.numel(), stream_of(pos)),
          "rglru_hip_block_flags");
  return flags;
}

struct BlockResult {
  Tensor u, v, state, taps, pos, x_conv, y, h0, flags, kept, gated, h_last, new_conv;
};

BlockResult block_forward_pass(const Tensor& u, const Tensor& v, const Tensor& conv_state, const Tensor& weight,
                               const Tensor& bias, const Tensor& segment_pos, const Tensor& flags, bool first_reset,
                               const Tensor& w_a, const Tensor& b_a, const Tensor& w_x, const Tensor& b_x, const Tensor& lam,
                               const Tensor& h0, double c, const Tensor& image, const Tensor& rows, bool need_carry, bool training) {
  BlockResult r;
  c10::DeviceGuard guard(u.device());
  const int64_t B = u.size(0), T = u.size(1), W = u.size(2), K = weight.size(2), nb = w_a.size(0);
  const auto dtype = u.scalar_type();
  const int code = code_of(dtype);
  r.u = row_view(u), r.v = row_view(v);
  r.state = K == 1 ? Tensor() : as(conv_state, dtype);
  r.taps = operand(weight, dtype);
  Tensor b = as(bias, r.taps.scalar_type());
  r.pos = segment_pos.to(u.device(), at::kLong).contiguous();
  r.h0 = as(h0, at::kFloat);
  r.flags = first_reset ? Tensor() : flags.defined() ? flags : block_flags(r.pos);
  r.gated = fresh({B, T, W}, dtype, u);
  if (training) r.x_conv = fresh({B, T, W}, dtype, u), r.y = fresh({B, T, W}, dtype, u);
  r.new_conv = fresh({B, K - 1, W}, dtype, u);
  r.h_last = fresh({B, W}, at::kFloat, u);
  void* stream = stream_of(u);
  void* new_conv = K > 1 && !rows.defined() ? ptr(r.new_conv) : nullptr;   // of a padded row: not its last tokens, see below
  const uint8_t* fl = flags_ptr(r.flags, first_reset);
  if (training || !image.defined()) {
    Operands p(w_a, b_a, w_x, b_x, lam, dtype);
    Kept kept(u, B, T, W, nb, code);
    r.kept = kept.buffer;
    check(rglru_hip_prepare_block_fwd(ptr(p.w_a), ptr(p.b_a), ptr(p.w_x), ptr(p.b_x), ptr(p.lam), static_cast<float>(c), p.vec,
                                      kept.image, ptr(r.u), r.u.stride(1), ptr(r.v), r.v.stride(1), ptr(r.state), ptr(r.taps),
                                      ptr(b), K, fptr(r.h0), fl, ptr(r.x_conv), ptr(r.y), ptr(r.gated), new_conv,
                                      fptr(r.h_last), kept.ws, nullptr, nullptr, nullptr, 0, B, T, W, nb, code, stream), "rglru_hip_prepare_block_fwd");
  } else {
    Tensor ws = bytes(rglru_hip_workspace_bytes(B, T, W, nb), u);
    check(rglru_hip_block_fwd(ptr(r.u), r.u.stride(1), ptr(r.v), r.v.stride(1), ptr(r.state), ptr(r.taps), ptr(b), K,
                              code_of(r.taps.scalar_type()), ptr(image), fptr(r.h0), fl, ptr(r.x_conv), ptr(r.y), ptr(r.gated),
                              new_conv, fptr(r.h_last), ptr(ws), B, T, W, nb, code, stream), "rglru_hip_block_fwd");
  }
  if (rows.defined() && need_carry && K > 1)
    check(rglru_hip_conv_carry(ptr(r.u), r.u.stride(1), ptr(r.state), static_cast<const int32_t*>(ptr(rows)), ptr(r.new_conv), B, T, W, K,
                               code, stream), "rglru_hip_conv_carry");
  return r;
}

// The backward pass runs the three reverse kernels one after the other on the x and y the forward kept.
struct BlockForward : torch::autograd::Function<BlockForward> {
  static variable_list forward(AutogradContext* ctx, const Tensor& u, const Tensor& v, const MaybeTensor& conv_state_,
                               const Tensor& weight, const MaybeTensor& bias_, const Tensor& segment_pos,
                               const MaybeTensor& flags_, bool first_reset, const Tensor& w_a, const Tensor& b_a,
                               const Tensor& w_x, const Tensor& b_x, const Tensor& lam, const MaybeTensor& h0_, double c,
                               const MaybeTensor& rows_, bool need_carry) {
    Tensor conv_state = opt(conv_state_), bias = opt(bias_), flags = opt(flags_), h0 = opt(h0_), rows = opt(rows_);
    note_arguments(ctx, {true, true, conv_state.defined(), true, bias.defined(), true, flags.defined(), true, true, true, true,
                         true, h0.defined()});
    BlockResult r = block_forward_pass(u, v, conv_state, weight, bias, segment_pos, flags, first_reset, w_a, b_a, w_x, b_x, lam,
                                       h0, c, Tensor(), rows, need_carry, true);
    ctx->save_for_backward({r.u, r.v, r.state, r.taps, r.pos, r.x_conv, r.y, r.h0, r.flags, r.kept, rows});
    auto t = types_of(w_a, b_a, w_x, b_x, lam);
    pack(ctx, {first_reset, w_a.size(0), type_or_none(h0), (int64_t)t[0], (int64_t)t[1], (int64_t)t[2], (int64_t)t[3], (int64_t)t[4],
               type_or_none(conv_state), type_or_none(weight), type_or_none(bias)});
    ctx->mark_non_differentiable({r.new_conv});
    ctx->set_materialize_grads(false);
    return {r.gated, r.h_last, r.new_conv};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto s = ctx->get_saved_variables();
    auto m = unpack(ctx);
    const Tensor &u = s[0], &v = s[1], &state = s[2], &taps = s[3], &pos = s[4], &x_conv = s[5], &y = s[6], &h0 = s[7],
                 &flags = s[8], &kept = s[9];
    Needs need(ctx);  // by tensor argument of forward: u, v, conv_state, weight, bias, ... (12: h0)
    const bool need_u = need(0), need_v = need(1);
    Tensor dv;
    ParamGrads g;
    variable_list conv;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(y.device());
      const int64_t B = y.size(0), T = y.size(1), W = y.size(2);
      const auto dtype = y.scalar_type();
      Tensor dy, du_out;
      if (grads[0].defined()) {
        Tensor dout = as(grads[0], dtype);
        Tensor v_c = v.contiguous();
        dy = fresh_like(y);
        const int64_t row_bytes = W * y.element_size();
        if (need_u && need_v && row_bytes % 16 == 0 && B * T * 2 * row_bytes < (int64_t(1) << 31)) {
          // The gradients of the two projections as the halves of ONE [B, T, 2 W] matrix: the Linear layers' backward
          // then runs one GEMM each for dx and dW and one column sum (linear_pair).
          Tensor both = fresh({B, T, 2 * W}, dtype, y);
          du_out = both.narrow(2, 0, W), dv = both.narrow(2, W, W);
        } else {
          dv = fresh_like(v_c);
        }
        check(rglru_hip_gelu_gate_bwd(ptr(dout), ptr(y), ptr(v_c), ptr(dy), ptr(dv), y.numel(), W, dv.stride(1), code_of(dtype),
                                      stream_of(y)), "rglru_hip_gelu_gate_bwd");
      }
      g = rglru_backward(x_conv, y, m[1], h0, flags, m[0], kept, dy, grads[1],
                         {type_at(m, 3), type_at(m, 4), type_at(m, 5), type_at(m, 6), type_at(m, 7)}, need(12), false);
      if (g.dh0.defined() && type_at(m, 2) != at::kFloat) g.dh0 = g.dh0.to(type_at(m, 2));
      conv = conv_backward(u.contiguous(), state, taps, pos, g.dx, {m[8], m[9], m[10]}, need_u, need(2), need(3),
                           need(4), du_out, s[10]);
      if (!need_v) dv = Tensor();
    }
    return once({conv[0], dv, conv[1], conv[2], conv[3], Tensor(), Tensor(), Tensor(), g.dw_a, g.db_a, g.dw_x, g.db_x, g.dlam,
                 g.dh0, Tensor(), Tensor(), Tensor()});
  }
};

std::tuple<Tensor, Tensor, Tensor> block_forward(const Tensor& u, const Tensor& v, const MaybeTensor& conv_state_,
                                                 const Tensor& weight, const MaybeTensor& bias_, const Tensor& segment_pos,
                                                 const MaybeTensor& flags_, bool first_reset, const Tensor& w_a, const Tensor& b_a,
                                                 const Tensor& w_x, const Tensor& b_x, const Tensor& lam, const MaybeTensor& h0_,
                                                 double c, const MaybeTensor& image_, const MaybeTensor& rows_, bool need_carry) {
  Tensor conv_state = opt(conv_state_), bias = opt(bias_), flags = opt(flags_), h0 = opt(h0_), rows = opt(rows_);
  require_gpu("hip_block_forward", {&u, &v, &conv_state, &weight, &bias, &segment_pos, &w_a, &b_a, &w_x, &b_x, &lam, &h0});
  const Tensor image = opt(image_);
  require_device_of("hip_block_forward", u, {&v, &conv_state, &weight, &bias, &flags, &w_a, &b_a, &w_x, &b_x, &lam, &h0, &rows, &image});
  TORCH_CHECK_VALUE(u.dim() == 3 && u.sizes() == v.sizes() && u.scalar_type() == v.scalar_type(),
                    "hip_block_forward expects two [batch, sequence, width] tensors of one dtype");
  const int64_t B = u.size(0), T = u.size(1), W = u.size(2);
  check_conv("hip_block_forward", u, conv_state, weight, bias, segment_pos);
  check_gates(w_a, b_a, w_x, b_x, lam);
  TORCH_CHECK_VALUE(w_a.size(0) * w_a.size(1) == W, "gate weights ", w_a.sizes(), " do not match width ", W);
  TORCH_CHECK_VALUE(!h0.defined() || (h0.dim() == 2 && h0.size(0) == B && h0.size(1) == W), "initial state must have shape (", B, ", ", W, ")");
  TORCH_CHECK_VALUE(!flags.defined() || (flags.dim() == 2 && flags.size(0) == B && flags.size(1) == T && flags.scalar_type() == at::kByte && flags.is_contiguous()),
                    "flags must be a contiguous uint8 tensor of shape [batch, sequence]");
  if (wants_grad({&u, &v, &conv_state, &weight, &bias, &w_a, &b_a, &w_x, &b_x, &lam, &h0})) {
    auto out = BlockForward::apply(u, v, maybe(conv_state), weight, maybe(bias), segment_pos, maybe(flags), first_reset, w_a,
                                   b_a, w_x, b_x, lam, maybe(h0), c, maybe(rows), need_carry);
    return {out[0], out[1], out[2]};
  }
  at::NoGradGuard no_grad;
  BlockResult r = block_forward_pass(u, v, conv_state, weight, bias, segment_pos, flags, first_reset, w_a, b_a, w_x, b_x, lam, h0, c,
                                     image, rows, need_carry, false);
  return {r.gated, r.h_last, r.new_conv};
}

// One token per row through conv -> RG-LRU step -> output gate (no autograd), two kernel launches.
std::tuple<Tensor, Tensor, Tensor, Tensor> block_decode_step(const Tensor& u_in, const Tensor& v_in, const MaybeTensor& conv_state_,
                                                             const Tensor& weight, const MaybeTensor& bias_, const MaybeTensor& prev_pos_,
                                                             const MaybeTensor& segment_pos_, const MaybeTensor& active_,
                                                             const Tensor& image, int64_t width, int64_t blocks, at::ScalarType prep_dtype,
                                                             const MaybeTensor& rnn_state_) {
  Tensor conv_state = opt(conv_state_), bias = opt(bias_), prev_pos = opt(prev_pos_), segment_pos = opt(segment_pos_),
         active = opt(active_), rnn_state = opt(rnn_state_);
  require_gpu("hip_block_decode_step", {&u_in, &v_in, &conv_state, &weight, &bias, &prev_pos, &segment_pos, &active, &rnn_state});
  require_device_of("hip_block_decode_step", u_in, {&v_in, &conv_state, &weight, &bias, &prev_pos, &segment_pos, &active, &image, &rnn_state});
  TORCH_CHECK_VALUE(u_in.dim() == 2 && u_in.sizes() == v_in.sizes() && u_in.scalar_type() == v_in.scalar_type(),
                    "hip_block_decode_step expects two [batch, width] tensors of one dtype");
  const int64_t B = u_in.size(0), W = u_in.size(1), K = weight.size(2);
  TORCH_CHECK_VALUE(W == width && u_in.scalar_type() == prep_dtype, "the prepared RG-LRU parameters do not match the activations");
  TORCH_CHECK_VALUE(weight.dim() == 3 && weight.size(0) == W && weight.size(1) == 1, "weight must be that of a depthwise Conv1d: [width, 1, kernel_size]");
  TORCH_CHECK_VALUE(!bias.defined() || (bias.dim() == 1 && bias.size(0) == W), "bias must have shape [width]");
  TORCH_CHECK_VALUE(!conv_state.defined() || (conv_state.dim() == 3 && conv_state.size(0) == B && conv_state.size(1) == K - 1 && conv_state.size(2) == W),
                    "state must have shape [batch, kernel_size - 1, width]");
  TORCH_CHECK_VALUE(!rnn_state.defined() || (rnn_state.dim() == 2 && rnn_state.size(0) == B && rnn_state.size(1) == W), "the state must have shape (",
                    B, ", ", W, ")");
  for (const Tensor* t : {&prev_pos, &segment_pos})
    TORCH_CHECK_VALUE(!t->defined() || (t->numel() == B && t->scalar_type() == at::kLong && t->is_contiguous()), "positions must be ", B, " contiguous integers");
  active = token_bytes(active, B);
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(u_in.device());
  const auto dtype = u_in.scalar_type();
  const int code = code_of(dtype);
  // rows may be views into a wider buffer (the two halves of one fused projection)
  auto rows = [W](const Tensor& t) { return t.stride(1) == 1 && t.stride(0) >= W ? t : t.contiguous(); };
  Tensor u = rows(u_in), v = rows(v_in);
  Tensor state = K == 1 ? Tensor() : as(conv_state, dtype);
  Tensor taps = operand(weight, dtype);
  Tensor b = as(bias, taps.scalar_type());
  Tensor new_conv = fresh({B, K - 1, W}, dtype, u);
  Tensor new_pos = fresh({B}, at::kLong, u);
  Tensor h_in = rnn_state.defined() ? as(rnn_state, at::kFloat) : at::zeros({B, W}, u.options().dtype(at::kFloat));
  Tensor h_out = fresh({B, W}, at::kFloat, u);
  Tensor out = fresh({B, W}, dtype, u);
  const size_t x_bytes = round_up(B * W * u.element_size());
  Tensor scratch = bytes(x_bytes + B, u);
  char* x = static_cast<char*>(scratch.data_ptr());
  uint8_t* flags = reinterpret_cast<uint8_t*>(x + x_bytes);
  void* stream = stream_of(u);
  check(rglru_hip_decode_prepare(ptr(u), u.stride(0), ptr(state), ptr(taps), ptr(b), iptr(prev_pos), iptr(segment_pos), bptr(active),
                                 x, K > 1 ? ptr(new_conv) : nullptr, static_cast<int64_t*>(new_pos.data_ptr()), flags, B, W, K, code,
                                 code_of(taps.scalar_type()), stream), "rglru_hip_decode_prepare");
  check(rglru_hip_step_gated(x, ptr(image), fptr(h_in), fptr(h_out), flags, ptr(v), v.stride(0), ptr(out), B, W, blocks, code, stream),
        "rglru_hip_step_gated");
  return {out, h_out, new_conv, new_pos};
}

// A vector of n elements, or absent.
bool has(const Tensor& t, int64_t n) { return !t.defined() || (t.dim() == 1 && t.size(0) == n); }

// Whether the Linear layers and the convolution of a block belong together: [W, D] twice, [W, 1, K], [D, W], with biases to match.
bool block_shapes(int64_t D, const Tensor& w_x, const Tensor& b_x, const Tensor& w_y, const Tensor& b_y, const Tensor& conv_w, const Tensor& conv_b,
                  const Tensor& w_o, const Tensor& b_o) {
  if (w_x.dim() != 2 || w_x.size(1) != D || w_y.sizes() != w_x.sizes() || w_o.dim() != 2 || conv_w.dim() != 3) return false;
  const int64_t W = w_x.size(0);
  return has(b_x, W) && has(b_y, W) && conv_w.size(0) == W && conv_w.size(1) == 1 && conv_w.size(2) >= 1 && has(conv_b, W) && w_o.size(0) == D &&
         w_o.size(1) == W && has(b_o, D);
}

// ... and the carried state of B rows.
bool state_shapes(int64_t B, int64_t W, int64_t K, const Tensor& conv_state, const Tensor& rnn_state, const Tensor& positions) {
  if (conv_state.defined() && (conv_state.dim() != 3 || conv_state.size(0) != B || conv_state.size(1) != K - 1 || conv_state.size(2) != W)) return false;
  return (!rnn_state.defined() || (rnn_state.dim() == 2 && rnn_state.size(0) == B && rnn_state.size(1) == W)) && has(positions, B);
}

// The whole single-token step of the block around the RG-LRU (griffin/griffin.py:459-528 with T == 1, no autograd) in three
// launches: projections + positions + convolution, RG-LRU step + output gate, output projection.  Nothing is returned
// where the kernels do not take the operands (mixed types, unaligned rows, many rows): the caller then goes through the
// BLAS library.
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> block_step(
    const Tensor& x_in, const Tensor& w_x, const MaybeTensor& b_x_, const Tensor& w_y, const MaybeTensor& b_y_, const Tensor& conv_w,
    const MaybeTensor& conv_b_, const Tensor& w_o, const MaybeTensor& b_o_, const MaybeTensor& conv_state_, const MaybeTensor& prev_pos_,
    const MaybeTensor& segment_pos_, const MaybeTensor& active_, const Tensor& image, int64_t blocks, const MaybeTensor& rnn_state_) {
  Tensor b_x = opt(b_x_), b_y = opt(b_y_), conv_b = opt(conv_b_), b_o = opt(b_o_), conv_state = opt(conv_state_),
         prev_pos = opt(prev_pos_), segment_pos = opt(segment_pos_), active = opt(active_), rnn_state = opt(rnn_state_);
  const auto dtype = x_in.scalar_type();
  refuse_tangents("hip_block_step", std::initializer_list<Tensor>{x_in, w_x, b_x, w_y, b_y, conv_w, conv_b, w_o, b_o, conv_state, rnn_state});
  if (!block_shapes(x_in.size(2), w_x, b_x, w_y, b_y, conv_w, conv_b, w_o, b_o)) return std::nullopt;
  const int64_t B = x_in.size(0), D = x_in.size(2), W = w_x.size(0), K = conv_w.size(2);
  if (!state_shapes(B, W, K, conv_state, rnn_state, prev_pos) || !has(segment_pos, B)) return std::nullopt;
  for (const Tensor* t : std::initializer_list<const Tensor*>{&w_x, &b_x, &w_y, &b_y, &conv_w, &conv_b, &w_o, &b_o, &conv_state, &prev_pos, &segment_pos,
                                                              &active, &image, &rnn_state})
    if (!on_device_of(x_in, *t)) return std::nullopt;
  active = token_bytes(active, B);
  if (K > 4 || B >= (1 << 16) || !own_projections(B, 3.0 * B * W * D, dtype) || (D * x_in.element_size()) % 16 || (W * x_in.element_size()) % 16) return std::nullopt;
  for (const Tensor* t : std::initializer_list<const Tensor*>{&w_x, &b_x, &w_y, &b_y, &conv_w, &conv_b, &w_o, &b_o, &conv_state})
    if (t->defined() && (t->scalar_type() != dtype || !t->is_contiguous())) return std::nullopt;
  for (const Tensor* t : std::initializer_list<const Tensor*>{&w_x, &w_y, &w_o})
    if (!is_aligned(*t)) return std::nullopt;
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(x_in.device());
  const int code = code_of(dtype);
  Tensor x = x_in;
  if (x.stride(2) != 1 || (x.stride(0) * x.element_size()) % 16 || !is_aligned(x)) x = aligned(x);
  Tensor h_in = rnn_state.defined() ? as(rnn_state, at::kFloat) : at::zeros({B, W}, x.options().dtype(at::kFloat));
  Tensor h_out = fresh({B, W}, at::kFloat, x), new_conv = fresh({B, K - 1, W}, dtype, x), new_pos = fresh({B}, at::kLong, x);
  Tensor out = fresh({B, 1, D}, dtype, x);
  // x after the convolution, the second branch, their product with the state, one flag byte per row
  const size_t row_bytes = round_up(B * W * x.element_size());
  Tensor scratch = bytes(3 * row_bytes + B, x);
  char* sp = static_cast<char*>(scratch.data_ptr());
  uint8_t* flags = reinterpret_cast<uint8_t*>(sp + 3 * row_bytes);
  void* stream = stream_of(x);
  check(rglru_hip_decode_project(ptr(x), x.stride(0), ptr(w_x), ptr(b_x), ptr(w_y), ptr(b_y), ptr(conv_state), ptr(conv_w), ptr(conv_b),
                                 iptr(prev_pos), iptr(segment_pos), bptr(active), sp, sp + row_bytes, K > 1 ? ptr(new_conv) : nullptr,
                                 static_cast<int64_t*>(new_pos.data_ptr()), flags, B, D, W, K, code, stream), "rglru_hip_decode_project");
  check(rglru_hip_step_gated(sp, ptr(image), fptr(h_in), fptr(h_out), flags, sp + row_bytes, W, sp + 2 * row_bytes, B, W, blocks, code,
                             stream), "rglru_hip_step_gated");
  check(rglru_hip_decode_linear(sp + 2 * row_bytes, W, ptr(w_o), ptr(b_o), bptr(active), ptr(out), B, D, W, code, stream),
        "rglru_hip_decode_linear");
  return std::make_tuple(out, h_out, new_conv, new_pos);
}

// ---- single-token calls of the modules ----------------------------------------------------------------------------
// What a module's forward does around a decode step -- look up its parameters, check shapes, types and the prepared image --
// costs the interpreter more than the step's launches take (layer: 5 of 9 us, block: 8 of 18).  These read the module's own
// dictionaries and do it here.  None: not the plain case, the module's Python code goes on (and reports what is wrong).

std::atomic<uint64_t> usable_devices{0};                   // GPUs whose one-time self-test has passed
void mark_usable(int64_t device, bool usable) {
  if (device < 0 || device >= 64) return;
  if (usable) usable_devices |= uint64_t(1) << device; else usable_devices &= ~(uint64_t(1) << device);
}

// Members of an nn.Module as its instance dictionary holds them (borrowed references; null where missing).
struct Members {
  PyObject* dict;
  explicit Members(PyObject* module) : dict(nullptr) {
    PyObject** d = module != nullptr ? _PyObject_GetDictPtr(module) : nullptr;
    if (d != nullptr) dict = *d;
  }
  PyObject* at(const char* name) const { return dict != nullptr ? PyDict_GetItemString(dict, name) : nullptr; }
  static PyObject* in(PyObject* d, const char* name) { return d != nullptr && PyDict_Check(d) ? PyDict_GetItemString(d, name) : nullptr; }
  // a pass without gradients: the graph ends held for training keep nothing alive meanwhile
  void drop_leaves() const {
    PyObject* held = at("_leaves");
    if (held != nullptr && held != Py_None) PyDict_SetItemString(dict, "_leaves", Py_None);
  }
  PyObject* module(const char* name) const { return in(at("_modules"), name); }
  bool parameter(const char* name, Tensor& t) const {
    PyObject* p = in(at("_parameters"), name);
    if (p == nullptr || !THPVariable_Check(p)) return false;
    t = THPVariable_Unpack(p);
    return !t.key_set().has(c10::DispatchKey::Python);        // a tensor that dispatches itself (quantised weights) has no plain memory
  }
  // a plain number; anything else (an array scalar, a tensor, no such attribute) is left to the module's Python code
  std::optional<double> number(const char* name) const {
    PyObject* v = at(name);
    if (v == nullptr || !(PyFloat_Check(v) || PyLong_Check(v))) return std::nullopt;
    const double d = PyFloat_AsDouble(v);
    if (d == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return std::nullopt;
    }
    return d;
  }
  // calling the layer does more than its class's forward: hooks, or a forward of its own
  bool hooked() const {
    if (at("forward") != nullptr) return true;
    for (const char* name : {"_forward_hooks", "_forward_pre_hooks"}) {
      PyObject* h = at(name);
      if (h == nullptr || PyObject_Length(h) != 0) return true;
    }
    return false;
  }
};

bool usable_mode(const Members& lru, c10::Device device) {
  PyObject* mode = lru.at("scan_mode");
  if (mode == nullptr || !PyUnicode_Check(mode)) return false;
  if (PyUnicode_CompareWithASCIIString(mode, "auto") == 0) return (usable_devices.load(std::memory_order_relaxed) >> device.index()) & 1;
  return PyUnicode_CompareWithASCIIString(mode, "hip") == 0 || PyUnicode_CompareWithASCIIString(mode, "fused") == 0;
}

// The prepared image an RG_LRU module keeps, if it is that of its parameters as they are now.
const Stamp* current_stamp(const Members& lru, at::ScalarType dtype, c10::Device device) {
  PyObject* held = lru.at("_prep_key");
  if (held == nullptr || held == Py_None || !py::isinstance<Stamp>(held)) return nullptr;
  const Members r(lru.module("recurrence_gate")), i(lru.module("input_gate"));
  std::array<Tensor, 5> p;
  if (!r.parameter("weight", p[0]) || !r.parameter("bias", p[1]) || !i.parameter("weight", p[2]) || !i.parameter("bias", p[3]) ||
      !lru.parameter("Lambda", p[4]))
    return nullptr;
  const Stamp* s = py::handle(held).cast<const Stamp*>();
  const auto c = lru.number("c");
  return c && s->image.defined() && s->image.device() == device && s->holds(p, p.size(), *c, dtype) ? s : nullptr;
}

// RG_LRU on one token per row without masks: (y, state).
py::object lru_decode(py::handle module, const Tensor& x, const MaybeTensor& state) {
  if (at::GradMode::is_enabled()) return py::none();
  const Members lru(module.ptr());
  lru.drop_leaves();
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_cuda() || !known(x.scalar_type()) || x.numel() == 0) return py::none();
  if (lru.number("rnn_width") != double(x.size(2)) || !usable_mode(lru, x.device())) return py::none();
  if (state.has_value() && (state->dim() != 2 || state->size(0) != x.size(0) || state->size(1) != x.size(2) || state->scalar_type() != at::kFloat ||
                            state->device() != x.device()))
    return py::none();
  const Stamp* s = current_stamp(lru, x.scalar_type(), x.device());
  if (s == nullptr) return py::none();
  auto [y, h] = rglru_module_step(x, s->image, s->blocks, state, std::nullopt);
  return py::make_tuple(y, h);
}

// RecurrentBlock on one token per row, every row active, positions carried on: (output, rnn_state, conv_state, positions).
py::object block_decode(py::handle module, const Tensor& x, py::handle cache, py::handle linear_type) {
  if (at::GradMode::is_enabled()) return py::none();
  const Members block(module.ptr());
  block.drop_leaves();
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_cuda() || !known(x.scalar_type()) || x.numel() == 0 || at::autocast::is_autocast_enabled(at::kCUDA))
    return py::none();
  PyObject* layers[4] = {block.module("linear_x"), block.module("linear_y"), block.module("linear_out"), block.module("temporal_conv")};
  for (int i = 0; i < 3; ++i)
    if (layers[i] == nullptr || (PyObject*)Py_TYPE(layers[i]) != linear_type.ptr()) return py::none();
  const Members lx(layers[0]), ly(layers[1]), lo(layers[2]), conv(layers[3]), lru(block.module("rg_lru"));
  if (lx.hooked() || ly.hooked() || lo.hooked() || !usable_mode(lru, x.device())) return py::none();
  Tensor wx, bx, wy, by, cw, cb, wo, bo;
  if (!lx.parameter("weight", wx) || !lx.parameter("bias", bx) || !ly.parameter("weight", wy) || !ly.parameter("bias", by) ||
      !conv.parameter("weight", cw) || !conv.parameter("bias", cb) || !lo.parameter("weight", wo) || !lo.parameter("bias", bo))
    return py::none();
  const auto width = block.number("rnn_width"), taps = block.number("conv_kernel_size");
  if (!width || !taps) return py::none();
  const int64_t B = x.size(0), W = (int64_t)*width, K = (int64_t)*taps;
  if (wx.dim() != 2 || wx.size(0) != W || cw.dim() != 3 || cw.size(2) != K || wx.scalar_type() != x.scalar_type()) return py::none();
  MaybeTensor conv_state, prev, rnn;
  if (!cache.is_none()) {
    auto field = [&](const char* name, MaybeTensor& t) {
      py::object v = py::reinterpret_steal<py::object>(PyObject_GetAttrString(cache.ptr(), name));
      if (!v) { PyErr_Clear(); return false; }
      if (v.is_none()) return true;
      if (!THPVariable_Check(v.ptr())) return false;
      t = THPVariable_Unpack(v.ptr());
      return t->device() == x.device();
    };
    if (!field("conv_state", conv_state) || !field("segment_position", prev) || !field("rnn_state", rnn)) return py::none();
    if (!conv_state || !prev || !state_shapes(B, W, K, *conv_state, opt(rnn), *prev) || prev->scalar_type() != at::kLong || !prev->is_contiguous())
      return py::none();                                   // the module's Python code reports a wrong shape
  }
  if (!own_projections_captured(3.0 * B * W * x.size(2))) {
    // the module's Python code leaves the stacked projection that a capture of this step would go through
    PyObject* stacked = block.at("_stacked_projection");
    if (stacked == nullptr || stacked == Py_None) return py::none();
  }
  const Stamp* s = current_stamp(lru, x.scalar_type(), x.device());
  if (s == nullptr) return py::none();
  auto done = block_step(x, wx, bx, wy, by, cw, cb, wo, bo, conv_state, prev, std::nullopt, std::nullopt, s->image, s->blocks, rnn);
  if (!done.has_value()) return py::none();
  return py::cast(*done);
}

// ---- Linear layers of the block (griffin/griffin.py:379-389) ------------------------------------------------------

// sets.sum(0) of a contiguous [sets, ...] tensor in one pass; anything the kernel does not take goes to the generic one.
Tensor sum_sets(const Tensor& sets) {
  if (!sets.is_cuda() || !known(sets.scalar_type()) || !sets.is_contiguous() || sets.numel() == 0) return sets.sum(0);
  c10::DeviceGuard guard(sets.device());
  Tensor out = fresh(sets.sizes().slice(1), sets.scalar_type(), sets);
  check(rglru_hip_sum_sets(ptr(sets), ptr(out), sets.size(0), out.numel(), code_of(sets.scalar_type()), stream_of(sets)),
        "rglru_hip_sum_sets");
  return out;
}

// Whether products of `macs` multiply-adds each (tokens x width x model width) run on the library's own kernels.  The BLAS
// library is the faster one on long products (see rglru_linear.hip), but each call of it keeps the host for 17 us and a
// training step of the block has seven.  Without gradients and in fp32 the line lies where both ways take about equally long per layer in a
// stack of eight blocks, alone or with an MLP of three products behind each (profiles/block_products_own_vs_blas_in_stacks.txt, us own : BLAS,
// alone / with MLPs).  bf16, prefill 768 -> 1024: at 4.0e9 82 : 86 / 201 : 199, at 6.0e9
// 96 : 102 / 281 : 287, at 8.0e9 116 : 117 / 325 : 336, at 1.3e10 163 : 149 / 453 : 442;  2560 at 6.0e9 126 : 135 / 306 : 303, at 6.7e9 141 : 127 / 327 : 311.  So
// between 6e9 and 9e9 either way wins somewhere.  fp32, training 768 -> 1024: at 8e8 326 : 469 / 759 : 755, at 9e8 362 : 468 / 843 : 824, at 1.2e9
// 430 : 463, at 1.6e9 484 : 452;  wide and short ones lose below the line: 2560 -> 2560 at 5.8e8 (88 tokens) 481 : 466 / 1004 : 865, prefill
// 151 : 123.
// In a training step of the block in bf16, steps queued behind each other, us: gradients on the BLAS library : own, then the forward own as well.
// 768 -> 1024 at 6.3e9 374 : 317 : 305, 7.9e9 453 : 385 : 377, 9.7e9 442 : 443 : 439, 1.02e10 603 : 475 : 471, 1.3e10 516 : - : 542;  2560 -> 2560 at 6.0e9 482 :
// 401 : 340, 8.5e9 485 : 395 : 388, 1.18e10 541 : 460 : 474, 1.3e10 542 : - : 516;  1536 -> 2048 at 6.4e9 317 : 278 : 273, 7.5e9 346 : 318 : 331, 9.4e9 388 :
// 371 : 387, 1.3e10 447 : - : 477.
// A Linear layer by itself in bf16, forward and backward, gradients own : BLAS: 1024 x 768 at 7884 tokens 69 : 110, 8192 69 : 85, 14336 99 : 118; 2560 x 2560 at
// 948 79 : 84, 1812 107 : 126; 4096 x 1024 at 2836 109 : 110; the other way at 1024 x 4096, 2836 tokens, 111 : 107 and 4096 x 4096, 372 tokens, 85 : 82.
// Inside a captured graph host time is nothing.  The line there is where kernels took equally long whose slices went through registers; with those of
// today it is early.  Captured step in bf16, us, own : gradients alone own : BLAS: 768 -> 1024 at 2.0e9 155 : 167 : 175, 4.8e9 235 : 244 : 264, 9.7e9 406 :
// 421 : 424; 1536 -> 2048 at 4.7e9 229 : 233 : 229, 9.4e9 330 : 330 : 331, 1.3e10 432 : 428 : 406; 2560 -> 2560 at 5.0e9 270 : 272 : 292, 1.3e10 438 : 444 :
// 477; without gradients 768 -> 1024 at 4.8e9 66 : 76, 9.7e9 102 : 114; 2560 -> 2560 at 3.3e9 83 : 74, 6.7e9 106 : 95.
enum class Product { kInference, kTrainingForward, kGradient };
bool own_products(double macs, at::ScalarType dtype, Product use = Product::kInference) {
  if (!known(dtype)) return false;
  const bool bf16 = dtype == at::kBFloat16;
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return macs < (bf16 ? 2e9 : 4e8);
  if (!bf16) return macs < 9e8;
  return macs < (use == Product::kInference ? 6e9 : use == Product::kTrainingForward ? 9e9 : 1.2e10);
}

// Contiguous rows of whole 16-byte vectors, as rglru_hip_linear takes them.
bool vector_rows(const Tensor& t) {
  return t.is_contiguous() && (t.size(-1) * t.element_size()) % 16 == 0 && is_aligned(t);
}

// A tensor that dispatches itself (a subclass with __torch_dispatch__: quantised or distributed weights, wrapped inputs) or stands for a batch of
// them (vmap, batched gradients) has no memory for a kernel to read; PyTorch's product takes it.
bool plain(const Tensor& t) { return !t.defined() || (!t.key_set().has(c10::DispatchKey::Python) && t.has_storage()); }

// Whether the library takes y = x w^T + b (and its gradients) for these operands.
bool own_linear(const Tensor& x, const Tensor& w, const Tensor& b, Product use = Product::kInference) {
  const auto dtype = x.scalar_type();
  return plain(x) && plain(w) && plain(b) && w.dim() == 2 && x.size(-1) == w.size(1) && on_device_of(x, w) && on_device_of(x, b) && w.scalar_type() == dtype && has(b, w.size(0)) && (!b.defined() || (b.scalar_type() == dtype && b.is_contiguous())) &&
         x.numel() > 0 && own_products(double(x.numel()) * w.size(0), dtype, use) && vector_rows(w) && vector_rows(x) &&
         (w.size(0) * x.element_size()) % 16 == 0 && !at::autocast::is_autocast_enabled(at::kCUDA);
}

void linear_forward(const Tensor& x, const Tensor& w0, const Tensor& b0, const Tensor& w1, const Tensor& b1, const Tensor& active, void* y0,
                    void* y1) {
  const int64_t K = x.size(-1), N = w0.size(0);
  check(rglru_hip_linear(RGLRU_LINEAR_FORWARD, ptr(x), nullptr, K, ptr(w0), ptr(w1), K, ptr(b0), ptr(b1), bptr(active), y0, y1, N,
                         nullptr, nullptr, x.numel() / K, N, K, code_of(x.scalar_type()), stream_of(x)), "rglru_hip_linear");
}

// Sizes that rglru_hip_linear addresses.
bool own_rows(int64_t rows, int64_t n, int64_t k) { return rows < (int64_t(1) << 30) && n < (1 << 22) && k < (1 << 22); }

// Weight and bias gradients of one or two Linear layers on one input x [rows, K]: dy_i [rows, N], rows `ld` elements apart.
struct WeightGrad {
  int64_t splits, sets_bytes, sums_bytes, N, K, problems;
  WeightGrad(int64_t rows, int64_t n, int64_t k, int64_t n_problems, at::ScalarType dtype) : N(n), K(k), problems(n_problems) {
    splits = rglru_hip_linear_splits(RGLRU_LINEAR_WEIGHT_GRAD, N, K, rows, problems, code_of(dtype));
    sets_bytes = splits > 1 ? splits * problems * N * K * 4 : 0;
    sums_bytes = splits * problems * N * 4;
  }
  // dw (problems x N x K, contiguous) is written here where nothing is left to add up
  void run(const void* dy0, const void* dy1, int64_t ld, const void* x, const uint8_t* active, void* dw, void* sets, void* sums,
           int64_t rows, at::ScalarType dtype, void* stream) const {
    char* second = problems == 2 ? static_cast<char*>(dw) + N * K * c10::elementSize(dtype) : nullptr;
    check(rglru_hip_linear(RGLRU_LINEAR_WEIGHT_GRAD, dy0, dy1, ld, x, nullptr, K, nullptr, nullptr, active, dw, second, K,
                           static_cast<float*>(sets), static_cast<float*>(sums), N, K, rows, code_of(dtype), stream), "rglru_hip_linear");
  }
  rglru_sum weight_sum(void* sets, void* dw) const { return {sets, splits > 1 ? dw : nullptr, splits, problems * N * K, RGLRU_F32}; }
  rglru_sum bias_sum(void* sums, void* db) const { return {sums, db, splits, problems * N, RGLRU_F32}; }
};

// dW = dy^T x contracts over all tokens: one GEMM of the BLAS library with K = rows runs at a fraction of the rate of the same
// work as a batch of GEMMs with K = 2048 whose results are added (100 us against 43 us for 16384 x 1024 x 768 in bf16), so
// long contractions are split into this many.  Other numbers of tokens (1) take the library's own kernel in bf16: two of 1024 x 768 at 8704 tokens 39
// us, the BLAS library 66; at 8192 37 : 34, at 16384 59 : 52.  Own : one product of the BLAS library over 90 sizes of 512 to 10000 channels and 2063 to 60000
// tokens: 0.27 to 0.98 of its time in 84 of them (1024 x 768 at 4851 24 : 39, 2 x 2560 x 2496 at 5539 155 : 188, 4992 x 4608 at 43097 1932 : 2622), 1.03 to
// 1.12 in six that have no size in common (2 x 3968 x 2688 at 5707 304 : 270); 1.02 to 1.05 at 4096 x 4096 and 8192 x 4096 from 20000 tokens on.
int64_t contraction_chunks(int64_t rows) {
  int64_t chunks = rows % 2048 == 0 ? rows / 2048 : 1;
  while (chunks > 16 && chunks % 2 == 0) chunks /= 2;
  return chunks;
}

// (dW, db) of y = x W^T + b for the incoming dy; bias_type kNone skips db.
std::tuple<Tensor, Tensor> linear_parameter_grads(const Tensor& x, at::ScalarType weight_type, const Tensor& dy, bool need_w, int64_t bias_type) {
  Tensor dy2 = dy.reshape({-1, dy.size(-1)});
  Tensor dw, db;
  const int64_t rows = dy2.size(0), width = dy2.size(1);
  if (need_w) {
    Tensor x2 = x.reshape({-1, x.size(-1)}).to(dy.scalar_type());
    const int64_t chunks = dy2.is_contiguous() && x2.is_contiguous() ? contraction_chunks(rows) : 1;
    if (chunks == 1 && rows >= 2048 && own_rows(rows, width, x2.size(1)) && x2.scalar_type() == at::kBFloat16 && plain(x) && plain(dy) && on_device_of(x2, dy2) && vector_rows(x2) && vector_rows(dy2)) {
      const WeightGrad own(rows, width, x2.size(1), 1, at::kBFloat16);
      Tensor sets = own.splits > 1 ? fresh({own.splits, width, x2.size(1)}, at::kFloat, dy2) : Tensor();
      dw = fresh({width, x2.size(1)}, at::kBFloat16, dy2);
      own.run(ptr(dy2), nullptr, width, ptr(x2), nullptr, ptr(dw), ptr(sets), nullptr, rows, at::kBFloat16, stream_of(dy2));
      if (own.splits > 1) {
        const rglru_sum job = own.weight_sum(ptr(sets), ptr(dw));
        check(rglru_hip_sums(&job, 1, RGLRU_BF16, stream_of(dy2)), "rglru_hip_sums");
      }
    } else if (chunks > 1) {
      const int64_t per = rows / chunks;
      dw = sum_sets(at::bmm(dy2.view({chunks, per, width}).transpose(1, 2), x2.view({chunks, per, x2.size(1)})));
    } else {
      dw = at::mm(dy2.t(), x2);
    }
    if (dw.scalar_type() != weight_type) dw = dw.to(weight_type);
  }
  if (bias_type != kNone) {
    const auto bt = static_cast<at::ScalarType>(bias_type);
    const auto ot = known(bt) ? bt : at::kFloat;
    Tensor dy_c = dy2.contiguous();
    db = fresh({width}, ot, dy);
    Tensor scratch = bytes(rglru_hip_colsum_scratch_bytes(rows, width), dy);
    check(rglru_hip_colsum(ptr(dy_c), ptr(scratch), ptr(db), rows, width, code_of(dy.scalar_type()), code_of(ot), stream_of(dy)),
          "rglru_hip_colsum");
    if (ot != bt) db = db.to(bt);
  }
  return {dw, db};
}

// src with the rows of inactive tokens zeroed, in a new tensor or in place.
Tensor masked_rows(const Tensor& src_in, const Tensor& active, bool in_place) {
  c10::DeviceGuard guard(src_in.device());
  Tensor src = src_in.contiguous();
  Tensor dst = in_place ? src : fresh_like(src);
  const int64_t D = src.size(-1);
  if (src.numel() > 0)
    check(rglru_hip_mask_rows(ptr(src), bptr(active), ptr(dst), src.numel() / D, D, code_of(src.scalar_type()), stream_of(src)),
          "rglru_hip_mask_rows");
  return dst;
}

// `active` (one byte per token): outputs of inactive tokens are zero, and so are the gradients that reach them.
struct Linear : torch::autograd::Function<Linear> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const MaybeTensor& bias, const MaybeTensor& active) {
    ctx->save_for_backward({x, weight, opt(active)});
    note_arguments(ctx, {true, true, bias.has_value()});
    pack(ctx, {type_or_none(opt(bias))});
    return values(x, weight, opt(bias), opt(active));
  }
  static Tensor values(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& active) {
    if (own_linear(x, weight, bias)) {
      c10::DeviceGuard guard(x.device());
      at::DimVector size(x.sizes());
      size.back() = weight.size(0);
      Tensor y = fresh(size, x.scalar_type(), x);
      linear_forward(x, weight, bias, Tensor(), Tensor(), active, ptr(y), nullptr);
      return y;
    }
    Tensor y = at::linear(x, weight, maybe(bias));
    return active.defined() ? masked_rows(y, active, true) : y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto s = ctx->get_saved_variables();
    Tensor dx, dw, db;
    {
      at::NoGradGuard no_grad;
      const Tensor &x = s[0], &weight = s[1];
      c10::DeviceGuard guard(x.device());
      Needs need(ctx);
      const int64_t bias_type = unpack(ctx)[0];
      if (own_linear(x, weight, Tensor(), Product::kGradient) && plain(grads[0]) && grads[0].scalar_type() == x.scalar_type() && (bias_type == kNone || bias_type == (int64_t)x.scalar_type())) {
        std::tie(dx, dw, db) = own_backward(x, weight, grads[0], s[2], need(0), need(1), need(2));
        return once({dx, dw, db, Tensor()});
      }
      Tensor dy = s[2].defined() ? masked_rows(grads[0], s[2], false) : grads[0];
      if (need(0)) dx = at::matmul(dy, weight.to(dy.scalar_type()));
      std::tie(dw, db) = linear_parameter_grads(x, weight.scalar_type(), dy, need(1), need(2) ? bias_type : kNone);
    }
    return once({dx, dw, db, Tensor()});
  }
  static std::tuple<Tensor, Tensor, Tensor> own_backward(const Tensor& x, const Tensor& weight, const Tensor& dy_in, const Tensor& active,
                                                         bool need_x, bool need_w, bool need_b) {
    const auto dtype = x.scalar_type();
    Tensor dy = aligned(dy_in), dx, dw, db;
    const int64_t K = x.size(-1), N = weight.size(0), rows = x.numel() / K;
    void* stream = stream_of(x);
    if (need_x) {
      dx = fresh_like(x);
      check(rglru_hip_linear(RGLRU_LINEAR_INPUT_GRAD, ptr(dy), nullptr, N, ptr(weight), nullptr, K, nullptr, nullptr, bptr(active), ptr(dx), nullptr,
                             K, nullptr, nullptr, rows, K, N, code_of(dtype), stream), "rglru_hip_linear");
    }
    if (need_w || need_b) {
      const WeightGrad wg(rows, N, K, 1, dtype);
      Parts scratch;
      scratch.add(wg.sets_bytes), scratch.add(wg.sums_bytes);
      scratch.allocate(x);
      dw = fresh({N, K}, dtype, x), db = fresh({N}, dtype, x);
      char *sets = scratch.raw(), *sums = scratch.raw();
      wg.run(ptr(dy), nullptr, N, ptr(x), bptr(active), ptr(dw), sets, sums, rows, dtype, stream);
      const rglru_sum jobs[] = {wg.weight_sum(sets, ptr(dw)), wg.bias_sum(sums, ptr(db))};
      check(rglru_hip_sums(jobs, 2, code_of(dtype), stream), "rglru_hip_sums");
      if (!need_w) dw = Tensor();
      if (!need_b) db = Tensor();
    }
    return {dx, dw, db};
  }
};

Tensor linear(const Tensor& x, const Tensor& weight, const MaybeTensor& bias_, const MaybeTensor& active_) {
  Tensor bias = opt(bias_);
  require_gpu("hip_linear", {&x, &weight, &bias});
  const Tensor mask = opt(active_);
  require_device_of("hip_linear", x, {&weight, &bias, &mask});
  code_of(x.scalar_type());
  MaybeTensor active;
  if (active_.has_value()) {
    TORCH_CHECK_VALUE(active_->numel() == x.numel() / x.size(-1) && active_->element_size() == 1, "active: one byte for each row of x");
    active = active_->contiguous();
  }
  if (!wants_grad({&x, &weight, &bias})) {
    at::NoGradGuard no_grad;
    return Linear::values(x, weight, bias, opt(active));
  }
  return Linear::apply(x, weight, maybe(bias), active);
}

// The [rows, 2 W] matrix whose column halves `a` and `b` ([..., W] each) are, or an undefined tensor if they are not
// laid out that way (same storage, b starts W elements behind a, rows 2 W elements apart).
Tensor stacked_halves(const Tensor& a, const Tensor& b) {
  if (!a.defined() || !b.defined() || a.sizes() != b.sizes() || a.scalar_type() != b.scalar_type() || a.dim() < 2 || a.numel() == 0)
    return Tensor();
  const int64_t W = a.size(-1);
  if (a.strides() != b.strides() || a.stride(-1) != 1 || b.storage_offset() != a.storage_offset() + W) return Tensor();
  if (!a.is_alias_of(b)) return Tensor();
  int64_t expect = 2 * W;  // every leading axis must continue the rows of the one before
  for (int64_t d = a.dim() - 2; d >= 0; --d) {
    if (a.size(d) != 1 && a.stride(d) != expect) return Tensor();
    expect *= a.size(d);
  }
  return a.as_strided({a.numel() / W, 2 * W}, {2 * W, 1}, a.storage_offset());
}

// Two Linear layers on one input (the block's two branches).  Their input gradients are one GEMM that accumulates into
// the other's result instead of two results and an addition.
struct LinearPair : torch::autograd::Function<LinearPair> {
  typedef std::tuple<Tensor, Tensor> Values;
  // `known`: the values, where the caller has them already
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w1, const MaybeTensor& b1, const Tensor& w2,
                               const MaybeTensor& b2, const Values* known) {
    ctx->save_for_backward({x, w1, w2});
    note_arguments(ctx, {true, true, b1.has_value(), true, b2.has_value()});
    pack(ctx, {type_or_none(opt(b1)), type_or_none(opt(b2))});
    ctx->set_materialize_grads(false);
    auto [u, v] = known != nullptr ? *known : values(x, w1, opt(b1), w2, opt(b2));
    return {u, v};
  }
  static bool own(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2, const Tensor& b2, Product use = Product::kInference) {
    return own_linear(x, w1, b1, use) && own_linear(x, w2, b2, use) && w1.sizes() == w2.sizes() && b1.defined() == b2.defined();
  }
  static std::tuple<Tensor, Tensor> values(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2, const Tensor& b2) {
    if (!own(x, w1, b1, w2, b2)) return {at::linear(x, w1, maybe(b1)), at::linear(x, w2, maybe(b2))};
    return own_values(x, w1, b1, w2, b2);
  }
  static std::tuple<Tensor, Tensor> own_values(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2, const Tensor& b2) {
    c10::DeviceGuard guard(x.device());
    at::DimVector size(x.sizes());
    size.back() = w1.size(0);
    Tensor u = fresh(size, x.scalar_type(), x), v = fresh(size, x.scalar_type(), x);
    linear_forward(x, w1, b1, w2, b2, Tensor(), ptr(u), ptr(v));
    return {u, v};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto s = ctx->get_saved_variables();
    auto m = unpack(ctx);
    const Tensor &x = s[0], &w1 = s[1], &w2 = s[2];
    Needs need(ctx);
    const bool need_x = need(0), need_w1 = need(1), need_b1 = need(2), need_w2 = need(3), need_b2 = need(4);
    Tensor dx, dw1, db1, dw2, db2;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(x.device());
      Tensor both = stacked_halves(grads[0], grads[1]);
      const auto dtype = x.scalar_type();
      auto usual = [&](int64_t t) { return t == kNone || t == (int64_t)dtype; };
      if (grads[0].defined() && grads[1].defined() && plain(grads[0]) && plain(grads[1]) && grads[0].scalar_type() == dtype && grads[1].scalar_type() == dtype &&
          own(x, w1, Tensor(), w2, Tensor(), Product::kGradient) && usual(m[0]) && usual(m[1])) {
        Tensor g0 = grads[0], g1 = grads[1];
        const int64_t N = w1.size(0), K = w1.size(1), rows = x.numel() / K;
        const int64_t ld = both.defined() ? 2 * N : N;
        if (!both.defined() || !is_aligned(g0)) g0 = aligned(g0), g1 = aligned(g1);
        void* stream = stream_of(x);
        const int code = code_of(dtype);
        if (need_x) {
          dx = fresh_like(x);
          check(rglru_hip_linear(RGLRU_LINEAR_INPUT_GRAD, ptr(g0), ptr(g1), ld, ptr(w1), ptr(w2), K, nullptr, nullptr, nullptr, ptr(dx), nullptr,
                                 K, nullptr, nullptr, rows, K, N, code, stream), "rglru_hip_linear");
        }
        if (need_w1 || need_w2 || need_b1 || need_b2) {
          const WeightGrad wg(rows, N, K, 2, dtype);
          Parts scratch;
          scratch.add(wg.sets_bytes), scratch.add(wg.sums_bytes);
          scratch.allocate(x);
          Tensor dw = fresh({2, N, K}, dtype, x), db = fresh({2, N}, dtype, x);      // the halves of one sum
          char *sets = scratch.raw(), *sums = scratch.raw();
          wg.run(ptr(g0), ptr(g1), ld, ptr(x), nullptr, ptr(dw), sets, sums, rows, dtype, stream);
          const rglru_sum jobs[] = {wg.weight_sum(sets, ptr(dw)), wg.bias_sum(sums, ptr(db))};
          check(rglru_hip_sums(jobs, 2, code, stream), "rglru_hip_sums");
          if (need_w1) dw1 = part(dw, 0, {N, K}, dtype);
          if (need_w2) dw2 = part(dw, N * K * x.element_size(), {N, K}, dtype);
          if (need_b1) db1 = part(db, 0, {N}, dtype);
          if (need_b2) db2 = part(db, N * x.element_size(), {N}, dtype);
        }
      } else if (both.defined() && w1.scalar_type() == w2.scalar_type() && w1.sizes() == w2.sizes() && need_w1 == need_w2 &&
          need_b1 == need_b2 && m[0] == m[1]) {
        // The halves of one matrix (the block's backward writes them so): one GEMM for dx against the stacked weights,
        // one for both weight gradients, one column sum.  At 16384 rows, 768 -> 2 x 1024: 49 against 65 us (dx), 60
        // against 83 us (dW), two launches instead of four (db).
        const int64_t n = w1.size(0);
        if (need_x) dx = at::mm(both, at::cat({w1, w2}).to(both.scalar_type())).view(x.sizes());
        Tensor dw, db;
        std::tie(dw, db) = linear_parameter_grads(x, w1.scalar_type(), both, need_w1, need_b1 ? m[0] : kNone);
        if (dw.defined()) dw1 = dw.narrow(0, 0, n), dw2 = dw.narrow(0, n, n);
        if (db.defined()) db1 = db.narrow(0, 0, n), db2 = db.narrow(0, n, n);
      } else {
        for (int i = 0; i < 2; ++i) {
          const Tensor& dy = grads[i];
          if (!need_x || !dy.defined()) continue;
          Tensor flat = dy.reshape({-1, dy.size(-1)});
          Tensor w = (i == 0 ? w1 : w2).to(dy.scalar_type());
          if (dx.defined()) dx.addmm_(flat, w);
          else dx = at::mm(flat, w);
        }
        if (dx.defined()) dx = dx.view(x.sizes());
        if (grads[0].defined()) std::tie(dw1, db1) = linear_parameter_grads(x, w1.scalar_type(), grads[0], need_w1, need_b1 ? m[0] : kNone);
        if (grads[1].defined()) std::tie(dw2, db2) = linear_parameter_grads(x, w2.scalar_type(), grads[1], need_w2, need_b2 ? m[1] : kNone);
      }
    }
    return once({dx, dw1, db1, dw2, db2, Tensor()});
  }
};

// The values alone, without a graph.
std::tuple<Tensor, Tensor> linear_pair_values(const Tensor& x, const Tensor& w1, const MaybeTensor& b1, const Tensor& w2, const MaybeTensor& b2) {
  const Tensor bias1 = opt(b1), bias2 = opt(b2);
  refuse_tangents("hip_linear_pair", std::initializer_list<Tensor>{x, w1, bias1, w2, bias2});
  require_device_of("hip_linear_pair", x, {&w1, &bias1, &w2, &bias2});
  at::NoGradGuard no_grad;
  return LinearPair::values(x, w1, opt(b1), w2, opt(b2));
}

std::tuple<Tensor, Tensor> linear_pair(const Tensor& x, const Tensor& w1, const MaybeTensor& b1_, const Tensor& w2, const MaybeTensor& b2_,
                                       const MaybeTensor& u, const MaybeTensor& v) {
  Tensor b1 = opt(b1_), b2 = opt(b2_);
  require_gpu("hip_linear_pair", {&x, &w1, &b1, &w2, &b2});
  require_device_of("hip_linear_pair", x, {&w1, &b1, &w2, &b2});
  code_of(x.scalar_type());
  TORCH_CHECK_VALUE(u.has_value() == v.has_value(), "hip_linear_pair expects both values or neither");
  const bool known = u.has_value();
  if (known)
    for (const auto& [y, w] : {std::tie(*u, w1), std::tie(*v, w2)})
      TORCH_CHECK_VALUE(!y.requires_grad() && y.numel() * x.size(-1) == x.numel() * w.size(0) && y.size(-1) == w.size(0) && y.scalar_type() == x.scalar_type(),
                        "hip_linear_pair: these are not the values of the two products");
  if (!wants_grad({&x, &w1, &b1, &w2, &b2})) return known ? std::make_tuple(*u, *v) : linear_pair_values(x, w1, b1_, w2, b2_);
  const LinearPair::Values values = known ? std::make_tuple(*u, *v) : LinearPair::Values();
  auto out = LinearPair::apply(x, w1, maybe(b1), w2, maybe(b2), known ? &values : nullptr);
  return {out[0], out[1]};
}

// ---- the whole block in training (griffin/griffin.py:459-528 without cache) ----------------------------------------

// One node for projections, convolution, RG-LRU, output gate and output projection, so that a step costs the host one pass
// of the engine, three allocations each way and the launches; the last sums of all parameter gradients are one launch.  bf16
// throughout, every row a document from its beginning or right-padded (rows, active).
struct BlockTrain : torch::autograd::Function<BlockTrain> {
  static constexpr at::ScalarType kType = at::kBFloat16;
  enum { X, WX, BX, WY, BY, CW, CB, WA, BA, WI, BI, LAM, WO, BO, kTensors };

  // what the forward keeps: x_conv, y, gated, then the parameter image with the workspace; u and v in front where it made them
  struct Saved {
    size_t tensor_bytes;
    char* at;
    Saved(const Tensor& buffer, int64_t M, int64_t W) : tensor_bytes(round_up(M * W * 2)), at(static_cast<char*>(buffer.data_ptr())) {}
    char* operator[](int i) const { return at + i * tensor_bytes; }
  };

  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& wx, const Tensor& bx, const Tensor& wy, const Tensor& by,
                        const Tensor& cw, const Tensor& cb, const Tensor& wa, const Tensor& ba, const Tensor& wi, const Tensor& bi,
                        const Tensor& lam, const Tensor& wo, const Tensor& bo, const Tensor& pos, const MaybeTensor& flags_,
                        const MaybeTensor& rows_, const MaybeTensor& active_, const MaybeTensor& u_, const MaybeTensor& v_, bool first_reset,
                        double c, int64_t packed) {
    if (packed == 0)
      return run(ctx, x, wx, bx, wy, by, cw, cb, wa, ba, wi, bi, lam, wo, bo, pos, opt(flags_), opt(rows_), opt(active_), opt(u_), opt(v_), first_reset, c,
                 Packed());
    // Right-padded rows that are documents from their beginning become ONE row of documents without the padding, so that every product
    // and scan runs on the tokens that count; rows_ starts with the number of them in each row, u_ is the first projection of all tokens, v_ the
    // second where it is there already.
    c10::DeviceGuard guard(x.device());
    const Packed p = {x.size(0), x.size(1), packed, *rows_, x, *u_, opt(v_)};
    Tensor tokens = fresh({1, packed, x.size(2)}, kType, x);
    Tensor positions = fresh({1, packed}, at::kLong, x), flags = fresh({1, packed}, at::kByte, x);
    Tensor live = run(ctx, tokens, wx, bx, wy, by, cw, cb, wa, ba, wi, bi, lam, wo, bo, positions, flags, Tensor(), Tensor(), Tensor(), Tensor(), false, c, p);
    return p.unpack(live);
  }

  struct Packed {
    int64_t B = 0, T = 0, rows = 0;                          // of the padded batch; rows: 0 where it was not packed
    Tensor counts, x, u, v;
    Tensor unpack(const Tensor& src) const {
      Tensor dst = fresh({B, T, src.size(-1)}, kType, src);
      check(rglru_hip_unpack_rows(static_cast<const int32_t*>(ptr(counts)), ptr(src), ptr(dst), src.size(-1) * 2, B, T, rows, stream_of(src)),
            "rglru_hip_unpack_rows");
      return dst;
    }
  };

  static Tensor run(AutogradContext* ctx, const Tensor& x, const Tensor& wx, const Tensor& bx, const Tensor& wy, const Tensor& by, const Tensor& cw,
                    const Tensor& cb, const Tensor& wa, const Tensor& ba, const Tensor& wi, const Tensor& bi, const Tensor& lam, const Tensor& wo,
                    const Tensor& bo, const Tensor& pos, Tensor flags, const Tensor& rows, const Tensor& active, const Tensor& u, const Tensor& v,
                    bool first_reset, double c, const Packed& packed) {
    c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), W = wx.size(0), K = cw.size(2), nb = wa.size(0), M = B * T;
    void* stream = stream_of(x);
    const size_t image_bytes = round_up(prep_bytes(W, nb, RGLRU_BF16));
    const size_t tensor_bytes = round_up(M * W * 2);
    const int own = u.defined() ? 3 : 5;
    const size_t ws_bytes = round_up(rglru_hip_workspace_bytes(B, T, W, nb));
    const bool own_forward = own_linear(x, wx, bx, Product::kTrainingForward);
    const bool stack = !own_linear(x, wx, bx, Product::kGradient);               // the weights stacked for the backward's GEMM of the BLAS library
    Tensor buffer = bytes(own * tensor_bytes + image_bytes + ws_bytes + (stack ? 2 * W * D * 2 : 0), x);
    Saved s(buffer, M, W);
    if (packed.rows) {
      check(rglru_hip_pack_rows(static_cast<const int32_t*>(ptr(packed.counts)), ptr(packed.x), ptr(x), D * 2, ptr(packed.u), s[3], W * 2,
                                static_cast<int64_t*>(pos.data_ptr()), static_cast<uint8_t*>(flags.data_ptr()), packed.B, packed.T, packed.rows, stream),
            "rglru_hip_pack_rows");
      if (packed.v.defined()) {
        check(rglru_hip_pack_rows(static_cast<const int32_t*>(ptr(packed.counts)), ptr(packed.v), s[4], W * 2, nullptr, nullptr, 0, nullptr, nullptr, packed.B,
                                  packed.T, packed.rows, stream), "rglru_hip_pack_rows");
      } else if (own_forward) {
        linear_forward(x, wy, by, Tensor(), Tensor(), Tensor(), s[4], nullptr);
      } else {
        Tensor out_v = part(buffer, 4 * tensor_bytes, {M, W}, kType);
        at::addmm_out(out_v, by, x.view({M, D}), wy.t());
      }
    } else if (!first_reset && !flags.defined()) {
      flags = block_flags(pos);
    }
    if (!u.defined() && !packed.rows) {
      if (own_forward) {
        linear_forward(x, wx, bx, wy, by, Tensor(), s[3], s[4]);
      } else {
        Tensor x2 = x.view({M, D});
        Tensor out_u = part(buffer, 3 * tensor_bytes, {M, W}, kType), out_v = part(buffer, 4 * tensor_bytes, {M, W}, kType);
        at::addmm_out(out_u, bx, x2, wx.t());
        at::addmm_out(out_v, by, x2, wy.t());
      }
    }
    void *up = u.defined() ? ptr(u) : s[3], *vp = v.defined() ? ptr(v) : s[4];
    char *image = s[own], *ws = image + image_bytes;
    const bool clears = kernel_path(B, T, W, nb, kType, true) != RGLRU_PATH_FAST_CHAIN;   // as in RGLRU
    if (clears) note_cleared(ctx, x);
    check(rglru_hip_prepare_block_fwd(ptr(wa), ptr(ba), ptr(wi), ptr(bi), ptr(lam), static_cast<float>(c), RGLRU_BF16, image, up, W, vp, W,
                                      nullptr, ptr(cw), ptr(cb), K, nullptr, flags_ptr(flags, first_reset), s[0], s[1], s[2], nullptr,
                                      nullptr, ws, ptr(wx), ptr(wy), ws + ws_bytes, stack ? W * D * 2 : 0, B, T, W, nb,
                                      RGLRU_BF16 | (clears ? RGLRU_BACKWARD_CLEAR : 0), stream),
          "rglru_hip_prepare_block_fwd");
    Tensor out;
    if (own_forward) {
      out = fresh_like(x);
      check(rglru_hip_linear(RGLRU_LINEAR_FORWARD, s[2], nullptr, W, ptr(wo), nullptr, W, ptr(bo), nullptr, bptr(active), ptr(out), nullptr, D,
                             nullptr, nullptr, M, D, W, RGLRU_BF16, stream), "rglru_hip_linear");
    } else {
      out = at::linear(part(buffer, 2 * tensor_bytes, {B, T, W}, kType), wo, bo);
      if (active.defined()) masked_rows(out, active, true);
    }
    ctx->save_for_backward({x, wx, wy, wo, cw, pos, flags, rows, active, u, v, buffer, packed.counts});
    pack(ctx, {first_reset, nb, stack, packed.B, packed.T, packed.rows});
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto saved = ctx->get_saved_variables();
    auto m = unpack(ctx);
    const Tensor &x = saved[0], &wx = saved[1], &wy = saved[2], &wo = saved[3], &cw = saved[4], &pos = saved[5], &flags = saved[6],
                 &rows = saved[7], &active = saved[8], &u = saved[9], &v = saved[10], &buffer = saved[11];
    const bool first_reset = m[0];
    const int64_t nb = m[1];
    const Packed packed = {m[3], m[4], m[5], saved[12], Tensor(), Tensor(), Tensor()};
    variable_list g(23);
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(x.device());
      const int64_t B = x.size(0), T = x.size(1), D = x.size(2), W = wx.size(0), K = cw.size(2), bw = W / nb, M = B * T;
      void* stream = stream_of(x);
      Saved s(buffer, M, W);
      void *up = u.defined() ? ptr(u) : s[3], *vp = v.defined() ? ptr(v) : s[4];
      char *image = s[u.defined() ? 3 : 5], *ws = image + round_up(prep_bytes(W, nb, RGLRU_BF16));
      Tensor dy = aligned(grads[0].to(kType));
      if (packed.rows) {
        Tensor live = fresh({1, packed.rows, D}, kType, x);
        check(rglru_hip_pack_rows(static_cast<const int32_t*>(ptr(packed.counts)), ptr(dy), ptr(live), D * 2, nullptr, nullptr, 0, nullptr, nullptr, packed.B,
                                  packed.T, packed.rows, stream), "rglru_hip_pack_rows");
        dy = live;
      }
      const bool own = !m[2];
      const bool own_weights = own || (contraction_chunks(M) == 1 && own_rows(M, 2 * W, D));       // the library's own weight gradients
      if (!own && active.defined()) dy = masked_rows(dy, active, false);

      // parameter gradients; those of the two input projections are the halves of one sum each
      Tensor dw_pair = fresh({2, W, D}, kType, x), db_pair = fresh({2, W}, kType, x);
      g[WX] = part(dw_pair, 0, {W, D}, kType), g[WY] = part(dw_pair, W * D * 2, {W, D}, kType);
      g[BX] = part(db_pair, 0, {W}, kType), g[BY] = part(db_pair, W * 2, {W}, kType);
      g[CW] = fresh({W, 1, K}, kType, x), g[CB] = fresh({W}, kType, x);
      take_gates(nb, bw, kType, x, g[WA], g[BA], g[WI], g[BI], g[LAM]);
      g[WO] = fresh({D, W}, kType, x), g[BO] = fresh({D}, kType, x);

      const WeightGrad go(M, D, W, 1, kType), gp(M, W, D, 2, kType);
      const size_t column_bytes_o = rglru_hip_colsum_scratch_bytes(M, D);
      Parts scratch;
      scratch.add(M * W * 2), scratch.add(2 * M * W * 2);
      scratch.add(rglru_hip_bwd_scratch_bytes(B, T, W, nb, RGLRU_BF16)), scratch.add(rglru_hip_conv_scratch_bytes(B, T, W, K));
      scratch.add(own_weights ? go.sets_bytes : 0), scratch.add(own_weights ? go.sums_bytes : column_bytes_o);
      scratch.add(own_weights ? gp.sets_bytes : 0), scratch.add(rglru_hip_block_sums_bytes(B, T, W, nb));
      scratch.allocate(x);
      char *dgated = scratch.raw(), *du = scratch.raw(), *gate_scratch = scratch.raw(), *conv_scratch = scratch.raw(), *sets_o = scratch.raw(),
           *sums_o = scratch.raw(), *sets_p = scratch.raw(), *sums_p = scratch.raw();
      char* dv = du + W * 2;                               // the halves of one [M, 2 W] matrix
      rglru_sum sums[3];
      Tensor held_o, held_p;                               // results of the BLAS library that the last launch reads

      // output projection
      if (own) {
        check(rglru_hip_linear(RGLRU_LINEAR_INPUT_GRAD, ptr(dy), nullptr, D, ptr(wo), nullptr, W, nullptr, nullptr, bptr(active), dgated, nullptr, W,
                               nullptr, nullptr, M, W, D, RGLRU_BF16, stream), "rglru_hip_linear");
      } else {
        Tensor dg = part(scratch.buffer, scratch.offsets[0], {M, W}, kType);
        at::mm_out(dg, dy.view({M, D}), wo);
      }
      if (own_weights) {
        go.run(ptr(dy), nullptr, D, s[2], own ? bptr(active) : nullptr, ptr(g[WO]), sets_o, sums_o, M, kType, stream);
        sums[0] = go.weight_sum(sets_o, ptr(g[WO])), sums[1] = go.bias_sum(sums_o, ptr(g[BO]));
      } else {
        Tensor dy2 = dy.view({M, D});
        held_o = contraction(dy2, part(buffer, 2 * s.tensor_bytes, {M, W}, kType));
        check(rglru_hip_colsum(ptr(dy), sums_o, nullptr, M, D, RGLRU_BF16, RGLRU_BF16, stream), "rglru_hip_colsum");
        sums[0] = {ptr(held_o), ptr(g[WO]), held_o.size(0), D * W, RGLRU_BF16};
        sums[1] = {sums_o, ptr(g[BO]), int64_t(column_bytes_o / (4 * D)), D, RGLRU_F32};
      }
      check(rglru_hip_block_bwd(dgated, s[1], up, vp, s[0], image, ptr(cw), iptr(pos), static_cast<const int32_t*>(ptr(rows)),
                                flags_ptr(flags, first_reset), ws, gate_scratch, conv_scratch, sums_p, du, dv, 2 * W,
                                take_cleared(ctx, x), B, T, W, nb, K, stream),
            "rglru_hip_block_bwd");
      // input projections
      const bool need_x = ctx->needs_input_grad(0);
      if (own) {
        if (need_x) {
          g[X] = fresh_like(x);
          check(rglru_hip_linear(RGLRU_LINEAR_INPUT_GRAD, du, dv, 2 * W, ptr(wx), ptr(wy), D, nullptr, nullptr, nullptr, ptr(g[X]), nullptr, D,
                                 nullptr, nullptr, M, D, W, RGLRU_BF16, stream), "rglru_hip_linear");
        }
      } else {
        Tensor both = part(scratch.buffer, scratch.offsets[1], {M, 2 * W}, kType);
        const size_t stacked = static_cast<size_t>(ws - s.at) + round_up(rglru_hip_workspace_bytes(B, T, W, nb));
        if (need_x) g[X] = at::mm(both, part(buffer, stacked, {2 * W, D}, kType)).view(x.sizes());
      }
      if (own_weights) {
        gp.run(du, dv, 2 * W, ptr(x), nullptr, ptr(dw_pair), sets_p, nullptr, M, kType, stream);
        sums[2] = gp.weight_sum(sets_p, ptr(dw_pair));
      } else {
        held_p = contraction(part(scratch.buffer, scratch.offsets[1], {M, 2 * W}, kType), x.view({M, D}));
        sums[2] = {ptr(held_p), ptr(dw_pair), held_p.size(0), 2 * W * D, RGLRU_BF16};
      }
      check(rglru_hip_block_finish(image, gate_scratch, conv_scratch, sums_p, ptr(g[WA]), ptr(g[WI]), ptr(g[BA]), ptr(g[BI]), ptr(g[LAM]),
                                   ptr(g[CW]), ptr(g[CB]), ptr(g[BX]), ptr(g[BY]), sums, 3, B, T, W, nb, K, stream), "rglru_hip_block_finish");
      if (packed.rows && need_x) g[X] = packed.unpack(g[X]);
      for (int i = 1; i < kTensors; ++i)
        if (!ctx->needs_input_grad(i)) g[i] = Tensor();
    }
    return once(std::move(g));
  }

  // a^T b over the rows, as the partial products [chunks, columns of a, columns of b] of the BLAS library (one chunk: the library's own kernel)
  static Tensor contraction(const Tensor& a, const Tensor& b) {
    const int64_t rows = a.size(0), chunks = contraction_chunks(rows), per = rows / chunks;
    return at::bmm(a.view({chunks, per, a.size(1)}).transpose(1, 2), b.view({chunks, per, b.size(1)}));
  }
};

// Whether the thirteen parameters p of a block (BlockTrain's tensors behind x) belong together and to inputs of model width D.
bool block_parameters(int64_t D, const std::vector<Tensor>& p) {
  typedef BlockTrain N;
  if (p.size() != N::kTensors - 1) return false;
  const Tensor &wa = p[N::WA - 1], &wi = p[N::WI - 1];
  if (!block_shapes(D, p[N::WX - 1], p[N::BX - 1], p[N::WY - 1], p[N::BY - 1], p[N::CW - 1], p[N::CB - 1], p[N::WO - 1], p[N::BO - 1])) return false;
  const int64_t W = p[N::WX - 1].size(0);
  if (wa.dim() != 3 || wa.size(1) != wa.size(2) || wa.size(0) * wa.size(1) != W || wi.sizes() != wa.sizes()) return false;
  for (int i : {N::BA, N::BI, N::LAM})
    if (p[i - 1].numel() != W) return false;
  return true;
}

// ... and whether the per-token operands have the shape of [B, T] tokens.
bool token_shapes(int64_t B, int64_t T, int64_t W, const Tensor& pos, const Tensor& flags, const Tensor& rows, const Tensor& active, const Tensor& u,
                  const Tensor& v) {
  auto tokens = [&](const Tensor& t) { return t.dim() == 2 && t.size(0) == B && t.size(1) == T; };
  auto width = [&](const Tensor& t) { return t.dim() == 3 && t.size(0) == B && t.size(1) == T && t.size(2) == W; };
  return (!pos.defined() || tokens(pos)) && (!flags.defined() || (tokens(flags) && flags.element_size() == 1 && flags.is_contiguous())) &&
         (!rows.defined() || (rows.numel() == 3 * B && rows.scalar_type() == at::kInt && rows.is_contiguous())) &&
         (!active.defined() || (tokens(active) && active.element_size() == 1)) && u.defined() == v.defined() &&
         (!u.defined() || (width(u) && width(v) && u.scalar_type() == v.scalar_type()));
}

// Nothing is returned where the node does not take the operands; the caller then goes layer by layer.
MaybeTensor block_train_node(const Tensor& x, const std::vector<Tensor>& p, const Tensor& pos, const MaybeTensor& flags, const MaybeTensor& rows,
                        const MaybeTensor& active, const MaybeTensor& u, const MaybeTensor& v, bool first_reset, double c, int64_t packed) {
  typedef BlockTrain N;
  const int64_t B = x.size(0), T = x.size(1), D = x.size(2);
  refuse_tangents("the recurrent block", p);
  refuse_tangents("the recurrent block", std::initializer_list<Tensor>{x, opt(u), opt(v)});
  if (!block_parameters(D, p) || !on_device_of(x, pos)) return std::nullopt;
  for (const Tensor& t : p)
    if (!on_device_of(x, t)) return std::nullopt;
  for (const MaybeTensor* t : {&flags, &rows, &active, &u, &v})
    if (t->has_value() && !on_device_of(x, **t)) return std::nullopt;
  for (const Tensor& t : p)
    if (t.scalar_type() != N::kType || !t.is_contiguous() || !is_aligned(t)) return std::nullopt;
  // p: the node's tensors behind x
  const Tensor &wx = p[N::WX - 1], &cw = p[N::CW - 1], &wa = p[N::WA - 1];
  const int64_t W = wx.size(0);
  // packed: the number of rows that the tokens that count are packed to; u may then be there alone
  if (packed > 0 && (!u.has_value() || !rows.has_value() || packed > B * T || rglru_hip_reproducible())) return std::nullopt;
  if (x.scalar_type() != N::kType || !vector_rows(x) || W % 8 ||
      !token_shapes(B, T, W, pos, opt(flags), opt(rows), opt(active), opt(u), packed > 0 && !v.has_value() ? opt(u) : opt(v)) ||
      (u.has_value() && u->scalar_type() != N::kType) || (B * T + 64) * 2 * W * 2 >= (int64_t(1) << 31) || B * T * W * 2 > (int64_t(1) << 30) || !rglru_hip_block_fwd_path(W, wa.size(0), cw.size(2), RGLRU_BF16))
    return std::nullopt;
  // the gated reverse scan in tiles adds the gradient of linear_y's bias up in the order of its tickets
  if (rglru_hip_reproducible() && kernel_path(B, T, W, wa.size(0), N::kType, true) != RGLRU_PATH_FAST_CHAIN) return std::nullopt;
  MaybeTensor live;
  if (active.has_value()) live = active->contiguous();
  Tensor positions = pos.to(at::kLong).contiguous();
  auto contiguous = [](const MaybeTensor& t) { return t.has_value() ? MaybeTensor(aligned(*t)) : t; };
  return BlockTrain::apply(x, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11], p[12], positions, flags, rows, live,
                           contiguous(u), contiguous(v), first_reset, c, packed);
}

MaybeTensor block_train(const Tensor& x, const std::vector<Tensor>& p, const Tensor& pos, const MaybeTensor& flags, const MaybeTensor& rows,
                        const MaybeTensor& active, const MaybeTensor& u, const MaybeTensor& v, bool first_reset, double c) {
  return block_train_node(x, p, pos, flags, rows, active, u, v, first_reset, c, 0);
}
MaybeTensor block_train_packed(const Tensor& x, const std::vector<Tensor>& p, const Tensor& pos, const Tensor& rows, const Tensor& u, const MaybeTensor& v,
                               int64_t packed, double c) {
  return packed <= 0 ? std::nullopt : block_train_node(x, p, pos, std::nullopt, rows, std::nullopt, u, v, false, c, packed);
}

// Right-padded batches are packed (BlockTrain::Packed) where products are long enough for the launches around it to pay, and a quarter of
// the tokens or more is padding.  Training step of the block, half of the tokens padding, us, not packed : packed (multiply-adds of a product of
// all tokens): 768 -> 1024 at 2.2e9 226 : 237, 3.1e9 243 : 237, 4.1e9 269 : 247, 6.8e9 374 : 296, 1.0e10 (64 rows) 507 : 359, 1.3e10 538 : 434; 512 ->
// 512 at 4.3e9 302 : 269.  With 30, 50, 60, 70 and 80 % of the tokens active: B8 T2048 768 -> 1024 537 : 307, 389, 449, 512, 547; B16 T2048 960 : 513,
// 656, 775, 898, 995; B6 T1000 2048 -> 2048 710 : 375, 493, 551, 616, 685.  Rows: multiples of 64, and of 512 from 8192 on.  A size
// that the BLAS library has not seen costs it 20 to 35 us once, a coarser grain up to 1 % of every step: 60 lengths, 1024 -> 2048, us a step the first time and
// later, 64 498 and 448, 512 476 and 452; 2560 -> 2560 838 and 822, 830 and 815.
bool block_may_pack(const Tensor& x, const Tensor& w) {
  return x.dim() == 3 && x.size(0) > 1 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 && double(x.numel()) * w.size(0) >= 3e9 && !rglru_hip_reproducible();
}
int64_t block_packed_rows(int64_t B, int64_t T, int64_t active_tokens) {
  const int64_t grain = active_tokens >= 8192 ? 512 : 64, rows = (std::max<int64_t>(active_tokens, 1) + grain - 1) / grain * grain;
  return 4 * rows <= 3 * B * T ? rows : 0;
}

// x w^T + b without a graph.
Tensor linear_values(const Tensor& x, const Tensor& w, const MaybeTensor& b) {
  const Tensor bias = opt(b);
  refuse_tangents("hip_linear", std::initializer_list<Tensor>{x, w, bias});
  require_device_of("hip_linear", x, {&w, &bias});
  at::NoGradGuard no_grad;
  return Linear::values(x, w, bias, Tensor());
}

// The input projections of a training batch that may be packed, queued before the mask's answer is there: both where they are one launch of the
// library, else the first alone, and the second follows on the tokens that turn out to count.  The first alone everywhere leaves the device idle
// until the host has woken up: steps, us, two processes each, alone : together, every token active (half of them in brackets): 768 -> 1024 at 3.2e9
// multiply-adds 218-234 : 197-222 (211-225 : 181-215), 4.1e9 250-254 : 232-241 (220-235 : 202-223), 5.5e9 271 : 266-269 (244 : 236-241), 7.1e9 346-349 :
// 319-321 (271 : 268-270); 1536 -> 2048 at 4.1e9 243-245 : 227-239 (227 : 212-226), 5.5e9 272 : 256-262 (234 : 221-233).  Past the library's line a BLAS product
// covers most of the wait (1.3e10, every token active: 489 to 500 with the first alone, 494 to 497 with both queued).
std::tuple<Tensor, MaybeTensor> block_projections(const Tensor& x, const Tensor& w1, const MaybeTensor& b1, const Tensor& w2, const MaybeTensor& b2) {
  const Tensor bias1 = opt(b1), bias2 = opt(b2);
  refuse_tangents("hip_linear_pair", std::initializer_list<Tensor>{x, w1, bias1, w2, bias2});
  require_device_of("hip_linear_pair", x, {&w1, &bias1, &w2, &bias2});
  at::NoGradGuard no_grad;
  if (!LinearPair::own(x, w1, bias1, w2, bias2, Product::kTrainingForward)) return {Linear::values(x, w1, bias1, Tensor()), std::nullopt};
  auto [u, v] = LinearPair::own_values(x, w1, bias1, w2, bias2);
  return {u, v};
}

// The whole block over sequences without gradients (griffin/griffin.py:459-528): projections, positions, convolution, RG-LRU
// and gate, output projection in three launches (four behind the BLAS library's products).  Every token active: positions follow prev_pos (or are segment_pos);
// right-padded: flags, rows, active and the projections u, v as the caller has them from TokenFacts.  Returns (output, final
// state, convolution state, last position); nothing where the kernels do not take the operands.
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> block_infer(
    const Tensor& x, const std::vector<Tensor>& p, const Tensor& image, const MaybeTensor& conv_state_, const MaybeTensor& rnn_state_,
    const MaybeTensor& prev_pos_, const MaybeTensor& segment_pos_, const MaybeTensor& flags_, const MaybeTensor& rows_, const MaybeTensor& active_,
    const MaybeTensor& u_, const MaybeTensor& v_, bool need_carry) {
  typedef BlockTrain N;
  const auto dtype = x.scalar_type();
  const int64_t B = x.size(0), T = x.size(1), D = x.size(2);
  refuse_tangents("the recurrent block", p);
  refuse_tangents("the recurrent block", std::initializer_list<Tensor>{x, opt(conv_state_), opt(rnn_state_), opt(u_), opt(v_)});
  if (!block_parameters(D, p) || !on_device_of(x, image)) return std::nullopt;
  for (const Tensor& t : p)
    if (!on_device_of(x, t)) return std::nullopt;
  for (const MaybeTensor* t : {&conv_state_, &rnn_state_, &prev_pos_, &segment_pos_, &flags_, &rows_, &active_, &u_, &v_})
    if (t->has_value() && !on_device_of(x, **t)) return std::nullopt;
  for (const Tensor& t : p)
    if (t.scalar_type() != dtype || !t.is_contiguous() || !is_aligned(t)) return std::nullopt;
  const Tensor &wx = p[N::WX - 1], &bx = p[N::BX - 1], &wy = p[N::WY - 1], &by = p[N::BY - 1], &cw = p[N::CW - 1], &cb = p[N::CB - 1],
               &wa = p[N::WA - 1], &wo = p[N::WO - 1], &bo = p[N::BO - 1];
  const int64_t W = wx.size(0), K = cw.size(2), nb = wa.size(0), M = B * T;
  if (!vector_rows(x) || W % 8 || !token_shapes(B, T, W, opt(segment_pos_), opt(flags_), opt(rows_), opt(active_), opt(u_), opt(v_)) ||
      (u_.has_value() && u_->scalar_type() != dtype) || !state_shapes(B, W, K, opt(conv_state_), opt(rnn_state_), opt(prev_pos_)) || !rglru_hip_block_fwd_path(W, nb, K, code_of(dtype)))
    return std::nullopt;
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(x.device());
  const int code = code_of(dtype);
  void* stream = stream_of(x);
  Tensor u = opt(u_), v = opt(v_), flags = opt(flags_), rows = opt(rows_), active = opt(active_), prev = opt(prev_pos_), seg = opt(segment_pos_);
  Tensor state = K == 1 ? Tensor() : as(opt(conv_state_), dtype), h0 = as(opt(rnn_state_), at::kFloat);
  if (prev.defined()) prev = prev.to(at::kLong).contiguous();
  if (seg.defined()) seg = seg.to(at::kLong).contiguous();
  const bool own = own_linear(x, wx, bx);
  Parts s;
  const size_t row_bytes = M * W * x.element_size();
  s.add(row_bytes), s.add(own && !u.defined() ? row_bytes : 0), s.add(own && !u.defined() ? row_bytes : 0);
  s.add(rglru_hip_workspace_bytes(B, T, W, nb)), s.add(M);
  s.allocate(x);
  char *gated = s.raw(), *up = s.raw(), *vp = s.raw(), *ws = s.raw();
  uint8_t* flag_bytes = reinterpret_cast<uint8_t*>(s.raw());
  if (u.defined()) {
    u = aligned(u), v = aligned(v);
  } else if (!own) {
    u = at::linear(x, wx, bx), v = at::linear(x, wy, by);
  }
  const bool projects = !u.defined() && !flags.defined();  // in one launch with the positions
  if (!u.defined() && !projects) linear_forward(x, wx, bx, wy, by, Tensor(), up, vp);
  if (u.defined()) up = static_cast<char*>(ptr(u)), vp = static_cast<char*>(ptr(v));
  Tensor h_last = fresh({B, W}, at::kFloat, x), new_conv = fresh({B, K - 1, W}, dtype, x), last;
  if (projects) {
    uint8_t* bytes_of_flags = prev.defined() || seg.defined() ? flag_bytes : nullptr;
    last = fresh({B}, at::kLong, x);
    check(rglru_hip_block_project(ptr(x), ptr(wx), ptr(wy), ptr(bx), ptr(by), up, vp, iptr(prev), iptr(seg), bytes_of_flags,
                                  static_cast<int64_t*>(last.data_ptr()), ws, B, T, D, W, nb, code, stream), "rglru_hip_block_project");
    check(rglru_hip_block_infer_projected(up, W, vp, W, ptr(state), ptr(cw), ptr(cb), K, code, ptr(image), fptr(h0), bytes_of_flags,
                                          gated, K > 1 ? ptr(new_conv) : nullptr, fptr(h_last), ws, B, T, W, nb, code, stream),
          "rglru_hip_block_infer_projected");
  } else if (!flags.defined()) {
    last = fresh({B}, at::kLong, x);
    check(rglru_hip_block_infer(up, W, vp, W, ptr(state), ptr(cw), ptr(cb), K, code, ptr(image), fptr(h0), iptr(prev), iptr(seg), flag_bytes, gated,
                                K > 1 ? ptr(new_conv) : nullptr, fptr(h_last), static_cast<int64_t*>(last.data_ptr()), ws, B, T, W, nb, code, stream),
          "rglru_hip_block_infer");
  } else {
    check(rglru_hip_block_fwd(up, W, vp, W, ptr(state), ptr(cw), ptr(cb), K, code, ptr(image), fptr(h0), bptr(flags), nullptr, nullptr, gated,
                              nullptr, fptr(h_last), ws, B, T, W, nb, code, stream), "rglru_hip_block_fwd");
    if (need_carry && K > 1)
      check(rglru_hip_conv_carry(up, W, ptr(state), static_cast<const int32_t*>(ptr(rows)), ptr(new_conv), B, T, W, K, code, stream),
            "rglru_hip_conv_carry");
  }
  Tensor out, live = active.defined() ? active.contiguous() : active;
  if (own) {
    out = fresh_like(x);
    check(rglru_hip_linear(RGLRU_LINEAR_FORWARD, gated, nullptr, W, ptr(wo), nullptr, W, ptr(bo), nullptr, bptr(live), ptr(out), nullptr, D, nullptr,
                           nullptr, M, D, W, code, stream), "rglru_hip_linear");
  } else {
    out = at::linear(part(s.buffer, 0, {B, T, W}, dtype), wo, bo);
    if (live.defined()) masked_rows(out, live, true);
  }
  return std::make_tuple(out, h_last, new_conv, last);
}

// ---- RMSNorm (griffin/griffin.py:68-80) ---------------------------------------------------------------------------

std::tuple<Tensor, Tensor, Tensor, Tensor> rmsnorm_forward(const Tensor& x_in, const Tensor& g, double eps, bool need_inv) {
  c10::DeviceGuard guard(x_in.device());
  Tensor x = x_in.contiguous();
  Tensor scale = operand(g, x.scalar_type());
  const int64_t D = x.size(-1), rows = x.numel() / D;
  Tensor y = fresh_like(x);
  Tensor inv = need_inv ? fresh({rows}, at::kFloat, x) : Tensor();
  if (rows > 0)
    check(rglru_hip_rmsnorm_fwd(ptr(x), ptr(scale), ptr(y), fptr(inv), rows, D, static_cast<float>(eps), code_of(x.scalar_type()),
                                code_of(scale.scalar_type()), stream_of(x)), "rglru_hip_rmsnorm_fwd");
  return {x, scale, y, inv};
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& g, double eps) {
    auto [x, scale, y, inv] = rmsnorm_forward(x_in, g, eps, true);
    ctx->save_for_backward({x, scale, inv});
    pack(ctx, {type_or_none(g)});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &scale = s[1], &inv = s[2];
    Tensor dx, dg;
    {
      at::NoGradGuard no_grad;
      c10::DeviceGuard guard(x.device());
      const int64_t D = x.size(-1), rows = x.numel() / D;
      Tensor dy = as(grads[0], x.scalar_type());
      const auto gt = scale.scalar_type();
      dx = fresh_like(x);
      if (ctx->needs_input_grad(1)) dg = fresh({D}, gt, x);
      if (rows > 0) {
        Tensor scratch = bytes(rglru_hip_rmsnorm_scratch_bytes(rows, D), x);
        check(rglru_hip_rmsnorm_bwd(ptr(x), ptr(scale), fptr(inv), ptr(dy), ptr(scratch), ptr(dx), ptr(dg), rows, D,
                                    code_of(x.scalar_type()), code_of(gt), code_of(gt), stream_of(x)), "rglru_hip_rmsnorm_bwd");
      } else if (dg.defined()) {
        dg.zero_();
      }
      if (dg.defined()) dg = dg.to(type_at(unpack(ctx), 0));
    }
    return once({dx, dg, Tensor()});
  }
};

Tensor rmsnorm(const Tensor& x, const Tensor& g, double eps) {
  require_gpu("hip_rmsnorm", {&x, &g});
  require_device_of("hip_rmsnorm", x, {&g});
  TORCH_CHECK_VALUE(g.dim() == 1 && x.dim() >= 1 && x.size(-1) == g.numel(), "hip_rmsnorm expects a scale of shape [",
                    x.dim() >= 1 ? x.size(-1) : 0, "], got ", g.sizes());
  code_of(x.scalar_type());
  if (wants_grad({&x, &g})) return RmsNorm::apply(x, g, eps);
  at::NoGradGuard no_grad;
  return std::get<2>(rmsnorm_forward(x, g, eps, false));
}

// RMSNorm.forward where the kernels take x.
py::object norm_forward(py::handle module, const Tensor& x) {
  if (!x.is_cuda() || !known(x.scalar_type()) || x.numel() == 0 || x.dim() < 1 || !((usable_devices.load(std::memory_order_relaxed) >> x.device().index()) & 1))
    return py::none();
  const Members norm(module.ptr());
  if (!at::GradMode::is_enabled()) norm.drop_leaves();
  Tensor g;
  if (!norm.parameter("g", g) || g.dim() != 1 || g.size(0) != x.size(-1) || !on_device_of(x, g)) return py::none();
  const bool bf16 = x.scalar_type() == at::kBFloat16;
  const int code = code_of(x.scalar_type());
  if (x.size(-1) > rglru_hip_rmsnorm_max_width(code, x.size(-1) % (bf16 ? 8 : 4) == 0)) return py::none();
  const auto eps = norm.number("eps");
  if (!eps) return py::none();
  if (g.requires_grad() && at::GradMode::is_enabled()) hold_leaves(py::reinterpret_borrow<py::dict>(norm.dict), {g});
  return py::cast(rmsnorm(x, g, *eps));
}

}  // namespace

PYBIND11_MODULE(_native, m) {
#define EXPORT(name) m.def(#name, torch::wrap_pybind_function(name))
  EXPORT(kernel_path);
  EXPORT(prepare);
  EXPORT(fingerprint);
  py::class_<Stamp>(m, "Stamp")
      .def(py::init<const std::vector<Tensor>&, const Tensor&, int64_t, double, at::ScalarType>())
      .def("matches", &Stamp::matches)
      // a copy of a module starts without what is kept for the original
      .def(py::pickle([](const Stamp&) { return py::tuple(); }, [](const py::tuple&) { return Stamp(); }));
  py::class_<Leaves>(m, "Leaves")
      .def(py::pickle([](const Leaves&) { return py::tuple(); }, [](const py::tuple&) { return Leaves(); }));
  m.def("hold_leaves", &hold_leaves);
  EXPORT(mark_usable);
  EXPORT(lru_decode);
  EXPORT(block_decode);
  EXPORT(norm_forward);
  EXPORT(rglru);
  EXPORT(rglru_step);
  EXPORT(rglru_steps);
  EXPORT(rglru_module_step);
  EXPORT(scan);
  EXPORT(pack_flags);
  py::class_<TokenFacts>(m, "TokenFacts")
      .def(py::init<const Tensor&, const MaybeTensor&, const MaybeTensor&>())
      .def("resolve", &TokenFacts::resolve)
      .def_readonly("positions", &TokenFacts::positions)
      .def_readonly("flags", &TokenFacts::flags)
      .def_readonly("conv_positions", &TokenFacts::conv_positions)
      .def_readonly("rows", &TokenFacts::rows)
      .def_readonly("last_position", &TokenFacts::last_position)
      .def_readonly("active_tokens", &TokenFacts::active_tokens);
  EXPORT(causal_conv);
  EXPORT(causal_conv_padded);
  EXPORT(gelu_gate);
  EXPORT(block_flags);
  EXPORT(block_forward);
  EXPORT(block_decode_step);
  EXPORT(block_step);
  EXPORT(own_projections_captured);
  EXPORT(sum_sets);
  EXPORT(stacked_halves);
  EXPORT(linear);
  EXPORT(linear_pair);
  EXPORT(linear_pair_values);
  EXPORT(linear_values);
  EXPORT(block_projections);
  EXPORT(block_may_pack);
  EXPORT(block_packed_rows);
  EXPORT(block_train);
  EXPORT(block_train_packed);
  EXPORT(block_infer);
  EXPORT(rmsnorm);
#undef EXPORT
}
