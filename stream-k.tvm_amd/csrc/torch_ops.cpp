// The operators' short way from the dispatcher to a launch: streamk::gemm_* for ordinary calls, in native code.
//
// An eager decode step of a small layer runs for a few microseconds on the device; through the operator's Python
// implementation alone a layer's call took 22.4 us (1 x 4096 x 4096, 4-bit weights; the kernel 4.0).  The
// implementations registered here check the operands, look the plan up, allocate C and launch; whatever is not the
// ordinary case -- a configuration or a plan of the caller's, a plan that is not known yet, a stream whose workspace is
// missing or too small, operands that have to be copied first or that the checks refuse -- goes, with its arguments as
// they are, to the Python implementation (streamk::<name>_general), which answers it or raises.  Kept here are plans, by
// shape, device and type, and the addresses of the workspaces that the Python layer owns, by device and stream; it tells
// of both and takes both back (sk_torch_*).  A call holds the tables' lock, shared, from the look-up until its kernels are
// enqueued; a workspace is taken back under the same lock, exclusively, before its memory goes to the allocator, which
// orders whatever uses it next on that stream behind them.
// (A call's host time now: 5.1 to 6.1 us through an operator, 9.8 through a layer, of which the launch is about 3; the Python
// implementation 16.3 to 16.9.)
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <map>
#include <mutex>
#include <shared_mutex>
#include <optional>
#include <string>
#include <tuple>

#include "streamk.h"

namespace {

using torch::jit::Stack;

// (M, N, K, dtype, layout, device)
typedef std::tuple<int64_t, int64_t, int64_t, int, int, int> PlanKey;
constexpr size_t MAX_PLANS = 4096;
std::shared_mutex g_mutex;
struct Buffer {
  void *ptr = nullptr;
  size_t bytes = 0;
};
std::map<PlanKey, sk_plan> g_plans;
std::map<std::pair<int, void *>, Buffer> g_workspaces;

// what a launch on the current stream takes beside the operands; the workspace is there as long as this is.  (Nothing but
// the launch happens while it lives: an allocation could run a caller's code, which may call an operator itself.)
struct Launch {
  std::shared_lock<std::shared_mutex> lock{g_mutex, std::defer_lock};
  sk_plan plan;
  Buffer ws;
  void *stream;
  bool find(int64_t M, int64_t N, int64_t K, int dtype, int layout) {
    const int device = (int)c10::hip::current_device();
    stream = (void *)c10::hip::getCurrentHIPStream().stream();
    lock.lock();
    const auto it = g_plans.find(PlanKey(M, N, K, dtype, layout, device));
    if (it == g_plans.end()) return false;
    plan = it->second;
    if (plan.workspace_bytes == 0) return true;
    const auto w = g_workspaces.find({device, stream});
    if (w == g_workspaces.end() || w->second.bytes < (size_t)plan.workspace_bytes) return false;
    ws = w->second;
    return true;
  }
};

bool is_matrix(const at::Tensor &t, at::ScalarType type) {
  return t.is_cuda() && t.scalar_type() == type && t.dim() == 2 && t.stride(1) == 1;
}
// rows that the kernels read in place: 16 bytes apart or in multiples of it, the first element 16-byte aligned
bool aligned_rows(const at::Tensor &A) {
  return A.size(0) > 0 && (A.size(0) == 1 || A.stride(0) * (int64_t)A.element_size() % 16 == 0) &&
         reinterpret_cast<uintptr_t>(A.data_ptr()) % 16 == 0;
}

// the epilogue operands: false if they are not what a launch takes as it is
bool epilogue(const c10::IValue &bias, const c10::IValue &activation, const at::Tensor &A, int64_t N, at::ScalarType type,
              sk_epilogue *epi, bool *used) {
  *epi = sk_epilogue{};
  const std::string &act = activation.toStringRef();
  if (act == "none") epi->activation = SK_ACT_NONE;
  else if (act == "relu") epi->activation = SK_ACT_RELU;
  else if (act == "gelu_tanh") epi->activation = SK_ACT_GELU_TANH;
  else if (act == "silu") epi->activation = SK_ACT_SILU;
  else return false;
  if (!bias.isNone()) {
    const at::Tensor &b = bias.toTensor();
    if (b.scalar_type() != type || b.dim() != 1 || b.size(0) != N || !b.is_contiguous() || b.device() != A.device()) return false;
    epi->bias = b.data_ptr();
  }
  *used = epi->bias != nullptr || epi->activation != SK_ACT_NONE;
  return true;
}

// C of a call: the caller's, or a new one.  Undefined where the caller's is not one a launch can write.
at::Tensor result(const at::Tensor *out, const at::Tensor &A, int64_t M, int64_t N, at::ScalarType type) {
  if (out == nullptr) return at::empty({M, N}, A.options().dtype(type));
  return is_matrix(*out, type) && out->size(0) == M && out->size(1) == N ? *out : at::Tensor();
}

// Each of these returns C, or an undefined tensor for a call that the general implementation has to answer.  a[]: the
// arguments behind the operands (and behind `out`).

// (layout, config, bias, activation)
at::Tensor gemm_16bit(const at::Tensor &A, const at::Tensor &B, const at::Tensor *out, const c10::IValue *a, at::ScalarType type, int dtype) {
  const std::string &layout = a[0].toStringRef();
  if (!a[1].toStringRef().empty() || (layout != "nt" && layout != "nn")) return {};
  if (!is_matrix(A, type) || !is_matrix(B, type) || !aligned_rows(A)) return {};
  const bool nt = layout == "nt";
  const int64_t M = A.size(0), K = A.size(1), N = B.size(nt ? 0 : 1);
  if (B.size(nt ? 1 : 0) != K) return {};
  sk_epilogue epi;
  bool used;
  if (!epilogue(a[2], a[3], A, N, type, &epi, &used)) return {};
  at::Tensor C = result(out, A, M, N, type);
  if (!C.defined()) return {};
  Launch l;
  if (!l.find(M, N, K, dtype, nt ? SK_LAYOUT_NT : SK_LAYOUT_NN)) return {};
  const int rc = (dtype == SK_F16 ? sk_gemm_f16_ex : sk_gemm_bf16_ex)(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0),
                                                                      B.stride(0), C.stride(0), &l.plan, l.ws.ptr, l.ws.bytes, l.stream,
                                                                      used ? &epi : nullptr);
  return rc == SK_OK ? C : at::Tensor();
}

// (layout, config)
at::Tensor gemm_f32(const at::Tensor &A, const at::Tensor &B, const at::Tensor *out, const c10::IValue *a) {
  const std::string &layout = a[0].toStringRef();
  if (!a[1].toStringRef().empty() || (layout != "nt" && layout != "nn")) return {};
  if (!is_matrix(A, at::kFloat) || !is_matrix(B, at::kFloat) || A.size(0) == 0) return {};
  const bool nt = layout == "nt";
  const int64_t M = A.size(0), K = A.size(1), N = B.size(nt ? 0 : 1);
  if (B.size(nt ? 1 : 0) != K) return {};
  at::Tensor C = result(out, A, M, N, at::kFloat);
  if (!C.defined()) return {};
  Launch l;
  if (!l.find(M, N, K, SK_F32, nt ? SK_LAYOUT_NT : SK_LAYOUT_NN)) return {};
  const int rc = sk_gemm_f32(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0), &l.plan, l.ws.ptr, l.ws.bytes, l.stream);
  return rc == SK_OK ? C : at::Tensor();
}

// (alpha, fmt, config, bias, activation); raw bytes, whose format only `fmt` tells, are left to the general implementation
at::Tensor gemm_f8(const at::Tensor &A, const at::Tensor &B, const at::Tensor *out, const c10::IValue *a) {
  const at::ScalarType type = A.scalar_type();
  if (type != at::kFloat8_e4m3fn && type != at::kFloat8_e5m2) return {};
  const std::string &fmt = a[1].toStringRef();
  if (!a[2].toStringRef().empty() || !(fmt.empty() || fmt == (type == at::kFloat8_e5m2 ? "e5m2" : "e4m3"))) return {};
  if (!is_matrix(A, type) || !is_matrix(B, type) || A.size(0) == 0) return {};
  const int64_t M = A.size(0), K = A.size(1), N = B.size(0);
  if (B.size(1) != K) return {};
  sk_epilogue epi;
  bool used;
  if (!epilogue(a[3], a[4], A, N, at::kHalf, &epi, &used)) return {};
  at::Tensor C = result(out, A, M, N, at::kHalf);
  if (!C.defined()) return {};
  Launch l;
  if (!l.find(M, N, K, type == at::kFloat8_e5m2 ? SK_F8E5M2 : SK_F8E4M3, SK_LAYOUT_NT)) return {};
  const int rc = sk_gemm_f8_ex(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0),
                               (float)a[0].toDouble(), &l.plan, l.ws.ptr, l.ws.bytes, l.stream, used ? &epi : nullptr);
  return rc == SK_OK ? C : at::Tensor();
}

// (config)
at::Tensor gemm_i8(const at::Tensor &A, const at::Tensor &B, const at::Tensor *out, const c10::IValue *a) {
  if (!a[0].toStringRef().empty() || !is_matrix(A, at::kChar) || !is_matrix(B, at::kChar) || A.size(0) == 0) return {};
  const int64_t M = A.size(0), K = A.size(1), N = B.size(0);
  if (B.size(1) != K) return {};
  at::Tensor C = result(out, A, M, N, at::kInt);
  if (!C.defined()) return {};
  Launch l;
  if (!l.find(M, N, K, SK_I8, SK_LAYOUT_NT)) return {};
  const int rc = sk_gemm_i8(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, A.stride(0), B.stride(0), C.stride(0), &l.plan, l.ws.ptr, l.ws.bytes, l.stream);
  return rc == SK_OK ? C : at::Tensor();
}

// operands A, Wq, scales, zeros; (zero, group, tiled, config, bias, activation).  One launch, row-major weights, as many rows as
// the Q4 tile kernels serve -- a shape that the general implementation answers with several launches never has a plan here
// under these types.
at::Tensor gemm_q4(const c10::IValue *operands, const at::Tensor *out, const c10::IValue *a) {
  const at::Tensor &A = operands[0].toTensor(), &Wq = operands[1].toTensor(), &scales = operands[2].toTensor();
  const int64_t zero = a[0].toInt(), group = a[1].toInt();
  if (a[2].toBool() || !a[3].toStringRef().empty() || group != 128 || zero < 0 || zero > 15) return {};
  if (!is_matrix(A, at::kHalf) || !aligned_rows(A) || !is_matrix(Wq, at::kByte) || !Wq.is_contiguous() ||
      !is_matrix(scales, at::kHalf) || !scales.is_contiguous())
    return {};
  const int64_t M = A.size(0), K = A.size(1), N = Wq.size(0);
  if (Wq.size(1) * 2 != K || scales.size(0) != N || scales.size(1) != K / group) return {};
  const bool zp = !operands[3].isNone();
  const void *zeros = nullptr;
  if (zp) {
    const at::Tensor &z = operands[3].toTensor();
    if (!is_matrix(z, at::kHalf) || !z.is_contiguous() || z.sizes() != scales.sizes()) return {};
    zeros = z.data_ptr();
  }
  if (M > 1024) return {};
  sk_epilogue epi;
  bool used;
  if (!epilogue(a[4], a[5], A, N, at::kHalf, &epi, &used)) return {};
  at::Tensor C = result(out, A, M, N, at::kHalf);
  if (!C.defined()) return {};
  Launch l;
  if (!l.find(M, N, K, zp ? SK_Q4_ZP : SK_Q4, SK_LAYOUT_NT)) return {};
  const int rc = sk_gemm_q4_ex(A.data_ptr(), Wq.data_ptr(), scales.data_ptr(), zeros, C.data_ptr(), M, N, K, A.stride(0), C.stride(0),
                               (int)group, zp ? 0 : (int)zero, &l.plan, l.ws.ptr, l.ws.bytes, l.stream, used ? &epi : nullptr);
  return rc == SK_OK ? C : at::Tensor();
}

enum Op { F16, BF16, F32, F8, I8, Q4 };

// boxed implementation of streamk::gemm_* (OUT: its _out twin): the arguments stay on the stack until the call is answered
template <Op OP, bool OUT>
void boxed(const c10::OperatorHandle &op, c10::DispatchKeySet, Stack *stack) {
  at::AutoDispatchBelowADInplaceOrView guard;   // (autograd is behind us, also for what is called from here)
  const size_t nargs = op.schema().arguments().size();
  const c10::IValue *args = stack->data() + (stack->size() - nargs);
  constexpr int operands = OP == Q4 ? 4 : 2;
  const c10::IValue *rest = args + operands + (OUT ? 1 : 0);
  at::Tensor C;
  const at::Tensor *out = OUT ? &args[operands].toTensor() : nullptr;
  if constexpr (OP == F16) C = gemm_16bit(args[0].toTensor(), args[1].toTensor(), out, rest, at::kHalf, SK_F16);
  if constexpr (OP == BF16) C = gemm_16bit(args[0].toTensor(), args[1].toTensor(), out, rest, at::kBFloat16, SK_BF16);
  if constexpr (OP == F32) C = gemm_f32(args[0].toTensor(), args[1].toTensor(), out, rest);
  if constexpr (OP == F8) C = gemm_f8(args[0].toTensor(), args[1].toTensor(), out, rest);
  if constexpr (OP == I8) C = gemm_i8(args[0].toTensor(), args[1].toTensor(), out, rest);
  if constexpr (OP == Q4) C = gemm_q4(args, out, rest);
  if (!C.defined()) {
    static const c10::OperatorHandle general =
        c10::Dispatcher::singleton().findSchemaOrThrow((op.schema().name() + "_general").c_str(), "");
    general.callBoxed(stack);
    return;
  }
  stack->erase(stack->end() - nargs, stack->end());
  if constexpr (!OUT) stack->push_back(c10::IValue(std::move(C)));
}

}  // namespace

TORCH_LIBRARY_IMPL(streamk, CUDA, m) {
#define IMPL(OP, NAME)                                                                         \
  m.impl(NAME, torch::CppFunction::makeFromBoxedFunction<&boxed<OP, false>>());                \
  m.impl(NAME "_out", torch::CppFunction::makeFromBoxedFunction<&boxed<OP, true>>());
  IMPL(F16, "gemm_f16")
  IMPL(BF16, "gemm_bf16")
  IMPL(F32, "gemm_f32")
  IMPL(F8, "gemm_f8")
  IMPL(I8, "gemm_i8")
  IMPL(Q4, "gemm_q4")
#undef IMPL
}

// plan of an operator call without a configuration of its own.  (Nothing is thrown through these C entries: a plan or a
// workspace that there is no memory to note is one that the general implementation serves.)
extern "C" __attribute__((visibility("default"))) void sk_torch_add_plan(const sk_plan *plan, int device) try {
  if (plan == nullptr) return;
  std::lock_guard<std::shared_mutex> lock(g_mutex);
  if (g_plans.size() < MAX_PLANS) g_plans[PlanKey(plan->M, plan->N, plan->K, plan->dtype, plan->layout, device)] = *plan;
} catch (...) {
}
extern "C" __attribute__((visibility("default"))) void sk_torch_clear_plans(void) try {
  std::lock_guard<std::shared_mutex> lock(g_mutex);
  g_plans.clear();
} catch (...) {
}
// the workspace that operator calls on a stream use, initialised (null: forget it); the caller keeps the memory alive
// until it has taken it back here
extern "C" __attribute__((visibility("default"))) void sk_torch_set_workspace(int device, void *stream, void *ptr, size_t bytes) try {
  std::lock_guard<std::shared_mutex> lock(g_mutex);
  if (ptr != nullptr) g_workspaces[{device, stream}] = Buffer{ptr, bytes};
  else g_workspaces.erase({device, stream});
} catch (...) {
}
