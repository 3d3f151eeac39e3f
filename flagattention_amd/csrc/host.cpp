// Host path of the operators for GPU tensors: argument checks, launch decisions, allocations and launches of one
// call in one native function, with native autograd nodes for the two operators that have gradients.
//
// Why it is native: the kernels of a short call take 10-40 us, and the same work done in Python through ctypes took
// longer than they do -- 38 us for a decode step, 20 us for a paged one, 195 us for a forward and backward over
// 512 tokens (of 42 us of kernels).
//
// The Python modules hold the reference form of the launch decisions made here (`flash.py`, `split_kv.py`, `paged.py`,
// `piecewise.py`).  It runs whenever a tile-config hook has been replaced, for tensors that are not on a GPU, where
// this extension is not built, and for every call this file does not take (it then answers NotImplemented, before any
// effect); arguments that are in error are among those, so that their messages have one source.  `decisions()` and the
// functions after it expose the numbers chosen here to the tests that compare them with the Python functions.  One
// decision is made only here: whether a dropout mask is kept for the backward (`keeps_mask`); the Python form always
// draws it again, with the same result.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <cmath>

#include "../../include/flagattn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Python callables bound once at import: abi.check (raises for an error code), the per-backward settings.
PyObject* g_check = nullptr;
PyObject* g_flash_settings = nullptr;
PyObject* g_piecewise_settings = nullptr;

// Thrown through code that does not hold the GIL; the Python error travels with it.
[[noreturn]] void throw_python_error() {
  python_error e;
  e.persist();
  throw std::move(e);
}

void check(int code, const char* what) {
  if (code == 0) return;
  pybind11::gil_scoped_acquire gil;
  PyObject* r = PyObject_CallFunction(g_check, "is", code, what);
  if (!r) throw_python_error();
  Py_DECREF(r);
  throw std::runtime_error(std::string(what) + ": the kernel library failed");
}

// ---------------------------------------------------------------------------------------------- decisions ----
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

constexpr int kSplitBlockM = 16, kSplitBlockN = 128;   // split_kv.SPLIT_BLOCK_M, SPLIT_BLOCK_N
constexpr int kDecodeMaxRows = 16;                     // split_kv.DECODE_MAX_ROWS

// split_kv.num_splits_heuristic
int num_splits_heuristic(int64_t B, int64_t H, int64_t M, int64_t N, int cus, int max_splits) {
  const int64_t base = B * H * cdiv(M, kSplitBlockM);
  if ((double)base >= 0.8 * cus) return 1;
  const int64_t units = cdiv(N, kSplitBlockN), limit = std::min<int64_t>({cus, units, max_splits});
  auto efficiency = [&](int64_t s) {
    const double waves = (double)(base * s) / cus;
    return waves / std::ceil(waves);
  };
  auto last_is_empty = [&](int64_t s) { const int64_t per = cdiv(units, s); return s > 1 && per * s - units >= per; };
  double best = 0.0;
  for (int64_t s = 1; s <= limit; ++s)
    if (!last_is_empty(s)) best = std::max(best, efficiency(s));
  for (int64_t s = 1; s <= limit; ++s)
    if (!last_is_empty(s) && efficiency(s) >= 0.85 * best) return (int)s;
  return 1;
}

// split_kv.choose_num_splits
int choose_num_splits(int64_t B, int64_t H, int64_t Hk, int64_t M, int64_t N, int cus) {
  const int64_t base = B * Hk * cdiv(H / Hk * M, 16), units = cdiv(N, kSplitBlockN);
  int64_t splits = std::min(cdiv(2 * (int64_t)cus, base), std::max<int64_t>(1, N / 512));
  if (N >= 1024) splits = std::max(splits, std::min(cdiv(cus, base), N / 128));
  splits = std::min<int64_t>({splits, 128, units});
  while (splits > 1 && cdiv(units, splits) * (splits - 1) >= units) --splits;
  return (int)splits;
}

// split_kv._split_size
int split_size(int64_t N, int splits) { return (int)(cdiv(cdiv(N, kSplitBlockN), splits) * kSplitBlockN); }

// flash.wide_key_splits
int wide_key_splits(int64_t B, int64_t H, int64_t M, int64_t N, int64_t D, int cus) {
  if (D != 128 || M < 256) return 1;
  const int64_t wgs = cdiv(M, 256) * H * B, pieces = std::min<int64_t>(cus / wgs, N / 1024);
  return pieces < 2 || 4 * pieces * wgs < 3 * (int64_t)cus ? 1 : (int)pieces;
}

// flash.forward_pieces (the reasons and figures stand there)
int forward_pieces(int64_t B, int64_t H, int64_t Hk, int64_t M, int64_t N, int64_t D, bool split, int cus) {
  if (M <= kDecodeMaxRows || (D == 128 && cdiv(M, 256) * H * B >= cus)) return 0;
  const int64_t wgs = cdiv(M, 128) * H * B, steps = cdiv(N, 64);
  const double alone = D == 128 ? 1.3 : D == 64 ? 0.93 : 0.75, shared = D == 128 ? 0.8 : D == 64 ? 0.45 : 0.36;
  const double decode = D == 128 ? 2.4e-3 : D == 64 ? 0.85e-3 : 0.3e-3;
  auto us = [&](int64_t pieces) {
    const int64_t per_unit = cdiv(wgs * pieces, cus);
    const double t = (double)cdiv(steps, pieces) * (alone + shared * (double)(per_unit - 1)) + 2.0 * (double)per_unit;
    return pieces == 1 ? t : t + 6.0 + (double)(B * H * M * pieces * D * 8) / 5e6;
  };
  int best = 0;
  double least = split ? 5.0 + (double)(B * Hk * cdiv(H / Hk * M, 16) * cdiv(N, 32)) * decode : us(1);
  for (int pieces = 2; pieces <= 32 && steps >= 3 * pieces && wgs * pieces <= 4 * (int64_t)cus; ++pieces)
    if (us(pieces) < 0.93 * least) { best = pieces; least = us(pieces); }
  return best;
}

// flash.dkdv_heads_per_slice
int dkdv_heads_per_slice(int64_t B, int64_t H, int group, int64_t N, int cus) {
  const int64_t blocks = cdiv(N, 128);
  for (int chunk = group; chunk > 0; --chunk)
    if (group % chunk == 0 && blocks * B * (H / chunk) >= 2 * (int64_t)cus) return chunk;
  return 1;
}

// flash._DKDV_128 and those after it: how a backward kernel's workgroups use a compute unit (what is measured stands there)
struct Pace { int slots; double alone, shared, around; };
constexpr Pace kDkdv128 = {1, 1.7, 2.1, 6.0}, kDkdv64 = {2, 1.05, 2.1, 5.0}, kDq = {2, 1.1, 1.6, 4.0}, kDqFromDs = {2, 1.15, 1.6, 4.0};

// flash._launch_us
double launch_us(const Pace& pace, int64_t tiles, double steps, bool causal, int pieces, double slice_bytes, int cus) {
  const double wgs = (double)tiles * pieces, per = steps / pieces, full = (double)cus * pace.slots;
  double t;
  if (causal) {
    t = std::max(per * pace.alone, tiles * steps / 2 / full * pace.shared);
  } else {
    const double rounds = std::floor(wgs / full), rest = wgs - rounds * full;
    t = per * (rounds * pace.shared + (rest <= 0 ? 0 : rest <= cus ? pace.alone : pace.shared));
  }
  t += pace.around * std::max(1.0, wgs / full);
  return pieces == 1 ? t : t + 3.0 + 2 * wgs * slice_bytes / 5e6;   // fp32 slices written and read back at 5 TB/s, and the launch that adds them
}
// flash._contraction_pieces
int contraction_pieces(const Pace& pace, int64_t tiles, int64_t steps, bool causal, double slice_bytes, int cus) {
  int best = 1;
  double least = launch_us(pace, tiles, (double)steps, causal, 1, slice_bytes, cus);
  for (int n = 2; n <= 16 && steps >= 8 * n; ++n) {
    const double t = launch_us(pace, tiles, (double)steps, causal, n, slice_bytes, cus);
    if (t < 0.95 * least) { best = n; least = t; }
  }
  return best;
}

// flash.gradient_pieces: of dK and dV, of dQ
struct GradientPieces { int kv, q; };
GradientPieces gradient_pieces(int64_t B, int64_t H, int64_t M, int64_t N, int64_t D, bool causal, int chunk, bool ds_kept, int cus) {
  return {chunk > 1 ? 1 : contraction_pieces(D == 128 ? kDkdv128 : kDkdv64, cdiv(N, 128) * B * H, cdiv(M, 64), causal, 2 * 4.0 * 128 * D, cus),
          contraction_pieces(ds_kept ? kDqFromDs : kDq, cdiv(M, 128) * B * H, cdiv(N, 64), causal, 4.0 * 128 * D, cus)};
}

// flash.ds_heads_per_launch
int64_t ds_heads_per_launch(int64_t B, int64_t H, int group, int64_t M, int64_t N, int64_t D, int64_t limit_mib, int grids) {
  if (D < 128 || M * N < 1024 * 1024 || limit_mib <= 0) return 0;
  const int64_t per_head = (int64_t)grids * fa_bwd_ds_workspace_mib(1, 1, (int)M, (int)N);
  const int64_t fit = limit_mib / per_head;
  return fit >= B * H ? B * H : fit / group * group;
}

// flash.even_heads
int64_t even_heads(int64_t fit, int64_t H, int group) {
  const int64_t launches = cdiv(H, std::min(fit, H));
  return cdiv(cdiv(H, launches), group) * group;
}

// paged.choose_launch: workgroups of the balanced launch, 0 = one workgroup per (sequence, kv head) pair
int balanced_workgroups(int64_t seqs, int64_t Hkv, int64_t group, int64_t D, int64_t max_context, int cus) {
  const int wgs = cus * (D <= 128 ? 2 : 1);
  return seqs * Hkv * cdiv(group, 16) >= 8 * (int64_t)wgs && max_context <= 2048 ? 0 : wgs;
}

// ------------------------------------------------------------------------------------------------ tensors ----
int dtype_code(const Tensor& t) { return t.scalar_type() == at::kHalf ? FA_F16 : FA_BF16; }

// _abi.is_kernel_ready
bool is_kernel_ready(const Tensor& t) {
  const auto sizes = t.sizes(), strides = t.strides();
  const int64_t last = t.dim() - 1;
  if (strides[last] != 1 || ((uintptr_t)t.const_data_ptr() & 15)) return false;
  for (int64_t i = 0; i < last; ++i)
    if (sizes[i] > 1 && strides[i] % 8) return false;
  return true;
}
Tensor kernel_ready(const Tensor& t) { return is_kernel_ready(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

fa_view4 view4(const Tensor& t) {
  const auto n = t.sizes(), s = t.strides();
  // the stride of a dimension of extent 1 is never used; torch leaves arbitrary values there
  return fa_view4{const_cast<void*>(t.const_data_ptr()), n[0] > 1 ? s[0] : 0, n[1] > 1 ? s[1] : 0, n[2] > 1 ? s[2] : 0};
}
// heads [h0, h1) of batch entry b
fa_view4 slice4(const Tensor& t, int64_t b, int64_t h0) {
  fa_view4 v = view4(t);
  v.ptr = (char*)v.ptr + (b * v.stride_b + h0 * v.stride_h) * (int64_t)t.element_size();
  return v;
}

Tensor empty(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}
// torch.empty_like(t) where the kernels can write that layout, otherwise contiguous
Tensor empty_result(const Tensor& t) {
  if (t.is_contiguous()) return empty(t.sizes(), t.scalar_type(), t);
  Tensor o = at::empty_like(t);
  return is_kernel_ready(o) ? o : empty(t.sizes(), t.scalar_type(), t);
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
float* f32(const Tensor& t) { return (float*)const_cast<void*>(t.const_data_ptr()); }

bool is_operand(const Tensor& t, const Tensor& first) {
  return t.is_cuda() && t.dim() == 4 && t.layout() == at::kStrided && t.device() == first.device() &&
         t.scalar_type() == first.scalar_type();
}
// The operators' kernels are launched past the dispatcher.  Where something listens there -- a tracer, a functorch
// transform, a dispatch mode, a tensor subclass, forward-mode tangents -- the Python form takes the call, and does with it
// what torch does with a Python autograd function: records it or refuses it.
bool plain_call(std::initializer_list<const Tensor*> ts) {
  using c10::impl::tls_is_dispatch_key_included;
  if (tls_is_dispatch_key_included(c10::DispatchKey::Tracer) ||
      tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || c10::impl::TorchDispatchModeTLS::any_modes_set())
    return false;
  for (const Tensor* t : ts)
    if (t->unsafeGetTensorImpl()->key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                                          c10::DispatchKey::FuncTorchGradWrapper})) ||
        t->_fw_grad(0).defined())
      return false;
  return true;
}
bool type_ok(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool fits_int(std::initializer_list<int64_t> xs) {
  for (int64_t x : xs)
    if (x <= 0 || x > 0x7fffffff) return false;
  return true;
}

// memory that a slower way does without: an undefined tensor when the allocator has none left
Tensor scratch(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  try {
    return empty(shape, type, like);
  } catch (const c10::OutOfMemoryError&) {
    return Tensor();
  }
}

// dS of `heads` heads, or an undefined tensor when the allocator has no memory left (the caller then recomputes)
Tensor ds_workspace(const Tensor& like, int64_t B, int64_t H, int64_t M, int64_t N, int grids) {
  const int mib = fa_bwd_ds_workspace_mib((int)B, (int)H, (int)M, (int)N);
  if (mib <= 0) check(mib ? mib : FA_ERR_BAD_ARGUMENT, "fa_bwd_ds_workspace_mib");
  return scratch({(int64_t)grids * ((int64_t)mib << 20)}, at::kByte, like);
}

// The settings a backward reads when it runs: calls the (replaceable) tile hook, returns the dS workspace limit.
int64_t backward_settings(PyObject* callable, int64_t B, int64_t H, int64_t M, int64_t N, int64_t D, bool causal) {
  pybind11::gil_scoped_acquire gil;
  PyObject* r = PyObject_CallFunction(callable, "LLLLLO", (long long)B, (long long)H, (long long)M, (long long)N,
                                      (long long)D, causal ? Py_True : Py_False);
  if (!r) throw_python_error();
  const int64_t limit = PyLong_AsLongLong(r);
  Py_DECREF(r);
  if (limit == -1 && PyErr_Occurred()) throw_python_error();
  return limit;
}

// ------------------------------------------------------------------------------------------ flash attention ----
struct FlashCall {
  bool causal, want_total;
  double scale, dropout_p;
  uint64_t seed, offset;
};

// pieces > 0: the split kernel over that many pieces of the key axis and the merge; tiles > 0: the 128-row kernel, the
// keys of every row block dealt to that many workgroups, and the merge; otherwise the dense kernel
struct FlashPlan { int pieces, tiles; };

// false: the combination is an error (dropout on a split shape)
bool plan_flash(FlashPlan& plan, int64_t B, int64_t H, int64_t Hk, int64_t M, int64_t N, int64_t D, bool dropout,
                double scale, int64_t row_bytes, int cus) {
  const int splits = num_splits_heuristic(B, H, M, N, cus, 128);
  plan.pieces = plan.tiles = 0;
  if (splits > 1 && dropout) return false;
  if (splits > 1) plan.tiles = forward_pieces(B, H, Hk, M, N, D, true, cus);
  if (plan.tiles > 0) return true;
  if (splits > 1 || (M <= kDecodeMaxRows && N >= 1024 && !dropout)) {
    plan.pieces = choose_num_splits(B, H, Hk, M, N, cus);
  } else if (!dropout && scale > 0 && row_bytes < (1 << 24)) {
    const int pieces = wide_key_splits(B, H, M, N, D, cus);
    if (pieces > 1) plan.pieces = pieces;
  }
  if (!dropout && plan.pieces == 0) plan.tiles = forward_pieces(B, H, Hk, M, N, D, false, cus);
  return true;
}

// The mask goes to the backward as bits where they take at most as much memory as q, k, v and o do, which are kept
// too: N / 8 bytes per query row against 8 D (equal heads).  Beyond that the backward draws it again.
bool keeps_mask(int64_t N, int64_t D) { return N <= 64 * D; }

// o, L and (if asked for) the column sums; with dropout, the mask for a backward if `keep` is given
variable_list flash_forward(const Tensor& q, const Tensor& k, const Tensor& v, const FlashCall& c, const FlashPlan& plan,
                            Tensor* keep = nullptr) {
  const int B = (int)q.size(0), H = (int)q.size(1), M = (int)q.size(2), D = (int)q.size(3);
  const int Hk = (int)k.size(1), N = (int)k.size(2), type = dtype_code(q);
  void* stream = stream_of(q);
  const fa_view4 vq = view4(q), vk = view4(k), vv = view4(v);
  Tensor o, L;
  if (plan.pieces > 0) {
    const int S = plan.pieces;
    Tensor part_lse = empty({B, H, S, M}, at::kFloat, q), part_o = empty({B, H, S, M, D}, at::kHalf, q);
    check(fa_splitkv_fwd(type, &vq, &vk, &vv, part_o.mutable_data_ptr(), f32(part_lse), B, H, Hk, M, N, D, c.causal,
                         (float)c.scale, S, split_size(N, S), stream), "fa_splitkv_fwd");
    if (S == 1) {   // nothing to merge: the single piece is the result (a cast at most)
      o = part_o.squeeze(2).to(q.scalar_type());
      L = part_lse.squeeze(2);
    } else {
      L = empty({B, H, M}, at::kFloat, q);
      o = empty_result(q);
      const fa_view4 vo = view4(o);
      check(fa_splitkv_combine(type, part_o.const_data_ptr(), f32(part_lse), &vo, f32(L), B, H, M, D, S, stream),
            "fa_splitkv_combine");
    }
  } else {
    o = empty_result(q);
    L = empty({B, H, M}, at::kFloat, q);
    const fa_view4 vo = view4(o);
    const Tensor ws = plan.tiles > 0 ? scratch({(int64_t)B * H * plan.tiles * M * (D + 1)}, at::kFloat, q) : Tensor();
    if (ws.defined()) {
      check(fa_fwd_pieces(type, &vq, &vk, &vv, &vo, f32(L), ws.mutable_data_ptr(), ws.numel() * 4, B, H, Hk, M, N, D, c.causal,
                          (float)c.scale, plan.tiles, stream), "fa_fwd_pieces");
    } else if (keep && c.dropout_p > 0 && keeps_mask(N, D) &&
               (*keep = scratch({(int64_t)B * H * fa_dropout_keep_words(M, N)}, at::kInt, q)).defined()) {
      check(fa_fwd_keep(type, &vq, &vk, &vv, &vo, f32(L), (uint32_t*)keep->mutable_data_ptr(), B, H, Hk, M, N, D, c.causal,
                        (float)c.scale, (float)c.dropout_p, c.seed, c.offset, stream), "fa_fwd_keep");
    } else {
      check(fa_fwd(type, &vq, &vk, &vv, &vo, f32(L), B, H, Hk, M, N, D, c.causal, (float)c.scale, (float)c.dropout_p,
                   c.seed, c.offset, 0, stream), "fa_fwd");
    }
  }
  variable_list out = {o, L};
  if (c.want_total) {
    Tensor tot = empty({B, H, N}, at::kFloat, q);
    check(fa_total_attn(type, &vq, &vk, f32(L), f32(tot), B, H, Hk, M, N, D, c.causal, (float)c.scale, stream),
          "fa_total_attn");
    out.push_back(tot);
  }
  return out;
}

variable_list flash_backward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& L,
                             const Tensor& keep, const Tensor& grad, const FlashCall& c, int64_t limit_mib) {
  const int B = (int)q.size(0), H = (int)q.size(1), M = (int)q.size(2), D = (int)q.size(3);
  const int Hk = (int)k.size(1), N = (int)k.size(2), group = H / Hk, type = dtype_code(q), cus = fa_num_cus();
  const Tensor g = kernel_ready(grad);
  void* stream = stream_of(q);
  const float scale = (float)c.scale, p = (float)c.dropout_p;
  Tensor delta = empty(L.sizes(), at::kFloat, q);
  const fa_view4 vo = view4(o), vg = view4(g);
  check(fa_bwd_delta(type, &vo, &vg, f32(delta), B, H, M, D, stream), "fa_bwd_delta");

  // dS kept (heads > 0), for all heads in one launch pair or for `hn` heads of one batch entry at a time; or recomputed,
  // where it is not worth keeping for this shape or there is no memory for it
  const int64_t heads = ds_heads_per_launch(B, H, group, M, N, D, limit_mib, 1);
  int bn = B, hn = H;   // batch entries and heads per launch
  Tensor ds;
  if (heads >= (int64_t)B * H) ds = ds_workspace(q, B, H, M, N, 1);
  else if (heads > 0) ds = ds_workspace(q, bn = 1, hn = (int)even_heads(heads, H, group), M, N, 1);
  if (!ds.defined()) { bn = B; hn = H; }

  // Slices of dK / dV: one per `chunk` query heads (the kernels that sum query heads are built without dropout) and
  // piece of the query axis; of dQ: one per piece of the key axis.  More than one per result: fp32, added at the end.
  int chunk = c.dropout_p > 0 ? 1 : dkdv_heads_per_slice(bn, hn, group, N, cus);
  auto [kv_pieces, q_pieces] = gradient_pieces(B, H, M, N, D, c.causal, chunk, ds.defined(), cus);
  int kv_slices = group / chunk * kv_pieces;   // per kv head
  Tensor dk = empty({B, Hk, N, D}, k.scalar_type(), q), dv = empty({B, Hk, N, D}, k.scalar_type(), q);
  Tensor dq = empty({B, H, M, D}, q.scalar_type(), q), dk_s = dk, dv_s = dv, dq_s = dq;
  int kv_type = type, q_type = type;
  if (kv_slices > 1) {
    dk_s = scratch({B, (int64_t)Hk * kv_slices, N, D}, at::kFloat, q);
    if (dk_s.defined()) dv_s = scratch({B, (int64_t)Hk * kv_slices, N, D}, at::kFloat, q);
    if (!dk_s.defined() || !dv_s.defined()) {   // no memory: whole sums, by as few slices as there are kernels for
      TORCH_CHECK_WITH(OutOfMemoryError, chunk == group || c.dropout_p == 0, "flash_attention backward: no memory for the slices of dK and dV");
      chunk = group;
      kv_pieces = kv_slices = 1;
      dk_s = dk;
      dv_s = dv;
    } else {
      kv_type |= FA_PIECES(kv_pieces);
    }
  }
  if (q_pieces > 1) {
    dq_s = scratch({B, (int64_t)H * q_pieces, M, D}, at::kFloat, q);
    if (dq_s.defined()) q_type |= FA_PIECES(q_pieces);
    else { q_pieces = 1; dq_s = dq; }
  }
  const uint32_t* bits = keep.defined() ? (const uint32_t*)keep.const_data_ptr() : nullptr;
  const int64_t head_bits = bits ? fa_dropout_keep_words(M, N) : 0;

  for (int b = 0; b < B; b += bn)
    for (int h0 = 0; h0 < H; h0 += hn) {
      const int n = std::min(H, h0 + hn) - h0, kn = n / group, k0 = h0 / group;   // whole groups of query heads
      const fa_view4 vq = slice4(q, b, h0), vk = slice4(k, b, k0), vv = slice4(v, b, k0), vg = slice4(g, b, h0),
                     vdk = slice4(dk_s, b, (int64_t)k0 * kv_slices), vdv = slice4(dv_s, b, (int64_t)k0 * kv_slices),
                     vdq = slice4(dq_s, b, (int64_t)h0 * q_pieces);
      const int64_t row = ((int64_t)b * H + h0) * M;
      const float *l = f32(L) + row, *d = f32(delta) + row;
      const uint32_t* w = bits ? bits + ((int64_t)b * H + h0) * head_bits : nullptr;
      // the dropout counter of a launch starts where its heads start in the (B, H, M, N) score tensor
      const uint64_t offset = c.offset + (uint64_t)row * (uint64_t)N;
      if (bits)
        check(fa_bwd_dkdv_keep(kv_type, &vq, &vk, &vv, &vg, l, d, &vdk, &vdv, ds.defined() ? ds.mutable_data_ptr() : nullptr,
                               ds.defined() ? ds.numel() : 0, w, bn, n, kn, M, N, D, c.causal, scale, p, stream), "fa_bwd_dkdv_keep");
      else if (ds.defined())
        check(fa_bwd_dkdv_ds(kv_type, &vq, &vk, &vv, &vg, l, d, &vdk, &vdv, chunk, ds.mutable_data_ptr(), ds.numel(), bn, n,
                             kn, M, N, D, c.causal, scale, p, c.seed, offset, stream), "fa_bwd_dkdv_ds");
      else
        check(fa_bwd_dkdv(kv_type, &vq, &vk, &vv, &vg, l, d, &vdk, &vdv, chunk, bn, n, kn, M, N, D, c.causal, scale, p,
                          c.seed, offset, stream), "fa_bwd_dkdv");
      if (ds.defined())
        check(fa_bwd_dq_from_ds(q_type, &vk, ds.const_data_ptr(), ds.numel(), &vdq, bn, n, kn, M, N, D, c.causal, scale,
                                stream), "fa_bwd_dq_from_ds");
      else if (bits)
        check(fa_bwd_dq_keep(q_type, &vq, &vk, &vv, &vg, l, d, &vdq, w, bn, n, kn, M, N, D, c.causal, scale, p, stream),
              "fa_bwd_dq_keep");
      else
        check(fa_bwd_dq(q_type, &vq, &vk, &vv, &vg, l, d, &vdq, bn, n, kn, M, N, D, c.causal, scale, p, c.seed, offset,
                        stream), "fa_bwd_dq");
    }

  const float* slices[3];
  void* out[3];
  int64_t outer[3], inner[3];
  int32_t count[3];
  int sums = 0;
  auto add_up = [&](const Tensor& s, const Tensor& r, int n) {
    slices[sums] = f32(s);
    out[sums] = r.mutable_data_ptr();
    outer[sums] = r.size(0) * r.size(1);
    inner[sums] = r.size(2) * r.size(3);
    count[sums++] = n;
  };
  if (kv_slices > 1) { add_up(dk_s, dk, kv_slices); add_up(dv_s, dv, kv_slices); }
  if (q_pieces > 1) add_up(dq_s, dq, q_pieces);
  if (sums) check(fa_sum_slices(type, slices, out, outer, count, inner, sums, stream), "fa_sum_slices");
  return {dq, dk, dv};
}

template <class Call>
struct Held : torch::CustomClassHolder {   // a call's parameters as one saved value of the autograd context
  explicit Held(const Call& c) : call(c) {}
  Call call;
};
template <class Call>
void hold(AutogradContext* ctx, const Call& c) {
  ctx->set_materialize_grads(false);   // no zeroes for the outputs whose gradients are ignored
  ctx->saved_data["call"] = c10::IValue::make_capsule(c10::make_intrusive<Held<Call>>(c));
}
// the gradient of the output o: zero where nothing flows into it
Tensor gradient_of(const Tensor& o, const Tensor& grad) { return grad.defined() ? grad : at::zeros_like(o); }
template <class Call>
const Call& held(AutogradContext* ctx) {
  return static_cast<Held<Call>*>(ctx->saved_data["call"].toCapsule().get())->call;
}

struct FlashNode : torch::autograd::Function<FlashNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q0, const Tensor& k0, const Tensor& v0,
                               const FlashCall& c, const FlashPlan& plan) {
    const Tensor q = kernel_ready(q0), k = kernel_ready(k0), v = kernel_ready(v0);
    Tensor keep;
    variable_list out = flash_forward(q, k, v, c, plan, &keep);
    ctx->save_for_backward({q, k, v, out[0], out[1], keep});
    hold(ctx, c);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const FlashCall& c = held<FlashCall>(ctx);
    const Tensor &q = saved[0], &k = saved[1];
    const c10::DeviceGuard guard(q.device());
    const int64_t limit = backward_settings(g_flash_settings, q.size(0), q.size(1), q.size(2), k.size(2), q.size(3), c.causal);
    variable_list r = flash_backward(q, k, saved[2], saved[3], saved[4], saved[5],
                                     gradient_of(saved[3], grads[0]), c, limit);
    return {r[0], r[1], r[2], Tensor(), Tensor()};
  }
};

bool needs_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

PyObject* not_taken() { Py_RETURN_NOTIMPLEMENTED; }

// Tensors and parameters.  A subclass of either gets its own type back from the Python form's torch.empty_like.
bool plain_tensors(PyObject* const* a, int n) {
  for (int i = 0; i < n; ++i)
    if (!THPVariable_CheckExact(a[i])) return false;
  return true;
}

// flash(q, k, v, causal, sm_scale or None, dropout_p, return_log_normalizer, return_total_attention, return_seed_offset)
PyObject* flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 9, "flash: nine arguments");
  if (!plain_tensors(a, 3)) return not_taken();
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  FlashCall c = {};
  const int causal = PyObject_IsTrue(a[3]), want_lse = PyObject_IsTrue(a[6]), want_total = PyObject_IsTrue(a[7]),
            want_seed = PyObject_IsTrue(a[8]);
  if (causal < 0 || want_lse < 0 || want_total < 0 || want_seed < 0) throw python_error();
  if (!plain_call({&q, &k, &v}) || !is_operand(q, q) || !is_operand(k, q) || !is_operand(v, q) || !type_ok(q)) return not_taken();
  const int64_t B = q.size(0), H = q.size(1), M = q.size(2), D = q.size(3), Hk = k.size(1), N = k.size(2);
  if (!fits_int({B, H, M, N, Hk}) || k.size(0) != B || v.sizes() != k.sizes() || k.size(3) != D || H % Hk ||
      !(D == 16 || D == 32 || D == 64 || D == 128))
    return not_taken();
  c.causal = causal;
  c.want_total = want_total;
  c.scale = a[4] == Py_None ? 1.0 / std::sqrt((double)D) : PyFloat_AsDouble(a[4]);
  c.dropout_p = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) { PyErr_Clear(); return not_taken(); }
  if (!(c.dropout_p >= 0.0 && c.dropout_p < 1.0)) return not_taken();
  const bool dropout = c.dropout_p > 0;

  variable_list out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(q.device());
    FlashPlan plan;
    // (a copy made for the kernels has unit-stride rows, so only a tensor used as it is can have distant rows)
    const int64_t row_bytes = 2 * std::max(is_kernel_ready(k) ? k.stride(2) : D, is_kernel_ready(v) ? v.stride(2) : D);
    const bool fine = plan_flash(plan, B, H, Hk, M, N, D, dropout, c.scale, row_bytes, fa_num_cus());
    if (fine) {
      if (dropout) {   // one Philox counter value per score element, from the device's default generator
        at::Generator gen = at::globalContext().defaultGenerator(q.device());
        std::lock_guard<std::mutex> lock(gen.mutex());
        c.seed = gen.current_seed();
        c.offset = gen.get_offset();
        gen.set_offset(c.offset + (uint64_t)((B * H * M * N + 3) / 4 * 4));
      }
      if (needs_grad({&q, &k, &v})) out = FlashNode::apply(q, k, v, c, plan);
      else out = flash_forward(kernel_ready(q), kernel_ready(k), kernel_ready(v), c, plan);
    }
  }
  if (out.empty()) return not_taken();
  if (!(want_lse || want_total || want_seed)) return THPVariable_Wrap(out[0]);
  PyObject* r = PyTuple_New(5);
  if (!r) throw python_error();
  auto none = [] { Py_INCREF(Py_None); return Py_None; };
  const bool seeded = dropout && want_seed;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out[0]));
  PyTuple_SET_ITEM(r, 1, want_lse ? THPVariable_Wrap(out[1]) : none());
  PyTuple_SET_ITEM(r, 2, want_total ? THPVariable_Wrap(out[2]) : none());
  PyTuple_SET_ITEM(r, 3, seeded ? PyLong_FromLongLong((long long)c.seed) : none());
  PyTuple_SET_ITEM(r, 4, seeded ? PyLong_FromLongLong((long long)c.offset) : none());
  return r;
  END_HANDLE_TH_ERRORS
}

// -------------------------------------------------------------------------------------- piecewise attention ----
struct PiecewiseCall {
  bool causal;
  int w;
  double scale;
};

struct PiecewiseNode : torch::autograd::Function<PiecewiseNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q1, const Tensor& k1, const Tensor& q2, const Tensor& k2,
                        const Tensor& v, const PiecewiseCall& c) {
    const Tensor ins[5] = {kernel_ready(q1), kernel_ready(k1), kernel_ready(q2), kernel_ready(k2), kernel_ready(v)};
    Tensor L;
    Tensor o = run(ins, c, L);
    ctx->save_for_backward({ins[0], ins[1], ins[2], ins[3], ins[4], o, L});
    hold(ctx, c);
    return o;
  }
  static Tensor run(const Tensor* t, const PiecewiseCall& c, Tensor& L) {
    const int B = (int)t[0].size(0), H = (int)t[0].size(1), M = (int)t[0].size(2), D = (int)t[0].size(3), N = (int)t[1].size(2);
    Tensor o = empty_result(t[0]);
    L = empty({B, H, M}, at::kFloat, t[0]);
    const fa_view4 a = view4(t[0]), b = view4(t[1]), x = view4(t[2]), y = view4(t[3]), v = view4(t[4]), vo = view4(o);
    check(pw_fwd(dtype_code(o), &a, &b, &x, &y, &v, &vo, f32(L), B, H, M, N, D, c.w, c.causal, (float)c.scale,
                 stream_of(o)), "pw_fwd");
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const PiecewiseCall& c = held<PiecewiseCall>(ctx);
    const Tensor &q1 = t[0], &k1 = t[1], &q2 = t[2], &k2 = t[3], &v = t[4], &o = t[5], &L = t[6];
    const int B = (int)q1.size(0), H = (int)q1.size(1), M = (int)q1.size(2), D = (int)q1.size(3), N = (int)k1.size(2);
    const c10::DeviceGuard guard(q1.device());
    const int64_t limit = backward_settings(g_piecewise_settings, B, H, M, N, D, c.causal);
    const Tensor g = kernel_ready(gradient_of(o, grads[0]));
    const int type = dtype_code(q1);
    const float scale = (float)c.scale;
    void* stream = stream_of(q1);
    Tensor delta = empty(L.sizes(), at::kFloat, q1);
    const fa_view4 vo = view4(o), vg = view4(g);
    check(fa_bwd_delta(type, &vo, &vg, f32(delta), B, H, M, D, stream), "fa_bwd_delta");
    Tensor dq1 = empty(q1.sizes(), q1.scalar_type(), q1), dq2 = empty(q2.sizes(), q1.scalar_type(), q1);
    Tensor dk1 = empty(k1.sizes(), q1.scalar_type(), q1), dk2 = empty(k2.sizes(), q1.scalar_type(), q1);
    Tensor dv = empty(v.sizes(), q1.scalar_type(), q1);
    // dS handed from the dK/dV kernel to the dQ kernels, one chunk grid per regime, when it pays
    int64_t heads = ds_heads_per_launch(B, H, 1, M, N, D, limit, 2);
    Tensor ds;
    int64_t nb = B, step = H;   // batch entries and heads per launch
    if (heads >= (int64_t)B * H) ds = ds_workspace(q1, B, H, M, N, 2);
    else if (heads > 0) ds = ds_workspace(q1, nb = 1, step = even_heads(heads, H, 1), M, N, 2);
    if (!ds.defined()) { nb = B; step = H; }
    for (int64_t b = 0; b < B; b += nb)
      for (int64_t h0 = 0; h0 < H; h0 += step) {
        const int n = (int)(std::min<int64_t>(H, h0 + step) - h0);
        auto at_slice = [&](const Tensor& x) { return slice4(x, b, h0); };
        const fa_view4 a = at_slice(q1), bk = at_slice(k1), x = at_slice(q2), y = at_slice(k2), vv = at_slice(v),
                       gg = at_slice(g), a1 = at_slice(dq1), b1 = at_slice(dk1), a2 = at_slice(dq2), b2 = at_slice(dk2),
                       v1 = at_slice(dv);
        const float *l = f32(L) + (b * H + h0) * M, *d = f32(delta) + (b * H + h0) * M;
        if (ds.defined()) {
          check(pw_bwd_dkdv_ds(type, &a, &bk, &x, &y, &vv, &gg, l, d, &b1, &b2, &v1, ds.mutable_data_ptr(), ds.numel(),
                               (int)nb, n, M, N, D, c.w, c.causal, scale, stream), "pw_bwd_dkdv_ds");
          check(pw_bwd_dq_from_ds(type, &bk, &y, ds.const_data_ptr(), ds.numel(), &a1, &a2, (int)nb, n, M, N, D, c.w,
                                  c.causal, scale, stream), "pw_bwd_dq_from_ds");
        } else {
          check(pw_bwd_dkdv(type, &a, &bk, &x, &y, &vv, &gg, l, d, &b1, &b2, &v1, (int)nb, n, M, N, D, c.w, c.causal,
                            scale, stream), "pw_bwd_dkdv");
          check(pw_bwd_dq(type, &a, &bk, &x, &y, &vv, &gg, l, d, &a1, &a2, (int)nb, n, M, N, D, c.w, c.causal, scale,
                          stream), "pw_bwd_dq");
        }
      }
    return {dq1, dk1, dq2, dk2, dv, Tensor()};
  }
};

// piecewise(q1, k1, q2, k2, v, dist_threshold, causal, sm_scale or None)
PyObject* piecewise(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 8, "piecewise: eight arguments");
  if (!plain_tensors(a, 5)) return not_taken();
  const Tensor &q1 = THPVariable_Unpack(a[0]), &k1 = THPVariable_Unpack(a[1]), &q2 = THPVariable_Unpack(a[2]),
               &k2 = THPVariable_Unpack(a[3]), &v = THPVariable_Unpack(a[4]);
  if (!plain_call({&q1, &k1, &q2, &k2, &v})) return not_taken();
  for (const Tensor* t : {&q1, &k1, &q2, &k2, &v})
    if (!is_operand(*t, q1)) return not_taken();
  const int64_t D = q1.size(3);
  if (!type_ok(q1) || !fits_int({q1.size(0), q1.size(1), q1.size(2), k1.size(2)}) || q2.sizes() != q1.sizes() ||
      k2.sizes() != k1.sizes() || v.sizes() != k1.sizes() || k1.size(0) != q1.size(0) || k1.size(1) != q1.size(1) ||
      k1.size(3) != D || !(D == 16 || D == 32 || D == 64 || D == 128))
    return not_taken();
  const int causal = PyObject_IsTrue(a[6]);
  if (causal < 0) throw python_error();
  if (!PyLong_Check(a[5])) return not_taken();
  int overflow = 0;
  const long long w = PyLong_AsLongLongAndOverflow(a[5], &overflow);
  if (overflow || w < INT32_MIN || w > INT32_MAX) return not_taken();
  PiecewiseCall c = {causal != 0, (int)w, a[7] == Py_None ? 1.0 / std::sqrt((double)D) : PyFloat_AsDouble(a[7])};
  if (PyErr_Occurred()) { PyErr_Clear(); return not_taken(); }
  Tensor o;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(q1.device());
    if (needs_grad({&q1, &k1, &q2, &k2, &v})) {
      o = PiecewiseNode::apply(q1, k1, q2, k2, v, c);
    } else {
      const Tensor ins[5] = {kernel_ready(q1), kernel_ready(k1), kernel_ready(q2), kernel_ready(k2), kernel_ready(v)};
      Tensor L;
      o = PiecewiseNode::run(ins, c, L);
    }
  }
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------ paged attention ----
bool row_ready(const Tensor& t) {   // a (num_seqs, heads, D) tensor the kernels read or write as it is
  return t.stride(2) == 1 && !((uintptr_t)t.const_data_ptr() & 15) && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0;
}

// paged(query, key_cache, value_cache, context_lens, block_tables, attn_scale, max_context_len), the launch chosen here
PyObject* paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 7, "paged: seven arguments");
  if (!plain_tensors(a, 5)) return not_taken();
  const Tensor &q = THPVariable_Unpack(a[0]), &kc = THPVariable_Unpack(a[1]), &vc = THPVariable_Unpack(a[2]),
               &lens = THPVariable_Unpack(a[3]), &bt = THPVariable_Unpack(a[4]);
  if (!plain_call({&q, &kc, &vc, &lens, &bt})) return not_taken();
  if (!q.is_cuda() || q.dim() != 3 || q.layout() != at::kStrided || !is_operand(kc, kc) || !is_operand(vc, kc) ||
      kc.device() != q.device() || kc.scalar_type() != q.scalar_type() || !type_ok(q))
    return not_taken();
  const int64_t seqs = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = kc.size(1), block = kc.size(2);
  if (!fits_int({seqs, Hq, Hkv, block}) || kc.size(3) != D || vc.sizes() != kc.sizes() || vc.strides() != kc.strides() ||
      kc.stride(3) != 1 || Hq % Hkv || !(D == 16 || D == 32 || D == 64 || D == 128 || D == 256 || D == 512) || !row_ready(q))
    return not_taken();
  if (lens.scalar_type() != at::kInt || lens.device() != q.device() || lens.dim() != 1 || lens.size(0) != seqs || !lens.is_contiguous() ||
      bt.device() != q.device() || bt.dim() != 2 || bt.size(0) != seqs || bt.stride(1) != 1 ||
      !(bt.scalar_type() == at::kInt || bt.scalar_type() == at::kLong))
    return not_taken();
  const double scale = PyFloat_AsDouble(a[5]);
  const long long longest = PyLong_Check(a[6]) ? PyLong_AsLongLong(a[6]) : -1;
  if (PyErr_Occurred()) { PyErr_Clear(); return not_taken(); }
  if (longest < 0) return not_taken();
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(q.device());
    out = q.is_contiguous() ? empty(q.sizes(), q.scalar_type(), q) : at::empty_like(q);   // the caller's layout, when the kernels can write it
    if (!row_ready(out)) out = empty(q.sizes(), q.scalar_type(), q);
    const int type = dtype_code(q), wgs = balanced_workgroups(seqs, Hkv, Hq / Hkv, D, longest, fa_num_cus());
    void* stream = stream_of(q);
    if (wgs > 0) {
      const int bytes = paged_attn_balanced_workspace(wgs, (int)D);
      Tensor ws = empty({bytes / 4}, at::kFloat, q);
      check(paged_attn_balanced(type, out.mutable_data_ptr(), out.stride(0), out.stride(1), q.const_data_ptr(), q.stride(0), q.stride(1),
                                kc.const_data_ptr(), vc.const_data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2),
                                (const int32_t*)lens.const_data_ptr(), bt.const_data_ptr(), bt.scalar_type() == at::kLong,
                                bt.stride(0), (float)scale, (int)seqs, (int)Hq, (int)Hkv, (int)D, (int)block,
                                ws.mutable_data_ptr(), (int64_t)bytes / 4 * 4, wgs, stream), "paged_attn_balanced");
    } else {
      check(paged_attn(type, out.mutable_data_ptr(), out.stride(0), out.stride(1), q.const_data_ptr(), q.stride(0), q.stride(1),
                       kc.const_data_ptr(), vc.const_data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2),
                       (const int32_t*)lens.const_data_ptr(), bt.const_data_ptr(), bt.scalar_type() == at::kLong,
                       bt.stride(0), (float)scale, (int)seqs, (int)Hq, (int)Hkv, (int)D, (int)block, 0, 1, nullptr,
                       nullptr, nullptr, stream), "paged_attn");
    }
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------- module ----
// decisions(B, H, Hk, M, N, D, num_cus, ds_limit_mib) -> every launch decision for that shape, for the test that
// holds them against the Python functions
PyObject* decisions(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  long long B, H, Hk, M, N, D, cus, limit;
  if (!PyArg_ParseTuple(args, "LLLLLLLL", &B, &H, &Hk, &M, &N, &D, &cus, &limit)) return nullptr;
  const int c = (int)cus, splits = num_splits_heuristic(B, H, M, N, c, 128), chosen = choose_num_splits(B, H, Hk, M, N, c);
  return Py_BuildValue("{s:i,s:i,s:i,s:i,s:i,s:L,s:L,s:i}", "num_splits_heuristic", splits, "choose_num_splits", chosen,
                       "split_size", split_size(N, chosen), "wide_key_splits", wide_key_splits(B, H, M, N, D, c),
                       "dkdv_heads_per_slice", dkdv_heads_per_slice(B, H, (int)(H / Hk), N, c), "ds_heads_per_launch",
                       (long long)ds_heads_per_launch(B, H, (int)(H / Hk), M, N, D, limit, 1), "ds_heads_per_launch_piecewise",
                       (long long)ds_heads_per_launch(B, H, 1, M, N, D, limit, 2), "balanced_workgroups",
                       balanced_workgroups(B, Hk, H / Hk, D, N, c));
  END_HANDLE_TH_ERRORS
}

// forward_pieces(B, H, Hk, M, N, D, split, num_cus), for the same test
PyObject* pieces_of_forward(PyObject*, PyObject* args) {
  long long B, H, Hk, M, N, D, cus;
  int split;
  if (!PyArg_ParseTuple(args, "LLLLLLpL", &B, &H, &Hk, &M, &N, &D, &split, &cus)) return nullptr;
  return PyLong_FromLong(forward_pieces(B, H, Hk, M, N, D, split, (int)cus));
}

// gradient_pieces(B, H, M, N, D, causal, chunk, ds_kept, num_cus) -> (dK/dV, dQ)
PyObject* pieces_of_gradients(PyObject*, PyObject* args) {
  long long B, H, M, N, D, cus;
  int causal, chunk, ds_kept;
  if (!PyArg_ParseTuple(args, "LLLLLpipL", &B, &H, &M, &N, &D, &causal, &chunk, &ds_kept, &cus)) return nullptr;
  const GradientPieces p = gradient_pieces(B, H, M, N, D, causal, chunk, ds_kept, (int)cus);
  return Py_BuildValue("(ii)", p.kv, p.q);
}

// keeps_mask(N, D)
PyObject* mask_is_kept(PyObject*, PyObject* args) {
  long long N, D;
  if (!PyArg_ParseTuple(args, "LL", &N, &D)) return nullptr;
  return PyBool_FromLong(keeps_mask(N, D));
}

// bind(abi.check, flash settings, piecewise settings)
PyObject* bind(PyObject*, PyObject* args) {
  if (!PyArg_ParseTuple(args, "OOO", &g_check, &g_flash_settings, &g_piecewise_settings)) return nullptr;
  for (PyObject* o : {g_check, g_flash_settings, g_piecewise_settings}) Py_INCREF(o);   // for the life of the process
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"flash", (PyCFunction)(void*)flash, METH_FASTCALL, nullptr},
    {"piecewise", (PyCFunction)(void*)piecewise, METH_FASTCALL, nullptr},
    {"paged", (PyCFunction)(void*)paged, METH_FASTCALL, nullptr},
    {"decisions", decisions, METH_VARARGS, nullptr},
    {"forward_pieces", pieces_of_forward, METH_VARARGS, nullptr},
    {"gradient_pieces", pieces_of_gradients, METH_VARARGS, nullptr},
    {"keeps_mask", mask_is_kept, METH_VARARGS, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  if (fa_version() != FA_ABI_VERSION)   // the two are built apart
    return PyErr_Format(PyExc_ImportError, "_host.so was built for revision %d of the C interface, the kernel library is revision %d",
                        FA_ABI_VERSION, fa_version());
  return PyModule_Create(&kModule);
}
