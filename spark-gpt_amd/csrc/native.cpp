// Torch-facing wrappers of the libsparkfp8 entry points that a training or
// evaluation step calls, as a CPython extension (imported by ops.py).
//
// Each wrapper checks its operands, allocates its outputs and workspaces with
// torch's caching allocator and launches on torch's current stream, as the
// Python wrappers of ops.py do for the remaining entry points: a refused
// argument raises ValueError, a refused call RuntimeError, before anything is
// launched.  A step of the block makes nine of these calls; through ctypes
// each took 11 to 39 us of host time (argument checks, 2 to 7 allocations, 10
// to 17 converted arguments), more than the kernels of a small batch run.
// The GIL is released around the launches, which may block on a full queue.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/pybind.h>

#include <string>
#include <tuple>
#include <vector>

#include "../../include/sparkfp8.h"

namespace py = pybind11;
using at::Tensor;
using c10::ScalarType;
using OptTensor = std::optional<Tensor>;

namespace {

constexpr auto kE4M3 = ScalarType::Float8_e4m3fn;
constexpr auto kE5M2 = ScalarType::Float8_e5m2;
constexpr auto kBF16 = ScalarType::BFloat16;
constexpr auto kF32 = ScalarType::Float;
constexpr int64_t kSlab = 64;        // bytes of K per slab row
constexpr int kFmtE4M3 = 0, kFmtE5M2 = 1;

[[noreturn]] void refuse(const std::string& msg) { throw py::value_error(msg); }
inline void need(bool ok, const char* msg) {
  if (__builtin_expect(!ok, 0)) refuse(msg);
}

std::string shape_of(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

// A contiguous ROCm device tensor of this type and rank.
void contig(const char* name, const Tensor& t, ScalarType dtype, int64_t ndim) {
  if (__builtin_expect(t.is_cuda() && t.scalar_type() == dtype && t.dim() == ndim && t.is_contiguous(), 1)) return;
  const std::string n(name);
  if (!t.is_cuda()) refuse(n + " must be a ROCm device tensor");
  if (t.scalar_type() != dtype)
    refuse(n + " must be " + c10::toString(dtype) + ", got " + c10::toString(t.scalar_type()));
  if (t.dim() != ndim) refuse(n + " must be " + std::to_string(ndim) + "-D, got shape " + shape_of(t));
  refuse(n + " must be contiguous");
}

// The 5 delayed scales and amax slots of one block.
void state(const Tensor& scale, const Tensor& amax) {
  for (const auto& [n, t] : {std::pair<const char*, const Tensor&>{"scale", scale}, {"amax", amax}})
    if (!(t.is_cuda() && t.scalar_type() == kF32 && t.is_contiguous() && t.numel() >= 5))
      refuse(std::string(n) + " must be a contiguous fp32 device tensor of 5 slots");
}

inline int64_t ldt_of(int64_t T) { return (T + 255) / 256 * 256; }
inline int64_t slab_rows(int64_t R) { return (R + 255) / 256 * 256; }
inline int64_t esize(ScalarType t) { return t == kBF16 ? 2 : t == kF32 ? 4 : 1; }

inline Tensor empty(at::IntArrayRef shape, ScalarType dtype, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(like.device()));
}
inline void k_extent(int64_t L, int64_t n) {
  if (L % n) refuse("K extent " + std::to_string(L) + " must be a multiple of " + std::to_string(n));
}
// The K-slab of a row-major [R, L] matrix: [L * size / 64, slab_rows(R), 64 / size].
Tensor kslab(int64_t R, int64_t L, ScalarType dtype, const Tensor& like) {
  const int64_t n = kSlab / esize(dtype);
  k_extent(L, n);
  return empty({L / n, slab_rows(R), n}, dtype, like);
}
Tensor kslabs(int64_t E, int64_t R, int64_t L, ScalarType dtype, const Tensor& like) {
  const int64_t n = kSlab / esize(dtype);
  k_extent(L, n);
  return empty({E, L / n, slab_rows(R), n}, dtype, like);
}
void is_kslab(const char* name, const Tensor& t, ScalarType dtype, int64_t R, int64_t L) {
  const int64_t n = kSlab / esize(dtype);
  contig(name, t, dtype, 3);
  if (!(t.size(0) == L / n && t.size(1) == slab_rows(R) && t.size(2) == n))
    refuse(std::string(name) + " must be a K-slab of [" + std::to_string(R) + ", " + std::to_string(L) + "]");
}

inline void* ptr(const Tensor& t) { return t.data_ptr(); }
inline void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }
inline float* fptr(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
inline float* fptr(const OptTensor& t) { return t ? static_cast<float*>(t->data_ptr()) : nullptr; }
inline int* iptr(const Tensor& t) { return static_cast<int*>(t.data_ptr()); }
inline int* iptr(const OptTensor& t) { return t ? static_cast<int*>(t->data_ptr()) : nullptr; }

inline void* stream_of(const Tensor& t) {
  if (!t.is_cuda()) throw std::runtime_error("libsparkfp8 kernels need ROCm device tensors");
  return c10::hip::getCurrentHIPStream(t.get_device()).stream();
}

// One call of the C ABI with the GIL released; a refused call raises.
template <class F, class... A>
void call(const char* name, F fn, A... args) {
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = fn(args...);
  }
  if (rc == 0) return;
  const char* known[] = {"null pointer argument", "unsupported shape",
                         "misaligned pointer (16-byte alignment required)", "workspace too small",
                         "shape beyond the allocation-free entry point's fixed scratch"};
  throw std::runtime_error(std::string(name) + " failed: " +
                           (rc < 0 && rc >= -5 ? std::string(known[-rc - 1]) : "HIP error " + std::to_string(rc)));
}
#define CALL(fn, ...) call(#fn, fn, __VA_ARGS__)

Tensor workspace(int64_t floats, const Tensor& like) { return empty({floats > 1 ? floats : 1}, kF32, like); }

// ------------------------------------------------------------------ quantizers
std::tuple<Tensor, OptTensor, Tensor> norm_quant(const Tensor& h, const Tensor& norm_w, const Tensor& scale,
                                                 const Tensor& amax, double eps, bool copy) {
  contig("h", h, kBF16, 2);
  contig("norm_w", norm_w, kF32, 1);
  state(scale, amax);
  const int64_t T = h.size(0), D = h.size(1), ldt = ldt_of(T);
  Tensor x8 = kslab(ldt, D, kE4M3, h);
  OptTensor x8t;
  if (copy) x8t = kslab(D, ldt, kE4M3, h);
  Tensor rstd = empty({T}, kF32, h);
  CALL(sfp8_norm_quant, ptr(h), fptr(norm_w), T, D, (float)eps, fptr(scale), fptr(amax), ptr(x8), ptr(x8t), ldt,
       fptr(rstd), stream_of(h));
  return {x8, x8t, rstd};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> block_weight_quant(const Tensor& w_gu, const Tensor& w_down,
                                                                      const OptTensor& scale, const OptTensor& amax) {
  contig("w_gu", w_gu, kF32, 2);
  contig("w_down", w_down, kF32, 2);
  const int64_t R0 = w_gu.size(0), C0 = w_gu.size(1), R1 = w_down.size(0), C1 = w_down.size(1);
  need(R0 % 64 == 0 && C0 % 64 == 0, "gate/up weight rows and columns must be multiples of 64");
  need(C1 % 64 == 0 && R1 % 32 == 0, "down weight columns must be a multiple of 64, rows of 32");
  need(w_down.device() == w_gu.device(), "weights on one device");
  if (scale || amax) {
    need(scale && amax, "scale and amax go together");
    state(*scale, *amax);
    need(scale->numel() == 5 && amax->numel() == 5, "one 5-slot set");
    need(scale->device() == w_gu.device() && amax->device() == w_gu.device(), "scale/amax on the weights' device");
  }
  Tensor w8 = kslab(R0, C0, kE4M3, w_gu), w8t = kslab(C0, R0, kE4M3, w_gu);
  Tensor wd8 = kslab(R1, C1, kE4M3, w_gu), wdt = kslab(C1, R1, kBF16, w_gu);
  Tensor wscale = empty({2}, kF32, w_gu), parts = empty({1024}, kF32, w_gu);
  CALL(sfp8_block_weight_quant, fptr(w_gu), R0, C0, fptr(w_down), R1, C1, fptr(parts), parts.numel(), fptr(wscale),
       ptr(w8), ptr(w8t), ptr(wd8), ptr(wdt), fptr(scale), fptr(amax), stream_of(w_gu));
  return {w8, w8t, wd8, wdt, wscale};
}

std::tuple<OptTensor, OptTensor, OptTensor> weight_quant_experts(const Tensor& w, const Tensor& q_out, bool w8,
                                                                 bool w8t, bool bf16t) {
  contig("w", w, kF32, 3);
  const int64_t E = w.size(0), R = w.size(1), C = w.size(2);
  need(q_out.numel() >= E && q_out.is_contiguous(), "q_out must hold E scales");
  OptTensor o8, o8t, obt;
  if (w8) o8 = kslabs(E, R, C, kE4M3, w);
  if (w8t) o8t = kslabs(E, C, R, kE4M3, w);
  if (bf16t) obt = kslabs(E, C, R, kBF16, w);
  Tensor parts = empty({512 * E}, kF32, w);
  CALL(sfp8_weight_quant_experts, fptr(w), E, R, C, fptr(parts), parts.numel(), fptr(q_out), ptr(o8), ptr(o8t),
       ptr(obt), stream_of(w));
  return {o8, o8t, obt};
}

// ------------------------------------------------------------------ GEMMs of the block
std::tuple<Tensor, Tensor, OptTensor> gateup_swiglu_fwd(const Tensor& x8, const Tensor& w8, const Tensor& scale,
                                                        const Tensor& wscale, const Tensor& amax, int64_t T, int64_t I,
                                                        bool copy) {
  need(x8.dim() == 3, "x8 must be a K-slab");
  const int64_t D = x8.size(0) * kSlab, ldt = ldt_of(T);
  is_kslab("x8", x8, kE4M3, ldt, D);
  is_kslab("w8", w8, kE4M3, 2 * I, D);
  need(D % 128 == 0 && I % 128 == 0, "D and I must be multiples of 128");
  Tensor gu8 = kslab(ldt, 2 * I, kE4M3, x8), h8 = kslab(ldt, I, kE4M3, x8);
  OptTensor h8t;
  if (copy) h8t = kslab(I, ldt, kE4M3, x8);
  CALL(sfp8_gemm_gateup_swiglu_fwd, ptr(x8), ptr(w8), T, D, I, fptr(scale), fptr(wscale), fptr(amax), ptr(gu8),
       ptr(h8), ptr(h8t), ldt, stream_of(x8));
  return {gu8, h8, h8t};
}

Tensor down_fwd(const Tensor& h8, const Tensor& wd8, const Tensor& res, const Tensor& scale, const Tensor& wscale) {
  contig("res", res, kBF16, 2);
  const int64_t T = res.size(0), D = res.size(1);
  need(h8.dim() == 3, "h8 must be a K-slab");
  const int64_t I = h8.size(0) * kSlab, ldt = ldt_of(T);
  is_kslab("h8", h8, kE4M3, ldt, I);
  is_kslab("wd8", wd8, kE4M3, D, I);
  need(I % 128 == 0, "I must be a multiple of 128");
  Tensor y = empty({T, D}, kBF16, h8);
  CALL(sfp8_gemm_down_fwd, ptr(h8), ptr(wd8), ptr(res), T, D, I, fptr(scale), fptr(wscale), ptr(y), ldt,
       stream_of(h8));
  return y;
}

std::tuple<Tensor, OptTensor> down_dgrad_swiglu(const Tensor& dy, const Tensor& wdt, const Tensor& gu8,
                                                const Tensor& scale, const Tensor& amax, bool copy) {
  contig("dy", dy, kBF16, 2);
  const int64_t T = dy.size(0), D = dy.size(1);
  need(gu8.dim() == 3, "gu8 must be a K-slab");
  const int64_t I = gu8.size(0) * kSlab / 2, ldt = ldt_of(T);
  is_kslab("gu8", gu8, kE4M3, ldt, 2 * I);
  is_kslab("wdt", wdt, kBF16, I, D);
  need(D % 64 == 0 && I % 128 == 0, "D must be a multiple of 64 and I of 128");
  Tensor dgu8 = kslab(ldt, 2 * I, kE5M2, dy);
  OptTensor dgu8t;
  if (copy) dgu8t = kslab(2 * I, ldt, kE5M2, dy);
  CALL(sfp8_gemm_down_dgrad_swiglu, ptr(dy), ptr(wdt), ptr(gu8), T, D, I, fptr(scale), fptr(amax), ptr(dgu8),
       ptr(dgu8t), ldt, stream_of(dy));
  return {dgu8, dgu8t};
}

Tensor gateup_dgrad(const Tensor& dgu8, const Tensor& w8t, const Tensor& scale, const Tensor& wscale, int64_t T,
                    int64_t D) {
  need(dgu8.dim() == 3, "dgu8 must be a K-slab");
  const int64_t I2 = dgu8.size(0) * kSlab, ldt = ldt_of(T);
  is_kslab("dgu8", dgu8, kE5M2, ldt, I2);
  is_kslab("w8t", w8t, kE4M3, D, I2);
  need(I2 % 128 == 0, "2I must be a multiple of 128");
  Tensor dxn = empty({T, D}, kBF16, dgu8);
  CALL(sfp8_gemm_gateup_dgrad, ptr(dgu8), ptr(w8t), T, D, I2 / 2, fptr(scale), fptr(wscale), ptr(dxn), ldt,
       stream_of(dgu8));
  return dxn;
}

Tensor wgrad_rows(const Tensor& a8, const Tensor& b8, int64_t M, int64_t N, const Tensor& sa, const Tensor& sb,
                  bool a_rows, bool b_rows) {
  contig("a8", a8, kE5M2, 3);
  contig("b8", b8, kE4M3, 3);
  need(a_rows || b_rows, "at least one row K-slab operand (else use wgrad)");
  const int64_t ldt = a_rows ? a8.size(1) : a8.size(0) * kSlab;
  need((b_rows ? b8.size(1) : b8.size(0) * kSlab) == ldt, "a8, b8 must cover the same tokens");
  need(!a_rows || a8.size(0) * kSlab == M, "a8 must be the row K-slab of [ldt, M]");
  need(!b_rows || b8.size(0) * kSlab == N, "b8 must be the row K-slab of [ldt, N]");
  Tensor out = empty({M, N}, kF32, a8);
  Tensor ws = workspace(sfp8_wgrad_rows_workspace_floats(M, N, ldt), a8);
  CALL(sfp8_gemm_wgrad_rows, ptr(a8), kFmtE5M2, (int)a_rows, ptr(b8), kFmtE4M3, (int)b_rows, M, N, ldt, fptr(sa),
       fptr(sb), fptr(out), fptr(ws), ws.numel(), stream_of(a8));
  return out;
}

std::tuple<Tensor, Tensor, Tensor> norm_bwd(const Tensor& h, const Tensor& rstd, const Tensor& dxn, const Tensor& dy,
                                            const Tensor& norm_w, const Tensor& scale, const Tensor& amax, bool rows) {
  contig("h", h, kBF16, 2);
  contig("dxn", dxn, kBF16, 2);
  contig("dy", dy, kBF16, 2);
  contig("rstd", rstd, kF32, 1);
  contig("norm_w", norm_w, kF32, 1);
  const int64_t T = h.size(0), D = h.size(1), ldt = ldt_of(T);
  Tensor dh = empty({T, D}, kBF16, h), dnw = empty({D}, kF32, h);
  Tensor dy8 = rows ? kslab(ldt, D, kE5M2, h) : kslab(D, ldt, kE5M2, h);
  const int64_t nparts = sfp8_norm_bwd_partials(D, ldt);
  if (nparts < 0) refuse("unsupported hidden size " + std::to_string(D));
  Tensor parts = workspace(nparts * D, h);
  CALL(sfp8_norm_bwd, ptr(h), fptr(rstd), ptr(dxn), ptr(dy), fptr(norm_w), T, D, fptr(scale), fptr(amax), ptr(dh),
       fptr(dnw), fptr(parts), parts.numel(), rows ? ptr(dy8) : nullptr, rows ? nullptr : ptr(dy8), ldt, stream_of(h));
  return {dh, dnw, dy8};
}

// ------------------------------------------------------------------ MoE experts (grouped)
Tensor moe_plan(const Tensor& offsets_in, int64_t R) {
  need(offsets_in.is_cuda() && offsets_in.dim() == 1, "offsets must be a 1-D device tensor");
  const Tensor offsets = offsets_in.to(ScalarType::Int).contiguous();
  const int64_t E = offsets.numel(), n = sfp8_moe_plan_ints(R, E);
  if (n <= 0) refuse("unsupported expert count " + std::to_string(E));
  Tensor plan = empty({n}, ScalarType::Int, offsets);
  CALL(sfp8_moe_plan, iptr(offsets), E, R, iptr(plan), n, stream_of(offsets));
  return plan;
}

std::tuple<OptTensor, OptTensor> moe_rows_quant(const Tensor& src, const OptTensor& index, const Tensor& plan,
                                                int64_t ldp, const Tensor& scale, int64_t sslot, const Tensor& amax,
                                                int64_t aslot, int64_t fmt, bool with_rows, bool with_copy) {
  contig("src", src, kBF16, 2);
  const int64_t n = src.size(0), D = src.size(1);
  need(with_rows || with_copy, "at least one output layout");
  OptTensor xs, xt, idx;
  if (with_rows) xs = kslab(ldp, D, kE4M3, src);
  if (with_copy) xt = kslab(D, ldp, fmt == kFmtE4M3 ? kE4M3 : kE5M2, src);
  if (index) {
    need(index->is_cuda() && index->scalar_type() == ScalarType::Long, "row index must be an int64 device tensor");
    idx = index->contiguous();
  }
  CALL(sfp8_moe_rows_quant, ptr(src), n, D, idx ? static_cast<const int64_t*>(idx->data_ptr()) : nullptr,
       idx ? idx->numel() : 0, iptr(plan), ldp, fptr(scale), (int)sslot, fptr(amax), (int)aslot, (int)fmt, ptr(xs),
       ptr(xt), stream_of(src));
  return {xs, xt};
}

std::tuple<Tensor, Tensor, OptTensor> moe_gateup_swiglu_fwd(const Tensor& x8, const Tensor& w8, const Tensor& plan,
                                                            const Tensor& scale, const Tensor& q_gu,
                                                            const Tensor& amax, int64_t I, bool copy) {
  const int64_t D = x8.size(0) * kSlab, ldp = x8.size(1), E = w8.size(0);
  Tensor gu8 = kslab(ldp, 2 * I, kE4M3, x8), h8 = kslab(ldp, I, kE4M3, x8);
  OptTensor h8t;
  if (copy) h8t = kslab(I, ldp, kE4M3, x8);
  CALL(sfp8_moe_gemm_gateup_swiglu_fwd, ptr(x8), ptr(w8), E, D, I, iptr(plan), ldp, fptr(scale), fptr(q_gu),
       fptr(amax), ptr(gu8), ptr(h8), ptr(h8t), stream_of(x8));
  return {gu8, h8, h8t};
}

Tensor moe_down_fwd(const Tensor& h8, const Tensor& wd8, const Tensor& plan, const Tensor& scale, const Tensor& q_d,
                    int64_t R, int64_t D) {
  const int64_t I = h8.size(0) * kSlab, ldp = h8.size(1), E = wd8.size(0);
  Tensor out = empty({R, D}, kBF16, h8);
  CALL(sfp8_moe_gemm_down_fwd, ptr(h8), ptr(wd8), E, D, I, iptr(plan), ldp, fptr(scale), fptr(q_d), ptr(out), R,
       stream_of(h8));
  return out;
}

std::tuple<Tensor, OptTensor> moe_down_dgrad_swiglu(const Tensor& dout, const Tensor& wdt, const Tensor& gu8,
                                                    const Tensor& plan, const Tensor& scale, const Tensor& amax,
                                                    bool copy) {
  contig("dout", dout, kBF16, 2);
  const int64_t R = dout.size(0), D = dout.size(1), I2 = gu8.size(0) * kSlab, ldp = gu8.size(1), E = wdt.size(0);
  Tensor dgu8 = kslab(ldp, I2, kE5M2, dout);
  OptTensor dgu8t;
  if (copy) dgu8t = kslab(I2, ldp, kE5M2, dout);
  CALL(sfp8_moe_gemm_down_dgrad_swiglu, ptr(dout), ptr(wdt), ptr(gu8), E, D, I2 / 2, R, iptr(plan), ldp, fptr(scale),
       fptr(amax), ptr(dgu8), ptr(dgu8t), stream_of(dout));
  return {dgu8, dgu8t};
}

Tensor moe_gateup_dgrad(const Tensor& dgu8, const Tensor& w8t, const Tensor& plan, const Tensor& scale,
                        const Tensor& q_gu, int64_t R, int64_t D) {
  const int64_t I2 = dgu8.size(0) * kSlab, ldp = dgu8.size(1), E = w8t.size(0);
  Tensor dx = empty({R, D}, kBF16, dgu8);
  CALL(sfp8_moe_gemm_gateup_dgrad, ptr(dgu8), ptr(w8t), E, D, I2 / 2, iptr(plan), ldp, fptr(scale), fptr(q_gu),
       ptr(dx), R, stream_of(dgu8));
  return dx;
}

Tensor moe_wgrad_rows(const Tensor& a8, const Tensor& b8, int64_t M, int64_t N, int64_t E, const Tensor& plan,
                      const Tensor& sa, const Tensor& sb, bool a_rows, bool b_rows) {
  contig("a8", a8, kE5M2, 3);
  contig("b8", b8, kE4M3, 3);
  need(a_rows || b_rows, "at least one row K-slab operand (else use moe_wgrad)");
  const int64_t ldp = a_rows ? a8.size(1) : a8.size(0) * kSlab;
  need((b_rows ? b8.size(1) : b8.size(0) * kSlab) == ldp, "a8, b8 must cover the same padded rows");
  need(!a_rows || a8.size(0) * kSlab == M, "a8 must be the row K-slab of [ldp, M]");
  need(!b_rows || b8.size(0) * kSlab == N, "b8 must be the row K-slab of [ldp, N]");
  Tensor out = empty({E, M, N}, kF32, a8);
  Tensor ws = workspace(sfp8_moe_wgrad_rows_workspace_floats(M, N, E), a8);
  CALL(sfp8_moe_gemm_wgrad_rows, ptr(a8), kFmtE5M2, (int)a_rows, ptr(b8), kFmtE4M3, (int)b_rows, M, N, E, iptr(plan),
       ldp, fptr(sa), fptr(sb), fptr(out), fptr(ws), ws.numel(), stream_of(a8));
  return out;
}

Tensor moe_topk_sum(const Tensor& dx, const Tensor& inverse_permutation, int64_t T, int64_t top_k) {
  contig("dx", dx, kBF16, 2);
  const Tensor inv = inverse_permutation.to(ScalarType::Long).contiguous();
  const int64_t R = dx.size(0), D = dx.size(1);
  Tensor out = empty({T, D}, kBF16, dx);
  CALL(sfp8_moe_topk_sum, ptr(dx), R, D, static_cast<const int64_t*>(inv.data_ptr()), T, top_k, ptr(out),
       stream_of(dx));
  return out;
}

// ------------------------------------------------------------------ bf16 SwiGLU path
std::tuple<OptTensor, OptTensor> bf16_weight_slabs(const Tensor& w, const OptTensor& norm_w, bool rows,
                                                   bool transposed) {
  need(w.is_cuda() && w.dim() == 3 && w.is_contiguous() && (w.scalar_type() == kF32 || w.scalar_type() == kBF16),
       "w must be a contiguous [E, R, C] fp32 or bf16 device tensor");
  const int64_t E = w.size(0), R = w.size(1), C = w.size(2);
  if (R % 64 || C % 64)
    refuse("weight dims " + std::to_string(R) + " x " + std::to_string(C) + " must be multiples of 64");
  if (norm_w) contig("norm_w", *norm_w, kF32, 1);
  OptTensor ws, wt;
  if (rows) ws = kslabs(E, R, C, kBF16, w);
  if (transposed) wt = kslabs(E, C, R, kBF16, w);
  CALL(sfp8_bf16_weight_slabs, ptr(w), (int)(w.scalar_type() == kBF16), fptr(norm_w), E, R, C, ptr(ws), ptr(wt),
       stream_of(w));
  return {ws, wt};
}

std::tuple<OptTensor, OptTensor, OptTensor> bf16_rows_prep(const Tensor& x, const OptTensor& plan, int64_t ldp,
                                                           std::optional<double> eps, bool copy, bool rows) {
  contig("x", x, kBF16, 2);
  const int64_t n = x.size(0), D = x.size(1);
  need(copy || rows || eps, "nothing to compute");
  OptTensor xt, xs, rstd;
  if (copy) xt = kslab(D, ldp, kBF16, x);
  if (rows) xs = kslab(ldp, D, kBF16, x);
  if (eps) rstd = empty({n}, kF32, x);
  CALL(sfp8_bf16_rows_prep, ptr(x), n, D, iptr(plan), ldp, (float)eps.value_or(0.0), fptr(rstd), ptr(xt), ptr(xs),
       stream_of(x));
  return {rstd, xt, xs};
}

std::tuple<Tensor, Tensor> bf16_swiglu_fwd(const Tensor& x, const Tensor& ws, int64_t I, const OptTensor& rstd,
                                           const OptTensor& plan, int64_t ldp, const OptTensor& xs) {
  contig("x", x, kBF16, 2);
  const int64_t n = x.size(0), D = x.size(1);
  Tensor gu = empty({n, 2 * I}, kBF16, x), h = empty({n, I}, kBF16, x);
  if (!plan) {
    if (xs) is_kslab("xs", *xs, kBF16, ldt_of(n), D);
    CALL(sfp8_bf16_gemm_swiglu_fwd, ptr(xs ? *xs : x), (int)xs.has_value(), ptr(ws), n, D, I, fptr(rstd), ptr(gu),
         ptr(h), stream_of(x));
  } else {
    CALL(sfp8_bf16_moe_gemm_swiglu_fwd, ptr(x), ptr(ws), ws.size(0), D, I, iptr(plan), ldp, ptr(gu), ptr(h),
         stream_of(x));
  }
  return {gu, h};
}

Tensor bf16_swiglu_eval(const Tensor& x, const Tensor& w) {
  contig("x", x, kBF16, 2);
  contig("w", w, kBF16, 2);
  const int64_t T = x.size(0), D = x.size(1), I = w.size(0) / 2;
  need(w.size(0) % 2 == 0 && w.size(1) == D, "w must be [2I, D]");
  need(w.device() == x.device(), "x and w on one device");
  Tensor h = empty({T, I}, kBF16, x);
  CALL(sfp8_bf16_swiglu_eval, ptr(x), ptr(w), T, D, I, ptr(h), stream_of(x));
  return h;
}

std::tuple<Tensor, OptTensor> bf16_swiglu_bwd(const Tensor& gu, const Tensor& dout, const OptTensor& rstd,
                                              const OptTensor& plan, int64_t ldp, bool copy) {
  contig("gu", gu, kBF16, 2);
  contig("dout", dout, kBF16, 2);
  const int64_t n = gu.size(0), I2 = gu.size(1);
  need(dout.size(0) == n && dout.size(1) == I2 / 2, "dout must be [rows, I]");
  Tensor gs = kslab(ldp, I2, kBF16, gu);
  OptTensor gt;
  if (copy) gt = kslab(I2, ldp, kBF16, gu);
  CALL(sfp8_bf16_swiglu_bwd, ptr(gu), ptr(dout), n, I2 / 2, fptr(rstd), iptr(plan), ldp, ptr(gs), ptr(gt),
       stream_of(gu));
  return {gs, gt};
}

Tensor bf16_gemm(const Tensor& a, const Tensor& b, int64_t rows, int64_t N, int64_t K, const OptTensor& plan) {
  const int64_t lda = a.size(1);
  Tensor out = empty({rows, N}, kBF16, a);
  if (!plan)
    CALL(sfp8_bf16_gemm, ptr(a), ptr(b), rows, N, K, lda, ptr(out), stream_of(a));
  else
    CALL(sfp8_bf16_moe_gemm, ptr(a), ptr(b), b.size(0), N, K, iptr(plan), lda, ptr(out), stream_of(a));
  return out;
}

Tensor bf16_norm_dh(const Tensor& p, const Tensor& h, const Tensor& rstd) {
  contig("p", p, kBF16, 2);
  contig("h", h, kBF16, 2);
  const int64_t T = h.size(0), D = h.size(1);
  Tensor dh = empty({T, D}, kBF16, h);
  CALL(sfp8_bf16_norm_dh, ptr(p), ptr(h), fptr(rstd), T, D, ptr(dh), stream_of(h));
  return dh;
}

Tensor bf16_wgrad_rows(const Tensor& gs, const Tensor& b, int64_t M, int64_t N, const OptTensor& plan, int64_t E,
                       std::optional<int64_t> T) {
  contig("gs", gs, kBF16, 3);
  const int64_t ldp = gs.size(1);
  need(gs.size(0) * (kSlab / 2) == M, "gs must be the bf16 K-slab of [ldp, M]");
  if (!plan) {
    const bool x_rows = b.dim() == 2;
    contig("x", b, kBF16, x_rows ? 2 : 3);
    if (x_rows) {
      need(b.size(1) == N && b.size(0) <= ldp, "x must be [T, N] with T <= the padded rows");
      T = b.size(0);
    } else {
      need(b.size(0) * (kSlab / 2) == ldp && T, "xt must cover the padded rows; give T");
    }
    Tensor out = empty({M, N}, kBF16, gs);
    Tensor ws = workspace(sfp8_bf16_wgrad_workspace_floats(M, N, ldp), gs);
    CALL(sfp8_bf16_gemm_wgrad_rows, ptr(gs), ptr(b), (int)x_rows, M, N, *T, ldp, ptr(out), fptr(ws), ws.numel(),
         stream_of(gs));
    return out;
  }
  contig("bt", b, kBF16, 3);
  need(b.size(0) * (kSlab / 2) == ldp, "bt must cover the same padded rows");
  Tensor out = empty({E, M, N}, kBF16, gs);
  Tensor ws = workspace(sfp8_bf16_moe_wgrad_workspace_floats(M, N, E), gs);
  CALL(sfp8_bf16_moe_gemm_wgrad_rows, ptr(gs), ptr(b), M, N, E, iptr(plan), ldp, ptr(out), fptr(ws), ws.numel(),
       stream_of(gs));
  return out;
}

std::tuple<Tensor, Tensor> bf16_fold_grads(const Tensor& dwp, const Tensor& w, const Tensor& norm_w) {
  const int64_t M = dwp.size(0), N = dwp.size(1);
  Tensor dw = empty({M, N}, kF32, dwp), dnw = empty({N}, kF32, dwp);
  Tensor part = empty({sfp8_bf16_fold_partials(M, N)}, kF32, dwp);
  CALL(sfp8_bf16_fold_grads, ptr(dwp), fptr(w), fptr(norm_w), M, N, fptr(dw), fptr(dnw), fptr(part), part.numel(),
       stream_of(dwp));
  return {dw, dnw};
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  using py::arg;
  const auto kw = py::kw_only();
  m.def("norm_quant", &norm_quant, arg("h"), arg("norm_w"), arg("scale"), arg("amax"), arg("eps"), kw,
        arg("copy") = true,
        "(x8 K-slab of [T, D] ([D/64, ldt, 64]), x8t K-slab of [D, ldt], rstd [T]); amax[0] max-accumulated.  "
        "copy=False skips the token-contiguous x8t (None): the weight gradient then reads x8 itself (wgrad_rows).");
  m.def("block_weight_quant", &block_weight_quant, arg("w_gu"), arg("w_down"), arg("scale") = py::none(),
        arg("amax") = py::none(),
        "Both weight quantizations of a dense block in two launches: (w8, w8t, wd8, wdt, wscale) as "
        "weight_quant(w_gu, w8=True, w8t=True) and weight_quant(w_down, w8=True, bf16t=True) return them, wscale = "
        "[q_gu, q_d]; with scale and amax, also the delayed-scale roll of those 5 slots (update_scales), in the "
        "first launch.");
  m.def("weight_quant_experts", &weight_quant_experts, arg("w"), arg("q_out"), kw, arg("w8") = true,
        arg("w8t") = false, arg("bf16t") = false,
        "Per-expert e4m3 copies of fp32 masters [E, R, C] (stacked K-slabs, as weight_quant per expert); the pow2 "
        "scales land in q_out[0:E].");
  m.def("gateup_swiglu_fwd", &gateup_swiglu_fwd, arg("x8"), arg("w8"), arg("scale"), arg("wscale"), arg("amax"),
        arg("T"), arg("I"), kw, arg("copy") = true,
        "(gu8 K-slab of [T, 2I], h8 K-slab of [T, I], h8t K-slab of [I, ldt]); x8 is the K-slab of [T, D], w8 that "
        "of [2I, D]; amax[1], amax[2] max-accumulated.  copy=False skips the token-contiguous h8t (None): the weight "
        "gradient then reads h8 itself (wgrad_rows).");
  m.def("down_fwd", &down_fwd, arg("h8"), arg("wd8"), arg("res"), arg("scale"), arg("wscale"),
        "y = bf16(res + bf16(h8 @ wd8^T / (s2 * q_d))), [T, D] bf16; h8 is the K-slab of [T, I], wd8 that of [D, I].");
  m.def("down_dgrad_swiglu", &down_dgrad_swiglu, arg("dy"), arg("wdt"), arg("gu8"), arg("scale"), arg("amax"), kw,
        arg("copy") = true,
        "(dgu8 K-slab of [T, 2I] e5m2, dgu8t K-slab of [2I, ldt] e5m2); wdt is the bf16 K-slab of W_down^T [I, D], "
        "gu8 the e4m3 K-slab of [T, 2I] the forward wrote; amax[3] max-accumulated.  copy=False skips the "
        "token-contiguous dgu8t (None): the weight gradient then reads dgu8 itself (wgrad_rows).");
  m.def("gateup_dgrad", &gateup_dgrad, arg("dgu8"), arg("w8t"), arg("scale"), arg("wscale"), arg("T"), arg("D"),
        "dxn = bf16(dgu8 @ w8 / (s3 * q_gu)), [T, D] bf16; dgu8 is the K-slab of [T, 2I], w8t that of W8^T [D, 2I].");
  m.def("wgrad_rows", &wgrad_rows, arg("a8"), arg("b8"), arg("M"), arg("N"), arg("sa"), arg("sb"), kw,
        arg("a_rows") = true, arg("b_rows") = true,
        "out [M, N] fp32 = sum over tokens of a8[t, m] b8[t, n] / (sa * sb): a8 (e5m2) and b8 (e4m3) each either the "
        "row K-slab of the token-major activation ([rows/64, ldt, 64]: read through transposing LDS reads) or, with "
        "a_rows / b_rows False, the token-contiguous copy ([ldt/64, slab_rows, 64], as for wgrad).");
  m.def("norm_bwd", &norm_bwd, arg("h"), arg("rstd"), arg("dxn"), arg("dy"), arg("norm_w"), arg("scale"), arg("amax"),
        kw, arg("rows") = false,
        "(dh [T, D] bf16, dnw [D] fp32, dy8 e5m2); amax[4] = max|dy|.  dy8 is the token-contiguous K-slab copy of D "
        "rows ([ldt/64, slab_rows(D), 64]), or with rows=True the K-slab of [T, D] ([D/64, ldt, 64], read by "
        "wgrad_rows).");
  m.def("moe_plan", &moe_plan, arg("offsets"), arg("R"),
        "The tile table of padded expert order, built on the device from the experts' inclusive row-count prefix "
        "sums (int32 [E]); no host sync.");
  m.def("moe_rows_quant", &moe_rows_quant, arg("src"), arg("index"), arg("plan"), arg("ldp"), arg("scale"),
        arg("sslot"), arg("amax"), arg("aslot"), arg("fmt"), arg("with_rows"), arg("with_copy") = true,
        "fp8 copies of gathered rows in padded expert order: (xs, xt) = (K-slab of [ldp, D] or None, "
        "token-contiguous K-slab of [D, ldp] or None); row u of the expert order is src[index[u]] (or src[u] without "
        "index).");
  m.def("moe_gateup_swiglu_fwd", &moe_gateup_swiglu_fwd, arg("x8"), arg("w8"), arg("plan"), arg("scale"), arg("q_gu"),
        arg("amax"), arg("I"), kw, arg("copy") = true,
        "(gu8, h8, h8t) over padded expert order; x8 the K-slab of [ldp, D], w8 the stacked per-expert K-slabs of "
        "[2I, D].  copy=False skips h8t (None).");
  m.def("moe_down_fwd", &moe_down_fwd, arg("h8"), arg("wd8"), arg("plan"), arg("scale"), arg("q_d"), arg("R"),
        arg("D"), "out [R, D] bf16 expert-order rows (no residual).");
  m.def("moe_down_dgrad_swiglu", &moe_down_dgrad_swiglu, arg("dout"), arg("wdt"), arg("gu8"), arg("plan"),
        arg("scale"), arg("amax"), kw, arg("copy") = true,
        "(dgu8, dgu8t) e5m2 over padded expert order; dout [R, D] bf16 expert-order rows, wdt the stacked bf16 "
        "K-slabs of W_down[e]^T.  copy=False skips dgu8t (None).");
  m.def("moe_gateup_dgrad", &moe_gateup_dgrad, arg("dgu8"), arg("w8t"), arg("plan"), arg("scale"), arg("q_gu"),
        arg("R"), arg("D"), "dx [R, D] bf16 expert-order rows.");
  m.def("moe_wgrad_rows", &moe_wgrad_rows, arg("a8"), arg("b8"), arg("M"), arg("N"), arg("E"), arg("plan"), arg("sa"),
        arg("sb"), kw, arg("a_rows") = true, arg("b_rows") = true,
        "moe_wgrad with a8 (e5m2) and/or b8 (e4m3) the row K-slab of the expert-order activation over padded rows "
        "([rows/64, ldp, 64]: read through transposing LDS reads) instead of the token-contiguous copy.");
  m.def("moe_topk_sum", &moe_topk_sum, arg("dx"), arg("inverse_permutation"), arg("T"), arg("top_k"),
        "out[t] = sum of the top_k expert-order rows of token t (bf16 [T, D]).");
  m.def("bf16_weight_slabs", &bf16_weight_slabs, arg("w"), arg("norm_w") = py::none(), kw, arg("rows") = true,
        arg("transposed") = true,
        "bf16 K-slabs of W [E, R, C] (fp32, times norm_w[c] when given, or bf16): (ws: stacked K-slabs of W[e] [R, C] "
        "or None, wt: of W[e]^T [C, R] or None).");
  m.def("bf16_rows_prep", &bf16_rows_prep, arg("x"), arg("plan"), arg("ldp"), arg("eps") = py::none(), kw,
        arg("copy") = true, arg("rows") = false,
        "(rstd [rows] fp32 or None, xt or None, xs or None): xt the token-contiguous bf16 K-slab of x^T over ldp "
        "padded rows (copy=False skips it: bf16_wgrad_rows reads x itself); xs (rows=True) the row K-slab of x over "
        "the ldp rows, for bf16_swiglu_fwd; rstd = 1/sqrt(mean(x^2) + eps) when eps is given (dense rows only).");
  m.def("bf16_swiglu_fwd", &bf16_swiglu_fwd, arg("x"), arg("ws"), arg("I"), arg("rstd") = py::none(),
        arg("plan") = py::none(), arg("ldp") = 0, arg("xs") = py::none(),
        "(gu [rows, 2I], h [rows, I]) bf16: the gate/up GEMM with the SwiGLU epilogue, rows scaled by rstd when given "
        "(dense) or grouped by a plan.  Dense: xs, the row K-slab of x from bf16_rows_prep(rows=True), when given is "
        "read instead of x (the same result, a faster read).");
  m.def("bf16_swiglu_eval", &bf16_swiglu_eval, arg("x"), arg("w"),
        "h [T, I] bf16 = silu(x Wg^T) * (x Wu^T) for x [T, D] and W [2I, D] bf16 row-major, when no gradient will be "
        "taken: nothing is saved, W is read as it is.");
  m.def("bf16_swiglu_bwd", &bf16_swiglu_bwd, arg("gu"), arg("dout"), arg("rstd"), arg("plan"), arg("ldp"), kw,
        arg("copy") = true,
        "(gs, gt): G' = bf16 SwiGLU gradient of the rows (times rstd when given) as the K-slab over ldp padded rows "
        "and its token-contiguous transpose (copy=False skips gt, None: the weight gradient then reads gs itself).");
  m.def("bf16_gemm", &bf16_gemm, arg("a"), arg("b"), arg("rows"), arg("N"), arg("K"), arg("plan") = py::none(),
        "out [rows, N] bf16 = A @ B^T, A a bf16 K-slab over padded rows (dense: the first `rows` rows; a plan: the "
        "expert-order rows of each tile), B the (stacked per expert) bf16 K-slab of [N, K].");
  m.def("bf16_norm_dh", &bf16_norm_dh, arg("p"), arg("h"), arg("rstd"),
        "dh = bf16(p - rstd^2 * sum(h * p) / D * h) per row.");
  m.def("bf16_wgrad_rows", &bf16_wgrad_rows, arg("gs"), arg("b"), arg("M"), arg("N"), arg("plan") = py::none(),
        arg("E") = 1, arg("T") = py::none(),
        "bf16_wgrad with A read from gs, the bf16 K-slab of G' over the padded rows, through transposing LDS reads.  "
        "Dense (no plan): b is x itself, row-major [T, N] bf16, also transposed on read, or (3-d) the "
        "token-contiguous K-slab of x^T (bf16_rows_prep; T then gives the tokens); with a plan b is the "
        "token-contiguous K-slab of x^T over the padded rows.");
  m.def("bf16_fold_grads", &bf16_fold_grads, arg("dwp"), arg("w"), arg("norm_w"),
        "(dw = f32(dwp) * norm_w, dnorm_w = sum over rows of f32(dwp) * w): the gradients of the fp32 gate/up master "
        "and the norm weight from the bf16 gradient of the folded weight.");
}
