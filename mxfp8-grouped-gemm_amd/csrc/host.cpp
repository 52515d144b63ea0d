// Native host path of the Python entry points: checks, output allocation and
// the library call in one step.
//
// A small call (a few hundred tokens, small layers) is bound by the host: in
// Python an op spends 20 to 60 us on attribute reads, allocations and a ctypes
// call of 20 to 30 arguments, for kernels of 3 to 20 us.  Each function below
// takes the plain case of its op (device tensors of the right type, laid out as
// the kernels read them).  For anything else it returns None and touches
// nothing: the caller then runs the Python form, which converts, splits or
// raises.  A result is a tensor or a tuple; an int is a library status.
// Like torch's own ops, the functions run without the GIL (an allocation or a
// launch on a full queue can block) and raise torch's exceptions (a trainer
// catches torch.OutOfMemoryError).
//
// Library functions are reached through addresses handed in once by bind(), so
// this module does not link against libmxgg.so; bind() refuses a library of
// another ABI version than the header this module was compiled with.
#include <torch/extension.h>

#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <variant>
#include <vector>

#include "../../include/mxgg.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

struct Lib {
#define MXGG_FN(name) decltype(&::mxgg_##name) name = nullptr;
#define MXGG_FNS                                                                            \
  MXGG_FN(quant_dim0) MXGG_FN(quant_dim1) MXGG_FN(quant_dual) MXGG_FN(zero_rows_past_groups) \
  MXGG_FN(grouped_fwd) MXGG_FN(grouped_fwd_split) MXGG_FN(grouped_fwd_swiglu_quant)          \
  MXGG_FN(grouped_fwd_swiglu_quant_keep_h) MXGG_FN(grouped_wgrad) MXGG_FN(swiglu_bwd_quant)  \
  MXGG_FN(gather_quant_dual) MXGG_FN(gather_quant_dim0) MXGG_FN(combine)
  MXGG_FNS
#undef MXGG_FN
};
Lib lib;

void bind(const py::dict& address) {
  const auto version = reinterpret_cast<decltype(&::mxgg_abi_version)>(
      address["mxgg_abi_version"].cast<uintptr_t>())();
  if (version != MXGG_ABI_VERSION)
    throw std::runtime_error("built for ABI version " + std::to_string(MXGG_ABI_VERSION) +
                             ", the library has " + std::to_string(version));
  Lib l;
#define MXGG_FN(name) \
  l.name = reinterpret_cast<decltype(l.name)>(address["mxgg_" #name].cast<uintptr_t>());
  MXGG_FNS
#undef MXGG_FN
  lib = l;
}

constexpr int64_t kMaxOperandBytes = 0x7FFFFFF0;  // the C ABI's bound on (rows - 1) * ld + K

// A device tensor with memory of its own behind it (no fake, batched or
// otherwise wrapped tensor).
bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == c10::kStrided && t.has_storage() &&
         !t.key_set().has(c10::DispatchKey::Python) && t.numel() > 0 &&
         t.const_data_ptr() != nullptr;
}
bool aligned(const void* p, uintptr_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; }
// 2-D bf16 rows the kernels read in place.
bool bf16_rows(const Tensor& t) {
  return plain(t) && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.stride(1) == 1 &&
         t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) && aligned(t.const_data_ptr(), 16);
}
bool bytes(const Tensor& t) {
  const auto d = t.scalar_type();
  return plain(t) && (d == at::kFloat8_e4m3fn || d == at::kByte);
}
// Group ends used as they are.
bool ends_ok(const OptTensor& e, const Tensor& like) {
  return !e || (plain(*e) && e->scalar_type() == at::kInt && e->dim() == 1 &&
                e->is_contiguous() && e->device() == like.device());
}
const int32_t* ends_ptr(const OptTensor& e) { return e ? e->const_data_ptr<int32_t>() : nullptr; }

int64_t ld16(int64_t n) { return std::max<int64_t>(16, (n + 15) / 16 * 16); }
int64_t padded_capacity(int64_t tokens, int64_t groups) {
  return groups == 0 ? (tokens + 31) / 32 * 32 : (tokens + 31 * groups + 127) / 128 * 128;
}
Tensor empty(at::IntArrayRef size, const Tensor& like, at::ScalarType type) {
  return at::empty(size, like.options().dtype(type).requires_grad(false));
}
// Storage of block-major scales, [nblk][round_up(rows, 16)], and the logical
// [rows, nblk] view of it.
Tensor block_major(int64_t rows, int64_t nblk, const Tensor& like) {
  return empty({nblk, ld16(rows)}, like, at::kByte);
}
Tensor rows_view(const Tensor& buf, int64_t rows) {
  return buf.as_strided({rows, buf.size(0)}, {1, buf.stride(0)});
}
void* vp(const Tensor& t) { return t.data_ptr(); }
const void* cp(const Tensor& t) { return t.const_data_ptr(); }
void* st(int64_t stream) { return reinterpret_cast<void*>(stream); }

using Result = std::variant<std::monostate, int, Tensor, std::tuple<Tensor, Tensor>,
                            std::tuple<Tensor, Tensor, Tensor>,
                            std::tuple<Tensor, Tensor, OptTensor>,
                            std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>,
                            std::tuple<Tensor, Tensor, Tensor, Tensor, OptTensor>,
                            std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, OptTensor>>;
Result none() { return std::monostate{}; }

// E8M0 scales [rows, nblk] (or [E, rows, nblk]) stored block-major, as the
// library's casts return them; the conditions are the Python form's.
int64_t readable(const Tensor& t) {
  return (int64_t)t.storage().nbytes() - t.storage_offset() * t.element_size();
}
bool scale_bytes(const Tensor& s, const Tensor& of) {
  const auto d = s.scalar_type();
  return plain(s) && s.device() == of.device() &&
         (d == at::kByte || d == at::kFloat8_e8m0fnu || d == at::kFloat8_e4m3fn || d == at::kChar);
}
bool scales_2d(const Tensor& s, const Tensor& of, int64_t rows, int64_t nblk) {
  return scale_bytes(s, of) && s.dim() == 2 && s.size(0) == rows &&
         s.size(1) == nblk && (s.stride(0) == 1 || rows == 1) && s.stride(1) >= rows &&
         s.stride(1) % 4 == 0 && aligned(cp(s), 4) &&
         readable(s) >= (nblk - 1) * s.stride(1) + (rows + 3) / 4 * 4;
}
bool scales_3d(const Tensor& s, const Tensor& of, int64_t E, int64_t rows, int64_t nblk) {
  return scale_bytes(s, of) && s.dim() == 3 && s.size(0) == E &&
         s.size(1) == rows && s.size(2) == nblk && (s.stride(1) == 1 || rows == 1) &&
         s.stride(2) % 4 == 0 && (E == 1 || s.stride(0) % 4 == 0) && aligned(cp(s), 4) &&
         s.stride(2) >= rows && (E == 1 || s.stride(0) >= rows) &&
         readable(s) >= (E - 1) * s.stride(0) + (nblk - 1) * s.stride(2) + (rows + 3) / 4 * 4;
}

Result dim0(const Tensor& x, bool block, int mode, int64_t stream) {
  if (!plain(x) || x.scalar_type() != at::kBFloat16 || x.dim() < 1 || !x.is_contiguous() ||
      x.size(-1) % 32 != 0 || !aligned(cp(x), 16))
    return none();
  const int64_t K = x.size(-1), rows = x.numel() / K, nblk = K / 32;
  Tensor q = empty(x.sizes(), x, at::kFloat8_e4m3fn);
  auto size = x.sizes().vec();
  size.back() = nblk;
  Tensor s;
  int64_t lds;
  if (block) {
    lds = ld16(rows);
    Tensor buf = block_major(rows, nblk, x);
    std::vector<int64_t> stride(size.size());
    int64_t acc = 1;
    for (size_t d = size.size() - 1; d-- > 0;) {
      stride[d] = acc;
      acc *= size[d];
    }
    stride.back() = lds;
    s = buf.as_strided(size, stride);
  } else {
    lds = nblk;
    s = empty(size, x, at::kByte);
  }
  const int rc = lib.quant_dim0(cp(x), rows, K, K, vp(q), K, vp(s), lds,
                                block ? MXGG_SCALES_BLOCK_MAJOR : MXGG_SCALES_ROW_MAJOR, mode,
                                st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(q, s);
}

// cap: columns of the token-axis cast, 0 = padded_capacity.
Result dim1(const Tensor& x, const OptTensor& ends, bool block, int64_t cap, int mode,
                int64_t stream) {
  if (!bf16_rows(x) || x.size(1) % 8 != 0 || !ends_ok(ends, x)) return none();
  const int64_t M = x.size(0), C = x.size(1), E = ends ? ends->numel() : 0;
  if (cap == 0) cap = padded_capacity(M, E);
  Tensor qt = empty({C, cap}, x, at::kFloat8_e4m3fn);
  Tensor buf = block ? block_major(C, cap / 32, x) : empty({C, cap / 32}, x, at::kByte);
  OptTensor pad;
  if (ends) pad = empty({E}, x, at::kInt);
  const int rc = lib.quant_dim1(
      cp(x), M, C, x.stride(0), ends_ptr(ends), E, cap, vp(qt), cap, vp(buf), buf.stride(0),
      block ? MXGG_SCALES_BLOCK_MAJOR : MXGG_SCALES_ROW_MAJOR,
      pad ? pad->data_ptr<int32_t>() : nullptr, mode, st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(qt, block ? rows_view(buf, C) : buf, pad);
}

Result dual(const Tensor& x, const OptTensor& ends, int64_t cap, int mode, int64_t stream) {
  if (!bf16_rows(x) || x.size(1) % 32 != 0 || !ends_ok(ends, x)) return none();
  const int64_t M = x.size(0), C = x.size(1), E = ends ? ends->numel() : 0;
  if (cap == 0) cap = padded_capacity(M, E);
  Tensor q = empty({M, C}, x, at::kFloat8_e4m3fn), qt = empty({C, cap}, x, at::kFloat8_e4m3fn);
  Tensor sb = block_major(M, C / 32, x), stb = block_major(C, cap / 32, x);
  OptTensor pad;
  if (ends) pad = empty({E}, x, at::kInt);
  const int rc = lib.quant_dual(cp(x), M, C, x.stride(0), ends_ptr(ends), E, cap, vp(q), C, vp(sb),
                                sb.stride(0), vp(qt), cap, vp(stb), stb.stride(0),
                                MXGG_SCALES_BLOCK_MAJOR, pad ? pad->data_ptr<int32_t>() : nullptr,
                                mode, st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(q, rows_view(sb, M), qt, rows_view(stb, C), pad);
}

// Operands of the grouped forward, checked.
struct FwdIn {
  int64_t M, K, E, N;
  const void *as = nullptr, *ws = nullptr;
  int64_t ldas = 0, wsg = 0, ldws = 0;
};
bool fwd_in(const Tensor& a, const Tensor& w, const OptTensor& ends, const OptTensor& as,
            const OptTensor& ws, FwdIn& in) {
  if (!bytes(a) || !bytes(w) || a.dim() != 2 || w.dim() != 3 || a.stride(1) != 1 ||
      w.stride(2) != 1 || a.size(1) != w.size(2) || a.device() != w.device() ||
      as.has_value() != ws.has_value() || !ends_ok(ends, a))
    return false;
  in.M = a.size(0);
  in.K = a.size(1);
  in.E = w.size(0);
  in.N = w.size(1);
  if (in.K % 32 != 0 || (ends ? ends->numel() != in.E : in.E != 1) ||
      (in.M - 1) * a.stride(0) + in.K > kMaxOperandBytes)
    return false;
  if (as) {
    if (!scales_2d(*as, a, in.M, in.K / 32) || !scales_3d(*ws, a, in.E, in.N, in.K / 32)) return false;
    in.as = cp(*as);
    in.ldas = as->stride(1);
    in.ws = cp(*ws);
    in.wsg = ws->stride(0);
    in.ldws = ws->stride(2);
  }
  return true;
}

// split: workspace bytes of the split entry, 0 for the unsplit one.
Result mm(const Tensor& a, const Tensor& w, const OptTensor& ends, const OptTensor& as,
              const OptTensor& ws, bool f32, int64_t split, int64_t stream) {
  FwdIn in;
  if (!fwd_in(a, w, ends, as, ws, in) || in.N % 4 != 0) return none();
  Tensor out = empty({in.M, in.N}, a, f32 ? at::kFloat : at::kBFloat16);
  const int type = f32 ? MXGG_OUT_F32 : MXGG_OUT_BF16;
  int rc;
  if (split > 0) {
    Tensor scratch = empty({split}, a, at::kByte);
    rc = lib.grouped_fwd_split(cp(a), a.stride(0), in.as, in.ldas, cp(w), w.stride(0), w.stride(1),
                               in.ws, in.wsg, in.ldws, ends_ptr(ends), in.E, in.M, in.N, in.K,
                               vp(out), in.N, type, vp(scratch), split, st(stream));
  } else {
    rc = lib.grouped_fwd(cp(a), a.stride(0), in.as, in.ldas, cp(w), w.stride(0), w.stride(1),
                         in.ws, in.wsg, in.ldws, ends_ptr(ends), in.E, in.M, in.N, in.K, vp(out),
                         in.N, type, st(stream));
  }
  if (rc != MXGG_OK) return rc;
  return out;
}

Result mm_swiglu(const Tensor& a, const Tensor& w, const OptTensor& ends, const OptTensor& as,
                     const OptTensor& ws, int mode, bool keep, int64_t stream) {
  FwdIn in;
  if (!fwd_in(a, w, ends, as, ws, in) || in.N % 256 != 0) return none();
  const int64_t F = in.N / 2;
  Tensor q = empty({in.M, F}, a, at::kFloat8_e4m3fn), buf = block_major(in.M, F / 32, a);
  Tensor h;
  int rc;
  if (keep) {
    h = empty({in.M, in.N}, a, at::kBFloat16);
    rc = lib.grouped_fwd_swiglu_quant_keep_h(
        cp(a), a.stride(0), in.as, in.ldas, cp(w), w.stride(0), w.stride(1), in.ws, in.wsg,
        in.ldws, ends_ptr(ends), in.E, in.M, F, in.K, vp(h), in.N, vp(q), F, vp(buf),
        buf.stride(0), MXGG_SCALES_BLOCK_MAJOR, mode, st(stream));
    // the kernel writes no row past the last group end
    if (rc == MXGG_OK && ends)
      rc = lib.zero_rows_past_groups(vp(h), in.M, 2 * in.N, 2 * in.N, ends_ptr(ends), in.E,
                                     st(stream));
  } else {
    rc = lib.grouped_fwd_swiglu_quant(
        cp(a), a.stride(0), in.as, in.ldas, cp(w), w.stride(0), w.stride(1), in.ws, in.wsg,
        in.ldws, ends_ptr(ends), in.E, in.M, F, in.K, vp(q), F, vp(buf), buf.stride(0),
        MXGG_SCALES_BLOCK_MAJOR, mode, st(stream));
  }
  if (rc != MXGG_OK) return rc;
  if (keep) return std::make_tuple(q, rows_view(buf, in.M), h);
  return std::make_tuple(q, rows_view(buf, in.M));
}

// Unsplit weight gradient into a new dW.
Result wgrad(const Tensor& go, const Tensor& ia, const Tensor& ends, const OptTensor& gs,
                 const OptTensor& is, bool f32, int64_t stream) {
  if (!bytes(go) || !bytes(ia) || go.dim() != 2 || ia.dim() != 2 || go.stride(1) != 1 ||
      ia.stride(1) != 1 || go.size(1) != ia.size(1) || go.device() != ia.device() ||
      gs.has_value() != is.has_value() || !ends_ok(ends, go))
    return none();
  const int64_t N = go.size(0), K = ia.size(0), M = go.size(1), E = ends.numel();
  if (K % 4 != 0 || M % 32 != 0 || (N - 1) * go.stride(0) + M > kMaxOperandBytes ||
      (K - 1) * ia.stride(0) + M > kMaxOperandBytes)
    return none();
  if (gs && (!scales_2d(*gs, go, N, M / 32) || !scales_2d(*is, go, K, M / 32))) return none();
  Tensor dw = empty({E, N, K}, go, f32 ? at::kFloat : at::kBFloat16);
  const int rc = lib.grouped_wgrad(
      cp(go), go.stride(0), gs ? cp(*gs) : nullptr, gs ? gs->stride(1) : 0, cp(ia), ia.stride(0),
      is ? cp(*is) : nullptr, is ? is->stride(1) : 0, ends.const_data_ptr<int32_t>(), E, M, N, K,
      vp(dw), f32 ? MXGG_OUT_F32 : MXGG_OUT_BF16, 0, st(stream));
  if (rc != MXGG_OK) return rc;
  return dw;
}

Result swiglu_bwd(const Tensor& h, const Tensor& da, const OptTensor& ends, int mode,
                      int64_t stream) {
  if (!bf16_rows(h) || !bf16_rows(da) || h.size(1) % 64 != 0 || da.size(0) != h.size(0) ||
      da.size(1) != h.size(1) / 2 || !ends_ok(ends, h) || h.device() != da.device())
    return none();
  const int64_t M = h.size(0), F = da.size(1), E = ends ? ends->numel() : 0;
  const int64_t cap = padded_capacity(M, E);
  const uint16_t* gate = static_cast<const uint16_t*>(cp(h));
  Tensor q = empty({M, 2 * F}, h, at::kFloat8_e4m3fn), sb = block_major(M, 2 * F / 32, h);
  Tensor qt = empty({2 * F, cap}, h, at::kFloat8_e4m3fn), stb = block_major(2 * F, cap / 32, h);
  Tensor at = empty({F, cap}, h, at::kFloat8_e4m3fn), atb = block_major(F, cap / 32, h);
  OptTensor pad;
  if (ends) pad = empty({E}, h, at::kInt);
  const int rc = lib.swiglu_bwd_quant(
      gate, gate + F, h.stride(0), cp(da), da.stride(0), M, F, ends_ptr(ends), E, cap, vp(q), 2 * F,
      vp(sb), sb.stride(0), vp(qt), cap, vp(stb), stb.stride(0), vp(at), cap, vp(atb),
      atb.stride(0), pad ? pad->data_ptr<int32_t>() : nullptr, nullptr, 2 * F,
      MXGG_SCALES_BLOCK_MAJOR, mode, st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(q, rows_view(sb, M), qt, rows_view(stb, 2 * F), at, rows_view(atb, F), pad);
}

Result zero_rows(const Tensor& out, const Tensor& ends, int64_t stream) {
  if (!plain(out) || out.dim() != 2 || out.stride(1) != 1 || !ends_ok(ends, out)) return none();
  const int64_t e = out.element_size();
  const int rc = lib.zero_rows_past_groups(vp(out), out.size(0), out.size(1) * e, out.stride(0) * e,
                                           ends.const_data_ptr<int32_t>(), ends.numel(),
                                           st(stream));
  return rc;
}

// Routing: src / perm / offs are a plan's tensors.
bool row_scores(const Tensor& s, const Tensor& of, int64_t slots) {
  return plain(s) && s.scalar_type() == at::kFloat && s.is_contiguous() && s.numel() == slots &&
         s.device() == of.device();
}
Result gather_dual(const Tensor& x, const Tensor& src, const Tensor& offs, int topk,
                       const OptTensor& scale, int mode, int64_t stream) {
  if (!bf16_rows(x) || x.size(1) % 32 != 0 || !ends_ok(src, x) || !ends_ok(offs, x) ||
      (scale && !row_scores(*scale, x, x.size(0) * topk)))
    return none();
  const int64_t M = src.numel(), C = x.size(1), E = offs.numel(), cap = padded_capacity(M, E);
  Tensor q = empty({M, C}, x, at::kFloat8_e4m3fn), qt = empty({C, cap}, x, at::kFloat8_e4m3fn);
  Tensor sb = block_major(M, C / 32, x), stb = block_major(C, cap / 32, x);
  Tensor pad = empty({E}, x, at::kInt);
  const int rc = lib.gather_quant_dual(
      cp(x), x.size(0), C, x.stride(0), src.const_data_ptr<int32_t>(), topk,
      scale ? scale->const_data_ptr<float>() : nullptr, M, offs.const_data_ptr<int32_t>(), E, cap,
      vp(q), C, vp(sb), sb.stride(0), vp(qt), cap, vp(stb), stb.stride(0),
      MXGG_SCALES_BLOCK_MAJOR, pad.data_ptr<int32_t>(), mode, st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(q, rows_view(sb, M), qt, rows_view(stb, C), pad);
}

Result gather_dim0(const Tensor& x, const Tensor& src, int topk, int mode, int64_t stream) {
  if (!bf16_rows(x) || x.size(1) % 32 != 0 || !ends_ok(src, x)) return none();
  const int64_t M = src.numel(), C = x.size(1);
  Tensor q = empty({M, C}, x, at::kFloat8_e4m3fn), sb = block_major(M, C / 32, x);
  const int rc = lib.gather_quant_dim0(cp(x), x.size(0), C, x.stride(0),
                                       src.const_data_ptr<int32_t>(), topk, M, vp(q), C, vp(sb),
                                       sb.stride(0), MXGG_SCALES_BLOCK_MAJOR, mode, st(stream));
  if (rc != MXGG_OK) return rc;
  return std::make_tuple(q, rows_view(sb, M));
}

Result combine(const Tensor& y, const Tensor& perm, int64_t tokens, int topk,
                   const OptTensor& scores, int64_t stream) {
  if (!bf16_rows(y) || y.size(1) % 8 != 0 || !ends_ok(perm, y) || perm.numel() != tokens * topk ||
      (scores && !row_scores(*scores, y, tokens * topk)))
    return none();
  Tensor out = empty({tokens, y.size(1)}, y, at::kBFloat16);
  const int rc = lib.combine(cp(y), y.size(0), y.size(1), y.stride(0),
                             perm.const_data_ptr<int32_t>(),
                             scores ? scores->const_data_ptr<float>() : nullptr, tokens, topk,
                             vp(out), out.stride(0), st(stream));
  if (rc != MXGG_OK) return rc;
  return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", &bind);
  m.def("dim0", torch::wrap_pybind_function_no_gil(&dim0));
  m.def("dim1", torch::wrap_pybind_function_no_gil(&dim1));
  m.def("dual", torch::wrap_pybind_function_no_gil(&dual));
  m.def("mm", torch::wrap_pybind_function_no_gil(&mm));
  m.def("mm_swiglu", torch::wrap_pybind_function_no_gil(&mm_swiglu));
  m.def("wgrad", torch::wrap_pybind_function_no_gil(&wgrad));
  m.def("swiglu_bwd", torch::wrap_pybind_function_no_gil(&swiglu_bwd));
  m.def("zero_rows", torch::wrap_pybind_function_no_gil(&zero_rows));
  m.def("gather_dual", torch::wrap_pybind_function_no_gil(&gather_dual));
  m.def("gather_dim0", torch::wrap_pybind_function_no_gil(&gather_dim0));
  m.def("combine", torch::wrap_pybind_function_no_gil(&combine));
}
