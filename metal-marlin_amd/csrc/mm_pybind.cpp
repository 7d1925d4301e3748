// Python binding of the per-call hot path (marlin_gemm_fp4 / marlin_gemm_int4,
// the fused QKV and gate/up projections and the row-packed product) for callers
// that issue one projection per Python call.  It does in C++ what the
// ctypes path does in Python -- shape checks, the output allocation, the
// per-(device, stream) workspace -- and calls the same C ABI entry points of
// libmmfp4.so (mm_fp4_gemm / mm_u4_gemm).  torch is used only for tensor
// arguments and the output allocation; the stream comes from the caller.
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <sstream>
#include <utility>

#include "mmfp4.h"

namespace {

std::mutex g_mu;
std::map<std::pair<int, int64_t>, at::Tensor> g_ws;   // (device index, stream) -> workspace

// One workspace per (device, stream), shared with the ctypes path (which
// asks for it through workspace_for below); kept until release_workspaces().
at::Tensor workspace_dev(int dev, int64_t stream, size_t nbytes, const at::TensorOptions& opt) {
  std::lock_guard<std::mutex> lock(g_mu);
  const auto key = std::make_pair(dev, stream);
  auto it = g_ws.find(key);
  if (it != g_ws.end() && (size_t)it->second.numel() >= nbytes) return it->second;
  size_t size = nbytes < ((size_t)1 << 20) ? ((size_t)1 << 20) : nbytes;
  if (it != g_ws.end() && size < 2 * (size_t)it->second.numel()) size = 2 * it->second.numel();
  // Zero-filled once: the split-K arrival counters at its head must start at
  // zero, and every call leaves them at zero.
  at::Tensor buf = at::zeros({(int64_t)size}, opt.dtype(at::kByte));
  g_ws[key] = buf;
  return buf;
}

at::Tensor workspace(const at::Tensor& like, int64_t stream, size_t nbytes) {
  return workspace_dev((int)like.get_device(), stream, nbytes, like.options());
}

at::Tensor workspace_for(int64_t device, int64_t stream, int64_t nbytes) {
  return workspace_dev((int)device, stream, (size_t)nbytes,
                       at::TensorOptions().device(at::kCUDA, (int)device));
}

void release_workspaces() {
  std::lock_guard<std::mutex> lock(g_mu);
  g_ws.clear();
}

[[noreturn]] void fail(int rc) {
  const char* msg = mm_last_error();
  if (rc == 1) throw pybind11::value_error(msg);
  throw std::runtime_error(msg);
}

void check_groups(const char* name, const at::Tensor& t, int64_t K, int64_t N, int64_t g) {
  if (g <= 0 || K % g != 0) {
    std::ostringstream os;
    os << name << ": K=" << K << " must be divisible by group_size=" << g;
    throw pybind11::value_error(os.str());
  }
  if (t.dim() != 2 || t.size(0) != K / g || t.size(1) != N) {
    std::ostringstream os;
    os << name << ": " << name << " shape " << t.sizes() << " != (" << K / g << ", " << N
       << ") for K=" << K << ", group_size=" << g;
    throw pybind11::value_error(os.str());
  }
}

at::Tensor half_contig(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf && t.is_contiguous() ? t : t.to(at::kHalf).contiguous();
}

// C = A . dequant(B, S[, Z]) for A [*, K], B [K/8, N] words; fp16 [*, N].
// SZ (INT4 only, optional): the scales and zeros interleaved [K/g, N/4, 8]
// for the decode kernels (mm_u4_gemm_sz).
at::Tensor gemm(const at::Tensor& A, const at::Tensor& B, const at::Tensor& S,
                const c10::optional<at::Tensor>& Z, const c10::optional<at::Tensor>& SZ,
                int64_t group_size, int64_t stream) {
  const int dev = A.get_device();
  if (dev < 0 || B.get_device() != dev || S.get_device() != dev ||
      (Z && Z->get_device() != dev)) {
    std::ostringstream os;
    os << "tensor on " << (dev < 0 ? A.device() : B.device())
       << ": the FP4/INT4 kernels run on the GPU only, with every operand on one device";
    throw std::runtime_error(os.str());
  }
  if (B.dim() != 2) throw pybind11::value_error("B_packed must be [K/8, N]");
  if (B.scalar_type() != at::kInt && B.scalar_type() != at::kUInt32)
    throw pybind11::type_error("packed weights must be int32/uint32 words");
  const int64_t K = A.size(-1);
  const int64_t M = K ? A.numel() / K : 0;
  const int64_t N = B.size(1);
  if (B.size(0) * 8 != K) {
    std::ostringstream os;
    os << "Packed K " << B.size(0) * 8 << " does not match activations K " << K;
    throw pybind11::value_error(os.str());
  }
  check_groups("scales", S, K, N, group_size);
  if (Z) check_groups("zeros", *Z, K, N, group_size);
  const at::Tensor a = half_contig(A);
  const at::Tensor b = B.is_contiguous() ? B : B.contiguous();
  const at::Tensor s = half_contig(S);
  std::vector<int64_t> oshape(A.sizes().begin(), A.sizes().end());
  oshape.back() = N;
  at::Tensor out = at::empty(oshape, a.options());
  const size_t need = mm_gemm_workspace_bytes((int)M, (int)N, (int)K);
  at::Tensor ws = workspace(a, stream, need);
  int rc;
  if (!Z) {
    rc = mm_fp4_gemm((const uint16_t*)a.data_ptr(), (const uint32_t*)b.data_ptr(),
                     (const uint16_t*)s.data_ptr(), (uint16_t*)out.data_ptr(), (int)M, (int)N,
                     (int)K, (int)group_size, ws.data_ptr(), (size_t)ws.numel(),
                     (void*)stream);
  } else if (SZ) {
    const at::Tensor z = half_contig(*Z);
    if (SZ->scalar_type() != at::kHalf || !SZ->is_contiguous() || SZ->numel() != 2 * z.numel() ||
        SZ->get_device() != dev)
      throw pybind11::value_error("SZ must be contiguous fp16 [K/g, 2N] on the operands' device");
    rc = mm_u4_gemm_sz((const uint16_t*)a.data_ptr(), (const uint32_t*)b.data_ptr(),
                       (const uint16_t*)s.data_ptr(), (const uint16_t*)z.data_ptr(),
                       (const uint16_t*)SZ->data_ptr(), (uint16_t*)out.data_ptr(), (int)M,
                       (int)N, (int)K, (int)group_size, ws.data_ptr(), (size_t)ws.numel(),
                       (void*)stream);
  } else {
    const at::Tensor z = half_contig(*Z);
    rc = mm_u4_gemm((const uint16_t*)a.data_ptr(), (const uint32_t*)b.data_ptr(),
                    (const uint16_t*)s.data_ptr(), (const uint16_t*)z.data_ptr(),
                    (uint16_t*)out.data_ptr(), (int)M, (int)N, (int)K, (int)group_size,
                    ws.data_ptr(), (size_t)ws.numel(), (void*)stream);
  }
  if (rc) fail(rc);
  return out;
}

// The fused projections below take the plain form of their operands only --
// contiguous fp16 activations and scales and packed words on one device, shapes
// that agree -- and return None for anything else, which their Python callers
// then convert or refuse.
bool plain(const at::Tensor& t, at::ScalarType type, int dev, int64_t d0, int64_t d1) {
  return t.dim() == 2 && t.size(0) == d0 && t.size(1) == d1 && t.get_device() == dev &&
         t.is_contiguous() && t.scalar_type() == type;
}
bool plain_words(const at::Tensor& t, int dev, int64_t d0, int64_t d1) {
  return plain(t, t.scalar_type() == at::kUInt32 ? at::kUInt32 : at::kInt, dev, d0, d1);
}
// [M, K] of the activations, or M = -1.
std::pair<int64_t, int64_t> plain_acts(const at::Tensor& A) {
  if (A.dim() != 2 || A.get_device() < 0 || !A.is_contiguous() || A.scalar_type() != at::kHalf ||
      A.size(0) == 0 || A.size(1) == 0)
    return {-1, 0};
  return {A.size(0), A.size(1)};
}

// Q, K, V = A . dequant(W[p], S[p]) in one mm_fp4_gemm_multi call.
pybind11::object qkv(const at::Tensor& A, const std::array<at::Tensor, 3>& W,
                     const std::array<at::Tensor, 3>& S, int64_t g, int64_t stream) {
  const auto [M, K] = plain_acts(A);
  if (M < 0 || g <= 0 || K % g != 0 || K % 8 != 0) return pybind11::none();
  const int dev = (int)A.get_device();
  const uint32_t* b[3];
  const uint16_t* s[3];
  uint16_t* c[3];
  int n[3];
  int64_t ntot = 0;
  for (int p = 0; p < 3; ++p) {
    const int64_t N = W[p].dim() == 2 ? W[p].size(1) : 0;
    if (N <= 0 || N % 4 != 0 || !plain_words(W[p], dev, K / 8, N) ||
        !plain(S[p], at::kHalf, dev, K / g, N))
      return pybind11::none();
    n[p] = (int)N;
    ntot += N;
  }
  at::Tensor out[3];
  size_t need = mm_gemm_workspace_bytes((int)M, (int)ntot, (int)K);
  for (int p = 0; p < 3; ++p) {
    out[p] = at::empty({M, n[p]}, A.options());
    need = std::max(need, mm_gemm_workspace_bytes((int)M, n[p], (int)K));
    b[p] = (const uint32_t*)W[p].data_ptr();
    s[p] = (const uint16_t*)S[p].data_ptr();
    c[p] = (uint16_t*)out[p].data_ptr();
  }
  at::Tensor ws = workspace(A, stream, need);
  const int rc = mm_fp4_gemm_multi((const uint16_t*)A.data_ptr(), 3, b, s, c, n, (int)M, (int)K,
                                   (int)g, ws.data_ptr(), (size_t)ws.numel(), (void*)stream);
  if (rc) fail(rc);
  return pybind11::make_tuple(out[0], out[1], out[2]);
}

// The gate/up pair: Marlin [K/8, N] words, or row-packed [N, K/8] ones.
pybind11::object gate_up(const at::Tensor& A, const at::Tensor& Wg, const at::Tensor& Sg,
                         const at::Tensor& Wu, const at::Tensor& Su, int64_t g, bool rows,
                         bool act, int64_t stream) {
  const auto [M, K] = plain_acts(A);
  if (M < 0 || g <= 0 || K % g != 0 || K % 8 != 0 || Wg.dim() != 2) return pybind11::none();
  const int dev = (int)A.get_device();
  const int64_t N = Wg.size(rows ? 0 : 1), d0 = rows ? N : K / 8, d1 = rows ? K / 8 : N;
  if (N <= 0 || N % 8 != 0 || !plain_words(Wg, dev, d0, d1) || !plain_words(Wu, dev, d0, d1) ||
      !plain(Sg, at::kHalf, dev, K / g, N) || !plain(Su, at::kHalf, dev, K / g, N))
    return pybind11::none();
  at::Tensor out = at::empty({M, act ? N : 2 * N}, A.options());
  at::Tensor ws = workspace(A, stream, mm_gemm_workspace_bytes((int)M, (int)(2 * N), (int)K));
  const auto fn = rows ? mm_fp4_gate_up_rowpacked : mm_fp4_gate_up;
  const int rc = fn((const uint16_t*)A.data_ptr(), (const uint32_t*)Wg.data_ptr(),
                    (const uint16_t*)Sg.data_ptr(), (const uint32_t*)Wu.data_ptr(),
                    (const uint16_t*)Su.data_ptr(), (uint16_t*)out.data_ptr(), (int)M, (int)N,
                    (int)K, (int)g, act, ws.data_ptr(), (size_t)ws.numel(), (void*)stream);
  if (rc) fail(rc);
  return pybind11::cast(out);
}

// Row-packed product: W [N, K/8], scales [K/g, N].
pybind11::object rowpacked(const at::Tensor& A, const at::Tensor& W, const at::Tensor& S,
                           int64_t g, int64_t stream) {
  const auto [M, K] = plain_acts(A);
  if (M < 0 || g <= 0 || K % g != 0 || K % 8 != 0 || W.dim() != 2) return pybind11::none();
  const int dev = (int)A.get_device();
  const int64_t N = W.size(0);
  if (N <= 0 || !plain_words(W, dev, N, K / 8) || !plain(S, at::kHalf, dev, K / g, N))
    return pybind11::none();
  at::Tensor out = at::empty({M, N}, A.options());
  at::Tensor ws = workspace(A, stream, mm_gemm_workspace_bytes((int)M, (int)N, (int)K));
  const int rc = mm_fp4_gemm_rowpacked(
      (const uint16_t*)A.data_ptr(), (const uint32_t*)W.data_ptr(), (const uint16_t*)S.data_ptr(),
      (uint16_t*)out.data_ptr(), (int)M, (int)N, (int)K, (int)g, 0, ws.data_ptr(),
      (size_t)ws.numel(), (void*)stream);
  if (rc) fail(rc);
  return pybind11::cast(out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "Per-call binding of libmmfp4's FP4 / INT4 GEMM entry points";
  m.def("gemm", &gemm, "C = A . dequant(B, S[, Z]) on the given stream", pybind11::arg("A"),
        pybind11::arg("B"), pybind11::arg("S"), pybind11::arg("Z"), pybind11::arg("SZ"),
        pybind11::arg("group_size"), pybind11::arg("stream"));
  m.def("qkv", &qkv, "mm_fp4_gemm_multi on plain operands, else None");
  m.def("gate_up", &gate_up, "mm_fp4_gate_up[_rowpacked] on plain operands, else None");
  m.def("rowpacked", &rowpacked, "mm_fp4_gemm_rowpacked on plain operands, else None");
  m.def("workspace", &workspace_for,
        "the zero-initialised workspace of (device index, raw stream), at least nbytes",
        pybind11::arg("device"), pybind11::arg("stream"), pybind11::arg("nbytes"));
  m.def("release_workspaces", &release_workspaces, "drop every cached workspace");
}
