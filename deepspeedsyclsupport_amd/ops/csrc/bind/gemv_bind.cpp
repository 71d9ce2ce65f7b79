// Module of the bf16 products of the hybrid decoders: decode products (up to 48 token rows), with activation epilogues, and those of
// short prompts; a batch's tables on their way to the device.
#include "bind_util.h"
#include "narrow_bind.h"

extern "C" {
int ds_skinny_gemm(const void*, const void*, const void*, const void*, const void*, const void*, void*, void*, int, int,
                   int, int, int, int, float, hipStream_t);
int ds_decode_gemm_ok(int, int);
int ds_decode_gemm(const void*, const void*, const void*, const void*, float, const void*, void*, int, int, int, int, int, float,
                   void*, hipStream_t);
int64_t ds_decode_gemm_scratch(int, int, int, int, int);
int ds_upload_most();
int ds_upload(const void*, void*, int, hipStream_t);
int ds_skinny_mfma_ok(int, int, int);
int ds_skinny_mfma(const void*, const void*, const void*, const void*, const void*, const void*, void*, void*, int, int,
                   int, int, int, int, float, hipStream_t);
}

namespace {
bool decode_linear_ok(int64_t M, int64_t K) {
  return M >= 1 && K % 8 == 0 && (M <= 8 || (M <= 16 && ds_skinny_mfma_ok((int)M, (int)K, 0)));
}
constexpr int CLAMPED_GLU = 5;  // DS_ACT_CLAMPED_GLU
constexpr int UNARY = 16;       // DS_ACT_UNARY

// x [M, K] . w [N, K]^T for M <= 16 bf16 rows: the vector kernel up to two rows (or where K does not tile), else MFMA.
// act: an activation code applied to the result. With a limit instead, w is a fused [gate | up] weight and the result its
// clamped gated activation [M, N / 2].
Tensor decode_linear(Tensor x, Tensor w, std::optional<double> glu_limit, std::optional<int64_t> act) {
  need(x, "x"); need(w, "w");
  const int64_t N = w.size(0), K = w.size(1), M = x.numel() / K;
  const bool glu = glu_limit.has_value();
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && x.size(-1) == K, "decode_linear");
  TORCH_CHECK(decode_linear_ok(M, K), "decode_linear: up to 8 rows with K % 8 == 0 (16 with K % 256 == 0)");
  TORCH_CHECK(!glu || N % 2 == 0, "decode_linear: [gate | up] rows");
  auto sizes = x.sizes().vec();
  sizes.back() = glu ? N / 2 : N;
  auto y = torch::empty(sizes, x.options());
  TORCH_CHECK(!(glu && act.has_value()), "decode_linear: one epilogue");
  const int code = glu ? CLAMPED_GLU : act.has_value() ? UNARY + (int)*act : 0;
  auto fn = M > 2 && ds_skinny_mfma_ok((int)M, (int)K, 0) ? ds_skinny_mfma : ds_skinny_gemm;
  check(fn(w.data_ptr(), x.data_ptr(), nullptr, nullptr, nullptr, nullptr, y.data_ptr(), nullptr, (int)M, (int)N, (int)K,
           0, glu ? 1 : 0, code, glu ? (float)*glu_limit : 0.f, stream()), "decode_linear");
  return y;
}

// The same for M <= 48 over a weight in the shuffled decode layout (ops/bf16_gemv.py: preshuffle16), w [N, K], K % 64 == 0;
// with a limit: N % 2 == 0
Tensor decode_linear_sh(Tensor x, Tensor wsh, int64_t N, std::optional<double> glu_limit, std::optional<int64_t> act) {
  need(x, "x"); need(wsh, "wsh");
  const int64_t K = x.size(-1), M = x.numel() / K, NB = (N + 15) / 16;
  const bool glu = glu_limit.has_value();
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && wsh.scalar_type() == at::kBFloat16 && wsh.numel() == NB * 16 * K &&
              ds_decode_gemm_ok((int)M, (int)K), "decode_linear_sh: up to 48 bf16 rows, K % 64 == 0");
  TORCH_CHECK(NB * K < ((int64_t)1 << 40) && N < ((int64_t)1 << 31) / 16, "decode_linear_sh: matrix too large");
  TORCH_CHECK(!(glu && act.has_value()), "decode_linear_sh: one epilogue");
  TORCH_CHECK(!glu || N % 2 == 0, "decode_linear_sh: [gate | up] rows");
  if ((uintptr_t)x.data_ptr() % 16) x = x.clone();  // (its rows go to LDS in pieces of 16 bytes as they lie)
  auto sizes = x.sizes().vec();
  sizes.back() = glu ? N / 2 : N;
  auto y = torch::empty(sizes, x.options());
  const int code = glu ? CLAMPED_GLU : act.has_value() ? UNARY + (int)*act : -1;
  Tensor part;
  if (const int64_t bytes = ds_decode_gemm_scratch((int)M, (int)N, (int)K, glu, 0))
    part = torch::empty({bytes}, x.options().dtype(at::kByte));
  check(ds_decode_gemm(x.data_ptr(), wsh.data_ptr(), nullptr, nullptr, 0.f, nullptr, y.data_ptr(), (int)M, (int)N, (int)K, glu, code,
                       glu ? (float)*glu_limit : 0.f, part.defined() ? part.data_ptr() : nullptr, stream()), "decode_linear_sh");
  return y;
}
// Whether decode_linear_sh takes a product and is the faster one. Every workgroup reads all of x, or its part of it: over deep
// contractions that are not cut the library's blocking wins from 17 rows on ([4096, 14336] uncut, us: 24 rows 30 here, 29 there; 40
// rows 41 and 33; cut 25 and 27.5), over short ones the stream up to its 48 ([14368, 4096] 32 rows 26 and 27, 48 rows 25 and 28.0; [2048,
// 5632], 40 rows: 11.4 and 15).
bool decode_linear_sh_ok(int64_t M, int64_t N, int64_t K, bool glu) {
  if (M > 48 || K >= ((int64_t)1 << 31) || !ds_decode_gemm_ok((int)M, (int)K) || (glu && N % 2)) return false;
  if (M <= 16) return true;
  if (glu && N % 32) return false;
  return ds_decode_gemm_scratch((int)M, (int)N, (int)K, glu, 0) > 0 || K <= 8192;
}

// 32-bit words on the host -> on the device, in a launch; the host's may change as soon as this returns. Longer ones: undefined
OptT upload(Tensor words, int64_t device) {
  TORCH_CHECK(words.device().is_cpu() && words.dim() == 1 && words.is_contiguous() && words.scalar_type() == at::kInt, "upload: int32 words on the host");
  if (words.numel() > ds_upload_most()) return std::nullopt;
  const c10::Device dev(c10::kCUDA, (c10::DeviceIndex)device);
  const c10::DeviceGuard guard(dev);
  auto out = torch::empty({words.numel()}, words.options().device(dev));
  check(ds_upload(words.data_ptr(), out.data_ptr(), (int)words.numel(), stream()), "upload");
  return out;
}
}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("decode_linear", &decode_linear, py::arg("x"), py::arg("w"), py::arg("glu_limit") = py::none(),
        py::arg("act") = py::none());
  m.def("decode_linear_ok", &decode_linear_ok);
  m.def("decode_linear_sh_ok", &decode_linear_sh_ok);
  m.def("decode_linear_sh", &decode_linear_sh, py::arg("x"), py::arg("wsh"), py::arg("N"),
        py::arg("glu_limit") = py::none(), py::arg("act") = py::none());
  m.def("linear", &linear_product);
  m.def("upload", &upload);
  m.def("upload_most", &ds_upload_most);
}
