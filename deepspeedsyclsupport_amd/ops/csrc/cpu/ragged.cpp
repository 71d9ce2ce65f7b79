// Index tables of one ragged batch (reference `inference/v2/ragged/ragged_wrapper.py:31-193` and its C++ counterpart
// `inference/v2/ragged/csrc/fast_host_buffer.cu`): a step of a few sequences is bound by the host, and of that the tables were a
// fifth when lists of integers were put together in Python (12 decodes of 600 tokens: 75 us a step; here 15).
#include <torch/extension.h>

#include <algorithm>
#include <optional>
#include <stdexcept>
#include <string>
#include <vector>

namespace {

using Ints = std::vector<int64_t>;
using torch::Tensor;

int64_t narrow(int64_t v) {
  if ((int32_t)v != v) throw std::overflow_error("ragged_tables: " + std::to_string(v) + " does not fit 32 bits");
  return v;
}

// See RaggedMeta (inference/model_implementations/transformer.py) for the tables. One array of 32-bit integers behind the 64-bit
// ones (logit rows, then the tokens), taken to the device by `upload` where it has up to `most` words (a decode step's: 12 sequences
// of 600 tokens 400), else by one copy from pinned memory, so that no step waits for the steps before it.
// -> (the tables in the order of RaggedMeta.build, logit rows, tokens or None, offsets, n_short, end of the long contexts, width of
// the block tables, whether the logit rows are all rows)
pybind11::tuple ragged_tables(const Ints& starts, const Ints& n_new, const std::vector<Ints>& blocks, int64_t n_decode, const Ints& slots,
                              const std::optional<Ints>& logit_rows, const std::vector<Tensor>& ids, const std::optional<c10::Device>& device,
                              int64_t short_tokens, int64_t step_tokens, int64_t state_chunk, const std::optional<pybind11::function>& upload,
                              int64_t most) {
  const size_t S = starts.size();
  TORCH_CHECK(S > 0 && n_new.size() == S && blocks.size() == S && (slots.empty() || slots.size() == S), "ragged_tables: one entry a sequence");
  Ints cu(S + 1, 0);
  size_t width = 1;
  for (size_t i = 0; i < S; ++i) {
    TORCH_CHECK(n_new[i] >= 0, "ragged_tables: token counts");
    cu[i + 1] = cu[i] + narrow(n_new[i]);
    narrow(cu[i + 1]);
    narrow(narrow(starts[i]) + n_new[i]);
    width = std::max(width, blocks[i].size());
  }
  const int64_t T = cu[S];
  std::vector<int32_t> flat;
  flat.reserve(2 * T + S * (width + 8) + T / 32 + 64);
  std::vector<int64_t> ends;
  auto put = [&](int64_t v) { flat.push_back((int32_t)narrow(v)); };
  auto part = [&] { ends.push_back((int64_t)flat.size()); };
  for (size_t i = 0; i < S; ++i)
    for (int64_t j = 0; j < n_new[i]; ++j) put(starts[i] + j);
  part();
  for (size_t i = 0; i < S; ++i)
    for (int64_t j = 0; j < n_new[i]; ++j) put((int64_t)i);
  part();
  for (int64_t v : starts) put(v);
  part();
  for (size_t i = 0; i < S; ++i) put(starts[i] + n_new[i]);
  part();
  for (int64_t v : cu) put(v);
  part();
  for (size_t i = (size_t)n_decode; i < S; ++i)
    for (int64_t b = 0; b * 128 < n_new[i]; ++b) {
      put((int64_t)i);
      put(b);
    }
  part();
  Ints last;
  if (logit_rows) last = *logit_rows;
  else
    for (size_t i = 0; i < S; ++i) last.push_back(cu[i + 1] - 1);
  for (int64_t v : last) put(v);
  part();
  for (const Ints& b : blocks) {
    for (int64_t v : b) put(v);
    flat.resize(flat.size() + width - b.size(), 0);
  }
  part();
  for (int64_t v : slots) put(v);
  part();
  // states: short portions go token by token, the others by chunks
  Ints chunk_seqs, chunks;
  if (!slots.empty())
    for (size_t i = 0; i < S; ++i) {
      if (n_new[i] <= step_tokens) {
        put((int64_t)i);
        continue;
      }
      chunk_seqs.push_back((int64_t)i);
      chunk_seqs.push_back((int64_t)chunks.size() / 2);
      for (int64_t c = 0; c * state_chunk < n_new[i]; ++c) {
        chunks.push_back((int64_t)i);
        chunks.push_back(c);
      }
    }
  part();
  for (int64_t v : chunk_seqs) put(v);
  part();
  for (int64_t v : chunks) put(v);
  part();
  // (a sequence is only counted as short if everything before it in the batch is)
  size_t n_short = S;
  for (size_t i = (size_t)n_decode; i < S; ++i)
    if (n_new[i] > short_tokens) {
      n_short = i;
      break;
    }
  int64_t kv = 0;
  put(0);
  for (size_t i = n_short; i < S; ++i) put(kv += starts[i] + n_new[i]);
  part();

  int64_t tokens = 0;
  for (const Tensor& t : ids) {
    TORCH_CHECK(t.device().is_cpu() && t.scalar_type() == at::kLong, "ragged_tables: 64-bit tokens on the host");
    tokens += t.numel();
  }
  const int64_t wide = (int64_t)last.size() + tokens;
  const bool cuda = device && device->is_cuda();
  const int64_t words = 2 * wide + (int64_t)flat.size();
  const bool small = cuda && upload && words <= most;
  Tensor buf = torch::empty({words}, torch::TensorOptions().dtype(at::kInt).pinned_memory(cuda && !small));
  int64_t* w = reinterpret_cast<int64_t*>(buf.data_ptr<int32_t>());
  w = std::copy(last.begin(), last.end(), w);
  for (const Tensor& t : ids) {
    const Tensor c = t.contiguous();
    w = std::copy(c.data_ptr<int64_t>(), c.data_ptr<int64_t>() + c.numel(), w);
  }
  std::copy(flat.begin(), flat.end(), buf.data_ptr<int32_t>() + 2 * wide);
  if (small) buf = (*upload)(buf, device->index()).cast<Tensor>();
  else if (cuda) buf = buf.to(*device, /*non_blocking=*/true);
  const Tensor head = buf.narrow(0, 0, 2 * wide).view(at::kLong);
  std::vector<Tensor> views;
  int64_t at = 2 * wide, from = 0;
  for (int64_t end : ends) {
    views.push_back(buf.narrow(0, at + from, end - from));
    from = end;
  }
  views[5] = views[5].view({-1, 2});
  views[7] = views[7].view({(int64_t)S, (int64_t)width});
  views[10] = views[10].view({-1, 2});
  views[11] = views[11].view({-1, 2});
  bool all = (int64_t)last.size() == T;
  for (int64_t i = 0; all && i < T; ++i) all = last[i] == i;
  pybind11::object toks = pybind11::none();
  if (!ids.empty()) toks = pybind11::cast(head.narrow(0, (int64_t)last.size(), tokens));
  return pybind11::make_tuple(views, head.narrow(0, 0, (int64_t)last.size()), toks, cu, n_short, kv, width, all);
}

// Smallest and largest of integer tensors on the host: (0, -1) where there are none
std::pair<int64_t, int64_t> int_range(const std::vector<Tensor>& ts) {
  int64_t lo = INT64_MAX, hi = INT64_MIN;
  for (const Tensor& t : ts) {
    TORCH_CHECK(t.device().is_cpu(), "int_range: host tensors");
    const Tensor c = t.scalar_type() == at::kLong ? t.contiguous() : t.to(at::kLong).contiguous();
    const int64_t* p = c.data_ptr<int64_t>();
    for (int64_t i = 0; i < c.numel(); ++i) {
      lo = std::min(lo, p[i]);
      hi = std::max(hi, p[i]);
    }
  }
  return lo > hi ? std::make_pair((int64_t)0, (int64_t)-1) : std::make_pair(lo, hi);
}

}  // namespace

void register_ragged(pybind11::module& m) {
  m.def("ragged_tables", &ragged_tables);
  m.def("int_range", &int_range);
}
