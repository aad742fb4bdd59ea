// Text chunking for ingestion (N11 in SURVEY.md §2.B):
//  * token windows with overlap (SentenceTransformersTokenTextSplitter semantics: windows of
//    tokens_per_chunk tokens advancing by tokens_per_chunk - overlap —
//    RetrievalAugmentedGeneration/common/utils.py:321-331);
//  * recursive character splitting (separator hierarchy "\n\n", "\n", " ", "" with chunk
//    size / overlap in characters — the 1000/100 splitter of
//    examples/multimodal_rag/vectorstore/vectorstore_updater.py:49-59).
// And the inputs of an encoder's packed batch, from lists of token ids into one staging buffer.
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

namespace py = pybind11;

namespace {

std::vector<std::pair<int, int>> token_windows(int n_tokens, int chunk, int overlap) {
  std::vector<std::pair<int, int>> out;
  if (chunk <= 0) return out;
  if (overlap >= chunk) overlap = chunk - 1;
  const int step = chunk - overlap;
  for (int s = 0; s < n_tokens; s += step) {
    const int e = std::min(n_tokens, s + chunk);
    out.push_back({s, e});
    if (e == n_tokens) break;
  }
  return out;
}

void split_rec(const std::string& text, const std::vector<std::string>& seps, size_t sep_i,
               std::vector<std::string>& pieces, size_t chunk) {
  if (text.size() <= chunk) {
    if (!text.empty()) pieces.push_back(text);
    return;
  }
  if (sep_i >= seps.size() || seps[sep_i].empty()) {
    for (size_t i = 0; i < text.size(); i += chunk) pieces.push_back(text.substr(i, chunk));
    return;
  }
  const std::string& sep = seps[sep_i];
  size_t start = 0;
  while (start <= text.size()) {
    size_t p = text.find(sep, start);
    std::string part = text.substr(start, p == std::string::npos ? std::string::npos : p - start);
    if (p != std::string::npos) part += sep;  // keep the separator with the left piece
    if (!part.empty()) {
      if (part.size() > chunk)
        split_rec(part, seps, sep_i + 1, pieces, chunk);
      else
        pieces.push_back(part);
    }
    if (p == std::string::npos) break;
    start = p + sep.size();
  }
}

// Greedy merge of pieces into chunks of <= chunk chars with ~overlap chars carried over.
std::vector<std::string> char_split(const std::string& text, int chunk, int overlap,
                                    std::vector<std::string> seps) {
  if (seps.empty()) seps = {"\n\n", "\n", " ", ""};
  std::vector<std::string> pieces;
  split_rec(text, seps, 0, pieces, (size_t)chunk);
  std::vector<std::string> out;
  std::vector<std::string> cur;
  size_t cur_len = 0;
  auto flush = [&]() {
    std::string s;
    for (auto& p : cur) s += p;
    // strip
    size_t a = s.find_first_not_of(" \n\t\r"), b = s.find_last_not_of(" \n\t\r");
    if (a != std::string::npos) out.push_back(s.substr(a, b - a + 1));
  };
  for (auto& p : pieces) {
    if (cur_len + p.size() > (size_t)chunk && !cur.empty()) {
      flush();
      while (!cur.empty() && (cur_len > (size_t)overlap || cur_len + p.size() > (size_t)chunk)) {
        cur_len -= cur.front().size();
        cur.erase(cur.begin());
      }
    }
    cur.push_back(p);
    cur_len += p.size();
  }
  if (!cur.empty()) flush();
  return out;
}

// The batch seqs[order[0]], seqs[order[1]], ... into int32 words of `buf`: at 0 the places `order` (int64), at cu_at the offsets of
// the sequences, at ids_at, pos_at and (types given) types_at a value a token. Returns (longest sequence, least and largest id, least
// and largest type). What isn't a list of whole numbers of 32 bits, or does not fit, raises TypeError, OverflowError or ValueError.
py::tuple pack_tokens(const std::vector<py::object>& seqs, const std::vector<int64_t>& order, const py::object& types, py::buffer buf,
                      int64_t cu_at, int64_t ids_at, int64_t pos_at, int64_t types_at, int64_t tokens) {
  py::buffer_info info = buf.request(true);
  const int64_t n = (int64_t)order.size(), size = info.size;
  if (info.itemsize != 4 || info.ndim != 1 || info.strides[0] != 4) throw py::value_error("pack_tokens: one run of 32-bit words");
  const bool typed = !types.is_none();
  auto room = [&](int64_t at, int64_t len) {
    if (at < 0 || at > size || len > size - at) throw py::value_error("pack_tokens: a piece outside the buffer");
  };
  room(0, 2 * n);
  room(cu_at, n + 1);
  room(ids_at, tokens);
  room(pos_at, tokens);
  if (typed) room(types_at, tokens);
  int32_t* const base = static_cast<int32_t*>(info.ptr);
  auto list = [](const py::handle& o) {
    PyObject* f = PySequence_Fast(o.ptr(), "pack_tokens: a sequence of token ids");
    if (f == nullptr) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(f);
  };
  auto copy = [](PyObject* f, int64_t len, int32_t* to, int32_t& lo, int32_t& hi) {
    for (int64_t i = 0; i < len; ++i) {
      const long v = PyLong_AsLong(PySequence_Fast_GET_ITEM(f, i));
      if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
      if (v < INT32_MIN || v > INT32_MAX) throw py::value_error("pack_tokens: more than 32 bits");
      to[i] = (int32_t)v;
      lo = std::min(lo, to[i]);
      hi = std::max(hi, to[i]);
    }
  };
  py::object tlists = typed ? list(types) : py::object();
  int64_t at = 0, longest = 0;
  int32_t lo = INT32_MAX, hi = INT32_MIN, tlo = INT32_MAX, thi = INT32_MIN;
  base[cu_at] = 0;
  for (int64_t b = 0; b < n; ++b) {
    const int64_t i = order[b];
    if (i < 0 || i >= (int64_t)seqs.size()) throw py::value_error("pack_tokens: no such sequence");
    std::copy_n(reinterpret_cast<const int32_t*>(&i), 2, base + 2 * b);
    const py::object f = list(seqs[i]);
    const int64_t len = PySequence_Fast_GET_SIZE(f.ptr());
    if (len > tokens - at) throw py::value_error("pack_tokens: more tokens than said");
    copy(f.ptr(), len, base + ids_at + at, lo, hi);
    if (typed) {
      if (i >= PySequence_Fast_GET_SIZE(tlists.ptr())) throw py::value_error("pack_tokens: a sequence without types");
      const py::object t = list(PySequence_Fast_GET_ITEM(tlists.ptr(), i));
      if (PySequence_Fast_GET_SIZE(t.ptr()) != len) throw py::value_error("pack_tokens: one type a token");
      copy(t.ptr(), len, base + types_at + at, tlo, thi);
    }
    for (int64_t k = 0; k < len; ++k) base[pos_at + at + k] = (int32_t)k;
    at += len;
    base[cu_at + b + 1] = (int32_t)at;
    longest = std::max(longest, len);
  }
  return py::make_tuple(longest, lo, hi, tlo, thi);
}

}  // namespace

void register_text(py::module_& m) {
  m.def("token_windows", &token_windows, py::arg("n_tokens"), py::arg("chunk"),
        py::arg("overlap"));
  m.def("char_split", &char_split, py::arg("text"), py::arg("chunk_size"), py::arg("overlap"),
        py::arg("separators") = std::vector<std::string>{});
  m.def("pack_tokens", &pack_tokens);
}
