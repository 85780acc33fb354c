// A step's batch from the sequences' lists, put together in pinned memory and taken to the
// device in one copy. In Python every token's id, position and place in the cache was a step
// of the interpreter and every tensor a copy of its own, before the GPU had anything to do: a
// step of 6176 tokens of 8 prompts took 18.9 ms and takes 17.0, 27700 tokens of 200 texts 8.35
// and 7.36, 1600 tokens of 3 prompts beside 41 decoding sequences 3.45 and 2.83.
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>

namespace {

// Integers side by side, each array from a multiple of 64 bytes on
struct Layout {
  std::vector<std::pair<long, long>> at;  // first byte, bytes
  long size = 0;
  void add(long bytes) {
    at.emplace_back(size, bytes);
    size += (bytes + 63) / 64 * 64;
  }
};

struct Pack {
  torch::Tensor host;
  char* base;
  const Layout& layout;
  explicit Pack(const Layout& l)
      : host(torch::empty({l.size}, torch::dtype(torch::kUInt8).pinned_memory(true))),
        base((char*)host.data_ptr()), layout(l) {}
  int* i32(int k) { return (int*)(base + layout.at[k].first); }
  int64_t* i64(int k) { return (int64_t*)(base + layout.at[k].first); }
};

// plain ints of list[a:b]; false where there is anything else
bool read_ints(PyObject* list, long a, long b, int64_t* to) {
  const bool is_list = PyList_CheckExact(list);
  for (long i = a; i < b; ++i) {
    PyObject* o = is_list ? PyList_GET_ITEM(list, i) : PyTuple_GET_ITEM(list, i);
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    *to++ = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow) return false;
  }
  return true;
}

torch::Tensor part(const torch::Tensor& all, const Layout& l, int k, torch::ScalarType type) {
  return all.narrow(0, l.at[k].first, l.at[k].second).view(type);
}

}  // namespace

// The next tokens ``first[i] .. end[i]`` of sequences whose ids and pages are lists; the first
// ``prompts`` of them are portions of prompts, the others single tokens. -> [ids (int64),
// positions, cache slots], then of the prompts and of the others, where there are any, [block
// table, context lengths, state slots], then of the prompts where their tokens begin. None
// where a list holds anything but plain integers, or a token has no page.
py::object pack_batch(py::list ids, std::vector<long> first, std::vector<long> end,
                      py::list pages, std::vector<long> states, long prompts, long page,
                      torch::Device device) {
  const long n = first.size();
  TORCH_CHECK((long)ids.size() == n && (long)end.size() == n && (long)pages.size() == n &&
              (long)states.size() == n && prompts >= 0 && prompts <= n && page > 0);
  long tokens = 0, width[2] = {0, 0};
  for (long i = 0; i < n; ++i) {
    PyObject *t = ids[i].ptr(), *p = pages[i].ptr();
    if (!PyList_CheckExact(t) || !PyList_CheckExact(p) || first[i] < 0 || end[i] <= first[i] ||
        end[i] > PyList_GET_SIZE(t) || (end[i] + page - 1) / page > PyList_GET_SIZE(p) ||
        end[i] > INT_MAX)
      return py::none();
    tokens += end[i] - first[i];
    width[i >= prompts] = std::max(width[i >= prompts], (long)PyList_GET_SIZE(p));
  }
  if (tokens == 0) return py::none();
  const long count[2] = {prompts, n - prompts};
  Layout l;
  l.add(tokens * 8);
  l.add(tokens * 4);
  l.add(tokens * 4);
  for (int k = 0; k < 2; ++k)
    for (long each : {width[k], 1l, 1l}) l.add(count[k] * each * 4);
  l.add((prompts + 1) * 4);
  Pack pack(l);
  int64_t* id = pack.i64(0);
  int *pos = pack.i32(1), *slot = pack.i32(2), *begin = pack.i32(9);
  std::vector<int64_t> own;
  long done = 0;
  for (long i = 0; i < n; ++i) {
    const int k = i >= prompts;
    const long j = k ? i - prompts : i, len = end[i] - first[i], w = width[k];
    own.resize(PyList_GET_SIZE(pages[i].ptr()));
    if (!read_ints(ids[i].ptr(), first[i], end[i], id + done) ||
        !read_ints(pages[i].ptr(), 0, own.size(), own.data()))
      return py::none();
    int* row = pack.i32(3 + 3 * k) + j * w;
    for (long x = 0; x < w; ++x) row[x] = x < (long)own.size() ? (int)own[x] : 0;
    pack.i32(4 + 3 * k)[j] = (int)end[i];
    pack.i32(5 + 3 * k)[j] = (int)states[i];
    if (!k) begin[j] = (int)done;
    for (long t = 0; t < len; ++t) {
      const long at = first[i] + t;
      pos[done + t] = (int)at;
      slot[done + t] = (int)(own[at / page] * page + at % page);
    }
    done += len;
    if (!k) begin[j + 1] = (int)done;
  }
  const c10::DeviceGuard on(device);
  const auto all = pack.host.to(device, /*non_blocking=*/true);
  py::list out;
  out.append(part(all, l, 0, torch::kInt64));
  for (int k = 1; k < 3; ++k) out.append(part(all, l, k, torch::kInt32));
  for (int k = 0; k < 2; ++k) {
    if (!count[k]) continue;
    out.append(part(all, l, 3 + 3 * k, torch::kInt32).view({count[k], width[k]}));
    for (int x = 4; x < 6; ++x) out.append(part(all, l, x + 3 * k, torch::kInt32));
  }
  if (prompts) out.append(part(all, l, 9, torch::kInt32));
  return out;
}

// Texts as lists or tuples of ids, cut to ``most``, an empty one as [0] -> [ids (int64), where
// texts begin, positions]; None where they hold anything but plain integers.
py::object pack_texts(py::list texts, long most, torch::Device device) {
  const long n = texts.size();
  std::vector<long> len(n);
  long tokens = 0;
  for (long i = 0; i < n; ++i) {
    PyObject* t = texts[i].ptr();
    if (!PyList_CheckExact(t) && !PyTuple_CheckExact(t)) return py::none();
    tokens += len[i] = std::max(1l, std::min(most, (long)PySequence_Fast_GET_SIZE(t)));
  }
  if (tokens == 0 || most < 1 || tokens > INT_MAX) return py::none();
  Layout l;
  l.add(tokens * 8);
  l.add((n + 1) * 4);
  l.add(tokens * 4);
  Pack pack(l);
  int64_t* id = pack.i64(0);
  int *begin = pack.i32(1), *pos = pack.i32(2);
  long done = 0;
  for (long i = 0; i < n; ++i) {
    PyObject* t = texts[i].ptr();
    if (PySequence_Fast_GET_SIZE(t) == 0) id[done] = 0;
    else if (!read_ints(t, 0, len[i], id + done)) return py::none();
    begin[i] = (int)done;
    for (long x = 0; x < len[i]; ++x) pos[done + x] = (int)x;
    done += len[i];
  }
  begin[n] = (int)done;
  const c10::DeviceGuard on(device);
  const auto all = pack.host.to(device, /*non_blocking=*/true);
  py::list out;
  out.append(part(all, l, 0, torch::kInt64));
  for (int k = 1; k < 3; ++k) out.append(part(all, l, k, torch::kInt32));
  return out;
}
