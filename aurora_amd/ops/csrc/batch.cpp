// A step's batch from the sequences' lists, put together in pinned memory and taken to the
// device in one copy. In Python every token's id, position and place in the cache was a step
// of the interpreter and every tensor a copy of its own, before the GPU had anything to do: a
// step of 6176 tokens of 8 prompts took 18.9 ms and takes 17.0, 27700 tokens of 200 texts 8.35
// and 7.36, 1600 tokens of 3 prompts beside 41 decoding sequences 3.45 and 2.83. The rows of a
// captured decode step are staged here too: in Python 30 us of 1 sequence, 40 of 23, 65 of 96,
// with the GPU waiting, now 27, 30 and 40 (a third of it the caller's own).
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

bool is_int(int64_t x) { return x >= INT_MIN && x <= INT_MAX; }

torch::Tensor part(const torch::Tensor& all, const Layout& l, int k, torch::ScalarType type) {
  return all.narrow(0, l.at[k].first, l.at[k].second).view(type);
}

}  // namespace

// The next tokens ``first[i] .. end[i]`` of sequences whose ids and pages are lists; the first
// ``prompts`` of them are portions of prompts, the others single tokens. -> [ids (int64),
// positions, cache slots], then of the prompts and of the others, where there are any, [block
// table, context lengths, state slots], then of the prompts where their tokens begin. None
// where a list holds anything but plain integers, a token has no page, or a page, cache or state
// slot is not of 32 bits (Python says so).
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
    // (a page's last slot; with pages of 32 bits the product fits 64)
    for (const int64_t x : own)
      if (!is_int(x) || !is_int(x * page + page - 1)) return py::none();
    if (!is_int(states[i])) return py::none();
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

// Integers on the device, on their way when this returns: nothing waits for what runs there.
py::object pack_rows(py::list rows, torch::Device device) {
  const long n = py::len(rows);
  if (n == 0) return py::none();
  Layout l;
  l.add(n * 8);
  Pack pack(l);
  if (!read_ints(rows.ptr(), 0, n, pack.i64(0))) return py::none();
  const c10::DeviceGuard on(device);
  return py::cast(part(pack.host.to(device, /*non_blocking=*/true), l, 0, torch::kInt64));
}

// Stages the next token of every sequence in ``host``, pinned, and sends it to ``inputs``: the
// bucket's ids (int64, past the sequences those of ``ids``, which takes theirs first), then as
// int32 positions, cache slots, context lengths, state slots and block tables of ``width``
// pages. Rows past the sequences are idle: they write the scratch slot and touch no state. A
// table's row is written again only when its sequence's serial, generation or number of pages,
// ``keys`` [bucket, 3], has changed; keys of -1 are idle rows', of -2 nobody's. False, and nothing
// sent, where a sequence holds anything but lists of plain integers that fit: tables before its
// own may have been written, each with its key.
bool stage_decode(py::list seqs, torch::Tensor ids, torch::Tensor host, torch::Tensor keys,
                  torch::Tensor inputs, long width, long page, long scratch_page,
                  long scratch_slot) {
  const long n = seqs.size(), bucket = keys.size(0);
  for (auto* t : {&ids, &host, &keys})
    TORCH_CHECK(t->device().is_cpu() && t->dtype() == torch::kInt64 && t->is_contiguous());
  TORCH_CHECK(n <= bucket && bucket <= ids.numel() && keys.numel() == 3 * bucket && page > 0 &&
              width >= 0 && host.numel() == bucket + ((4 + width) * bucket + 1) / 2 &&
              inputs.numel() == host.numel() && inputs.dtype() == torch::kInt64);
  static PyObject* const names[] = {
      PyUnicode_InternFromString("token_ids"), PyUnicode_InternFromString("pages"),
      PyUnicode_InternFromString("state_slot"), PyUnicode_InternFromString("serial"),
      PyUnicode_InternFromString("page_gen")};
  struct Row {
    py::object pages;
    int64_t id, tokens, slot, state, key[3];
  };
  std::vector<Row> rows(n);
  for (long i = 0; i < n; ++i) {
    Row& r = rows[i];
    py::object got[5];
    for (int k = 0; k < 5; ++k) {
      got[k] = py::reinterpret_steal<py::object>(PyObject_GetAttr(seqs[i].ptr(), names[k]));
      if (!got[k]) throw py::error_already_set();
    }
    if (!PyList_CheckExact(got[0].ptr()) || !PyList_CheckExact(got[1].ptr())) return false;
    r.pages = got[1];
    r.tokens = PyList_GET_SIZE(got[0].ptr());
    r.key[2] = PyList_GET_SIZE(got[1].ptr());
    const long last = r.tokens - 1;
    int64_t at;
    py::list rest;
    for (int k = 2; k < 5; ++k) rest.append(got[k]);
    int64_t numbers[3];
    if (last < 0 || last / page >= r.key[2] || !is_int(r.tokens) ||
        !read_ints(got[0].ptr(), last, last + 1, &r.id) ||
        !read_ints(got[1].ptr(), last / page, last / page + 1, &at) ||
        !read_ints(rest.ptr(), 0, 3, numbers))
      return false;
    r.slot = is_int(at) ? at * page + last % page : INT64_MAX;
    r.state = numbers[0];
    r.key[0] = numbers[1];
    r.key[1] = numbers[2];
    if (!is_int(r.slot) || !is_int(r.state) || r.key[0] < 0) return false;
  }
  int64_t *id = ids.data_ptr<int64_t>(), *base = host.data_ptr<int64_t>(),
          *key = keys.data_ptr<int64_t>();
  int *pos = (int*)(base + bucket), *slot = pos + bucket, *ctx = slot + bucket,
      *state = ctx + bucket, *table = state + bucket;
  std::vector<int64_t> own;
  for (long i = 0; i < n; ++i) {  // all tables before anything else: they can still be refused
    const Row& r = rows[i];
    int64_t* k = key + 3 * i;
    if (k[0] == r.key[0] && k[1] == r.key[1] && k[2] == r.key[2]) continue;
    own.resize(std::min<long>(r.key[2], width));
    bool fit = read_ints(r.pages.ptr(), 0, own.size(), own.data());
    for (const int64_t x : own) fit = fit && is_int(x);
    k[0] = -2;  // of nobody while it is written
    if (!fit) return false;
    int* row = table + i * width;
    for (long x = 0; x < width; ++x) row[x] = x < (long)own.size() ? (int)own[x] : (int)scratch_page;
    std::copy(r.key, r.key + 3, k);
  }
  for (long i = n; i < bucket; ++i) {
    if (key[3 * i] == -1) continue;
    std::fill(table + i * width, table + (i + 1) * width, (int)scratch_page);
    std::fill(key + 3 * i, key + 3 * i + 3, -1);
  }
  for (long i = 0; i < bucket; ++i) {
    const bool there = i < n;
    if (there) id[i] = rows[i].id;
    base[i] = id[i];
    pos[i] = there ? (int)(rows[i].tokens - 1) : 0;
    slot[i] = there ? (int)rows[i].slot : (int)scratch_slot;
    ctx[i] = there ? (int)rows[i].tokens : 1;
    state[i] = there ? (int)rows[i].state : -1;
  }
  inputs.copy_(host, /*non_blocking=*/true);
  return true;
}
