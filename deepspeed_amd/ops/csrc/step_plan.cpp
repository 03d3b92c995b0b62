// The plan of a serving step over the paged pool (StepPlan in
// ops/paged_attention.py): where its new rows go and the work items of its
// attention. The first kernel that reads it waits for it on the host, so it is made
// here: 7 us for 1 request, 13 for 32 of 500 keys, where the same by numpy's calls
// on arrays as short takes 112 and 163.

#include <torch/extension.h>
#include <pybind11/numpy.h>

#include <algorithm>
#include <cstdint>
#include <unordered_map>
#include <utility>
#include <vector>

namespace {

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int64_t as_int(PyObject* o) {
  const Py_ssize_t v = PyNumber_AsSsize_t(o, PyExc_IndexError);
  if (v == -1 && PyErr_Occurred()) throw pybind11::error_already_set();
  return v;
}

struct Blocks { int64_t at, count; };     // of a slot
struct Run { int64_t row0, rows, keys, blocks; };
struct Tile { int64_t run, tile, end, splits; };

int64_t most_keys(const std::vector<Tile>& tiles) {
  int64_t most = 0;
  for (auto& t : tiles) most = std::max(most, t.end);
  return most;
}

}  // namespace

// slots and pos: request slot and position of every row; tables[slot]: its blocks.
// lines: ROUND of one and of two tiles, FEWER, KEYS, MIN_SPLIT, BLOCK, BLOCK_WORK,
// CUS, WORKGROUPS, LONG, STEP of one and of two tiles, HELD of these, BYTES, MERGE,
// MERGED, ROOMS. -> (int32 values on the host: items, runs, merges, blocks,
// places of the rows; items, runs, merges, whether any history is split, nq, index of
// the places).
std::tuple<at::Tensor, int64_t, int64_t, int64_t, bool, int64_t, int64_t>
step_plan(const pybind11::sequence& slots,
          pybind11::array_t<int64_t, pybind11::array::c_style |
                                         pybind11::array::forcecast> pos,
          const pybind11::object& tables, int64_t block_size, int64_t heads,
          int64_t kv_heads, const std::vector<int64_t>& lines, bool pinned) {
  namespace py = pybind11;
  const int64_t T = py::len(slots), G = kv_heads > 0 ? heads / kv_heads : 0;
  if (T < 1 || pos.ndim() != 1 || pos.size() != T || block_size < 1 || G < 1 ||
      lines.size() < 19)
    throw py::value_error("step_plan: a step of rows, each with its position");
  const int64_t* at = pos.data();
  const int64_t min_split = lines[4];

  // the rows' places and the runs of neighbours
  std::vector<int64_t> slot(T), offset(T);
  std::vector<int32_t> blocks;
  std::unordered_map<int64_t, Blocks> lists;
  Blocks list = {0, 0};
  std::vector<Run> runs;
  const py::list rows(slots);
  for (int64_t i = 0; i < T; ++i) {
    PyObject* s = PyList_GET_ITEM(rows.ptr(), i);
    slot[i] = as_int(s);
    const bool same = i && slot[i] == slot[i - 1];
    if (!same) {
      const auto [it, unseen] =
          lists.emplace(slot[i], Blocks{(int64_t)blocks.size(), 0});
      if (unseen) {
        const py::list own(py::object(
            tables[py::reinterpret_borrow<py::object>(s)]));
        for (Py_ssize_t j = 0; j < PyList_GET_SIZE(own.ptr()); ++j)
          blocks.push_back((int32_t)as_int(PyList_GET_ITEM(own.ptr(), j)));
        it->second.count = (int64_t)blocks.size() - it->second.at;
      }
      list = it->second;
    }
    offset[i] = list.at;
    if (at[i] < 0 || at[i] / block_size >= list.count)
      throw py::index_error("step_plan: a position outside its slot's blocks");
    if (!same || at[i] != at[i - 1] + 1)
      runs.push_back({i, 0, 0, offset[i]});
    ++runs.back().rows;
  }

  int64_t most = 0, least = T, work = 0;
  for (auto& r : runs) {
    r.keys = at[r.row0] + r.rows;
    most = std::max(most, r.rows);
    least = std::min(least, r.rows);
    work += r.rows * (r.keys - r.rows / 2);
  }
  // two tiles of 16 columns share the loads of a key tile where runs are long
  // enough, eight where they are longer
  int64_t nq = most * G > 16 ? 2 : 1;
  if (least * G >= lines[5] && kv_heads * G * work >= lines[6]) nq = 8;
  const int64_t width = 16 * nq;
  std::vector<Tile> tiles;
  int64_t total = 0;
  for (int64_t r = 0; r < (int64_t)runs.size(); ++r) {
    const int64_t columns = runs[r].rows * G;
    for (int64_t t = 0; t * width < columns; ++t) {
      const int64_t tok = std::min((t + 1) * width, columns) - 1;
      const int64_t end = runs[r].keys - runs[r].rows + tok / G + 1;
      tiles.push_back({r, t, end, 1});
      total += end;
    }
  }

  // split long histories until the chip is full
  const int64_t n = tiles.size();
  auto splits = [&](int64_t per) {
    int64_t sum = 0;
    for (auto& t : tiles) sum += t.splits = ceil_div(t.end, per);
    return sum;
  };
  int64_t grain = 32;
  if (nq == 8) {
    // the longest first; at most one round of workgroups, steps of 128
    std::stable_sort(tiles.begin(), tiles.end(),
                     [](const Tile& a, const Tile& b) { return a.end > b.end; });
    const int64_t room = lines[7] / kv_heads, longest = tiles[0].end;
    int64_t per = longest;
    grain = min_split;
    if (n < room) {
      per = std::max(min_split, total / room);
      while (per < longest && splits(per) > room) per += min_split;
    }
    splits(per);
  } else if (n * kv_heads < lines[8]) {
    int64_t full = lines[nq - 1];
    const int64_t fewer = lines[2];
    if (total * kv_heads < lines[3] * full) full = fewer;
    const int64_t room = ceil_div(n * kv_heads, full) * full / kv_heads;
    // half a split more for each tile, where it ends unevenly
    int64_t per = std::max(min_split,
                           total / std::max<int64_t>(1, room - n / 2));
    while (splits(per) > std::max(room, n)) per += per / 16;
    const bool few = block_size % 32 == 0 && n * kv_heads <= fewer &&
        (nq == 1 || runs.size() > 1);
    if (few) {
      // ns that the tiles take in these parts
      const int64_t held = lines[13 + nq], slots_ = held * lines[7];
      auto cost = [&] {
        int64_t count = 0, longest = 0;
        bool any = false;
        for (auto& t : tiles) {
          const int64_t step = ceil_div(ceil_div(t.end, t.splits), grain) * grain;
          count += ceil_div(t.end, step);
          longest = std::max(longest, std::min(step, t.end));
          any |= t.end > step;
        }
        count *= kv_heads;
        longest = ceil_div(longest, 128);
        const int64_t keys = total * kv_heads;
        const int64_t each = lines[8 + 2 * nq] +
            lines[9 + 2 * nq] * std::min(held, ceil_div(count, lines[7]));
        int64_t ns = std::max(longest * each, keys * 512 / lines[16]);
        if (count > slots_)     // behind one another
          ns = std::max(ns, (keys + 64 * count) / 128 * each / slots_ +
                                5 * longest * each / 8);
        return ns + (any ? lines[17] + lines[18] * count : 0);
      };
      int64_t best = most_keys(tiles);
      splits(best);
      int64_t least = cost();
      for (size_t i = 19; i < lines.size(); ++i) {
        if (lines[i] > full) continue;
        const int64_t cut = std::max(min_split, ceil_div(total * kv_heads, lines[i]));
        if (splits(cut) > room) continue;
        const int64_t ns = cost();
        if (ns < least) {
          least = ns;
          best = cut;
        }
      }
      splits(best);
    }
    // keys of the longest part, and rounds of two tiles' workgroups
    auto rounds = [&] {
      int64_t longest = 0, count = 0;
      for (auto& t : tiles) {
        longest = std::max(longest, ceil_div(t.end, t.splits));
        count += t.splits;
      }
      return std::make_pair(longest, ceil_div(count * kv_heads, fewer));
    };
    if (nq == 2 && !few) {
      const auto [longest, k] = rounds();
      if (k > 1 && longest > lines[9] &&
          10 * total * kv_heads < 7 * k * fewer * longest) {
        const auto before = tiles;
        splits(std::max(min_split, total * kv_heads / lines[8]));
        const auto [longest2, k2] = rounds();
        if (longest2 * k2 >= longest * k) tiles = before;
      }
    }
  }
  int64_t items = 0;
  bool any = false;
  for (auto& t : tiles) {
    const int64_t step = ceil_div(ceil_div(t.end, t.splits), grain) * grain;
    t.splits = ceil_div(t.end, step);
    items += t.splits;
    any |= t.splits > 1;
  }

  const int64_t head = 4 * items + 4 * (int64_t)runs.size() + 2 * n +
                       (int64_t)blocks.size();
  auto out = at::empty({head + T},
                       at::TensorOptions().dtype(at::kInt).pinned_memory(pinned));
  int32_t* p = out.data_ptr<int32_t>();
  for (auto& t : tiles) {
    const int64_t step = ceil_div(ceil_div(t.end, t.splits), grain) * grain;
    for (int64_t lo = 0; lo < t.end; lo += step) {
      const int64_t hi = std::min(lo + step, t.end);
      *p++ = (int32_t)t.run;
      *p++ = (int32_t)t.tile;
      *p++ = (int32_t)lo;
      *p++ = (int32_t)(t.splits == 1 ? -hi : hi);
    }
  }
  for (auto& r : runs)
    for (int64_t v : {r.row0, r.rows, r.keys, r.blocks}) *p++ = (int32_t)v;
  int64_t before = 0;
  for (auto& t : tiles) {
    *p++ = (int32_t)before;
    *p++ = (int32_t)t.splits;
    before += t.splits;
  }
  p = std::copy(blocks.begin(), blocks.end(), p);
  for (int64_t i = 0; i < T; ++i)
    *p++ = (int32_t)(blocks[offset[i] + at[i] / block_size] * block_size +
                     at[i] % block_size);
  return {out, items, (int64_t)runs.size(), n, any, nq, head};
}
