// The even-share line's integer logic (csrc/even_line.h) on the host: 64 lanes
// in lockstep as fibers, walking every share of a batch whose row lengths may
// change under the walk.  usage: even_line_host; exit status 1 and a line on
// stderr at the first rule broken.
#include <ucontext.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <memory>
#include <random>
#include <tuple>
#include <vector>

#define __device__
#define __forceinline__ inline
using std::max;
using std::min;

// ------------------------------------------------------------ lane emulation
namespace {
constexpr int kLanes = 64, kStack = 64 << 10;
ucontext_t g_main, g_lane[kLanes];
int g_cur;
bool g_done[kLanes];
int64_t g_slot[2][kLanes];
int g_parity[kLanes];
int g_calls[kLanes];       // collectives of this launch, per lane
int g_phase_at = 1 << 30;  // the lengths change after this many readlanes
int g_reads[kLanes];
std::function<void(int)> g_body;
std::vector<std::unique_ptr<char[]>> g_stacks;

[[noreturn]] void fail(const char* what) {
  std::fprintf(stderr, "even_line_host: %s\n", what);
  std::exit(1);
}

void next_lane() {
  const int from = g_cur;
  for (int i = 1; i <= kLanes; ++i) {
    const int to = (from + i) % kLanes;
    if (g_done[to]) continue;
    g_cur = to;
    if (to != from) swapcontext(&g_lane[from], &g_lane[to]);
    return;
  }
  setcontext(&g_main);
}

// every lane's value of this collective
const int64_t* gather(int64_t mine) {
  const int lane = g_cur, p = g_parity[lane];
  if (++g_calls[lane] > 1 << 20) fail("a wave does not come to an end");
  g_slot[p][lane] = mine;
  g_parity[lane] ^= 1;
  next_lane();
  return g_slot[p];
}

void entry() {
  g_body(g_cur);
  g_done[g_cur] = true;
  next_lane();
}

void run_wave(const std::function<void(int)>& body) {
  g_body = body;
  if (g_stacks.empty())
    for (int i = 0; i < kLanes; ++i) g_stacks.emplace_back(new char[kStack]);
  for (int i = 0; i < kLanes; ++i) {
    g_done[i] = false;
    g_parity[i] = g_calls[i] = g_reads[i] = 0;
    getcontext(&g_lane[i]);
    g_lane[i].uc_stack.ss_sp = g_stacks[i].get();
    g_lane[i].uc_stack.ss_size = kStack;
    g_lane[i].uc_link = nullptr;
    makecontext(&g_lane[i], entry, 0);
  }
  g_cur = 0;
  swapcontext(&g_main, &g_lane[0]);
}
}  // namespace

inline int __builtin_amdgcn_readlane(int x, int lane) {
  const int y = static_cast<int>(gather(x)[lane]);
  ++g_reads[g_cur];
  return y;
}
inline uint64_t __ballot(bool x) {
  const int64_t* all = gather(x);
  uint64_t m = 0;
  for (int i = 0; i < kLanes; ++i) m |= static_cast<uint64_t>(all[i] != 0) << i;
  return m;
}
// row_shr:n (0x111..) and row_bcast15 / 31 (0x142 / 0x143), as even_scan uses them
inline int __builtin_amdgcn_update_dpp(int old, int src, int ctrl, int row_mask, int, bool) {
  const int lane = g_cur;
  const int64_t* all = gather(src);
  if (!(row_mask >> (lane / 16) & 1)) return old;
  if (ctrl == 0x142) return lane >= 16 ? static_cast<int>(all[lane / 16 * 16 - 1]) : old;
  if (ctrl == 0x143) return lane >= 32 ? static_cast<int>(all[31]) : old;
  const int n = ctrl - 0x110;
  return lane % 16 >= n ? static_cast<int>(all[lane - n]) : 0;
}

namespace {
// what the lengths are before and after the change; kBase stands for either
std::vector<int> g_lens[2];
const char kBase = 0;
int length(int64_t i) {
  const auto& v = g_lens[g_reads[g_cur] >= g_phase_at];
  if (i < 0 || i >= static_cast<int64_t>(v.size())) fail("a length is read past the batch");
  return v[i];
}
}  // namespace

namespace fd {
inline int load_index(const void*, int64_t i, int) { return length(i); }
inline int load_index_uniform(const void*, int64_t i, int) { return length(i); }
}  // namespace fd

#include "even_line.h"

using namespace fd;

namespace {

struct Walk {
  std::vector<EvenCut> cuts;  // per share
  std::vector<char> written;
  std::map<std::tuple<int, int, int>, int> tiles;  // (kv head, row, tile) -> times attended
  std::map<std::pair<int, int>, std::vector<int>> slots;  // (kv head, row) -> partial slots
};

// Every share's walk, as even_decode_kernel drives it (wave by wave).
template <int UNIT, int W>
Walk walk(const EvenArgs& a) {
  Walk r;
  r.cuts.assign(a.shares, EvenCut{a.num_seqs - 1, a.hkv - 1, 1 << 20, 0});  // a cut that nobody writes may hold anything
  r.written.assign(a.shares, 0);
  const int64_t rows = static_cast<int64_t>(a.num_seqs) * a.hkv;
  for (int block = 0; block < a.shares; ++block) {
    for (int wave = 0; wave < W; ++wave) {
      run_wave([&](int lane) {
        const int mine = lane < a.num_seqs ? length(lane) : 0;
        int share, per, share_end, pad;
        EvenCursor cur = even_first<false>(a, block, lane, min(max(mine, 0), a.cap), share, per, share_end, pad);
        const bool says = lane == 0;
        if (share < 0 || share >= a.shares) fail("share out of range");
        auto write = [&](const EvenCut& c) {
          if (!says || wave != 0) return;
          if (r.written[share]++) fail("a share's cut is written twice");
          r.cuts[share] = c;
        };
        if (!cur.valid) {
          write(EvenCut{0, 0, 0, 0});
          return;
        }
        even_enter<UNIT, W>(cur, wave);
        int64_t segments = 0;
        while (cur.valid) {
          if (cur.b < 0 || cur.b >= a.num_seqs || cur.kvh < 0 || cur.kvh >= a.hkv) fail("row out of range");
          if (cur.unit < 0 || cur.t_begin < 0) fail("unit out of range");
          if (even_last<W>(cur)) {
            if (++segments > rows) fail("a share walks more rows than there are");
            const int tiles = even_tiles(cur.len, pad);
            const bool whole = cur.t_begin == 0 && cur.t_end == tiles;
            if (cur.left == 0) write(even_cut(cur, tiles, whole, share, share_end, per));
            if (says && wave == 0) {
              for (int t = cur.t_begin; t < cur.t_end; ++t) ++r.tiles[{cur.kvh, cur.b, t}];
              if (!whole) r.slots[{cur.kvh, cur.b}].push_back(2 * share + (cur.t_begin == 0 ? 1 : 0));
            }
          }
          cur = even_next<false, UNIT, W>(a, cur, pad, wave);
        }
      });
    }
  }
  return r;
}

EvenArgs args(int rows, int hkv, int cap, int shares) {
  EvenArgs a{};
  a.sl = &kBase;
  a.num_seqs = rows;
  a.hkv = hkv;
  a.cap = cap;
  a.shares = shares;
  a.min_tiles = 4;
  a.sls = 1;
  return a;
}

// The merges of a launch may read any slot up to 2 * (shares + early); whatever
// a cut holds, they stay inside it and store a row of the batch.
void check_merges(const EvenArgs& a, const std::vector<EvenCut>& cuts) {
  for (int s = 0; s < a.shares; ++s) {
    const int parts = even_cut_parts(cuts[s], s, a.shares, a.num_seqs, a.hkv);
    if (parts <= 0) continue;
    if (cuts[s].b < 0 || cuts[s].b >= a.num_seqs || cuts[s].kvh < 0 || cuts[s].kvh >= a.hkv)
      fail("a merge stores a row out of range");
    if (s + parts > a.shares) fail("a merge reads parts past the last share");
  }
}

template <int UNIT, int W>
Walk check(std::vector<int> before, std::vector<int> after, int phase_at, int hkv, int cap, int shares) {
  g_lens[0] = before;
  g_lens[1] = after;
  g_phase_at = phase_at;
  const int rows = static_cast<int>(before.size());
  const EvenArgs a = args(rows, hkv, cap, shares);
  const Walk w = walk<UNIT, W>(a);
  check_merges(a, w.cuts);
  for (int s = 0; s < shares; ++s)
    if (before == after && !w.written[s]) fail("a share's cut is not written");
  if (before != after) return w;
  // unchanged lengths: every tile attended once, and every cut row's parts are its merge's
  std::map<std::pair<int, int>, std::vector<int>> merged;
  for (int s = 0; s < shares; ++s) {
    const int parts = even_cut_parts(w.cuts[s], s, shares, rows, hkv);
    auto& to = merged[{w.cuts[s].kvh, w.cuts[s].b}];
    for (int j = 0; j < parts; ++j) to.push_back(j == 0 ? 2 * s + 1 : 2 * (s + j));
    if (to.empty()) merged.erase({w.cuts[s].kvh, w.cuts[s].b});
  }
  for (auto x : w.slots) {
    std::sort(x.second.begin(), x.second.end());
    auto got = merged[x.first];
    std::sort(got.begin(), got.end());
    if (got != x.second) fail("a row's parts are not what its merge reads");
    merged.erase(x.first);
  }
  if (!merged.empty()) fail("a merge of a row that no share cut");
  for (int h = 0; h < hkv; ++h)
    for (int b = 0; b < rows; ++b) {
      const int tiles = even_tiles(min(max(before[b], 0), cap), 0);
      for (int t = 0; t < tiles; ++t) {
        const auto it = w.tiles.find({h, b, t});
        if (it == w.tiles.end() || it->second != 1) fail("a tile is not attended once");
      }
    }
  return w;
}

}  // namespace

int main() {
  std::mt19937 rng(7);
  auto some = [&](int n, int hi) {
    std::vector<int> v(n);
    for (int& x : v) x = static_cast<int>(rng() % (hi + 1));
    return v;
  };
  for (int rows : {1, 3, 64, 65, 130, 300, 4100}) {
    const int hkv = rows > 1000 ? 1 : 2, shares = rows == 3 ? 12 : 16, hi = rows > 1000 ? 40 : 900;
    const std::vector<int> lens = some(rows, hi), none(rows, 0), full(rows, 1 << 20);
    check<16, 8>(lens, lens, 1 << 30, hkv, 960, shares);
    check<32, 4>(lens, lens, 1 << 30, hkv, 960, shares);
    // the lengths change after the scan (1), after the share's lane is known (2), while the rows are walked
    for (int at : {1, 2, 3, 5, 6}) {
      if (rows > 1000 && at > 2) break;
      for (const auto& later : {none, full, some(rows, hi)}) {
        check<16, 4>(lens, later, at, hkv, 960, shares);
        check<16, 4>(none, later, at, hkv, 960, shares);
        check<16, 4>(full, later, at, hkv, 960, shares);
      }
    }
    if (rows > 100) continue;
    // a short line: rows in shares of their own
    const std::vector<int> few = some(rows, 150);
    const Walk own = check<16, 8>(few, few, 1 << 30, hkv, 960, 2 * hkv * rows);
    for (const auto& x : own.slots)
      if (even_tiles(few[x.first.second], 0) <= 4) fail("a row of one share is cut");
  }
  // a merge's record that no workgroup of the launch wrote
  const EvenArgs a = args(5, 2, 960, 16);
  for (int i = 0; i < 20000; ++i) {
    std::vector<EvenCut> cuts(a.shares);
    for (EvenCut& c : cuts)
      c = EvenCut{static_cast<int32_t>(rng()), static_cast<int32_t>(rng()), static_cast<int32_t>(rng()), 0};
    for (EvenCut& c : cuts)
      if (i & 1) c.b = static_cast<int32_t>(rng() % 7) - 1, c.kvh = static_cast<int32_t>(rng() % 4) - 1;
    check_merges(a, cuts);
  }
  std::puts("ok");
  return 0;
}
