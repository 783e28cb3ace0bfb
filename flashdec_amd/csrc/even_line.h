// The even-share kernel's line of tiles: which part of it a workgroup takes and
// how its waves walk that part.  Integer logic over the rows' lengths only; the
// includer brings the index loads and the lane operations (tests/native runs it
// on the host).
//
// Each wave reads the lengths for itself, some of them twice, so a caller that
// changes them under the launch (the next step's update on another stream) may
// show it different ones.  Its rows are then wrong, as any kernel's would be, but
// every walk ends, and every row, slot and part stays in range.
#pragma once

namespace fd {

// Launch arguments of both kernels, strides in elements.  The host checks that
// every stride fits 32 bits.
struct EvenArgs {
  const void* q;
  void* k;
  void* v;
  const void* bt;
  const void* sl;
  const void* ak;
  const void* av;
  const void* slot;
  int32_t num_blocks;
  int32_t qs0, qs1, ks0, ks1, ks2, vs0, vs1, vs2, bts0, bts1;
  int32_t aks0, aks1, avs0, avs1, sls, slots;
  int32_t num_seqs, hkv, group, width, cap;
  int32_t shares, min_tiles;
  int32_t full_tiles, full_per, full_used;  // tiles of a full table row; the plan where every row is full
  int32_t bt_i64, sl_i64, slot_i64;
  float scale_log2;
};

// The row that a share's last segment starts but does not finish: its parts are
// that segment (the share's slot 1) and the first segments of the parts - 1
// shares after it (their slots 0).
struct EvenCut {
  int32_t b, kvh;
  int32_t parts;  // 0: no such row
  int32_t unused;
};

// Tokens row b attends: 0 for an empty row, a padding slot (fused append), at
// most what its block-table row holds.
template <bool FUSE, bool UNIFORM>
__device__ __forceinline__ int even_row_len(const EvenArgs& a, int b) {
  auto at = [&](const void* base, int64_t i, int i64) {
    return UNIFORM ? load_index_uniform(base, i, i64) : load_index(base, i, i64);
  };
  int n = at(a.sl, static_cast<int64_t>(b) * a.sls, a.sl_i64);
  if constexpr (FUSE) {
    const int slot = at(a.slot, static_cast<int64_t>(b) * a.slots, a.slot_i64);
    n = slot < 0 ? 0 : n;
  }
  n = n > 0 ? n : 0;
  return n < a.cap ? n : a.cap;
}

// 32-token tiles of a row; an empty row counts one (nothing in it attends, and
// its zero output row is stored by whoever walks it).  In a short batch's line
// (pad = min_tiles - 1, even_first) every row counts whole min_tiles, the last of
// them without tokens.
__device__ __forceinline__ int even_tiles(int len, int pad) { return (max(1, (len + 31) >> 5) + pad) & ~pad; }

// Where a wave is on its share's line (wave-uniform).
struct EvenCursor {
  int b, kvh;          // row, KV head
  int len;             // tokens row b attends
  int t_begin, t_end;  // the segment's tiles within the row
  int unit;            // this wave's unit of the segment
  int u_end;           // units end here (unit >= u_end: the wave has none, all of it is masked)
  int phase;           // units of the share before this segment, mod W
  int left;            // tiles of the share after this segment
  int valid;
};

// A wave without units in the segment takes one past its end, whose loads are
// empty and whose tokens are masked: every step computes the unit it loaded.
template <int UNIT, int W>
__device__ __forceinline__ void even_enter(EvenCursor& c, int wave) {
  constexpr int UPT = 32 / UNIT;
  c.u_end = min(c.t_end * UPT, (c.len + UNIT - 1) / UNIT);
  c.unit = c.t_begin * UPT + ((wave - c.phase) & (W - 1));
}

template <int W>
__device__ __forceinline__ bool even_last(const EvenCursor& c) {
  return c.unit + W >= c.u_end;
}

// The wave's next step on the line: its next unit of this segment, else the
// next segment.
template <bool FUSE, int UNIT, int W>
__device__ __forceinline__ EvenCursor even_next(const EvenArgs& a, EvenCursor c, int pad, int wave) {
  constexpr int UPT = 32 / UNIT;
  if (c.valid && !even_last<W>(c)) {
    c.unit += W;
    return c;
  }
  if (!c.valid || c.left <= 0) {
    c.valid = 0;
    return c;
  }
  c.phase = (c.phase + max(c.u_end - c.t_begin * UPT, 0)) & (W - 1);
  if (++c.b == a.num_seqs) {
    c.b = 0;
    if (++c.kvh == a.hkv) {  // only if a length changed under the launch
      c.valid = 0;
      return c;
    }
  }
  c.len = even_row_len<FUSE, true>(a, c.b);
  c.t_begin = 0;
  c.t_end = min(even_tiles(c.len, pad), c.left);
  c.left -= c.t_end;
  even_enter<UNIT, W>(c, wave);
  return c;
}

// Inclusive sum over the wave's lanes: shifts within each 16-lane row (DPP
// row_shr), then the row totals carried across (row_bcast), six VALU steps
// with no LDS round trip.
__device__ __forceinline__ int even_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

// Workgroup to share.  The hardware deals consecutive workgroups round the 8
// XCDs.  Each XCD takes a run of consecutive shares (rows and their tables
// through one L2), and a batch too small for the whole grid is spread over all
// of them; the workgroups left over take the ids after it.
__device__ __forceinline__ int even_share(int block, int shares, int used) {
  if (shares & 7) return block;
  const int each = (used + 7) >> 3;
  const int x = block & 7, i = block >> 3;
  return i < each ? x * each + i : block;
}

// The share's first segment and the batch's plan, from the row lengths (every
// wave computes them by itself: no barrier).  Lane l adds up rows [l*n, l*n+n)
// and a scan over the lanes finds the one holding the share's first tile.
template <bool FUSE>
__device__ __forceinline__ EvenCursor even_first(const EvenArgs& a, int block, int lane, int lane_len, int& share,
                                                 int& per, int& share_end, int& pad) {
  const int n = (a.num_seqs + 63) >> 6;  // rows per lane
  const int r0 = lane * n;
  const int short_pad = a.min_tiles - 1;  // min_tiles is a power of two
  int mine = 0, padded = 0;
  int len = 0;  // of the lane's row, when it has one
  if (n == 1) {
    len = lane_len;
    mine = lane < a.num_seqs ? even_tiles(len, 0) : 0;
    padded = (mine + short_pad) & ~short_pad;
  }
  for (int i = 0; n > 1 && i < n; i += 4) {
    int t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = r0 + i + j;
      const bool in = i + j < n && r < a.num_seqs;
      t[j] = even_tiles(even_row_len<FUSE, false>(a, in ? r : 0), 0);
      t[j] = in ? t[j] : 0;
    }
    mine += (t[0] + t[1]) + (t[2] + t[3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) padded += (t[j] + short_pad) & ~short_pad;
  }
  int incl = even_scan(mine);
  int total = __builtin_amdgcn_readlane(incl, 63);
  pad = 0;
  // A short batch: shares of min_tiles (or twice that) end where rows do, so that
  // no wave walks the ends of several rows one after the other and a row of one
  // share is not cut.  The tiles without tokens take no time, and at that length
  // there are workgroups to spare.  MI355X, graph replays, us/call as one line /
  // with rows padded / row kernel, Hq 16, Hkv 2, tables of 2048 to 4096 tokens: 48
  // rows of 1 .. 256 tokens 14.4 / 9.0 / 11.6, of 8 .. 2048 16.6 / 13.7 / 18.4; 100
  // rows of 256 13.9 / 12.0 / 15.6, of 4 .. 1024 18.9 / 14.0 / 18.0.  (Up to one
  // round of min_tiles instead of two: 9.0, 16.6, 14.1 and 18.9.)
  if (total * a.hkv <= 2 * a.shares * a.min_tiles) {
    pad = short_pad;
    mine = padded;
    incl = even_scan(mine);
    total = __builtin_amdgcn_readlane(incl, 63);
  }
  const int line = total * a.hkv;
  per = (max(a.min_tiles, (line + a.shares - 1) / a.shares) + pad) & ~pad;
  EvenCursor c{};
  share = even_share(block, a.shares, (line + per - 1) / per);
  const int pos = share * per;
  share_end = min(pos + per, line);
  if (pos >= line) return c;  // past the batch's last share
  c.kvh = pos / total;
  const int at = pos - c.kvh * total;  // the share's first tile among its KV head's
  const uint64_t hit = __ballot(at >= incl - mine && at < incl);
  const int l = __builtin_ctzll(hit);
  int base = __builtin_amdgcn_readlane(incl - mine, l);
  int b = l * n;
  int row_len = __builtin_amdgcn_readlane(len, l);
  // the row among the lane's own (if none is it, a length changed since the scan)
  for (int i = 0; n > 1 && i < n; i += 64) {
    const int r = l * n + i + lane;
    const bool in = i + lane < n && r < a.num_seqs;
    const int rl = even_row_len<FUSE, false>(a, in ? r : 0);
    const int t = in ? even_tiles(rl, pad) : 0;
    const int sum = even_scan(t);
    const uint64_t m = __ballot(in && at < base + sum);
    if (m) {
      const int k = __builtin_ctzll(m);
      b = l * n + i + k;
      base += __builtin_amdgcn_readlane(sum - t, k);
      row_len = __builtin_amdgcn_readlane(rl, k);
      break;
    }
    base += __builtin_amdgcn_readlane(sum, 63);
  }
  c.valid = 1;
  c.b = b;
  c.len = row_len;
  const int tiles = even_tiles(c.len, pad);
  c.t_begin = min(at - base, tiles);
  c.left = share_end - pos;
  c.t_end = min(tiles, c.t_begin + c.left);
  c.left -= c.t_end - c.t_begin;
  return c;
}

// The cut of a share whose last segment is cu's.
__device__ __forceinline__ EvenCut even_cut(const EvenCursor& cu, int tiles, bool whole, int share, int share_end,
                                            int per) {
  const bool starts = cu.t_begin == 0 && !whole;
  const int parts = (share_end - cu.t_end + tiles - 1) / per - share + 1;
  return EvenCut{cu.b, cu.kvh, starts ? parts : 0, 0};
}

// Parts that a share's merge takes, 0 or less for no merge.  The cut may be one
// that no workgroup of this launch wrote (lengths that changed: a walk that ended
// early, another share than the workgroup's id stands for): whatever it holds,
// the parts end with the last share's and the row is one of the batch's.
__device__ __forceinline__ int even_cut_parts(const EvenCut& cut, int share, int shares, int num_seqs, int hkv) {
  // (one load of the cut and no branch before the parts are known)
  const bool row = (static_cast<uint32_t>(cut.b) < static_cast<uint32_t>(num_seqs)) &
                   (static_cast<uint32_t>(cut.kvh) < static_cast<uint32_t>(hkv));
  return min(cut.parts, shares - share) & -static_cast<int>(row);
}

}  // namespace fd
