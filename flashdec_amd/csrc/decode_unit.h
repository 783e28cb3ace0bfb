// Device code shared by the token-major decode kernels: the kernel parameters,
// a wave's K/V unit (loads, QK^T, online softmax, PV), the fused append and
// RoPE operands, and the pieces of the wave merge.
#pragma once

#include <type_traits>

#include "fd_common.h"
#include "rope_math.h"

namespace fd {

// Per-wave timeline of the MFMA row kernel and the cascade kernel, in a
// measurement build only (FD_TIMELINE: libflashdec_timeline.so, read by
// bench.py's c2-timeline and c4-timeline workloads; the product library
// compiles none of it).  Lane 0 of each wave writes s_memrealtime (100 MHz)
// at the phase boundaries of decode_role / process_unit into slot
// (workgroup * 8 + wave) * 16 + phase: phases 0-9 as named at the stamps,
// 10-14 the end of the wave's units 0-4 (later units in 14), and in the
// cascade kernel slot 15 the wave's role (1 prefix, 2 tail) instead of a
// time.
#ifdef FD_TIMELINE
constexpr bool kTimeline = true;
constexpr int kTimelineWorkgroups = 8192;
__device__ uint64_t g_timeline[kTimelineWorkgroups * 8 * 16];
#else
constexpr bool kTimeline = false;
#endif

__device__ __forceinline__ void timeline_put([[maybe_unused]] int k, [[maybe_unused]] bool mark,
                                             [[maybe_unused]] uint64_t v) {
#ifdef FD_TIMELINE
  if ((threadIdx.x & 63) == 0 && blockIdx.x < kTimelineWorkgroups)
    g_timeline[(blockIdx.x * 8 + (threadIdx.x >> 6)) * 16 + k] = mark ? v : __builtin_amdgcn_s_memrealtime();
#endif
}

template <int K>
__device__ __forceinline__ void timeline_stamp() {
  timeline_put(K, false, 0);
}

struct DecodeParams {
  const void* q;
  int64_t qs0, qs1, qs2;
  void* k;
  int64_t ks0, ks1, ks2, ks3;
  void* v;
  int64_t vs0, vs1, vs2, vs3;
  const void* bt;
  int64_t bts0, bts1;
  const void* sl;
  int64_t sls;
  void* out;
  int64_t os0, os1, os2;
  float* acc;
  int64_t as0, as1, as2, as3;
  float* mx;
  float* sm;
  int64_t ss0, ss1, ss2;
  uint32_t* counters;  // in-launch merge arrival counters (nullptr: reducer kernel)
  const void* ak;
  int64_t aks0, aks1, aks2;
  const void* av;
  int64_t avs0, avs1, avs2;
  const void* slot;
  int64_t slots;
  int bt_i64, sl_i64, slot_i64, fuse;
  int num_seqs, hq, hkv, group, head_dim, block_size;
  int64_t num_blocks, max_blocks_per_seq;
  int splits;
  int hint_tiles;    // ceil(bound / 32): bound = max_seq_len or the table capacity
  int hint_tps;      // tiles per split
  // workgroup-index divisions by splits and hkv as multiply-high and shifts
  // (fast_div; set for the MFMA row kernel only)
  uint32_t div_splits_m, div_hkv_m;
  int div_shifts;  // bits 0-7 / 8-15: splits' shifts, 16-23 / 24-31: hkv's
  // cascade tail pass: row b attends tokens [tb[b], seq_len); its partials
  // take workspace splits [0, splits), the prefix pass's come after them
  const int32_t* tb;
  int hint_tb;       // guess of tb / 32 for the first unit's early loads
  // balanced splits (> 0): row b gets clamp(ceil(tiles_b / T), 1, splits)
  // splits, T = ceil(total tiles / bal_target); workgroup w takes KV head
  // w % hkv of the batch's (w / hkv)-th split
  int bal_target;
  float scale_log2;  // sm_scale * log2(e): scores live in the base-2 domain
  // fused RoPE (rope_dim 64 or 128, with the fused append): q and append_k
  // arrive unrotated and are rotated at position seq_len - 1
  int rope_dim;
  float rope_base;
  const float* rope_tab;  // optional cos/sin table [2, rope_tab_rows, rope_dim / 2]
  int64_t rope_tab_rows;
};

// Row-level bookkeeping shared by the decode kernels.
struct RowInfo {
  int64_t eff_len;     // tokens attended (0 => zero output row)
  int64_t app_tok;     // token taken from append_k/v (-1: none)
  int64_t slot;        // cache slot receiving the appended token
  int t_begin, t_end;  // 32-token tiles [t_begin, t_end) of this split
};

__device__ __forceinline__ int64_t effective_len(const DecodeParams& p, int64_t seq_len, int64_t slot) {
  bool active = seq_len > 0;
  if (p.fuse) active = active && slot >= 0;
  int64_t eff = active ? seq_len : 0;
  // never walk past the block-table row, whatever seq_lens says
  const int64_t cap = p.max_blocks_per_seq * p.block_size;
  return eff < cap ? eff : cap;
}

// Split s covers tiles [s * tps, (s + 1) * tps) of the row, tps = ceil(T / S),
// T = the row's own 32-token tile count (flashdec/kernels/paged_decode.py:
// 408-411).  The host bound (hint_tiles / hint_tps) never decides the range:
// the MFMA kernel uses it only to guess where its first tile is, so that
// tile's loads can be issued before seq_lens arrives.
// (first_tile > 0: the cascade tail pass, whose rows start after their prefix)
__device__ __forceinline__ void split_tiles(int splits, int split, int64_t eff, int first_tile, int& t0, int& t1) {
  const int total = static_cast<int>((eff + 31) / 32);
  const int span = max(total - first_tile, 0);
  const int tps = (span + splits - 1) / splits;
  t0 = first_tile + split * tps;
  t1 = min(t0 + tps, total);
}

__device__ __forceinline__ void split_range(const DecodeParams& p, int split, int64_t eff, int& t0, int& t1) {
  split_tiles(p.splits, split, eff, 0, t0, t1);
}

__device__ __forceinline__ RowInfo row_info(const DecodeParams& p, int b, int split) {
  RowInfo r;
  const int64_t seq_len = load_index(p.sl, b * p.sls, p.sl_i64);
  r.slot = p.fuse ? load_index(p.slot, b * p.slots, p.slot_i64) : -1;
  r.eff_len = effective_len(p, seq_len, r.slot);
  r.app_tok = (p.fuse && r.eff_len > 0) ? r.eff_len - 1 : -1;
  split_range(p, split, r.eff_len, r.t_begin, r.t_end);
  const int live = static_cast<int>((r.eff_len + 31) / 32);
  r.t_end = min(r.t_end, live);
  return r;
}

// ===================================================== MFMA fast path ====
template <typename T>
__device__ __forceinline__ f32x4 mfma16x16x32(u32x4 a, u32x4 b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma16x16x32<__bf16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16x16x32<_Float16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                               __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// 16x16x16 MFMA (k = 16): A rows lane % 16, k = 4 * (lane / 16) + j; the
// D layout is the same as the 16x16x32 product's.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f32x4 mfma16x16x16(u32x2 a, u32x2 b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma16x16x16<__bf16>(u32x2 a, u32x2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c,
                                                   0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16x16x16<_Float16>(u32x2 a, u32x2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h16x4, a), __builtin_bit_cast(h16x4, b), c, 0,
                                               0, 0);
}

// Work unit of one wave: UNIT = 16 or 32 consecutive tokens.  Register
// footprint for one lane (lane = 16*g + c), MT = UNIT / 16 row blocks, head
// dim D = 128 or 64:
//   kf[mt][s]: K row (token UNIT*u + 16*mt + c), dims [32*s + 8*g, +8), s < D/32  (QK A)
//   vf[i]    : V row (token UNIT*u + vrow(g, i)), dims [(D/16)*c, +D/16)  (PV, transposed)
// vrow(g, i) = 4*g + i (i < 4) or 16 + 4*g + (i - 4): the tokens whose scores
// this lane holds after QK (MFMA D layout: rows 4*g + r of each 16-row
// block), so P needs no cross-lane movement.  Four waves of 32-token units
// suit splits of about one unit per wave (their compute runs on four SIMDs
// at once); eight waves of 16-token units stream better on long splits (a
// 16.8 MB read: 4.1 vs 4.8 us) and use the 16x16x16 PV product.
//
// Load addresses depend only on the block table, never on seq_lens: tokens
// past the row's length and rows whose block id is out of range are masked
// in registers at compute time, so the K/V loads of the first unit can be in
// flight before the row length arrives.
// A lane's piece of one V row: D/16 dims (16 bytes at D = 128, 8 at 64)
template <int D>
using VPiece = std::conditional_t<D == 128, u32x4, u32x2>;

template <int UNIT, int D = 128>
struct UnitRegs {
  static_assert(D == 128 || D == 64, "head_dim 128 or 64");
  static constexpr int MT = UNIT / 16;
  static constexpr int VR = UNIT / 4;  // V rows per lane: 4 (UNIT 16) or 8 (UNIT 32)
  static constexpr int KS = D / 32;    // 32-dim pieces of a K row (QK k-steps)
  u32x4 kf[MT][KS];
  VPiece<D> vf[VR];
  uint32_t bmask;  // bit i: V row i lies in a valid physical block
};

__device__ __forceinline__ int vrow(int g, int i) { return i < 4 ? 4 * g + i : 12 + 4 * g + i; }

template <int UNIT>
constexpr int waves_for() {
  return UNIT == 32 ? 4 : 8;
}

// One K/V vector load (16 or 8 bytes).  NT: non-temporal, for K/V that a
// launch reads once (streamed past the caches: a 550 MB read runs at 6.8
// instead of 6.1 TB/s on MI355X); plain loads where rows re-read shared
// blocks.
template <bool NT, typename V = u32x4>
__device__ __forceinline__ V kv_load(const void* a) {
  if constexpr (NT)
    return __builtin_nontemporal_load(reinterpret_cast<const V*>(a));
  else
    return *reinterpret_cast<const V*>(a);
}

// Physical block ids a unit needs (wave-uniform; SCALAR: read through the
// scalar cache); pages are clamped to the table row so the read is in bounds
// whatever the row's length.  A unit spans one block, or UNIT / BS
// consecutive ones (at most four: the dim-major kernel's 32-token units on
// 8-token blocks).
struct UnitPages {
  int32_t a, b, c, d;
};

template <int BS, int UNIT, bool SCALAR = false>
__device__ __forceinline__ UnitPages fetch_pages(const DecodeParams& p, int b, int unit) {
  static_assert(BS >= UNIT / 4, "a unit spans at most four blocks");
  constexpr int kPages = BS < UNIT ? UNIT / BS : 1;
  UnitPages up{0, 0, 0, 0};
  const int64_t row = b * p.bts0;
  const int64_t width = p.max_blocks_per_seq;
  const int64_t first = (static_cast<int64_t>(unit) * UNIT) / BS;
  auto entry = [&](int i) -> int32_t {
    const int64_t pg = first + i < width ? first + i : width - 1;
    const int64_t at = row + pg * p.bts1;
    return SCALAR ? load_index_uniform(p.bt, at, p.bt_i64) : load_index(p.bt, at, p.bt_i64);
  };
  up.a = entry(0);
  if constexpr (kPages >= 2) up.b = entry(1);
  if constexpr (kPages == 4) {
    up.c = entry(2);
    up.d = entry(3);
  }
  return up;
}

template <typename T, int BS, int UNIT, bool NT, int D>
__device__ __forceinline__ void load_unit(const DecodeParams& p, int kvh, int unit, const UnitPages& up, int c,
                                          int g, UnitRegs<UNIT, D>& t) {
  const T* kbase = static_cast<const T*>(p.k);
  const T* vbase = static_cast<const T*>(p.v);
  // tt: token within the unit; its block and the row inside that block
  auto block_of = [&](int tt) -> int32_t { return (BS < UNIT && tt >= BS) ? up.b : up.a; };
  auto row_in_block = [&](int tt) -> int { return (UNIT * unit + tt) % BS; };
  // K rows 16*mt + c.  Rows in invalid blocks read row 0 of the cache (in
  // bounds, value discarded by the score mask).
#pragma unroll
  for (int mt = 0; mt < UnitRegs<UNIT, D>::MT; ++mt) {
    const int tt = 16 * mt + c;
    const int32_t blk = block_of(tt);
    const bool ok = blk >= 0 && blk < p.num_blocks;
    const int64_t off = ok ? blk * p.ks0 + kvh * p.ks1 + row_in_block(tt) * p.ks2 : 0;
    const T* row = kbase + off;
#pragma unroll
    for (int s = 0; s < UnitRegs<UNIT, D>::KS; ++s) t.kf[mt][s] = kv_load<NT>(row + 32 * s + 8 * g);
  }
  // V rows vrow(g, i)
  uint32_t bm = 0;
#pragma unroll
  for (int i = 0; i < UnitRegs<UNIT, D>::VR; ++i) {
    const int tt = vrow(g, i);
    const int32_t blk = block_of(tt);
    const bool ok = blk >= 0 && blk < p.num_blocks;
    const int64_t off = ok ? blk * p.vs0 + kvh * p.vs1 + row_in_block(tt) * p.vs2 : 0;
    bm |= ok ? (1u << i) : 0u;
    t.vf[i] = kv_load<NT, VPiece<D>>(vbase + off + (D / 16) * c);
  }
  t.bmask = bm;
}

// Byte offsets of a lane's K and V rows inside their block (head kvh, the
// row's token slot, the lane's dims).  They are the same for every unit a
// wave takes: units advance by kWaves * UNIT = 128 tokens, a multiple of the
// block size, so (UNIT * unit) % BS depends only on the wave.  The host
// checks that they fit in 32 bits.
template <int UNIT>
struct UnitOffsets {
  uint32_t k[UnitRegs<UNIT>::MT];
  uint32_t v[UnitRegs<UNIT>::VR];
};

template <typename T, int BS, int UNIT, int D>
__device__ __forceinline__ UnitOffsets<UNIT> unit_offsets(const DecodeParams& p, int kvh, int wave, int c, int g) {
  UnitOffsets<UNIT> o;
  const int u0 = UNIT * wave;
#pragma unroll
  for (int mt = 0; mt < UnitRegs<UNIT>::MT; ++mt) {
    const int row = (u0 + 16 * mt + c) % BS;
    o.k[mt] = static_cast<uint32_t>((kvh * p.ks1 + row * p.ks2 + 8 * g) * static_cast<int64_t>(sizeof(T)));
  }
#pragma unroll
  for (int i = 0; i < UnitRegs<UNIT>::VR; ++i) {
    const int row = (u0 + vrow(g, i)) % BS;
    o.v[i] = static_cast<uint32_t>((kvh * p.vs1 + row * p.vs2 + (D / 16) * c) * static_cast<int64_t>(sizeof(T)));
  }
  return o;
}

// load_unit for block sizes of 16 and 32: each 16-token row group of a unit
// lies in one block (a 32-token unit on 16-token blocks: rows < 16 in the
// first, the rest in the second), so a row's address is a uniform block base
// (scalar) plus the lane's fixed 32-bit offset -- no per-unit vector
// address arithmetic.
template <typename T, int BS, int UNIT, bool NT, int D>
__device__ __forceinline__ void load_unit_fixed(const DecodeParams& p, const UnitPages& up,
                                                const UnitOffsets<UNIT>& o, UnitRegs<UNIT, D>& t) {
  static_assert(BS >= 16, "a 16-token row group must lie in one block");
  constexpr bool kTwo = BS < UNIT;
  const bool oka = up.a >= 0 && up.a < p.num_blocks;
  const bool okb = kTwo ? (up.b >= 0 && up.b < p.num_blocks) : oka;
  constexpr int64_t E = sizeof(T);
  const char* ka = static_cast<const char*>(p.k) + (oka ? up.a : 0) * p.ks0 * E;
  const char* va = static_cast<const char*>(p.v) + (oka ? up.a : 0) * p.vs0 * E;
  const char* kb = kTwo ? static_cast<const char*>(p.k) + (okb ? up.b : 0) * p.ks0 * E : ka;
  const char* vb = kTwo ? static_cast<const char*>(p.v) + (okb ? up.b : 0) * p.vs0 * E : va;
#pragma unroll
  for (int mt = 0; mt < UnitRegs<UNIT, D>::MT; ++mt) {
    const char* base = (kTwo && mt == 1) ? kb : ka;
#pragma unroll
    for (int s = 0; s < UnitRegs<UNIT, D>::KS; ++s) t.kf[mt][s] = kv_load<NT>(base + o.k[mt] + 64 * s);
  }
  uint32_t bm = 0;
#pragma unroll
  for (int i = 0; i < UnitRegs<UNIT, D>::VR; ++i) {
    const bool second = kTwo && i >= 4;  // V rows 16 + 4g + (i - 4)
    t.vf[i] = kv_load<NT, VPiece<D>>((second ? vb : va) + o.v[i]);
    bm |= (second ? okb : oka) ? (1u << i) : 0u;
  }
  t.bmask = bm;
}

// The appended token's pieces in this lane's operand layout: akf[s] = dims
// [32*s + 8*g, +8) of append_k, avf = dims [(D/16)*c, +D/16) of append_v.
template <int D = 128>
struct AppendRegs {
  u32x4 akf[D / 32];
  VPiece<D> avf;
};

// Fused append: store the newest token's K/V at the request's slot.  Lanes
// c == 0 write the K row (4 x D/32 x 16 B), lanes g == 0 the V row
// (16 x 2D/16 B).
template <typename T, int BS, int D>
__device__ __forceinline__ void store_append(const DecodeParams& p, int kvh, int32_t slot, int c, int g,
                                             const AppendRegs<D>& ar) {
  const int64_t blk = slot / BS, off = slot % BS;
  if (blk >= p.num_blocks) return;
  if (c == 0) {
    T* dst = static_cast<T*>(p.k) + blk * p.ks0 + kvh * p.ks1 + off * p.ks2;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) *reinterpret_cast<u32x4*>(dst + 32 * s + 8 * g) = ar.akf[s];
  }
  if (g == 0) {
    T* dst = static_cast<T*>(p.v) + blk * p.vs0 + kvh * p.vs1 + off * p.vs2;
    *reinterpret_cast<VPiece<D>*>(dst + (D / 16) * c) = ar.avf;
  }
}

// Fused RoPE: rotate this lane's Q^T operand pieces and the appended K row
// in place, at position seq_len - 1 (the row's length counts the appended
// token), with the RoPE kernel's arithmetic (rope_math.h) so the cached K
// bytes and the scores are those of RoPE + append followed by decode.  Piece
// s of a lane holds dims [32*s + 8*g, +8); with half = rope_dim / 2 its
// rotation partner is piece s + half / 32 (rope_dim 64: 0 <-> 1, dims 64-127
// unrotated; 128: 0 <-> 2 and 1 <-> 3).  Lane l evaluates frequency l in
// float64 (or reads it from the caller's cos/sin table), and ds_bpermute
// hands each lane the 8 frequencies of a piece.
template <typename T>
__device__ __forceinline__ void rope_operands(const DecodeParams& p, int32_t seq_len, int lane, int g,
                                              u32x4 (&qf)[4], AppendRegs<128>& ar) {
  const int half = p.rope_dim / 2;  // 32 or 64, checked on the host
  const int64_t pos = seq_len > 0 ? seq_len - 1 : 0;
  float cl, sl;
  if (p.rope_tab != nullptr)
    rope_table_cos_sin(p.rope_tab, p.rope_tab_rows, half, pos, lane < half ? lane : 0, cl, sl);
  else
    rope_cos_sin(p.rope_base, p.rope_dim, pos, lane < half ? lane : 0, cl, sl);
  const int ci = __builtin_bit_cast(int, cl), si = __builtin_bit_cast(int, sl);
  auto rotate = [&](u32x4& lo_w, u32x4& hi_w, const float (&c)[8], const float (&sn)[8]) {
    u32x4 a = lo_w, b = hi_w;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t ua = a[w], ub = b[w];
      float l0, h0, l1, h1;
      rope_rotate(lo_f32<T>(ua), lo_f32<T>(ub), c[2 * w], sn[2 * w], l0, h0);
      rope_rotate(hi_f32<T>(ua), hi_f32<T>(ub), c[2 * w + 1], sn[2 * w + 1], l1, h1);
      a[w] = pack2<T>(l0, l1);
      b[w] = pack2<T>(h0, h1);
    }
    lo_w = a;
    hi_w = b;
  };
  auto piece = [&](int s, int partner) {
    float c[8], sn[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int src = (32 * s + 8 * g + j) * 4;
      c[j] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src, ci));
      sn[j] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src, si));
    }
    rotate(qf[s], qf[partner], c, sn);
    rotate(ar.akf[s], ar.akf[partner], c, sn);
  };
  if (half == 64) {
    piece(0, 2);
    piece(1, 3);
  } else {
    piece(0, 1);
  }
}

// Online-softmax state of one lane: query head c, dims (D/4)*g + (D/16)*r + n.
template <int D = 128>
struct WaveState {
  f32x4 acc[D / 16];  // acc[n][r]
  float m;            // running max (base-2 domain), uniform over g
  float l;            // partial denominator of this lane's tokens
};

// Reductions over the four lanes c, c + 16, c + 32, c + 48 (one query
// column), every lane receiving the result.  With both operands the same
// value, v_permlane16_swap leaves rows 2k and 2k + 1 of each 32-lane half in
// its two results (and v_permlane32_swap the two halves), so combining the
// pair is the xor-16 (xor-32) butterfly step, with no LDS round trip.
__device__ __forceinline__ float pair_rows16_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return fmaxf(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}
__device__ __forceinline__ float pair_rows32_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return fmaxf(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}
__device__ __forceinline__ float pair_rows16_sum(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float pair_rows32_sum(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float column_max(float x) { return pair_rows32_max(pair_rows16_max(x)); }
__device__ __forceinline__ float column_sum(float x) { return pair_rows32_sum(pair_rows16_sum(x)); }

// 2^x on the hardware's v_exp_f32: results below 2^-126 flush to zero, which
// only drops probabilities that small relative to the running maximum.  The
// merges (the wave merge, the split reducer and the in-launch merge) weight
// their partials with it too: the library's exp2f adds a range reduction of
// about five instructions per weight, on the merges' dependent chains (C2
// 7.58 -> 7.51 us per call), for weights that only matter above 2^-126.
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// 1 / x on the hardware's v_rcp_f32 (1 ulp), for the softmax denominators of
// the stored rows: the division's correctly rounded sequence is about ten
// dependent instructions ahead of every output store.
__device__ __forceinline__ float rcp_fast(float x) { return __builtin_amdgcn_rcpf(x); }

// w * l rounded on its own (the empty asm keeps it out of any fused
// multiply-add): the terms of a merge's denominator.  Callers form it
// unconditionally and select the result: the compiler does not speculate the
// asm, so under a uniform test it became a branch per term, and the in-launch
// merge spilled its running sums around each one.
__device__ __forceinline__ float merge_term(float w, float l) {
  float t = w * l;
  asm volatile("" : "+v"(t));
  return t;
}

// The sum of 16 terms in the order a DPP row reduction gives its first lane
// (rotations by 8, 4, 2, 1): ((x0+x8)+(x4+x12)) + ((x2+x10)+(x6+x14)) and the
// same over the odd terms, then the two.  The in-launch merge sums its
// per-thread terms this way so that it matches the reducer bit for bit.
__device__ __forceinline__ float tree_sum16(const float (&x)[16]) {
  float a[8], b[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = x[i] + x[i + 8];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = a[i] + a[i + 4];
  return (b[0] + b[2]) + (b[1] + b[3]);
}

// Online-softmax step over one unit's scores of a lane (base-2 domain): the
// probabilities pr, and st updated for them.  The reference's kernels move
// the running maximum to every new block maximum and rescale acc and l each
// time (flashdec/kernels/paged_decode.py:293-312).  Here the maximum st.m
// moves only when a column's maximum exceeds it by more than kRescaleSlack:
// the probabilities, taken against st.m, stay below 2^kRescaleSlack (no
// overflow in fp32, the same relative rounding in the cache dtype), and the
// accumulator's multiply runs only on such moves instead of on most units.
// acc and l are always taken against the same st.m, so the partial they
// stand for is the same up to rounding.  LAZY false moves the maximum to every
// new one, so that a peak's probability is 1 and the cache dtype holds it
// exactly: even_decode.hip and wide_tile.h, whose waves take more units of a
// row (relative error against 64 bits, bf16, lazy / not / row kernels: 193 rows
// of 256 .. 511 tokens 0.0022 / 0.0018 / 0.0019, 54.6 us either way, the rescales
// hide behind the loads; 64 rows on a 16384-token prefix 0.0022 / 0.0018 /
// 0.0021, 30.5 / 32.5 / 34.2 us).
constexpr float kRescaleSlack = 8.f;

template <int VR, int D, bool LAZY = true>
__device__ __forceinline__ void softmax_step(const float (&sc)[VR], float (&pr)[VR], WaveState<D>& st) {
  float mx = sc[0];
#pragma unroll
  for (int i = 1; i < VR; ++i) mx = fmaxf(mx, sc[i]);
  mx = column_max(mx);
  // st.m == -inf: -inf + slack is -inf, so the first live unit moves it
  const bool move = mx > (LAZY ? st.m + kRescaleSlack : st.m);
  const float m_ref = move ? mx : st.m;
  const float m_use = m_ref == -INFINITY ? 0.f : m_ref;
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    pr[i] = exp2_fast(sc[i] - m_use);
    psum += pr[i];
  }
  // while st.m is -inf, acc and l are zero: nothing to rescale
  if (__ballot(move && st.m != -INFINITY)) {
    const float alpha = exp2_fast(st.m - m_use);  // 1 where st.m stays
#pragma unroll
    for (int n = 0; n < D / 16; ++n) st.acc[n] *= alpha;
    st.l *= alpha;
  }
  st.l += psum;
  st.m = m_ref;
}

// One unit for NCB 16-column blocks of query rows: mask (row length, invalid
// blocks), splice in the appended token, QK^T, online softmax, PV.  The
// blocks share the unit's K/V registers, its mask and its V^T operands.
// `last` is the last attended token, `first` the first (0: from the row's
// start), `app` the token taken from the append registers (-1: none).  The
// probabilities enter the PV product rounded to the cache dtype, as the
// reference's grouped kernels do (flashdec/kernels/paged_decode.py:308-310);
// the denominator sums them in fp32.  Masking is skipped for units whose
// tokens are all live (wave-uniform test).
template <typename T, bool FUSE, int UNIT, int D, int NCB, bool TL = false, bool LAZY = true>
__device__ __forceinline__ void process_unit(UnitRegs<UNIT, D>& t, const u32x4 (&qf)[NCB][D / 32],
                                             float scale_log2, int tok0, int first, int last, int app,
                                             const AppendRegs<D>& ar, int c, int g, WaveState<D> (&st)[NCB]) {
  constexpr int MT = UnitRegs<UNIT, D>::MT;
  constexpr int VR = UnitRegs<UNIT, D>::VR;
  constexpr int KS = UnitRegs<UNIT, D>::KS;
  constexpr int NW = D / 32;  // 32-bit words of a lane's V piece
  constexpr int NTILE = D / 16;  // PV output tiles (16 dims each)
  constexpr uint32_t kAll = (1u << VR) - 1u;
  uint32_t vmask = t.bmask;
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    const int tok = tok0 + vrow(g, i);
    vmask &= (tok <= last && (first == 0 || tok >= first)) ? ~0u : ~(1u << i);
  }
  if constexpr (FUSE) {
    const int at = app - tok0;  // in [0, UNIT) only for the unit holding it
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const bool hit = at == 16 * mt + c;
#pragma unroll
      for (int s = 0; s < KS; ++s) t.kf[mt][s] = hit ? ar.akf[s] : t.kf[mt][s];
    }
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      const bool hit = at == vrow(g, i);
      t.vf[i] = hit ? ar.avf : t.vf[i];
      vmask |= hit ? (1u << i) : 0u;
    }
  }
  // S^T[token][head] = K . Q^T  (MT 16-token row blocks)
  float sc[NCB][VR];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4 sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) sb = mfma16x16x32<T>(t.kf[mt][s], qf[cb][s], sb);
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[cb][4 * mt + r] = sb[r] * scale_log2;
    }
  if constexpr (TL) {
    asm volatile("" ::"v"(sc[0][0]), "v"(sc[0][VR - 1]));
    timeline_stamp<3>();  // K landed, QK done
  }
  // masked tokens: -inf scores and zero V rows (their memory may hold
  // NaN/Inf, and 0 * NaN is NaN)
  if (__ballot(vmask != kAll)) {
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      const bool keep = (vmask >> i) & 1u;
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) sc[cb][i] = keep ? sc[cb][i] : -INFINITY;
#pragma unroll
      for (int k = 0; k < NW; ++k) t.vf[i][k] = keep ? t.vf[i][k] : 0u;
    }
  }
  // P^T operands (k = VR*g + i: this lane's tokens)
  uint32_t ph[NCB][VR / 2];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    float pr[VR];
    softmax_step<VR, D, LAZY>(sc[cb], pr, st[cb]);
#pragma unroll
    for (int j = 0; j < VR / 2; ++j) ph[cb][j] = pack2<T>(pr[2 * j], pr[2 * j + 1]);
  }
  if constexpr (TL) {
    asm volatile("" ::"v"(ph[0][0]));
    timeline_stamp<4>();  // softmax done
  }
  // V^T operands: vt_n holds dim (D/16)*c + n of the lane's tokens
#pragma unroll
  for (int n = 0; n < NTILE; ++n) {
    const int w = n >> 1;
    const uint32_t sel = (n & 1) ? 0x07060302u : 0x05040100u;
    if constexpr (UNIT == 32) {
      u32x4 vt;
#pragma unroll
      for (int j = 0; j < 4; ++j) vt[j] = __builtin_amdgcn_perm(t.vf[2 * j + 1][w], t.vf[2 * j][w], sel);
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        u32x4 pp;
#pragma unroll
        for (int j = 0; j < 4; ++j) pp[j] = ph[cb][j];
        st[cb].acc[n] = mfma16x16x32<T>(vt, pp, st[cb].acc[n]);
      }
    } else {
      u32x2 vt;
#pragma unroll
      for (int j = 0; j < 2; ++j) vt[j] = __builtin_amdgcn_perm(t.vf[2 * j + 1][w], t.vf[2 * j][w], sel);
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        u32x2 pp;
#pragma unroll
        for (int j = 0; j < 2; ++j) pp[j] = ph[cb][j];
        st[cb].acc[n] = mfma16x16x16<T>(vt, pp, st[cb].acc[n]);
      }
    }
  }
}

// Floats per head row of the LDS merge slots (16-byte pieces, written and
// merged with 128-bit LDS accesses), and where a head's dims sit in its row:
// the 16-byte piece of dims [d, d + 4) starts at float acc_spread<D>() * d.
// Measured on MI355X (SQ_LDS_BANK_CONFLICT of a one-wave probe): a
// ds_write_b128 is conflict-free when each 8 consecutive lanes cover the 32
// banks once; a ds_read_b128 where each 16 lanes read 16 bytes at a 32-byte
// stride from rows 528 bytes apart is conflict-free, while 16 lanes reading
// 256 contiguous bytes from such rows is not.  So the rows are 132 floats
// apart, and head_dim-64 rows keep their pieces 32 bytes apart as head_dim
// 128's are (the merge then reads them with the same pattern).
template <int D>
constexpr int acc_pitch() {
  return 132;
}
template <int D>
constexpr int acc_spread() {
  return D == 64 ? 2 : 1;
}
// An output row's eight elements.  ``out`` may be any strided view (the
// reference indexes it through its strides), so with unit dim stride the
// 16-byte store can be unaligned: gfx9+ global memory runs in the
// unaligned-access mode, which splits such a store in hardware (checked on
// views one element past an aligned base in tests/test_unaligned_views_gpu.py;
// the split partials' 16-byte stores below take caller workspaces the same way).
// N: the first 4 or all 8 elements of o.
template <typename T, int N = 8>
__device__ __forceinline__ void store_row(const DecodeParams& p, int b, int qh, int d0, const float (&o)[8],
                                          float inv) {
  static_assert(N == 4 || N == 8, "4 or 8 elements");
  T* dst = static_cast<T*>(p.out) + b * p.os0 + qh * p.os1 + d0 * p.os2;
  if (p.os2 == 1) {
    if constexpr (N == 8) {
      u32x4 w;
      w[0] = pack2<T>(o[0] * inv, o[1] * inv);
      w[1] = pack2<T>(o[2] * inv, o[3] * inv);
      w[2] = pack2<T>(o[4] * inv, o[5] * inv);
      w[3] = pack2<T>(o[6] * inv, o[7] * inv);
      *reinterpret_cast<u32x4*>(dst) = w;
    } else {
      u32x2 w;
      w[0] = pack2<T>(o[0] * inv, o[1] * inv);
      w[1] = pack2<T>(o[2] * inv, o[3] * inv);
      *reinterpret_cast<u32x2*>(dst) = w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) dst[j * p.os2] = from_f32<T>(o[j] * inv);
  }
}

__device__ __forceinline__ int wave_sum_i32(int x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

__device__ __forceinline__ int wave_inclusive_scan_i32(int x, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    x += lane >= o ? y : 0;
  }
  return x;
}

// The hardware dispatches consecutive workgroup ids round-robin over the
// XCDs (8 on MI355X, each with its own L2).  With per_xcd = grid / 8 (a grid
// of a multiple of 8 workgroups), the i-th workgroup on XCD x takes logical
// index x * per_xcd + i, so each run of per_xcd consecutive logical
// workgroups shares one XCD; per_xcd 0 keeps the hardware order.
__device__ __forceinline__ int xcd_logical_block(int block, int per_xcd) {
  return per_xcd > 0 ? (block & 7) * per_xcd + (block >> 3) : block;
}

}  // namespace fd
