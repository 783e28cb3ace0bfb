// Even-share paged decode for gfx950: batches whose K/V keeps every CU busy.
//
// The row kernel (paged_decode.hip) gives every row the same number of splits,
// so a batch of unequal rows ends waiting on its longest ones, and a batch of
// many short rows spends its time starting and merging workgroups.  Here the
// batch's 32-token tiles -- KV head by KV head, row by row -- form one line
// (rows that share blocks then find one KV head's blocks in an XCD's L2: 40 rows
// on 5984 shared tokens, Hkv 4, cached loads: 43.4 us a call, row by row 57.1),
// and a fixed grid of workgroups cuts it into equal shares.  A workgroup walks
// its share across row boundaries ("segments": the part of one (row, KV head)
// that lies in the share), its waves taking 16-token units in turn.  The next
// unit's K/V loads (of the next segment too) are in flight while a unit is
// computed, so the memory pipeline does not drain between rows.  A segment that
// is a whole row goes straight to the output; the others leave fp32 partials in
// the share's two slots (a share cuts at most the row it starts in and the row
// it ends in), which even_reduce_kernel merges.  (Merging them inside the
// launch, by the last workgroup to arrive at a cut row, measured slower: 32
// rows of 128 .. 32768 tokens 45.7 us against 40.4, 48 rows with the fused append
// 25.4 against 23.0.)
//
// Reference semantics followed (cysong2025/flashdec):
//   flashdec/kernels/paged_decode.py:124-327  grouped decode + fused append
//   flashdec/kernels/paged_decode.py:546-642  LSE merge; zero rows for
//                                             seq_len == 0 / slot < 0
#include "decode_host.h"
#include "even_line.h"

namespace fd {

// Waves of a workgroup, W: 4 (two workgroups per CU) or 8 (one).
constexpr int kEvenWavesPerCU = 8;

// What only the merges need; fetched from the argument buffer there, so that it
// takes no scalar registers from the unit loop.
struct EvenOut {
  void* out;
  EvenCut* cuts;  // [shares]
  float* acc;     // [2 * shares][heads][D] partial rows
  float* stats;   // [2 * shares][heads][max, sum]
  int32_t os0, os1, os2;
  int32_t heads;  // query heads per KV head
};

// Physical block ids of a unit, through the scalar cache (fetched a step before
// the unit's K/V loads, so their wait never holds those up).
template <int BS, int UNIT>
__device__ __forceinline__ UnitPages even_pages(const EvenArgs& a, const EvenCursor& c) {
  constexpr int N = BS < UNIT ? UNIT / BS : 1;
  UnitPages up{-1, -1, -1, -1};
  if (!c.valid) return up;
  const int64_t row = static_cast<int64_t>(c.b) * a.bts0;
  const int first = c.unit * UNIT / BS;
  auto entry = [&](int i) {
    const int pg = min(first + i, a.width - 1);
    return load_index_uniform(a.bt, row + static_cast<int64_t>(pg) * a.bts1, a.bt_i64);
  };
  up.a = entry(0);
  if constexpr (N >= 2) up.b = entry(1);
  if constexpr (N == 4) {
    up.c = entry(2);
    up.d = entry(3);
  }
  return up;
}

// One 16- or 8-byte piece of a K/V row; NT: streamed past the caches (aux 2: nt).
template <bool NT, typename V>
__device__ __forceinline__ V even_buffer_load(__amdgpu_buffer_rsrc_t rsrc, int voff, int soff) {
  if constexpr (sizeof(V) == 16)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, soff, NT ? 2 : 0));
  else
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff, soff, NT ? 2 : 0));
}

// Buffer descriptor at a wave-uniform address of `bytes` bytes: -1 (the host
// checks that a block's rows span less than 2^32 bytes), or 0, with which loads
// return zero and read nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t even_rsrc(const char* at, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(at), 0, bytes, 0x00020000);
}

// A unit's K/V (UnitRegs layout), issued on every step: a step without a live
// unit (the wave has none in the segment, or the share is at its end) loads
// nothing through empty descriptors, but the number of loads in flight is the
// same on every path, so that a step's first use of its unit waits for that
// unit's loads alone and not for the next one's.
//
// Blocks of 16 and 32 tokens: every 16-token half lies in one block, so a
// half's rows are a buffer descriptor at the block (uniform) plus the lane's
// fixed offset; an invalid block's descriptor is empty.  Blocks of 8: the
// lane's quarter picks the address.
template <typename T, int BS, int UNIT, int D, bool NT>
__device__ __forceinline__ void even_load(const EvenArgs& a, const EvenCursor& cu, const UnitPages& up, int c, int g,
                                          UnitRegs<UNIT, D>& t) {
  constexpr int MT = UnitRegs<UNIT, D>::MT;
  constexpr int KS = UnitRegs<UNIT, D>::KS;
  constexpr int E = sizeof(T);
  // -1 for a live unit's valid block, else 0: integer arithmetic keeps it, and
  // the descriptors made from it, in scalar registers
  const int some = -cu.valid & ((cu.unit - cu.u_end) >> 31);
  auto live = [&](int32_t blk) { return some & ~(blk >> 31) & ((blk - a.num_blocks) >> 31); };
  const char* kh = static_cast<const char*>(a.k) + static_cast<int64_t>(cu.kvh) * a.ks1 * E;
  const char* vh = static_cast<const char*>(a.v) + static_cast<int64_t>(cu.kvh) * a.vs1 * E;
  uint32_t bm = 0;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    if constexpr (BS >= 16) {
      const int32_t page = (BS == 16 && j == 1) ? up.b : up.a;
      const int ok = live(page);
      const int64_t blk = page & ok;
      const __amdgpu_buffer_rsrc_t kr = even_rsrc(kh + blk * a.ks0 * E, ok);
      const __amdgpu_buffer_rsrc_t vr = even_rsrc(vh + blk * a.vs0 * E, ok);
      const uint32_t row0 = static_cast<uint32_t>(UNIT * cu.unit + 16 * j) % BS;
      // 32-bit unsigned byte offsets (the host checks that they fit)
      const uint32_t ks2 = a.ks2, vs2 = a.vs2;
      const uint32_t ko = (c * ks2 + 8 * g) * E;
      const uint32_t vo = (4 * g * vs2 + (D / 16) * c) * E;
#pragma unroll
      for (int s = 0; s < KS; ++s) t.kf[j][s] = even_buffer_load<NT, u32x4>(kr, ko + 64 * s, row0 * ks2 * E);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.vf[4 * j + i] = even_buffer_load<NT, VPiece<D>>(vr, vo, (row0 + i) * vs2 * E);
      bm |= static_cast<uint32_t>(ok) & (0xfu << (4 * j));
    } else {
      const int32_t lo = j == 0 ? up.a : up.c, hi = j == 0 ? up.b : up.d;
      const int32_t kpage = c < 8 ? lo : hi, vpage = g < 2 ? lo : hi;
      const bool kok = live(kpage) != 0, vok = live(vpage) != 0;
      // dead rows read the start of the cache: one line
      const char* kp = kok ? kh + (static_cast<int64_t>(kpage) * a.ks0 + (c & 7) * a.ks2 + 8 * g) * E
                           : static_cast<const char*>(a.k);
      const char* vp = vok ? vh + (static_cast<int64_t>(vpage) * a.vs0 + 4 * (g & 1) * a.vs2 + (D / 16) * c) * E
                           : static_cast<const char*>(a.v);
      const int64_t vstep = vok ? static_cast<int64_t>(a.vs2) * E : 0;
#pragma unroll
      for (int s = 0; s < KS; ++s) t.kf[j][s] = kv_load<NT>(kp + 64 * s);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.vf[4 * j + i] = kv_load<NT, VPiece<D>>(vp + i * vstep);
      bm |= vok ? (0xfu << (4 * j)) : 0u;
    }
  }
  t.bmask = bm;
}

// The appended token's cache row.
template <typename T, int BS, int D>
__device__ __forceinline__ void even_store_append(const EvenArgs& a, int kvh, int slot, int c, int g,
                                                  const AppendRegs<D>& ar) {
  const int64_t blk = slot / BS, off = slot % BS;
  if (blk >= a.num_blocks) return;
  if (c == 0) {
    T* dst = static_cast<T*>(a.k) + blk * a.ks0 + static_cast<int64_t>(kvh) * a.ks1 + off * a.ks2;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) *reinterpret_cast<u32x4*>(dst + 32 * s + 8 * g) = ar.akf[s];
  }
  if (g == 0) {
    T* dst = static_cast<T*>(a.v) + blk * a.vs0 + static_cast<int64_t>(kvh) * a.vs1 + off * a.vs2;
    *reinterpret_cast<VPiece<D>*>(dst + (D / 16) * c) = ar.avf;
  }
}

// One merged row piece (d0 .. d0 + N) to the output.
template <typename T, int N>
__device__ __forceinline__ void even_store_row(const EvenOut& w, int b, int qh, int d0, const float (&o)[8], float L) {
  const float inv = L > 0.f ? rcp_fast(L) : 0.f;
  T* dst = static_cast<T*>(w.out) + static_cast<int64_t>(b) * w.os0 + static_cast<int64_t>(qh) * w.os1 +
           static_cast<int64_t>(d0) * w.os2;
  if (w.os2 == 1) {
    const u32x2 lo{pack2<T>(o[0] * inv, o[1] * inv), pack2<T>(o[2] * inv, o[3] * inv)};
    if constexpr (N == 8)
      *reinterpret_cast<u32x4*>(dst) =
          u32x4{lo[0], lo[1], pack2<T>(o[4] * inv, o[5] * inv), pack2<T>(o[6] * inv, o[7] * inv)};
    else
      *reinterpret_cast<u32x2*>(dst) = lo;
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) dst[static_cast<int64_t>(j) * w.os2] = from_f32<T>(o[j] * inv);
  }
}

// FUSE: fused append of the current token.  The leading scalars repeat what the
// length scan needs: the command processor preloads them into SGPRs.
template <typename T, int BS, bool FUSE, int UNIT, int D, int W, bool NT>
__global__ __launch_bounds__(64 * W, kEvenWavesPerCU / W) void even_decode_kernel(
    const void* sl, int32_t num_seqs, int32_t sls, int32_t sl_i64, int32_t cap, int32_t hkv,
    int32_t shares, int32_t min_tiles, EvenArgs args, EvenOut) {
  constexpr int KS = D / 32;
  constexpr int P = acc_pitch<D>();
  // two sets of slots: one barrier per segment (the set of the segment before
  // last is free again once its merge's readers have passed this one)
  __shared__ __attribute__((aligned(16))) float s_acc[2][W][16][P];
  __shared__ float s_m[2][W][16];
  __shared__ float s_l[2][W][16];

  EvenArgs a = args;
  a.sl = sl;
  a.num_seqs = num_seqs;
  a.sls = sls;
  a.sl_i64 = sl_i64;
  a.cap = cap;
  a.hkv = hkv;
  a.shares = shares;
  a.min_tiles = min_tiles;
  auto out_args = [&]() {
    constexpr int kAt = (sizeof(void*) + 7 * sizeof(int32_t) + sizeof(EvenArgs) + 7) / 8 * 8;
    using Const = const __attribute__((address_space(4))) char*;
    Const base = (Const)__builtin_amdgcn_kernarg_segment_ptr() + kAt;
    asm volatile("" : "+s"(base));  // read here, not at the kernel's start
    const auto* p = (const __attribute__((address_space(4))) EvenOut*)base;
    return EvenOut{p->out, p->cuts, p->acc, p->stats, p->os0, p->os1, p->os2, p->heads};
  };
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  // the lane's row length (batches of up to 64 rows): asked for before all else
  const int my_row = lane < num_seqs ? lane : 0;
  int raw_len = load_index(sl, static_cast<int64_t>(my_row) * sls, sl_i64);
  [[maybe_unused]] int raw_slot = 0;
  if constexpr (FUSE) raw_slot = load_index(a.slot, static_cast<int64_t>(my_row) * a.slots, a.slot_i64);
  // While it is on its way: the block ids of the first unit as they are if
  // every row fills its table (a uniform batch, tables as wide as its rows),
  // one round trip less there.
  EvenCursor guess{};
  {
    const int pos = even_share(blockIdx.x, shares, args.full_used) * args.full_per;
    const int pair = pos / args.full_tiles;
    guess.b = pair % num_seqs;
    guess.t_begin = pos - pair * args.full_tiles;
    guess.unit = guess.t_begin * (32 / UNIT) + wave;
    guess.valid = pair < hkv * num_seqs;
  }
  const UnitPages guessed = even_pages<BS, UNIT>(a, guess);
  if constexpr (FUSE) raw_len = raw_slot < 0 ? 0 : raw_len;
  int share, per, share_end, pad;
  EvenCursor cur =
      even_first<FUSE>(a, blockIdx.x, lane, min(max(raw_len, 0), a.cap), share, per, share_end, pad);
  if (!cur.valid) {  // every wave of the workgroup
    if (threadIdx.x == 0) out_args().cuts[share].parts = 0;
    return;
  }
  even_enter<UNIT, W>(cur, wave);

  // columns past the group's last head take the KV head's first query head;
  // their results are dropped
  AppendRegs<D> ar;  // the appended token's rows
  auto load_q = [&](const EvenCursor& cu, u32x4 (&q)[1][KS]) {
    const T* row = static_cast<const T*>(a.q) + static_cast<int64_t>(cu.b) * a.qs0 +
                   static_cast<int64_t>(cu.kvh * a.group + (c < a.group ? c : 0)) * a.qs1;
#pragma unroll
    for (int s = 0; s < KS; ++s) q[0][s] = *reinterpret_cast<const u32x4*>(row + 32 * s + 8 * g);
    if constexpr (FUSE) {
      const T* ak = static_cast<const T*>(a.ak) + static_cast<int64_t>(cu.b) * a.aks0 + static_cast<int64_t>(cu.kvh) * a.aks1;
      const T* av = static_cast<const T*>(a.av) + static_cast<int64_t>(cu.b) * a.avs0 + static_cast<int64_t>(cu.kvh) * a.avs1;
#pragma unroll
      for (int s = 0; s < KS; ++s) ar.akf[s] = *reinterpret_cast<const u32x4*>(ak + 32 * s + 8 * g);
      ar.avf = *reinterpret_cast<const VPiece<D>*>(av + (D / 16) * c);
    }
  };

  UnitRegs<UNIT, D> ra, rb;
  u32x4 qf[1][KS];
  UnitPages pages = guessed;
  if (cur.b != guess.b || cur.unit != guess.unit || !guess.valid) pages = even_pages<BS, UNIT>(a, cur);
  load_q(cur, qf);
  even_load<T, BS, UNIT, D, NT>(a, cur, pages, c, g, ra);
  EvenCursor nxt = even_next<FUSE, UNIT, W>(a, cur, pad, wave);
  pages = even_pages<BS, UNIT>(a, nxt);

  WaveState<D> st[1];
  auto clear = [&]() {
#pragma unroll
    for (int n = 0; n < D / 16; ++n) st[0].acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    st[0].m = -INFINITY;
    st[0].l = 0.f;
  };
  clear();
  int set = 0;

  // merge the waves' states of segment `cu` and store its rows or partials
  auto flush = [&](const EvenCursor& cu) {
    constexpr int N = D == 128 ? 8 : 4;
    constexpr int kDimThreads = D / N;
    constexpr int kSpread = acc_spread<D>();
    const EvenOut w = out_args();
    const int tiles = even_tiles(cu.len, pad);
    const bool whole = cu.t_begin == 0 && cu.t_end == tiles;
    const int slot = 2 * share + (cu.t_begin == 0 ? 1 : 0);
    if (cu.left == 0 && threadIdx.x == 0) w.cuts[share] = even_cut(cu, tiles, whole, share, share_end, per);
    const float lt = column_sum(st[0].l);
    if (g == 0) {
      s_m[set][wave][c] = st[0].m;
      s_l[set][wave][c] = lt;
    }
    if (c < a.group) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        float* dst = &s_acc[set][wave][c][kSpread * ((D / 4) * g + (D / 16) * rr)];
        const WaveState<D>& x = st[0];
        *reinterpret_cast<f32x4*>(dst) = f32x4{x.acc[0][rr], x.acc[1][rr], x.acc[2][rr], x.acc[3][rr]};
        if constexpr (D == 128)
          *reinterpret_cast<f32x4*>(dst + 4) = f32x4{x.acc[4][rr], x.acc[5][rr], x.acc[6][rr], x.acc[7][rr]};
      }
    }
    // LDS only: the K/V loads in flight are not waited for
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int h = threadIdx.x / kDimThreads;
    const int d0 = (threadIdx.x % kDimThreads) * N;
    if (h < a.group) {
      float M = -INFINITY, L = 0.f;
      float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < W; ++x) M = fmaxf(M, s_m[set][x][h]);
      const float Mu = M == -INFINITY ? 0.f : M;
#pragma unroll
      for (int x = 0; x < W; ++x) {
        const float wt = exp2_fast(s_m[set][x][h] - Mu);
        L += wt * s_l[set][x][h];
        const f32x4 y = *reinterpret_cast<const f32x4*>(&s_acc[set][x][h][kSpread * d0]);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] += wt * y[j];
        if constexpr (N == 8) {
          const f32x4 z = *reinterpret_cast<const f32x4*>(&s_acc[set][x][h][d0 + 4]);
#pragma unroll
          for (int j = 0; j < 4; ++j) o[4 + j] += wt * z[j];
        }
      }
      if (whole) {
        even_store_row<T, N>(w, cu.b, cu.kvh * a.group + h, d0, o, L);
      } else {
        const int64_t at = static_cast<int64_t>(slot) * w.heads + h;
        float* dst = w.acc + at * D + d0;
        *reinterpret_cast<f32x4*>(dst) = f32x4{o[0], o[1], o[2], o[3]};
        if constexpr (N == 8) *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4], o[5], o[6], o[7]};
        if (d0 == 0) *reinterpret_cast<float2*>(w.stats + 2 * at) = float2{M, L};
      }
    }
    set ^= 1;
  };

  // One step: issue the next step's loads, then compute this step's unit; at
  // the wave's last unit of a segment the segment's merge.
  auto step = [&](UnitRegs<UNIT, D>& now, UnitRegs<UNIT, D>& ahead) -> bool {
    const bool last = even_last<W>(cur);
    const bool more = nxt.valid;
    even_load<T, BS, UNIT, D, NT>(a, nxt, pages, c, g, ahead);
    const EvenCursor after = even_next<FUSE, UNIT, W>(a, nxt, pad, wave);
    pages = even_pages<BS, UNIT>(a, after);
    const int app = FUSE && cur.unit < cur.u_end ? cur.len - 1 : -1;
    if constexpr (FUSE) {
      if (app >= 0 && app / UNIT == cur.unit) {
        const int slot = load_index_uniform(a.slot, static_cast<int64_t>(cur.b) * a.slots, a.slot_i64);
        even_store_append<T, BS, D>(a, cur.kvh, slot, c, g, ar);
      }
    }
    process_unit<T, FUSE, UNIT, D, 1, false, false>(now, qf, a.scale_log2, UNIT * cur.unit, 0,
                                                    min(cur.len, 32 * cur.t_end) - 1, app, ar, c, g, st);
    if (last) {
      if (more) load_q(nxt, qf);  // in flight during the merge
      flush(cur);
      clear();
    }
    cur = nxt;
    nxt = after;
    return more;
  };
  while (step(ra, rb) && step(rb, ra)) {
  }
}

// Merges the rows that shares cut: one workgroup per share, for the row that
// its last segment starts, every query head of the KV head.  Pure latency:
// the first EARLY parts' addresses need no data, so that their loads go out with
// the cut's own, one round trip in all for a row in so many shares; rows in more
// take the others kEvenParts at a time.  (The workspace holds EARLY slots after
// the last share's.)
constexpr int kEvenParts = 16;

template <typename T, int D, int EARLY>
__global__ __launch_bounds__(256) void even_reduce_kernel(const EvenCut* cuts, const float* acc, const float* stats,
                                                          int32_t heads, int32_t shares, int32_t num_seqs, int32_t hkv,
                                                          EvenOut w) {
  constexpr int N = 4;  // dims per thread
  constexpr int kDimThreads = D / N;
  const int share = blockIdx.x;
  struct Part {
    f32x4 x;
    float2 ml;
  };
  for (int i = threadIdx.x + 256 * blockIdx.y; i < heads * kDimThreads; i += 256 * gridDim.y) {
    const int head = i / kDimThreads, d0 = (i % kDimThreads) * N;
    auto part = [&](int j) {
      const int64_t at = static_cast<int64_t>(j == 0 ? 2 * share + 1 : 2 * (share + j)) * heads + head;
      Part r;
      r.x = *reinterpret_cast<const f32x4*>(acc + at * D + d0);
      r.ml = *reinterpret_cast<const float2*>(stats + 2 * at);
      return r;
    };
    // slots that this launch did not write may hold anything
    Part early[EARLY];
#pragma unroll
    for (int j = 0; j < EARLY; ++j) early[j] = part(j);
    asm volatile("" ::: "memory");  // the cut's load and its tests stay behind those loads
    const EvenCut cut = cuts[share];
    const int parts = even_cut_parts(cut, share, shares, num_seqs, hkv);
    if (parts <= 0) return;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int j = 0; j < EARLY; ++j) M = j < parts ? fmaxf(M, early[j].ml.x) : M;
    float mu = M == -INFINITY ? 0.f : M;
    float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < EARLY; ++j) {
      if (j >= parts) continue;
      const float wt = exp2_fast(early[j].ml.x - mu);
      L += wt * early[j].ml.y;
#pragma unroll
      for (int k = 0; k < N; ++k) o[k] += wt * early[j].x[k];
    }
    for (int j0 = EARLY; j0 < parts; j0 += kEvenParts) {
      Part p[kEvenParts];
#pragma unroll
      for (int j = 0; j < kEvenParts; ++j) p[j] = part(min(j0 + j, parts - 1));
      float nm = M;
#pragma unroll
      for (int j = 0; j < kEvenParts; ++j) nm = fmaxf(nm, p[j].ml.x);  // past the end: a part again, weight 0
      mu = nm == -INFINITY ? 0.f : nm;
      const float sc = exp2_fast(M - mu);
      L *= sc;
#pragma unroll
      for (int k = 0; k < N; ++k) o[k] *= sc;
#pragma unroll
      for (int j = 0; j < kEvenParts; ++j) {
        const float wt = j0 + j < parts ? exp2_fast(p[j].ml.x - mu) : 0.f;
        L += wt * p[j].ml.y;
#pragma unroll
        for (int k = 0; k < N; ++k) o[k] += wt * p[j].x[k];
      }
      M = nm;
    }
    even_store_row<T, N>(w, cut.b, cut.kvh * heads + head, d0, o, L);
  }
}

// ========================================================== host glue ====
namespace {

constexpr int kEvenMinTiles = 4;  // per share
// (row, KV head) pairs from which a share holds several rows as a rule: two
// 4-wave workgroups per CU hide each other's merges.  Below, one 8-wave
// workgroup: half as many cut rows and parts (us/call, 4 x 2 against 8 x 1: 64
// pairs of 4096 tokens 31.0 against 27.5, 1024 pairs of 2 .. 512 tokens 24 against 33).
constexpr int64_t kEvenFewPairs = 256;

struct EvenShape {
  int waves = 0;  // per workgroup; 0: the kernel does not take this call
  int shares = 0;
  int early = 0;  // parts of a cut row that the merge asks for at once
  int64_t acc_floats = 0, stats_floats = 0;
  int64_t floats() const { return acc_floats + stats_floats + 4 * static_cast<int64_t>(shares); }
};

bool fits32(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// Shape of the even-share launch, waves 0 where the call is not one for it.
EvenShape even_shape(const fd_paged_decode_args& a) {
  EvenShape s;
  if (a.num_kv_heads <= 0 || a.num_q_heads <= 0 || a.num_seqs <= 0) return s;
  const int64_t group = a.num_q_heads / a.num_kv_heads;
  if (a.rotary_dim != 0 || a.split_counters != nullptr || !fast_path_ok(a, group)) return s;
  if (group > 16 || (a.append_k && a.head_dim != 128)) return s;
  for (const int64_t* st : {a.k_stride, a.v_stride})
    for (int i = 0; i < 3; ++i)
      if (!fits32(st[i])) return s;
  for (int64_t x : {a.q_stride[0], a.q_stride[1], a.out_stride[0], a.out_stride[1], a.out_stride[2],
                    a.seq_lens_stride, a.num_seqs, a.num_q_heads, a.num_blocks})
    if (!fits32(x)) return s;
  if (a.append_k)
    for (int64_t x : {a.append_k_stride[0], a.append_k_stride[1], a.append_v_stride[0], a.append_v_stride[1],
                      a.slot_mapping_stride})
      if (!fits32(x)) return s;
  const int64_t cap = a.max_blocks_per_seq * a.block_size;
  const int64_t line = a.num_seqs * a.num_kv_heads * ((cap + 31) / 32);
  if (!fits32(cap) || line > (1 << 30)) return s;
  s.waves = a.num_seqs * a.num_kv_heads < kEvenFewPairs ? 8 : 4;
  s.shares = kEvenWavesPerCU / s.waves * device_cus();
  s.early = s.waves == 8 ? 4 : 2;
  s.acc_floats = int64_t{2} * (s.shares + s.early) * group * a.head_dim;
  s.stats_floats = int64_t{2} * (s.shares + s.early) * group * 2;
  return s;
}

template <typename T, int BS, int W, bool NT>
void launch_even_kernel(const fd_paged_decode_args& a, const EvenArgs& e, const EvenOut& w, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(e.shares)), block(64 * W);
  auto go = [&](auto kernel) {
    dispatch(kernel, grid, block, stream, a.timing_events[0], a.timing_events[1], e.sl, e.num_seqs, e.sls, e.sl_i64,
             e.cap, e.hkv, e.shares, e.min_tiles, e, w);
  };
  if (a.head_dim == 64)
    go(even_decode_kernel<T, BS, false, 32, 64, W, NT>);
  else
    a.append_k ? go(even_decode_kernel<T, BS, true, 16, 128, W, NT>)
               : go(even_decode_kernel<T, BS, false, 16, 128, W, NT>);
}

template <typename T, int BS, int W>
void launch_even_kernel(const fd_paged_decode_args& a, const EvenArgs& e, const EvenOut& w, hipStream_t stream) {
  a.kv_reuse ? launch_even_kernel<T, BS, W, false>(a, e, w, stream) : launch_even_kernel<T, BS, W, true>(a, e, w, stream);
}

template <typename T, int W>
void launch_even_kernel(const fd_paged_decode_args& a, const EvenArgs& e, const EvenOut& w, hipStream_t stream) {
  switch (a.block_size) {
    case 8: launch_even_kernel<T, 8, W>(a, e, w, stream); break;
    case 16: launch_even_kernel<T, 16, W>(a, e, w, stream); break;
    default: launch_even_kernel<T, 32, W>(a, e, w, stream); break;
  }
}

template <typename T>
int launch_even(const fd_paged_decode_args& a, const EvenArgs& e, const EvenOut& w, int waves, hipStream_t stream) {
  waves == 8 ? launch_even_kernel<T, 8>(a, e, w, stream) : launch_even_kernel<T, 4>(a, e, w, stream);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_error(FD_E_LAUNCH, "even-share decode launch failed: %s", hipGetErrorString(err));
  auto reduce = [&](auto kernel) {
    const unsigned per_share = static_cast<unsigned>((w.heads * a.head_dim / 4 + 255) / 256);
    dispatch(kernel, dim3(static_cast<unsigned>(e.shares), per_share), dim3(256), stream, a.timing_events[2],
             a.timing_events[3], static_cast<const EvenCut*>(w.cuts), static_cast<const float*>(w.acc),
             static_cast<const float*>(w.stats), w.heads, e.shares, e.num_seqs, e.hkv, w);
  };
  if (waves == 8)
    a.head_dim == 64 ? reduce(even_reduce_kernel<T, 64, 4>) : reduce(even_reduce_kernel<T, 128, 4>);
  else
    a.head_dim == 64 ? reduce(even_reduce_kernel<T, 64, 2>) : reduce(even_reduce_kernel<T, 128, 2>);
  err = hipGetLastError();
  if (err != hipSuccess) return set_error(FD_E_LAUNCH, "even-share reduce launch failed: %s", hipGetErrorString(err));
  return FD_OK;
}

}  // namespace
}  // namespace fd

using namespace fd;

extern "C" int fd_paged_decode_even_floats(const fd_paged_decode_args* args) {
  if (args == nullptr || args->struct_size != sizeof(fd_paged_decode_args))
    return set_error(FD_E_INVALID, "fd_paged_decode_even_floats: args is NULL or has another ABI's size");
  const EvenShape s = even_shape(*args);
  return s.waves ? static_cast<int>(s.floats()) : 0;  // about 2 M at most
}

// The host knows what the tables hold at most, not the rows' lengths.  Against
// the row kernel and its merge this one starts with one more round trip (the
// lengths) and merges with one more, about 2 us a call, and saves what rounds of
// workgroups that the rows do not fill cost the row kernel.  The rows may be far
// shorter than the tables, so a call goes here only where it gains at every
// length.  MI355X, graph replays, us/call of the row kernel / here, Hq 16, Hkv 2
// unless said otherwise; "mixed": lengths spread evenly over their logarithm.
//   Row kernel in one round (pairs x splits up to the CUs): never.  Full rows
//     gain little, rows shorter than the table lose: 8 x 2048 in 32768 9.4 /
//     12.7, 128 x 512 in 2048 15.1 / 18.6, 64 x 4096 full 47.1 / 46.7.
//   In more, two splits and more: always.  100 rows in 4096: x 64 12.5 / 9.7,
//     x 512 20.8 / 18.2, mixed to 1024 18.0 / 14.0, full 82.6 / 71.5.  Under 64
//     pairs from three rounds on: 1024 tokens in 32768, Hkv 1, 32 rows (two
//     rounds) 14.0 / 15.1, 48 rows 19.4 / 13.3.
//   One split: from 1024 pairs on, 2048 with more than 8 heads per KV head (more
//     to merge).  Rows of 64 to 128, pairs: 512 11.3 / 12.3, 768 15.8 / 17.4, 1024
//     20.5 / 19.2; Hkv 1, rows of 128 to 256: 1024 30.9 / 34.3, 2048 59.0 / 59.3.
//   64-dim heads (half the bytes, the same fixed time): from 64 pairs, in more
//     than three rounds, eight under four splits: 100 rows of 128 to 256, two splits
//     (tables of 4096) 9.6 / 10.9, five (8192) 13.2 / 10.9.
// A caller that says the lengths vary widely (balance_target) gets the balanced
// kernel otherwise, one round whatever the lengths: from 192 pairs on.  Below, one
// long row among short ones loses (64 pairs, 8192 in 32768: 14.3 / 16.3), and
// mixed ones to 4096 come out even (Hq 32, Hkv 8, 128 pairs 19.1 / 20.0, 192 25.6 /
// 24.0).
constexpr int64_t kEvenRaggedPairs = 192;
constexpr int64_t kEvenOneSplitPairs = 1024;

extern "C" int fd_paged_decode_even_pays(const fd_paged_decode_args* args) {
  if (args == nullptr || args->struct_size != sizeof(fd_paged_decode_args))
    return set_error(FD_E_INVALID, "fd_paged_decode_even_pays: args is NULL or has another ABI's size");
  const fd_paged_decode_args& a = *args;
  if (even_shape(a).waves == 0) return 0;
  const int64_t cap = a.max_blocks_per_seq * a.block_size;
  const int64_t pairs = a.num_seqs * a.num_kv_heads;
  const bool many_heads = a.num_q_heads > 8 * a.num_kv_heads;
  const int64_t tiles = pairs * ((cap + 31) / 32) * a.head_dim / 128;  // of 16 KB
  if (tiles < 12288 && (tiles < 4096 || pairs < 64 || pairs >= 448 || many_heads)) return 0;
  if (a.balance_target > 0) return pairs >= kEvenRaggedPairs ? 1 : 0;
  const int splits = fd_paged_decode_plan(a.num_seqs, a.num_q_heads, a.num_kv_heads, a.head_dim, cap, 0);
  const int64_t cus = device_cus(), wgs = pairs * splits;
  if (a.head_dim == 64) return pairs >= 64 && splits > 1 && wgs > (splits < 4 ? 8 : 3) * cus ? 1 : 0;
  if (splits == 1) return pairs >= (many_heads ? 2 : 1) * kEvenOneSplitPairs ? 1 : 0;
  return pairs < 64 ? wgs >= 3 * cus : wgs > cus;
}

extern "C" int fd_paged_decode_even(const fd_paged_decode_args* args, float* workspace, int64_t floats,
                                    fd_stream_t stream_) {
  clear_launch_record();
  static const char* fn = "fd_paged_decode_even";
  DecodeParams p;
  const int rc = fill_decode_params(args, fn, p);
  if (rc != FD_OK) return rc;
  const fd_paged_decode_args& a = *args;
  const EvenShape s = even_shape(a);
  if (s.waves == 0) return set_error(FD_E_UNSUPPORTED, "%s: the call's shape, strides or alignment need fd_paged_decode", fn);
  if (workspace == nullptr || floats < s.floats() || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return set_error(FD_E_INVALID, "%s: needs a 16-byte aligned workspace of %lld floats", fn,
                     static_cast<long long>(s.floats()));
  EvenArgs e{};
  EvenOut w{};
  e.q = a.q;
  e.k = a.k_cache;
  e.v = a.v_cache;
  e.bt = a.block_tables;
  e.sl = a.seq_lens;
  w.out = a.out;
  e.ak = a.append_k;
  e.av = a.append_v;
  e.slot = a.slot_mapping;
  w.acc = workspace;
  w.stats = workspace + s.acc_floats;
  w.cuts = reinterpret_cast<EvenCut*>(workspace + s.acc_floats + s.stats_floats);
  w.heads = static_cast<int32_t>(a.num_q_heads / a.num_kv_heads);
  auto i32 = [](int64_t x) { return static_cast<int32_t>(x); };
  e.num_blocks = i32(a.num_blocks);
  e.qs0 = i32(a.q_stride[0]);
  e.qs1 = i32(a.q_stride[1]);
  e.ks0 = i32(a.k_stride[0]);
  e.ks1 = i32(a.k_stride[1]);
  e.ks2 = i32(a.k_stride[2]);
  e.vs0 = i32(a.v_stride[0]);
  e.vs1 = i32(a.v_stride[1]);
  e.vs2 = i32(a.v_stride[2]);
  e.bts0 = i32(a.block_tables_stride[0]);
  e.bts1 = i32(a.block_tables_stride[1]);
  w.os0 = i32(a.out_stride[0]);
  w.os1 = i32(a.out_stride[1]);
  w.os2 = i32(a.out_stride[2]);
  if (a.append_k) {
    e.aks0 = i32(a.append_k_stride[0]);
    e.aks1 = i32(a.append_k_stride[1]);
    e.avs0 = i32(a.append_v_stride[0]);
    e.avs1 = i32(a.append_v_stride[1]);
    e.slots = i32(a.slot_mapping_stride);
    e.slot_i64 = a.slot_mapping_dtype == FD_INDEX_I64;
  }
  e.sls = i32(a.seq_lens_stride);
  e.num_seqs = i32(a.num_seqs);
  e.hkv = i32(a.num_kv_heads);
  e.group = i32(a.num_q_heads / a.num_kv_heads);
  e.width = i32(a.max_blocks_per_seq);
  e.cap = i32(a.max_blocks_per_seq * a.block_size);
  e.shares = s.shares;
  e.min_tiles = kEvenMinTiles;
  e.full_tiles = e.cap > 0 ? (e.cap + 31) / 32 : 1;
  const int line = e.num_seqs * e.hkv * e.full_tiles;  // even_shape checks that it fits
  e.full_per = (line + e.shares - 1) / e.shares;
  if (e.full_per < kEvenMinTiles) e.full_per = kEvenMinTiles;
  e.full_used = (line + e.full_per - 1) / e.full_per;
  e.bt_i64 = a.block_tables_dtype == FD_INDEX_I64;
  e.sl_i64 = a.seq_lens_dtype == FD_INDEX_I64;
  e.scale_log2 = p.scale_log2;
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (a.dtype == FD_DTYPE_BF16) return launch_even<__bf16>(a, e, w, s.waves, stream);
  return launch_even<_Float16>(a, e, w, s.waves, stream);
}
