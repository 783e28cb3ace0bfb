// Device code of the wide decode workgroup: many query rows on one read of a
// K/V range.  A group that shares a prefix brings hundreds of (member, head)
// rows to the same tokens.  The row kernels keep a wave's K/V unit in its
// registers, so every 32 of those rows read the tokens again; here the
// workgroup stages a batch of tokens in LDS once and each wave attends it with
// its own rows.  (The range is read again by the group's other chunks: plain
// loads.)
#pragma once

#include "decode_unit.h"

namespace fd {

// RG row groups of 16 * RB rows x TG token groups of 32 tokens: RG * TG waves,
// a batch of 32 * TG tokens staged at a time.  Two batches are in LDS (one
// barrier a batch), and a third and fourth on their way in registers.
template <int D, int RB, int RG, int TG>
struct WideShape {
  static constexpr int kColBlocks = RB;
  static constexpr int kWaves = RG * TG;
  static constexpr int kRows = 16 * RB * RG;
  static constexpr int kTokens = 32 * TG;
  static constexpr int kPieces = D / 8;           // 16-byte pieces of a K/V row
  static constexpr int kLoadRows = 64 / kPieces;  // rows of one wave-wide load
  // A wave brings the K and V rows of one run of 8 tokens, which lies in one
  // block: one block id, one pair of descriptors.
  static constexpr int kRun = 8;
  static constexpr int kRuns = kTokens / kRun;
  static constexpr int kLoads = kRun / kLoadRows;  // of K, and as many of V
  static_assert(kWaves == kRuns, "a run for each wave");
  static_assert(D == 128, "the tiles' swizzle");
  static constexpr int kTileBytes = kTokens * D * 2;
  static constexpr int kMergeBytes = (TG - 1) * kRows * D * 4;
  static constexpr int kStageBytes = 4 * kTileBytes > kMergeBytes ? 4 * kTileBytes : kMergeBytes;
};

template <typename S>
struct alignas(16) WideLds {
  uint8_t stage[S::kStageBytes];    // [2 batches][K, V][token][dim], swizzled; then the merge's accumulators
  int32_t live[2][S::kRuns];        // attended tokens of each run
  float m[S::kWaves][2 * S::kColBlocks][16];  // the waves' maxima and denominators
};

// A K/V row's 16-byte piece within a staged tile, in bytes.  K rows are read 16
// at a time at one piece (ds_read_b128: the row's low bits pick the banks); V
// is read 4 rows by 32 bytes at a time, transposed (ds_read_b64_tr_b16), so its
// 32-byte pairs of pieces are what moves.
template <int D>
__device__ __forceinline__ int wide_k_at(int row, int piece) {
  return row * (2 * D) + ((piece ^ (row & (D / 8 - 1))) << 4);
}
template <int D>
__device__ __forceinline__ int wide_v_at(int row, int pair) {
  return row * (2 * D) + ((pair ^ (row & 7)) << 5);
}

// Four rows of the lane's 16-lane group, transposed: the lane gives the address
// of row (lane % 16) / 4, dims 4 * (lane % 4), and receives dim lane % 16 of
// the four rows (checked against a plain read on gfx950).
__device__ __forceinline__ u32x2 wide_read_tr(const uint8_t* at) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(at)));
}

// What a workgroup attends: tokens [32 * t_begin, limit) of table row trow.
struct WideWork {
  int trow, kvh;
  int begin, limit;
};

// A wave's run of a batch.
template <typename S>
struct WideRegs {
  u32x4 k[S::kLoads], v[S::kLoads];
};

// First token of the wave's run.
template <typename S>
__device__ __forceinline__ int wide_run(const WideWork& w, int batch, int wave) {
  return w.begin + batch * S::kTokens + wave * S::kRun;
}

template <typename S, int BS>
__device__ __forceinline__ int32_t wide_page(const DecodeParams& p, const WideWork& w, int batch, int wave) {
  const int pg = min(wide_run<S>(w, batch, wave) / BS, static_cast<int>(p.max_blocks_per_seq) - 1);
  return load_index_uniform(p.bt, w.trow * p.bts0 + pg * p.bts1, p.bt_i64);
}

// -1 where the run at tok in block id has attended tokens, else 0.  Unsigned
// differences: from signed ones the compiler takes the comparisons, extends
// their conjunction in a vector register, and the descriptors made from it are
// read back lane by lane.
__device__ __forceinline__ int wide_some(const DecodeParams& p, const WideWork& w, int tok, int32_t id) {
  const int in = static_cast<int>(static_cast<uint32_t>(tok) - static_cast<uint32_t>(w.limit)) >> 31;
  const int blk = static_cast<int>(static_cast<uint32_t>(id) - static_cast<uint32_t>(p.num_blocks)) >> 31;
  return in & ~(id >> 31) & blk;
}

// How many.
template <typename S>
__device__ __forceinline__ int wide_live(const DecodeParams& p, const WideWork& w, int tok, int32_t id) {
  return min(w.limit - tok, S::kRun) & wide_some(p, w, tok, id);
}

// A batch's loads, issued whether or not it has tokens (a run with none, or in
// an invalid block, goes through empty descriptors: zeros and no read), so
// that the number in flight is the same on every path and the wait for a batch
// leaves the next one's loads in flight.
template <typename S, int BS>
__device__ __forceinline__ void wide_load(const DecodeParams& p, const WideWork& w, int batch, int wave, int lane,
                                          int32_t page, WideRegs<S>& r) {
  const int tok = wide_run<S>(w, batch, wave);
  const int some = wide_some(p, w, tok, page);
  const int64_t id = page & some;
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<char*>(p.k) + (id * p.ks0 + w.kvh * p.ks1) * 2, 0, some, 0x00020000);
  const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<char*>(p.v) + (id * p.vs0 + w.kvh * p.vs1) * 2, 0, some, 0x00020000);
  const uint32_t ks2 = static_cast<uint32_t>(p.ks2) * 2u, vs2 = static_cast<uint32_t>(p.vs2) * 2u;
  const uint32_t row = lane / S::kPieces, piece = (lane % S::kPieces) * 16u;
  const uint32_t row0 = static_cast<uint32_t>(tok) % BS;
#pragma unroll
  for (int j = 0; j < S::kLoads; ++j)
    r.k[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           kr, row * ks2 + piece, (row0 + j * S::kLoadRows) * ks2, 0));
#pragma unroll
  for (int j = 0; j < S::kLoads; ++j)
    r.v[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           vr, row * vs2 + piece, (row0 + j * S::kLoadRows) * vs2, 0));
}

// A batch's rows into its LDS tiles.  Rows past the attended tokens are stored
// as zeros: their scores are masked, but 0 * NaN in the PV product is not 0.
template <typename S, int D>
__device__ __forceinline__ void wide_stage(const DecodeParams& p, const WideWork& w, int batch, int wave, int lane,
                                           int32_t page, const WideRegs<S>& r, WideLds<S>& lds, int buf) {
  uint8_t* kt = lds.stage + buf * 2 * S::kTileBytes;
  const int live = wide_live<S>(p, w, wide_run<S>(w, batch, wave), page);
  const int row = lane / S::kPieces, piece = lane % S::kPieces;
#pragma unroll
  for (int j = 0; j < S::kLoads; ++j) {
    const int at = wave * S::kRun + j * S::kLoadRows + row;
    u32x4 v = r.v[j];
    if (live < S::kRun) v = j * S::kLoadRows + row < live ? v : u32x4{0u, 0u, 0u, 0u};
    *reinterpret_cast<u32x4*>(kt + wide_k_at<D>(at, piece)) = r.k[j];
    *reinterpret_cast<u32x4*>(kt + S::kTileBytes + wide_v_at<D>(at, piece >> 1) + (piece & 1) * 16) = v;
  }
  if (lane == 0) lds.live[buf][wave] = live;
}

// A wave's 32 tokens of a staged batch for its RB 16-row column blocks.
template <typename T, typename S, int D, int RB>
__device__ __forceinline__ void wide_compute(const u32x4 (&qf)[RB][D / 32], float scale_log2, int tg, int c, int g,
                                             const WideLds<S>& lds, int buf, WaveState<D> (&st)[RB]) {
  constexpr int KS = D / 32;
  const uint8_t* kt = lds.stage + buf * 2 * S::kTileBytes + tg * 32 * 2 * D;
  const uint8_t* vt = kt + S::kTileBytes;
  // Every K read issues ahead of the products, and every V read ahead of the
  // softmax (the scheduler leaves each beside its use: eight LDS round trips in
  // a row with nothing to hide them, two waves a SIMD).
  u32x4 kf[2][KS];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      kf[mt][s] = *reinterpret_cast<const u32x4*>(kt + wide_k_at<D>(16 * mt + c, 4 * s + g));
  // this lane's tokens: 4 * g + r of each 16
  const int first = (4 * g) % S::kRun;
  const int n0 = lds.live[buf][(32 * tg + 4 * g) / S::kRun] - first;
  const int n1 = lds.live[buf][(32 * tg + 16 + 4 * g) / S::kRun] - first;
  __builtin_amdgcn_sched_barrier(0);
  float sc[RB][8];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    f32x4 sb[RB];
#pragma unroll
    for (int cb = 0; cb < RB; ++cb) sb[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int cb = 0; cb < RB; ++cb) sb[cb] = mfma16x16x32<T>(kf[mt][s], qf[cb][s], sb[cb]);
#pragma unroll
    for (int cb = 0; cb < RB; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[cb][4 * mt + r] = sb[cb][r] * scale_log2;
  }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 vf[D / 16];
  const int i = 4 * g + (c >> 2);
#pragma unroll
  for (int n = 0; n < D / 16; ++n) {
    const uint8_t* at = vt + wide_v_at<D>(i, n) + (c & 3) * 8;
    const u32x2 lo = wide_read_tr(at), hi = wide_read_tr(at + 16 * 2 * D);
    vf[n] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
  __builtin_amdgcn_sched_barrier(0);
  if (__ballot(min(n0, n1) < 4)) {
#pragma unroll
    for (int cb = 0; cb < RB; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[cb][r] = r < n0 ? sc[cb][r] : -INFINITY;
        sc[cb][4 + r] = r < n1 ? sc[cb][4 + r] : -INFINITY;
      }
  }
  u32x4 ph[RB];
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) {
    float pr[8];
    softmax_step<8, D, false>(sc[cb], pr, st[cb]);
#pragma unroll
    for (int j = 0; j < 4; ++j) ph[cb][j] = pack2<T>(pr[2 * j], pr[2 * j + 1]);
  }
#pragma unroll
  for (int n = 0; n < D / 16; ++n)
#pragma unroll
    for (int cb = 0; cb < RB; ++cb) st[cb].acc[n] = mfma16x16x32<T>(vf[n], ph[cb], st[cb].acc[n]);
}

// The whole workgroup: rows (col_b, col_h) of every column, the range w, and
// the workspace split that takes the partials.
template <typename T, int BS, int D, int RB, int RG, int TG>
__device__ __forceinline__ void wide_attend(const DecodeParams& p, const WideWork& w, const int (&col_b)[RB],
                                            const int (&col_h)[RB], const bool (&col_ok)[RB], int ws,
                                            WideLds<WideShape<D, RB, RG, TG>>& lds) {
  using S = WideShape<D, RB, RG, TG>;
  constexpr int KS = D / 32;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int rg = wave % RG, tg = wave / RG;
  const int batches = max(0, w.limit - w.begin + S::kTokens - 1) / S::kTokens;

  int32_t page_a = wide_page<S, BS>(p, w, 0, wave);
  int32_t page_b = wide_page<S, BS>(p, w, 1, wave);
  int32_t next = wide_page<S, BS>(p, w, 2, wave);
  WideRegs<S> ra, rb;
  wide_load<S, BS>(p, w, 0, wave, lane, page_a, ra);
  wide_load<S, BS>(p, w, 1, wave, lane, page_b, rb);
  __builtin_amdgcn_sched_barrier(0);  // ahead of the rows' own loads and their wait
  u32x4 qf[RB][KS];
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) {
    const T* qrow = static_cast<const T*>(p.q) + col_b[cb] * p.qs0 +
                    (w.kvh * p.group + (col_ok[cb] ? col_h[cb] : 0)) * p.qs1;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * g);
      qf[cb][s] = col_ok[cb] ? x : u32x4{0u, 0u, 0u, 0u};
    }
  }
  WaveState<D> st[RB];
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) {
#pragma unroll
    for (int n = 0; n < D / 16; ++n) st[cb].acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    st[cb].m = -INFINITY;
    st[cb].l = 0.f;
  }
  // batch i: registers into LDS buffer i % 2, batch i + 2 into the registers,
  // then the barrier that also frees the other buffer
  int i = 0;
  // (a batch past the last is staged, empty, but not attended: one exit from the
  // loop, or the compiler merges the waits of an exit between the steps into the
  // next one's and drains the loads in flight)
  auto step = [&](int buf, WideRegs<S>& r, int32_t& page) {
    const int32_t after = wide_page<S, BS>(p, w, i + 3, wave);
    wide_stage<S, D>(p, w, i, wave, lane, page, r, lds, buf);
    page = next;
    next = after;
    wide_load<S, BS>(p, w, i + 2, wave, lane, page, r);
    __syncthreads();
    if (i < batches) wide_compute<T, S, D, RB>(qf, p.scale_log2, tg, c, g, lds, buf, st);
    ++i;
  };
  while (i < batches) {
    step(0, ra, page_a);
    step(1, rb, page_b);
  }

  // The token groups' states meet: column block cb in token group cb % TG, which
  // reads the other groups' accumulators from LDS (all of a block's reads ahead
  // of their first use).
  f32x4* slots = reinterpret_cast<f32x4*>(lds.stage);
  auto slot = [&](int cb, int t) { return slots + ((t * RG + rg) * RB + cb) * (D / 16) * 64 + lane; };
  float lt[RB];
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) lt[cb] = column_sum(st[cb].l);
  __syncthreads();  // every wave has read its last batch
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) {
    if (tg == cb % TG) continue;
    f32x4* to = slot(cb, (tg - cb % TG - 1 + TG) % TG);
#pragma unroll
    for (int n = 0; n < D / 16; ++n) to[n * 64] = st[cb].acc[n];
    if (g == 0) {
      lds.m[wave][2 * cb][c] = st[cb].m;
      lds.m[wave][2 * cb + 1][c] = lt[cb];
    }
  }
  __syncthreads();
#pragma unroll
  for (int cb = 0; cb < RB; ++cb) {
    if (tg != cb % TG) continue;
    f32x4 other[TG][D / 16];
    float om[TG], ol[TG];
#pragma unroll
    for (int t = 0; t < TG - 1; ++t) {
      const int from = (tg + 1 + t) % TG * RG + rg;
      om[t] = lds.m[from][2 * cb][c];
      ol[t] = lds.m[from][2 * cb + 1][c];
#pragma unroll
      for (int n = 0; n < D / 16; ++n) other[t][n] = slot(cb, t)[n * 64];
    }
    __builtin_amdgcn_sched_barrier(0);
    float M = st[cb].m;
#pragma unroll
    for (int t = 0; t < TG - 1; ++t) M = fmaxf(M, om[t]);
    const float Mu = M == -INFINITY ? 0.f : M;
    const float w0 = exp2_fast(st[cb].m - Mu);
    float L = w0 * lt[cb];
#pragma unroll
    for (int n = 0; n < D / 16; ++n) st[cb].acc[n] *= w0;
#pragma unroll
    for (int t = 0; t < TG - 1; ++t) {
      const float wt = exp2_fast(om[t] - Mu);
      L += wt * ol[t];
#pragma unroll
      for (int n = 0; n < D / 16; ++n) st[cb].acc[n] += other[t][n] * wt;
    }
    if (!col_ok[cb]) continue;
    const int qh = w.kvh * p.group + col_h[cb];
    float* a = p.acc + col_b[cb] * p.as0 + qh * p.as1 + ws * p.as2 + 4 * g;
#pragma unroll
    for (int n = 0; n < D / 16; ++n) *reinterpret_cast<f32x4*>(a + 16 * n) = st[cb].acc[n];
    if (g == 0) {
      const int64_t so = col_b[cb] * p.ss0 + qh * p.ss1 + ws * p.ss2;
      p.mx[so] = M;
      p.sm[so] = L;
    }
  }
}

}  // namespace fd
