// Co-ALiBi forward on gfx950.
//
// Semantics follow the reference forward (co_alibi_attn/co_alibi_fwd_kernel.py:46-127
// and model.py:13-40 with the per-head slope of co_alibi_attn.py:147):
//   p_ij   = sm_scale * q_i . k_j
//   s_ij   = sigmoid(p_ij) for valid (i, j), else 0     valid: j < Skv and (!causal or j <= i)
//   z_ij   = sum_{k >= j} s_ik                          (inclusive suffix over keys)
//   a_ij   = p_ij - slope_h * z_ij
//   O_i    = sum_j exp(a_ij - m_i) v_j / (sum_j exp(a_ij - m_i) + 1e-9)
//   LSE_i  = m_i + log(sum_j exp(a_ij - m_i) + 1e-9)
//
// One work-group = 128 query rows of one (batch, query head), 4 wavefronts of
// 32 rows.  Key tiles of 64 are walked from the causal diagonal leftwards so
// the suffix sum z is a running carry.  Per tile and wavefront:
//   S^T = K Q^T   (MFMA, keys on the accumulator rows: with the kRowOfReg
//                  permutation each lane holds 16 consecutive keys of one row)
//   sigmoid, suffix scan (in registers + one exchange with the other half),
//   penalty, online softmax (exp2, lazily rescaled), then
//   O^T += V^T P^T (MFMA, the P accumulators are reused as the B operand).
// K is staged in LDS row-major (rows permuted); V row-major, read as the
// transposed operand with ds_read_b64_tr_b16 (fp32 mode: V stored transposed).
// Besides O and LSE the kernel saves, per 128-row block, the first key it processed
// (kstart, the tail skip's record), and per row the sum R of the sigmoids of the keys it
// processed: backward pass 1 rebuilds z from it.  R is summed in fp64 over 32-key block
// totals, exactly the totals pass 1 computes (the same sigmoids summed in the same order), so
// the difference pass 1 takes is exact up to one rounding.
#include <algorithm>
#include <type_traits>

#include "coalibi_common.h"
#include "coalibi_kernels.h"

namespace coalibi {

namespace {

constexpr int kFwdBM = 128;  // query rows per work-group
constexpr int kFwdBN = 64;   // keys per tile
// Rescale O only when the running max grows by more than 2^8: P stays <= 256,
// exact in fp16/bf16 range, and O/LSE are renormalised to the true max at the end.
constexpr float kRescaleThreshold = 8.0f;

template <typename T, int D>
struct FwdCfg {
  static constexpr bool kTr = sizeof(T) == 2;  // V through LDS transpose reads
  static constexpr int CH = 16 / sizeof(T);
  // O^T is produced in 32-row tiles of the head dim: D = 16 runs on a 32-wide head dim whose
  // upper 16 columns of V are zero in LDS (written once, never loaded over).
  static constexpr int DP = D < 32 ? 32 : D;
  static constexpr int LDK = D + CH;       // sK row stride (elements)
  // sV: row-major [key][d] (stride keeps each 4-row transpose read on distinct
  // banks) or, in fp32 mode, transposed [d][key].
  static constexpr int LDV = kTr ? DP + 2 * CH : kFwdBN + CH;
  static constexpr int V_ELEMS = kTr ? kFwdBN * LDV : DP * LDV;
  static constexpr int KS = D / 16;        // k16 steps over the head dim
  static constexpr int DT = DP / 32;       // 32-row tiles of O^T
};

template <bool MASKED, bool CAUSAL>
__device__ __forceinline__ bool key_ok(int key, int row, int Skv) {
  if (!MASKED) return true;
  return key < Skv && (!CAUSAL || key <= row);
}

// One 64-key tile for one wavefront.  State: acc (O^T, scaled by 2^-m2), m2
// (log2-domain scale, -inf before the first visible key), lsum (this half's
// share of sum_j 2^(a_j - m2)), zr (sigmoid sum of all keys right of the tile, read only).
// Returns the sigmoid totals of the tile's two 32-key blocks, keys k0 + 32.. in btot[1] and k0..
// in btot[0] (the same values in both halves of the wavefront).
template <typename T, int D, bool CAUSAL, bool MASKED>
__device__ __forceinline__ void fwd_tile(const T* __restrict__ sK, const T* __restrict__ sV,
                                         const typename Mfma<T>::vec8 (&qf)[FwdCfg<T, D>::KS],
                                         f32x16 (&acc)[FwdCfg<T, D>::DT], float& m2, float& lsum,
                                         float zr, float (&btot)[2], int k0, int row, int lane, int Skv,
                                         float sc2, float lam2) {
  using C = FwdCfg<T, D>;
  using M = Mfma<T>;
  const int col = lane & 31, hh = lane >> 5;

  // S^T tile: two 32-key subtiles; register r of subtile st <-> key k0 + st*32 + hh*16 + r.
  f32x16 sacc[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    sacc[st] = f32x16{};
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks)
      sacc[st] = M::k16(ld_vec8(sK + (st * 32 + col) * C::LDK + ks * 16 + hh * 8), qf[ks], sacc[st]);
  }
  __builtin_amdgcn_sched_barrier(0);

  // sigma and its inclusive suffix sum inside each lane's 16-key run.
  float loc[2][16];
  float tot[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    float run = 0.f;
#pragma unroll
    for (int r = 15; r >= 0; --r) {
      float s = sigmoid_log2(sacc[st][r] * sc2);
      if (MASKED) s = key_ok<MASKED, CAUSAL>(k0 + st * 32 + hh * 16 + r, row, Skv) ? s : 0.f;
      run += s;
      loc[st][r] = run;
    }
    tot[st] = run;
  }
  // Run totals in key order (right to left): (1,1) (1,0) (0,1) (0,0), where (st, h) is
  // the 16-key run of subtile st held by wavefront half h.
  const float oth0 = other_half(tot[0]), oth1 = other_half(tot[1]);
  const float T11 = hh ? tot[1] : oth1, T10 = hh ? oth1 : tot[1];
  const float T01 = hh ? tot[0] : oth0, T00 = hh ? oth0 : tot[0];
  const float zst1 = (zr + T11) + T10;  // suffix sum from key k0 + 32
  const float off[2] = {hh ? zst1 : zst1 + T01, hh ? zr : zr + T11};
  btot[1] = T11 + T10;
  btot[0] = T01 + T00;

  // Log2-domain logit relative to the current scale:
  //   t - lam2 * (off + loc) - mb = fma(-lam2, loc, fma(s, sc2, -(mb + lam2 * off)))
  const float mb = m2 == kNegInf ? 0.f : m2;
  float mt = kNegInf;
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const float cst = mb + lam2 * off[st];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float av = fmaf(-lam2, loc[st][r], fmaf(sacc[st][r], sc2, -cst));
      if (MASKED) av = key_ok<MASKED, CAUSAL>(k0 + st * 32 + hh * 16 + r, row, Skv) ? av : kNegInf;
      sacc[st][r] = av;
      mt = fmaxf(mt, av);
    }
  }
  mt = fmaxf(mt, other_half(mt));
  const bool need = m2 == kNegInf ? mt > kNegInf : mt > kRescaleThreshold;
  if (__any(need)) {
    const float delta = need ? mt : 0.f;
    const float alpha = need ? (m2 == kNegInf ? 0.f : fast_exp2(-delta)) : 1.f;
    m2 = need ? mb + delta : m2;
    lsum *= alpha;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) acc[dt] *= alpha;
#pragma unroll
    for (int st = 0; st < 2; ++st) sacc[st] -= delta;
  }

  typename M::vec8 pb[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
#pragma unroll
    for (int mh = 0; mh < 2; ++mh) {
      f32x8 pv;
#pragma unroll
      for (int e = 0; e < 8; ++e) pv[e] = fast_exp2(sacc[st][mh * 8 + e]);
      pb[st][mh] = M::pack(pv);
      lsum = sum8(pb[st][mh], lsum);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // O^T[d][q] += V^T[d][key] P^T[key][q]; A rows are keys st*32 + hh*16 + mh*8 + e.
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int mh = 0; mh < 2; ++mh) {
        typename M::vec8 va;
        if constexpr (C::kTr)
          va = ld_kmajor<T, false>(sV, C::LDV, st * 32 + mh * 8, 16, dt * 32, lane);
        else
          va = ld_vec8(sV + (dt * 32 + col) * C::LDV + st * 32 + hh * 16 + mh * 8);
        acc[dt] = M::k16(va, pb[st][mh], acc[dt]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Work orders (coalibi_kernels.h), written by the first work-groups of the key-norm launch:
// one sorts the forward's and pass 1's row blocks, one pass 2's key blocks, largest
// predicted cost first.
constexpr int kOrderBuckets = 256;  // cost classes: ceil(extent / 256) keys or rows each
constexpr int kOrderLdsHeads = 1024;
constexpr int kOrderLdsItems = 8192;

struct ScheduleArgs {
  const float* slopes;
  int* row_order;  // NULL: not written
  int* key_order;  // NULL: not written
  int B, Hq, Hkv, Sq, Skv;
  int causal;
  int rows_sorted, keys_sorted;  // 0: the table holds its index order (too large to sort, or unused)
  float window;                  // order_window<T>()
};

// The lanes of the wavefront whose `b` equals this lane's (among the lanes with `ok`), matched
// bit by bit with ballots.
__device__ __forceinline__ unsigned long long same_bucket(int b, bool ok) {
  unsigned long long peers = __ballot(ok);
#pragma unroll
  for (int bit = 0; (1 << bit) < kOrderBuckets; ++bit) {
    const bool one = (b >> bit) & 1;
    const unsigned long long m = __ballot(one);
    peers &= one ? m : ~m;
  }
  return peers;
}

// Stable counting sort by one work-group of 256 threads: out[j] is the j-th of the n items in
// decreasing bucket order, the items of one bucket in index order.  Wavefront w takes the w-th
// quarter of the items and places them in chunks of 64, the lowest lane that holds a bucket moving
// its cursor.  The buckets are computed first, by all threads at once, and kept in LDS as bytes (for
// the first kOrderLdsItems items; the rest are computed again where they are needed), and counted
// with LDS atomics: computed chunk by chunk on each wavefront's critical path, twice, they made this
// work-group the longest of its launch (key-norm launch at the headline 19.5 -> 16.8 us, B1 H8 n
// 16384 D64 10.6 -> 7.2, B8 H12 n 1024 D64 10.5 -> 6.9).
// lds: 5 * kOrderBuckets ints.  cls: kOrderLdsItems bytes.
template <typename F>
__device__ void sort_items_desc(int n, const F& bucket, int* __restrict__ out, int* lds, unsigned char* cls, int tid) {
  constexpr int K = kOrderBuckets;
  static_assert(K == 256, "one thread per bucket in the scan, a byte per class");
  int* const cur = lds;          // [4][K]: per-wavefront counts, then per-wavefront cursors
  int* const part = lds + 4 * K;  // [4]: per-wavefront scan totals
  const int lane = tid & 63, wave = tid >> 6;
  const int per = (n + 3) / 4;
  const int lo = min(wave * per, n), hi = min(lo + per, n);
  for (int j = tid; j < 4 * K; j += 256) cur[j] = 0;
  __syncthreads();
  for (int i = tid; i < n; i += 256) {
    const int b = bucket(i);
    if (i < kOrderLdsItems) cls[i] = (unsigned char)b;
    atomicAdd(&cur[i / per * K + b], 1);
  }
  __syncthreads();
  auto bucket_of = [&](int i) { return i < kOrderLdsItems ? (int)cls[i] : bucket(i); };
  // Thread t owns bucket K - 1 - t (descending): its total over the wavefronts, an exclusive
  // scan over the threads, then each wavefront's cursor for the bucket.
  const int bk = K - 1 - tid;
  int c[4], tot = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) tot += (c[w] = cur[w * K + bk]);
  int incl = tot;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int start = incl - tot;
  for (int w = 0; w < wave; ++w) start += part[w];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    cur[w * K + bk] = start;
    start += c[w];
  }
  __syncthreads();
  int* const mine = cur + wave * K;
  int next = lo + lane < hi ? bucket_of(lo + lane) : 0;  // one chunk ahead
  for (int base = lo; base < hi; base += 64) {
    const int i = base + lane, b = next;
    const bool ok = i < hi;
    next = i + 64 < hi ? bucket_of(i + 64) : 0;
    const unsigned long long peers = same_bucket(b, ok);
    if (ok) {
      // LDS operations of the wavefront complete in program order: every lane reads the
      // cursor before its lowest lane moves it.
      const int before = __popcll(peers & ((1ull << lane) - 1));
      const int at = mine[b];
      out[at + before] = i;
      if (before == 0) mine[b] = at + __popcll(peers);
    }
  }
}

// Per query head, the keys (or rows) a row block (or key block) keeps at most: window / slope,
// or +inf for a slope that skips nothing (<= 0 or NaN).  Held in LDS for the first
// kOrderLdsHeads heads; the others are computed where they are needed.
struct HeadWindow {
  const float* __restrict__ slopes;
  const float* lds;
  float window;
  __device__ float operator()(int h) const {
    if (h < kOrderLdsHeads) return lds[h];
    const float lam = slopes[h];
    return lam > 0.f ? window / lam : __builtin_inff();
  }
};

// Cost class of a row block (item rank * heads + bh, rank 0 = the last row block): the keys
// it processes, up to its diagonal (causal) and at most its head's window, in units of
// ceil(Skv / kOrderBuckets) keys.
struct RowCost {
  HeadWindow win;
  int heads, Hq, nQB, Skv, causal;
  float unit;
  __device__ int operator()(int i) const {
    const int rank = i / heads, bh = i - rank * heads;
    const int qb = nQB - 1 - rank;
    const float keys = causal ? (float)min((qb + 1) * kSkipRows, Skv) : (float)Skv;
    return min((int)(fminf(keys, win(bh % Hq)) / unit), kOrderBuckets - 1);
  }
};

// Cost class of a 64-key block (item kb * heads + bh; one query head per key head): the query
// rows that see it (causal: rows from its first key on), at most the head's window, in units
// of ceil(Sq / kOrderBuckets) rows.
struct KeyCost {
  HeadWindow win;
  int heads, H, Sq, causal;
  float unit;
  __device__ int operator()(int i) const {
    const int kb = i / heads, bh = i - kb * heads;
    const float rows = causal ? (float)max(Sq - kb * kOrderKeyBlock, 0) : (float)Sq;
    return min((int)(fminf(rows, win(bh % H)) / unit), kOrderBuckets - 1);
  }
};

// Work-group 0 writes the row order, work-group 1 the key order.  Every element of both tables
// is written (the statistics are an output): a table that is not sorted holds its index order,
// and the key table's room for B*Hq*nKB entries past its B*Hkv*nKB items holds zeros.
__device__ void schedule_orders(const ScheduleArgs& s, int which, int tid) {
  __shared__ int lds[5 * kOrderBuckets];
  __shared__ float wlds[kOrderLdsHeads];
  __shared__ unsigned char cls[kOrderLdsItems];
  for (int h = tid; h < min(s.Hq, kOrderLdsHeads); h += 256) {
    const float lam = s.slopes[h];
    wlds[h] = lam > 0.f ? s.window / lam : __builtin_inff();
  }
  __syncthreads();
  const HeadWindow win{s.slopes, wlds, s.window};
  if (which == 0) {
    const int nQB = (s.Sq + kSkipRows - 1) / kSkipRows;
    const int n = nQB * s.B * s.Hq;
    if (s.rows_sorted) {
      const RowCost cost{win, s.B * s.Hq, s.Hq, nQB, s.Skv, s.causal,
                         (float)((s.Skv + kOrderBuckets - 1) / kOrderBuckets)};
      sort_items_desc(n, cost, s.row_order, lds, cls, tid);
    } else {
      for (int i = tid; i < n; i += 256) s.row_order[i] = i;
    }
  } else {
    const int nKB = stats_key_block_count(s.Skv);
    const int n = nKB * s.B * s.Hkv;
    if (s.keys_sorted) {
      const KeyCost cost{win, s.B * s.Hkv, s.Hkv, s.Sq, s.causal,
                         (float)((s.Sq + kOrderBuckets - 1) / kOrderBuckets)};
      sort_items_desc(n, cost, s.key_order, lds, cls, tid);
    } else {
      for (int i = tid; i < n; i += 256) s.key_order[i] = i;
    }
    for (int i = n + tid; i < nKB * s.B * s.Hq; i += 256) s.key_order[i] = 0;
  }
}

// max over each chunk of kNormKeys keys of |k|_2, per key head: the key side of the tail
// skip's bound.  One work-group per (head, chunk) over B*Hq heads: the buffer has room for
// B*Hq rows, and rows past the B*Hkv key heads are written as zero, so every element of
// the forward's statistics is written (deterministic outputs).  The D/CH lanes that hold one key row's 16-byte chunks
// sum their squares with xor shuffles.  A NaN norm is kept (fmaxf would drop it), so a
// non-finite key disables the skip for its head.
// The first nSched work-groups of the launch write the work orders instead.
template <typename T, int D>
__global__ __launch_bounds__(256) void coalibi_key_norm_kernel(const T* __restrict__ k, Layout kl,
                                                               float* __restrict__ knorm, int Skv, int nKC,
                                                               int nKeyHeads, int nSched, ScheduleArgs sched) {
  constexpr int CH = 16 / (int)sizeof(T);  // elements per 16-byte chunk
  constexpr int CPR = D / CH;              // chunks (lanes) per key row: 2 .. 32
  constexpr int RPP = 256 / CPR;           // key rows per pass of the work-group
  static_assert(CPR >= 2 && CPR <= 64 && (CPR & (CPR - 1)) == 0, "a key row spans a power-of-two lane group");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if ((int)blockIdx.x < nSched) {
    schedule_orders(sched, blockIdx.x, tid);
    return;
  }
  const int id = blockIdx.x - nSched;
  const int bhk = id / nKC, c = id - bhk * nKC;
  if (bhk >= nKeyHeads) {
    if (tid == 0) knorm[(size_t)bhk * nKC + c] = 0.f;
    return;
  }
  // Every load of the chunk goes out before any is used, through a buffer resource over the
  // chunk's valid rows (rows past Skv read as zero, whose norm 0 leaves the maximum alone).
  constexpr int NP = kNormKeys / RPP;  // passes over the chunk
  const int r0 = c * kNormKeys;
  const __amdgpu_buffer_rsrc_t rs = tile_rsrc(
      head_at(k, kl, bhk / sched.Hkv, bhk % sched.Hkv) + (size_t)r0 * kl.r, row_span(min(kNormKeys, Skv - r0), kl.r, D));
  u32x4 x[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p)
    x[p] = __builtin_amdgcn_raw_buffer_load_b128(rs, ((p * RPP + tid / CPR) * kl.r + (tid % CPR) * CH) * (int)sizeof(T),
                                                 0, 0);
  float best = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const typename VecOf<T, CH>::type xv = __builtin_bit_cast(typename VecOf<T, CH>::type, x[p]);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < CH; ++e) ss = fmaf((float)xv[e], (float)xv[e], ss);
#pragma unroll
    for (int off = CPR / 2; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
    best = ss != ss ? ss : fmaxf(best, ss);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float o = __shfl_xor(best, off);
    best = o != o ? o : fmaxf(best, o);
  }
  __shared__ float red[4];
  if (lane == 0) red[wave] = best;
  __syncthreads();
  if (tid == 0) {
    float m = red[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) m = red[w] != red[w] ? red[w] : fmaxf(m, red[w]);
    knorm[(size_t)bhk * nKC + c] = sqrtf(m);
  }
}

// One 128-row block (bh, qb) by a work-group of 4 wavefronts, 32 rows each, over tiles in sK and sV.
// SKIP: the tail skip (args.knorm holds the key norms); without it every key is processed and
// the code carries none of the skip's per-tile test.  PLAIN: every operand is contiguous, and the
// strides are constants (in registers they cost the grouped-query forward 1.7 %, n 8192 bf16).
template <typename T, int D, bool CAUSAL, bool SKIP, bool PLAIN>
__device__ __forceinline__ void fwd_row_block(const FwdArgs& args, int bh, int qb, T* __restrict__ sK,
                                              T* __restrict__ sV) {
  using C = FwdCfg<T, D>;
  using M = Mfma<T>;
  using vec8 = typename M::vec8;
  using KTile = TileLoader<T, D, kFwdBN>;
  using VTile = TileLoader<T, D, kFwdBN, !FwdCfg<T, D>::kTr>;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, hh = lane >> 5;
  const int Sq = args.Sq, Skv = args.Skv;
  const int nQB = (Sq + kFwdBM - 1) / kFwdBM;
  const int b = bh / args.Hq, hq = bh - b * args.Hq;
  const int hkv = hq / (args.Hq / args.Hkv);
  const Layout rows_q = contiguous_layout(args.Hq, Sq, D), rows_kv = contiguous_layout(args.Hkv, Skv, D);
  const Layout ql = PLAIN ? rows_q : args.ql, ol = PLAIN ? rows_q : args.ol;
  const Layout kl = PLAIN ? rows_kv : args.kl, vl = PLAIN ? rows_kv : args.vl;
  const T* __restrict__ Qp = head_at(static_cast<const T*>(args.q), ql, b, hq);
  const T* __restrict__ Kp = head_at(static_cast<const T*>(args.k), kl, b, hkv);
  const T* __restrict__ Vp = head_at(static_cast<const T*>(args.v), vl, b, hkv);
  const int ldk = kl.r, ldv = ldk;  // K and V share a row stride
  const float lam2 = args.slopes[hq] * kLog2e;
  const float sc2 = args.sc2;
  if constexpr (D < C::DP) {  // the padding columns of V stay zero: tiles only write the D real ones
    lds_zero(sV, C::V_ELEMS * (int)sizeof(T), tid, 256);
  }

  const int q0 = qb * kFwdBM;
  const int wrow0 = q0 + wave * 32;
  const int row = wrow0 + col;
  const bool row_ok = row < Sq;

  // 16-bit types: Q pre-scaled by sm_scale*log2(e) (one rounding per element, far below the
  // input precision's effect on q.k), so the tile math takes the scale 1 and multiplies by nothing.
  constexpr bool kPreScaled = sizeof(T) == 2;
  // The reads before the first tile go out together and share one round trip: the Q
  // fragments, the first K / V tile and (tail skip) the key-norm chunk maxima.
  // Q through a buffer resource over the block's valid rows: rows past Sq read as zero.
  vec8 qf[C::KS];
  {
    const __amdgpu_buffer_rsrc_t qrs = tile_rsrc(Qp + (size_t)q0 * ql.r, row_span(min(Sq - q0, kFwdBM), ql.r, D));
    const int qoffb = ((wave * 32 + col) * ql.r + hh * 8) * (int)sizeof(T);
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) qf[ks] = buffer_load_vec8<vec8>(qrs, qoffb + ks * 16 * (int)sizeof(T));
  }
  const int last_key = CAUSAL ? min(q0 + kFwdBM - 1, Skv - 1) : Skv - 1;
  const int nkt = last_key / kFwdBN + 1;
  KTile kt_regs;
  VTile vt_regs;
  kt_regs.template load<!PLAIN>(Kp, (nkt - 1) * kFwdBN, Skv, tid, ldk);
  vt_regs.template load<!PLAIN>(Vp, (nkt - 1) * kFwdBN, Skv, tid, ldv);
  const bool tail_skip = SKIP && lam2 > 0.f;
  float km = 0.f;
  if (tail_skip) {
    const float* kn = args.knorm + ((size_t)b * args.Hkv + hkv) * args.nKC;
    for (int c = tid; c < args.nKC; c += 256) km = kn[c] != kn[c] ? kn[c] : fmaxf(km, kn[c]);
  }
  if constexpr (kPreScaled) {
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) qf[ks] = scale_vec8<T>(qf[ks], sc2);
  }
  const float tile_sc2 = kPreScaled ? 1.0f : sc2;

  // Tail skip (coalibi_kernels.h): this row's bound on |t| in log2 units, |q| * max|k| with
  // the scale (folded into q in 16-bit types), with a margin for the rounding of the norms
  // and of the fp32 dot products.
  // The bound stays in LDS (one per row) rather than in a register across the tile loop.
  __shared__ float sKmax[4];
  __shared__ float sBound[kFwdBM];
  __shared__ int sDone[4];
  if (tail_skip) {
    float qq = 0.f;
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) qq = fmaf((float)qf[ks][e], (float)qf[ks][e], qq);
    qq += other_half(qq);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float o = __shfl_xor(km, off);
      km = o != o ? o : fmaxf(km, o);
    }
    if (lane == 0) sKmax[wave] = km;
    __syncthreads();
    km = sKmax[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) km = sKmax[w] != sKmax[w] ? sKmax[w] : fmaxf(km, sKmax[w]);
    if (hh == 0) sBound[wave * 32 + col] = sqrtf(qq) * km * (kPreScaled ? 1.0f : sc2) * 1.001f + 1e-3f;
  }
  int kfirst = 0;  // first key of the leftmost tile processed

  f32x16 acc[C::DT];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) acc[dt] = f32x16{};
  // zsum: the sigmoid sum of the keys processed so far (right of the current tile), in fp64;
  // zr, its fp32 value, is the running offset of the tile's z.
  float m2 = kNegInf, lsum = 0.f, zr = 0.f;
  double zsum = 0.0;
  if (args.flags != nullptr && blockIdx.x == 0 && tid < kStatsHeader) args.flags[tid] = tid == 0 ? args.order_flags : 0;

  int kt_end = 0;  // the loop's lower bound, raised by the tail skip
  for (int kt = nkt - 1; kt >= kt_end; --kt) {
    __syncthreads();
    // Every wavefront's rows passed the tail test after tile kt + 1: the keys left of it
    // carry weights below 2^-skip_log2<T>() (the vote is uniform, so all wavefronts leave here).
    // Leaving through the loop bound rather than a break keeps the loop's register
    // allocation as it is without the skip (a break costs 13 spilled registers at D = 128, the
    // test after the LDS stores 50).
    if (tail_skip && kt < nkt - 1 && (sDone[0] & sDone[1] & sDone[2] & sDone[3])) {
      kfirst = (kt + 1) * kFwdBN;
      kt_end = kt + 1;
      continue;
    }
    kt_regs.store_rows(sK, C::LDK, tid);
    if constexpr (C::kTr)
      vt_regs.template store_rows<false>(sV, C::LDV, tid);
    else
      vt_regs.store_cols(sV, C::LDV, tid);
    __syncthreads();
    // The next tile's K / V go into registers during this tile's math; at D = 256 those
    // registers do not fit beside the tile state, and the loads are issued after it.
    constexpr bool kPrefetchKV = D <= 128;
    if (kPrefetchKV && kt > 0) {
      kt_regs.template load<!PLAIN>(Kp, (kt - 1) * kFwdBN, Skv, tid, ldk);
      vt_regs.template load<!PLAIN>(Vp, (kt - 1) * kFwdBN, Skv, tid, ldv);
    }
    const int k0 = kt * kFwdBN;
    const bool skip = CAUSAL && k0 > wrow0 + 31;  // every key of the tile is above this wavefront's rows
    if (skip) {
      if (!kPrefetchKV && kt > 0) {
        kt_regs.template load<!PLAIN>(Kp, (kt - 1) * kFwdBN, Skv, tid, ldk);
        vt_regs.template load<!PLAIN>(Vp, (kt - 1) * kFwdBN, Skv, tid, ldv);
      }
      if (tail_skip && lane == 0) sDone[wave] = Sq <= wrow0;  // no visible key yet: only rows past Sq pass
      continue;
    }
    const bool masked = (CAUSAL && k0 + kFwdBN - 1 > wrow0) || (k0 + kFwdBN > Skv);
    float btot[2];
    if (masked)
      fwd_tile<T, D, CAUSAL, true>(sK, sV, qf, acc, m2, lsum, zr, btot, k0, row, lane, Skv, tile_sc2, lam2);
    else
      fwd_tile<T, D, CAUSAL, false>(sK, sV, qf, acc, m2, lsum, zr, btot, k0, row, lane, Skv, tile_sc2, lam2);
    zsum += (double)btot[1];  // right block first, as the keys are walked
    zsum += (double)btot[0];
    zr = (float)zsum;
    if (!kPrefetchKV && kt > 0) {
      kt_regs.template load<!PLAIN>(Kp, (kt - 1) * kFwdBN, Skv, tid, ldk);
      vt_regs.template load<!PLAIN>(Vp, (kt - 1) * kFwdBN, Skv, tid, ldv);
    }
    if (tail_skip) {
      // Every key left of k0 has z >= zr, so its weight is at most 2^(bound - lam2*zr - m2).
      const bool done =
          !row_ok || (m2 != kNegInf && sBound[wave * 32 + col] - lam2 * zr - m2 < -skip_log2<T>());
      const bool all = __all(done);
      if (lane == 0) sDone[wave] = all;
    }
  }
  if (args.kstart != nullptr && tid == 0) args.kstart[(size_t)bh * nQB + qb] = kfirst;

  // O = acc / l and LSE = m + log(l) with l = sum_j 2^(a_j - m2) >= 1 (m2 is one of
  // the a_j and at most 8 below their max): the reference's "+1e-9" in l + 1e-9
  // (co_alibi_fwd_kernel.py:115,120) is below fp32 resolution and is omitted.
  const float ltot = lsum + other_half(lsum);
  const float inv = ltot > 0.f ? 1.0f / ltot : 0.f;
  if (row_ok) {
    T* __restrict__ Orow = head_at(static_cast<T*>(args.o), ol, b, hq) + (size_t)row * ol.r;
    using vec4 = typename VecOf<T, 4>::type;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (dt * 32 + g * 8 >= D) continue;  // padding rows of O^T (D = 16)
        f32x4 v4 = {acc[dt][g * 4 + 0] * inv, acc[dt][g * 4 + 1] * inv, acc[dt][g * 4 + 2] * inv,
                    acc[dt][g * 4 + 3] * inv};
        *reinterpret_cast<vec4*>(Orow + dt * 32 + g * 8 + hh * 4) = __builtin_convertvector(v4, vec4);
      }
    }
    if (hh == 0 && args.lse != nullptr)
      args.lse[(size_t)bh * Sq + row] = ltot > 0.f ? (m2 + log2f(ltot)) * kLn2 : kNegInf;
    if (hh == 0 && args.rsum != nullptr) {  // R as hi + lo, exact to about 2^-48 of it
      const float hi = (float)zsum;
      args.rsum[(size_t)bh * Sq + row] = hi;
      args.rsum[(size_t)args.B * args.Hq * Sq + (size_t)bh * Sq + row] = (float)(zsum - (double)hi);
    }
  }
}

// PER_CU: work-groups per CU that the registers are to allow.
template <typename T, int D, bool CAUSAL, bool SKIP, bool PLAIN, int PER_CU>
__global__ __launch_bounds__(256, PER_CU) void coalibi_fwd_kernel(FwdArgs args) {
  using C = FwdCfg<T, D>;
  __shared__ __align__(16) T sK[kFwdBN * C::LDK];
  __shared__ __align__(16) T sV[C::V_ELEMS];
  const int nQB = (args.Sq + kFwdBM - 1) / kFwdBM;
  const WorkItem item = args.row_order ? table_item(args.row_order, blockIdx.x, args.B * args.Hq, gridDim.x)
                                       : lpt_item(blockIdx.x, args.B * args.Hq, 1);
  // rank 0: the longest causal rows
  fwd_row_block<T, D, CAUSAL, SKIP, PLAIN>(args, item.head, nQB - 1 - item.rank, sK, sV);
}

// ---------------------------------------------------------------------------
// Small grids.  With fewer row blocks than the GPU has room for, a 128-row block's walk over its
// keys is the time: one wavefront per SIMD takes about 2.4 us per 64-key tile, whatever the rest
// of the GPU does.  Here a row block is four work-groups of 32 rows, and a work-group's four
// wavefronts take the four 32-key tiles of every 128-key step, each from LDS tiles of its own
// filled by its own DMA (the decode's scheme).  The walk is a quarter as long, over four times the
// work-groups.  What it costs: K and V are read from L2 four times as often, so it loses where
// the GPU is full.
//   Per step each wavefront computes its tile's S^T and sigmoids; the tiles' sigmoid totals go
// through LDS (one barrier), so that z is absolute in every wavefront; the softmax state is a
// wavefront's own and the four are combined at the end.

template <typename T, int D>
struct SplitCfg {
  static constexpr bool kTr = sizeof(T) == 2;
  static constexpr int CH = 16 / (int)sizeof(T);
  static constexpr int DP = D < 32 ? 32 : D;
  static constexpr int LDK = DP + CH;
  static constexpr int LDV = kTr ? DP + 2 * CH : DP + CH;
  using KTile = DmaTile<T, D, kWaveKeys, LDK, 1, true>;
  using VTile = DmaTile<T, D, kWaveKeys, LDV, 1, false>;
  static constexpr int K_ELEMS = KTile::LDS_ELEMS;  // a wavefront's K tile
  static constexpr int V_ELEMS = VTile::LDS_ELEMS;
  static constexpr int KS = D / 16;
  static constexpr int DT = DP / 32;
  // At the end the O partials of rows 0..15 alias a wavefront's K tile, of rows 16..31 its V tile.
  static constexpr int LDO = DP + 4;  // floats
  static_assert(16 * LDO * 4 <= K_ELEMS * (int)sizeof(T) && 16 * LDO * 4 <= V_ELEMS * (int)sizeof(T),
                "O partials alias the tiles");
  // The whole-block form runs in the same LDS.
  static_assert(kSplitWaves * K_ELEMS >= kFwdBN * FwdCfg<T, D>::LDK && kSplitWaves * V_ELEMS >= FwdCfg<T, D>::V_ELEMS,
                "the 64-key tiles fit");
  static constexpr size_t kLds = (size_t)kSplitWaves * (K_ELEMS + V_ELEMS) * sizeof(T);
  // fp32 at D = 256 takes 266 KB, above a CU's 160.
  static constexpr bool kFits = split_fits(sizeof(T), D);
  static_assert(!kFits || kLds <= 155 * 1024, "the tiles fit a CU");
};

// Which row blocks a launch splits: those of `keys` visible keys, longer than `longer_than`, of a head
// that the tail skip stops after about window / slope keys, where that is not much sooner than the
// split walk's end.  The tail skip's record is per 128-row block, so the split form has no skip
// and records that it processed every key.  With the skip switched off the window is infinite.
struct SplitRule {
  float window;
  float reach, slack;  // split up to reach * window / slope + slack keys
  int longer_than;
  __device__ __forceinline__ bool operator()(int keys, float slope) const {
    return keys > longer_than && (!(slope > 0.f) || (float)keys <= reach * (window / slope) + slack);
  }
};

template <typename T, int D, bool CAUSAL>
__device__ __forceinline__ void fwd_split_rows(const FwdArgs& args, int bh, int q0, T* __restrict__ sK,
                                               T* __restrict__ sV) {
  using C = SplitCfg<T, D>;
  using M = Mfma<T>;
  using vec8 = typename M::vec8;
  __shared__ float sSig[2][kSplitWaves][kSplitRows];  // the tiles' sigmoid totals, by step parity
  __shared__ float sMax[kSplitWaves][kSplitRows];
  __shared__ float sSum[kSplitWaves][kSplitRows];
  __shared__ float sInv[kSplitRows];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hh = lane >> 5;
  const int Sq = args.Sq, Skv = args.Skv;
  const int b = bh / args.Hq, hq = bh - b * args.Hq;
  const int hkv = hq / (args.Hq / args.Hkv);
  const T* __restrict__ Kp = head_at(static_cast<const T*>(args.k), args.kl, b, hkv);
  const T* __restrict__ Vp = head_at(static_cast<const T*>(args.v), args.vl, b, hkv);
  const int ldq = args.ql.r, ldk = args.kl.r, ldv = ldk;
  T* const sKw = sK + wave * C::K_ELEMS;  // this wavefront's tiles
  T* const sVw = sV + wave * C::V_ELEMS;
  const float lam2 = args.slopes[hq] * kLog2e;
  const int row = q0 + col;

  // Tiles n32 - 1 .. 0, four per step from the right; tile t < 0 holds no key (zero rows).
  const int n32 = (CAUSAL ? min(q0 + kSplitRows - 1, Skv - 1) : Skv - 1) / kWaveKeys + 1;
  const int steps = (n32 + kSplitWaves - 1) / kSplitWaves;
  int t = n32 - kSplitWaves + wave;
  // Untracked DMA: the tiles are this wavefront's own, and the waits below order it.
  typename C::KTile kdma;
  typename C::VTile vdma;
  kdma.init(0, lane, ldk);
  vdma.init(0, lane, ldv);
  const unsigned lds_k = lds_address(sKw), lds_v = lds_address(sVw);
  auto issue_k = [&](int tt) { kdma.issue_untracked(Kp, max(tt, 0) * kWaveKeys, tt < 0 ? 0 : Skv, lds_k, 0, ldk); };
  auto issue_v = [&](int tt) { vdma.issue_untracked(Vp, max(tt, 0) * kWaveKeys, tt < 0 ? 0 : Skv, lds_v, 0, ldv); };
  vec8 qf[C::KS];
  {
    const __amdgpu_buffer_rsrc_t qrs =
        tile_rsrc(head_at(static_cast<const T*>(args.q), args.ql, b, hq) + (size_t)q0 * ldq,
                  row_span(min(Sq - q0, kSplitRows), ldq, D));
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks)
      qf[ks] = buffer_load_vec8<vec8>(qrs, (col * ldq + ks * 16 + hh * 8) * (int)sizeof(T));
  }
  issue_k(t);
  issue_v(t);
  constexpr bool kPreScaled = sizeof(T) == 2;  // as in fwd_row_block
  if constexpr (kPreScaled) {
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) qf[ks] = scale_vec8<T>(qf[ks], args.sc2);
  }
  const float sc2 = kPreScaled ? 1.0f : args.sc2;

  f32x16 acc[C::DT];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) acc[dt] = f32x16{};
  float m2 = kNegInf, lsum = 0.f;
  double zsum = 0.0;  // the sigmoids of the keys right of the step, as fwd_row_block sums them

  for (int s = 0; s < steps; ++s, t -= kSplitWaves) {
    const bool more = s + 1 < steps;
    const int key0 = t * kWaveKeys + hh * 16;  // key of register 0
    // This step's K has landed once at most its V (issued after it) is outstanding.
    wait_vm<C::VTile::NINSTR>();
    f32x16 sacc = f32x16{};
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks)
      sacc = M::k16(ld_vec8(sKw + col * C::LDK + ks * 16 + hh * 8), qf[ks], sacc);
    if (more) {  // the K tile has been read: the next one lands in it during this step's math
      wait_lds();
      issue_k(t - kSplitWaves);
    }
    // Register r is a visible key iff r < nvis.
    const bool masked = t < 0 || (CAUSAL && t * kWaveKeys + kWaveKeys - 1 > q0) || (t + 1) * kWaveKeys > Skv;
    const int nvis = t < 0 ? 0 : min(Skv, CAUSAL ? row + 1 : Skv) - key0;
    float loc[16], tot = 0.f;
    if (masked) {
#pragma unroll
      for (int r = 15; r >= 0; --r) loc[r] = tot += r < nvis ? sigmoid_log2(sacc[r] * sc2) : 0.f;
    } else {
#pragma unroll
      for (int r = 15; r >= 0; --r) loc[r] = tot += sigmoid_log2(sacc[r] * sc2);
    }
    const float oth = other_half(tot);
    const float upper = hh ? tot : oth, lower = hh ? oth : tot;  // keys 16..31 and 0..15 of the tile
    if (hh == 0) sSig[s & 1][wave][col] = upper + lower;
    lds_barrier();  // the DMA stays in flight
    float zr = 0.f;
#pragma unroll
    for (int w = kSplitWaves - 1; w >= 0; --w) {  // right to left
      if (w == wave) zr = (float)zsum;
      zsum += (double)sSig[s & 1][w][col];
    }

    // As fwd_tile, for one 32-key subtile.
    const float mb = m2 == kNegInf ? 0.f : m2;
    const float cst = mb + lam2 * (hh ? zr : zr + upper);
    float mt = kNegInf;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sacc[r] = fmaf(-lam2, loc[r], fmaf(sacc[r], sc2, -cst));
      if (masked) sacc[r] = r < nvis ? sacc[r] : kNegInf;
      mt = fmaxf(mt, sacc[r]);
    }
    mt = fmaxf(mt, other_half(mt));
    const bool need = m2 == kNegInf ? mt > kNegInf : mt > kRescaleThreshold;
    if (__any(need)) {
      const float delta = need ? mt : 0.f;
      const float alpha = need ? (m2 == kNegInf ? 0.f : fast_exp2(-delta)) : 1.f;
      m2 = need ? mb + delta : m2;
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt) acc[dt] *= alpha;
      sacc -= delta;
    }
    vec8 pb[2];
#pragma unroll
    for (int mh = 0; mh < 2; ++mh) {
      f32x8 pv;
#pragma unroll
      for (int e = 0; e < 8; ++e) pv[e] = fast_exp2(sacc[mh * 8 + e]);
      pb[mh] = M::pack(pv);
      lsum = sum8(pb[mh], lsum);
    }
    // This step's V has landed once at most the next step's K is outstanding.
    if (more)
      wait_vm<C::KTile::NINSTR>();
    else
      wait_vm<0>();
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
      for (int mh = 0; mh < 2; ++mh)
        acc[dt] = M::k16(ld_kmajor_any<T, false>(sVw, C::LDV, mh * 8, 16, dt * 32, lane), pb[mh], acc[dt]);
    if (more) {
      wait_lds();  // the V tile has been read
      issue_v(t - kSplitWaves);
    }
  }

  // Combine the four wavefronts' softmax states.
  const float lown = lsum + other_half(lsum);
  if (hh == 0) {
    sMax[wave][col] = m2;
    sSum[wave][col] = lown;
  }
  __syncthreads();
  float m = kNegInf, l = 0.f;
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) m = fmaxf(m, sMax[w][col]);
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) {
    const float mw = sMax[w][col];
    l += mw == kNegInf ? 0.f : sSum[w][col] * fast_exp2(mw - m);
  }
  const float own = m2 == kNegInf ? 0.f : fast_exp2(m2 - m);
  auto o_row = [&](int w, int r) {
    return reinterpret_cast<float*>(r < 16 ? sK + w * C::K_ELEMS : sV + w * C::V_ELEMS) + (r & 15) * C::LDO;
  };
  float* const orow = o_row(wave, col);
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(orow + dt * 32 + g * 8 + hh * 4) =
          f32x4{acc[dt][g * 4] * own, acc[dt][g * 4 + 1] * own, acc[dt][g * 4 + 2] * own, acc[dt][g * 4 + 3] * own};
  if (wave == 0 && hh == 0) {
    sInv[col] = l > 0.f ? 1.0f / l : 0.f;
    if (row < Sq) {
      const size_t at = (size_t)bh * Sq + row;
      if (args.lse != nullptr) args.lse[at] = l > 0.f ? (m + log2f(l)) * kLn2 : kNegInf;
      if (args.rsum != nullptr) {
        const float hi = (float)zsum;
        args.rsum[at] = hi;
        args.rsum[(size_t)args.B * args.Hq * Sq + at] = (float)(zsum - (double)hi);
      }
    }
  }
  __syncthreads();
  const int r = tid >> 3;
  if (q0 + r < Sq) {
    using vec4 = typename VecOf<T, 4>::type;
    T* __restrict__ Orow = head_at(static_cast<T*>(args.o), args.ol, b, hq) + (size_t)(q0 + r) * args.ol.r;
    const float inv = sInv[r];
#pragma unroll
    for (int c = (tid & 7) * 4; c < D; c += 32) {
      f32x4 v = *reinterpret_cast<const f32x4*>(o_row(0, r) + c);
#pragma unroll
      for (int w = 1; w < kSplitWaves; ++w) v += *reinterpret_cast<const f32x4*>(o_row(w, r) + c);
      *reinterpret_cast<vec4*>(Orow + c) = __builtin_convertvector(v * inv, vec4);
    }
  }
}

// Work-groups 8j .. 8j + 7 of every 32 run on the 8 XCDs: item (id / 32) * 8 + id % 8, so that the
// four parts of a row block share their K and V in one XCD's L2.  Within an XCD the ids go to its four
// shader engines in turn; which part takes which turn rotates, since a block that is not split runs
// as its part 0 alone (without the rotation all of them share one engine).
template <typename T, int D, bool CAUSAL, bool SKIP>
__global__ __launch_bounds__(256, D * sizeof(T) > 256 ? 1 : 2) void coalibi_fwd_split_kernel(FwdArgs args,
                                                                                               int items, SplitRule rule,
                                                                                               bool small) {
  const bool by_head = small && CAUSAL;
  using C = SplitCfg<T, D>;
  __shared__ __align__(16) T sK[kSplitWaves * C::K_ELEMS];
  __shared__ __align__(16) T sV[kSplitWaves * C::V_ELEMS];
  int i = (blockIdx.x >> 5) * 8 + (blockIdx.x & 7), part = ((blockIdx.x >> 3) + (blockIdx.x >> 5)) & 3;
  if (!small) {
    // Most blocks are whole, and a work-group that only exits still waits for a slot on its engine,
    // holding up the ids after it: every part 0 first, then the others.
    const int first = (items + 7) / 8 * 8, rest = (int)blockIdx.x - first;
    i = rest < 0 ? (int)blockIdx.x : rest / 24 * 8 + (rest & 7);
    part = rest < 0 ? 0 : 1 + (rest >> 3) % 3;
  }
  if (i >= items) return;
  // by_head: a head's blocks on one XCD where the heads are a multiple of 8 (on two with 4 or 12, on four
  // with 2 or 6), where its K and V stay in one L2 (fp32, B2 H12 n 1000:
  // 78.3 -> 58.4 us against the sorted order; n 512 to 2048 fp16: 3 to 13 %).  Non-causal heads differ
  // more in work, and the sorted order is ahead (333 x 2047: 41.2 against 48.8), as it is on larger grids.
  const WorkItem item = !by_head && args.row_order ? table_item(args.row_order, i, args.B * args.Hq, items)
                                                   : lpt_item(i, args.B * args.Hq, by_head ? 1 << 30 : 1);
  const int nQB = (args.Sq + kFwdBM - 1) / kFwdBM, qb = nQB - 1 - item.rank;
  const int q0 = qb * kFwdBM;
  const float slope = args.slopes[item.head % args.Hq];
  if (rule(CAUSAL ? min(q0 + kFwdBM, args.Skv) : args.Skv, slope)) {
    if (blockIdx.x == 0 && args.flags != nullptr && threadIdx.x < kStatsHeader)
      args.flags[threadIdx.x] = threadIdx.x == 0 ? args.order_flags : 0;
    if (part == 0 && args.kstart != nullptr && threadIdx.x == 0) args.kstart[(size_t)item.head * nQB + qb] = 0;
    if (q0 + part * kSplitRows < args.Sq) fwd_split_rows<T, D, CAUSAL>(args, item.head, q0 + part * kSplitRows, sK, sV);
  } else if (part == 0) {
    fwd_row_block<T, D, CAUSAL, SKIP, false>(args, item.head, qb, sK, sV);
  }
}

}  // namespace

template <typename T, int D, bool CAUSAL>
hipError_t launch_fwd(const FwdArgs& a, hipStream_t stream) {
  static_assert(kFwdBM == kSkipRows, "kstart entries are per forward row block");
  FwdArgs f = a;
  const bool rows_sorted = row_order_fits(a.B, a.Hq, a.Sq);
  f.order_flags = 0;
  if (a.knorm != nullptr) {
    const bool keys_sorted = key_order_used(a.B, a.Hq, a.Hkv, a.Skv);
    const ScheduleArgs sched{a.slopes, a.row_order, a.key_order, a.B, a.Hq, a.Hkv, a.Sq, a.Skv, CAUSAL ? 1 : 0,
                             rows_sorted ? 1 : 0, keys_sorted ? 1 : 0, order_window<T>()};
    // The key table needs the row table's work-group before it (work-group 1 writes it).
    const int nSched = a.row_order == nullptr ? 0 : (a.key_order != nullptr ? 2 : 1);
    hipLaunchKernelGGL((coalibi_key_norm_kernel<T, D>), dim3(nSched + a.nKC * a.B * a.Hq), dim3(256), 0, stream,
                       static_cast<const T*>(a.k), a.kl, const_cast<float*>(a.knorm), a.Skv, a.nKC, a.B * a.Hkv, nSched,
                       sched);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // The backward follows a table only where it was sorted; an unsorted one holds the index
    // order, which the fixed orders of the kernels beat (their heads rotate over the XCDs).
    if (a.row_order != nullptr && rows_sorted) f.order_flags |= kFlagRowOrder;
    if (a.key_order != nullptr && keys_sorted) f.order_flags |= kFlagKeyOrder;
    f.order_flags |= kFlagTailSkip;
  }
  if (a.knorm == nullptr || !rows_sorted) f.row_order = nullptr;  // no sorted table: the fixed order
  const int nQB = (a.Sq + kFwdBM - 1) / kFwdBM;
  const int grid = nQB * a.B * a.Hq;
  if constexpr (SplitCfg<T, D>::kFits) {
    const float window = a.every_key ? __builtin_inff() : order_window<T>();
    const int keys = CAUSAL ? std::min(a.Sq, a.Skv) : a.Skv;
    const bool small = split_fwd_grid(sizeof(T), D, grid, keys, CAUSAL, a.every_key);
    if (small || (CAUSAL && !a.every_key && split_fwd_long_rows(sizeof(T), D, grid, keys))) {
      const dim3 parts((grid + 7) / 8 * 32);
      const SplitRule rule = small ? SplitRule{window, 3.0f, 192.0f, 0} : SplitRule{window, 1.25f, 0.0f, keys / 2};
      auto* const kernel = a.knorm != nullptr ? coalibi_fwd_split_kernel<T, D, CAUSAL, true>
                                              : coalibi_fwd_split_kernel<T, D, CAUSAL, false>;
      hipLaunchKernelGGL(kernel, parts, dim3(256), 0, stream, f, grid, rule, small);
      return hipGetLastError();
    }
  }
  const bool plain = is_contiguous(a.ql, a.Hq, a.Sq, D) && is_contiguous(a.ol, a.Hq, a.Sq, D) &&
                     is_contiguous(a.kl, a.Hkv, a.Skv, D) && is_contiguous(a.vl, a.Hkv, a.Skv, D);
  constexpr int kPerCU = D * sizeof(T) > 256 ? 1 : 2;
  auto choose = [&](auto per_cu) {
    constexpr int N = decltype(per_cu)::value;
    return a.knorm != nullptr ? (plain ? coalibi_fwd_kernel<T, D, CAUSAL, true, true, N>
                                       : coalibi_fwd_kernel<T, D, CAUSAL, true, false, N>)
                              : (plain ? coalibi_fwd_kernel<T, D, CAUSAL, false, true, N>
                                       : coalibi_fwd_kernel<T, D, CAUSAL, false, false, N>);
  };
  auto* kernel = choose(std::integral_constant<int, kPerCU>{});
  if constexpr (has_roomy_form(sizeof(T), D)) {
    if (roomy_fwd_grid(grid, CAUSAL ? std::min(a.Sq, a.Skv) : a.Skv, CAUSAL, a.every_key))
      kernel = choose(std::integral_constant<int, 1>{});
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, stream, f);
  return hipGetLastError();
}

#define COALIBI_INST_FWD(T, D)                                           \
  template hipError_t launch_fwd<T, D, true>(const FwdArgs&, hipStream_t); \
  template hipError_t launch_fwd<T, D, false>(const FwdArgs&, hipStream_t);

COALIBI_INST_FWD(_Float16, 16)
COALIBI_INST_FWD(_Float16, 32)
COALIBI_INST_FWD(_Float16, 64)
COALIBI_INST_FWD(_Float16, 128)
COALIBI_INST_FWD(_Float16, 256)
COALIBI_INST_FWD(__bf16, 16)
COALIBI_INST_FWD(__bf16, 32)
COALIBI_INST_FWD(__bf16, 64)
COALIBI_INST_FWD(__bf16, 128)
COALIBI_INST_FWD(__bf16, 256)
COALIBI_INST_FWD(float, 16)
COALIBI_INST_FWD(float, 32)
COALIBI_INST_FWD(float, 64)
COALIBI_INST_FWD(float, 128)
COALIBI_INST_FWD(float, 256)

}  // namespace coalibi
