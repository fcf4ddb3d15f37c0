// Launch interface between the C ABI layer and the gfx950 kernels.
#pragma once

#include <algorithm>
#include <hip/hip_runtime.h>

namespace coalibi {

constexpr float kLog2eHost = 1.4426950408889634f;

// Tensors are contiguous row-major: q/o/dout/dq (B, Hq, Sq, D),
// k/v/dk/dv (B, Hkv, Skv, D).  Query head h reads key/value head h / (Hq/Hkv).
//
// Statistics the forward saves for the backward besides LSE ("stats", int32 / fp32 words,
// O(B*Hq*S) in all):
//   header (kStatsHeader words): word 0 holds flags -- bit 0: row_order is a work order the
//     key-norm launch wrote, bit 1: key_order likewise (without a bit the kernels that would
//     read the table use their fixed order instead), bit 2: the forward ran with the tail
//     skip; the other header words are zero;
//   kstart (B*Hq, nQB) int32, nQB = ceil(Sq/128): the first key the forward processed for
//     each 128-row block (0 when the tail skip is off).  Every key left of it has a softmax
//     weight below 2^-skip_log2 of its row's total in every row of the block (the tail skip
//     below); the backward passes skip the same keys;
//   knorm (B*Hq, nKC) fp32, nKC = ceil(Skv/kNormKeys): max_k |k|_2 over each chunk of
//     kNormKeys keys of key head b*Hkv + h in its first B*Hkv rows, zero in the rest;
//   row_order (B*Hq*nQB) int32: the work order of the forward and pass 1 (below);
//   key_order (B*Hq*nKB) int32, nKB = ceil(Skv/64): the work order of pass 2 over its
//     B*Hkv*nKB key blocks (written, and read, only when Hq == Hkv);
//   rsum (2, B*Hq, Sq) fp32: R_i, the sum of sigmoid(p_ik) over the keys the forward processed
//     (k >= kstart), summed with compensation and saved as hi + lo.  It takes the place of the
//     reference's RowSigTotal (co_alibi_attn.py:37): backward pass 1 walks the keys left to
//     right and rebuilds z at each block start as R minus the sigma it has passed.
//
// Tail skip.  In the log2 domain a row's logit for key k is a_k = t_k - lam2 * z_k with
// t_k = q.k * sm_scale * log2(e) and z_k = sum of sigmoids of the visible keys >= k.  The
// forward walks keys from the diagonal leftwards, so when it has processed every key from
// k_next on, z_k >= zr (the sum over those keys) for every k < k_next, as sigmoids are
// >= 0, and |t_k| <= |q| * max|k| * sm_scale * log2(e) =: bound (Cauchy-Schwarz).  With
// lam2 > 0 and m2 the running maximum, every later weight 2^(a_k - m2) is then at most
// 2^(bound - lam2 * zr - m2); once that is below 2^-skip_log2 for all rows of a 128-row
// block the forward stops.  The row total l is >= 1 at the final scale, so each skipped
// weight is below 2^-skip_log2 of it (the softmax probability s = 2^(a - LSE2) too).
// The threshold follows the type P is rounded to before it multiplies V:
//   fp16: 26 -- P < 2^-26 rounds to zero (below half the smallest subnormal, 2^-25), so
//     the forward's O is bit-identical to that of co_alibi_fwd without statistics, which skips
//     nothing (with the skip switched off, small grids take other forms: coalibi_fwd.hip);
//   bf16: 32 -- P keeps 8 bits, so each P carries a relative error up to 2^-9; the skipped
//     weights together are below S * 2^-32 of the row total (1e-6 at S = 4096);
//   fp32: 64 -- the validation mode stays within S * 2^-64 of the unskipped result.
// The backward leaves out the same keys; their dA = s (dS - D) terms are below the same
// fraction of the row's scale.
// The skip is a library setting (co_alibi_set_tail_skip, on by default): with it off the
// forward launches no key-norm kernel, processes every key and records kstart = 0.
constexpr int kStatsHeader = 4;
constexpr int kFlagRowOrder = 1;
constexpr int kFlagKeyOrder = 2;
constexpr int kFlagTailSkip = 4;  // the forward ran with the tail skip
constexpr int kNormKeys = 256;
template <typename T>
constexpr float skip_log2() {
  return sizeof(T) == 4 ? 64.0f : (__is_same(T, __bf16) ? 32.0f : 26.0f);
}
constexpr int kSkipRows = 128;  // rows per kstart entry: the forward's and pass 1's row block
// kstart as the backward kernels read it.  It is device data the host cannot check without a
// synchronisation: a value outside [0, Skv] (not written by the forward) counts as 0, so no
// value moves a tile or a record address past the key range.
__device__ __forceinline__ int valid_kstart(int ks, int Skv) { return ks >= 0 && ks <= Skv ? ks : 0; }
inline int stats_kstart_count(int Sq) { return (Sq + kSkipRows - 1) / kSkipRows; }
inline int stats_knorm_count(int Skv) { return (Skv + kNormKeys - 1) / kNormKeys; }
constexpr int kOrderKeyBlock = 64;  // keys per pass-2 work-group (16-bit kernels)
__host__ __device__ inline int stats_key_block_count(int Skv) { return (Skv + kOrderKeyBlock - 1) / kOrderKeyBlock; }

// Work orders.  The tail skip makes a work-group's cost depend on its head's slope: a
// 128-row block of a steep head processes a few key tiles, one of a flat head up to all of
// them.  The hardware hands consecutive work-group ids to the 8 XCDs in turn and, within an
// XCD, to its 4 shader engines in turn, and it dispatches in id order: when the engine
// that the next id is bound for has no free slot, dispatch waits even if other engines are
// idle.  Ids whose costs differ widely (the fixed orders of the kernels) therefore leave
// engines idle; ids in decreasing order of cost keep every engine's queue alike.  The
// key-norm launch writes such orders (coalibi_fwd.hip, schedule_rows / schedule_keys): entry
// j of a table is the item the work-group with id j processes, item = rank * heads + head in
// the fixed order's numbering, sorted by a cost predicted from the slope alone (the order is
// not needed to be exact, only close): a row keeps about W = kOrderWindow / slope keys left
// of its diagonal, where kOrderWindow = (T + 8) / (0.5 log2 e) for the threshold T of the
// type (the sigmoid sum z grows by about 0.5 a key, and the skip fires once slope*z*log2 e
// passes T plus the logit bound, a few units).
// A table is sorted for at most this many items (the sort runs on one wavefront); larger
// grids keep the fixed orders.
constexpr long long kOrderMaxItems = 1 << 20;
inline bool row_order_fits(int B, int Hq, int Sq) {
  return static_cast<long long>(B) * Hq * stats_kstart_count(Sq) <= kOrderMaxItems;
}
inline bool key_order_fits(int B, int Hkv, int Skv) {
  return static_cast<long long>(B) * Hkv * stats_key_block_count(Skv) <= kOrderMaxItems;
}
// Pass 2 follows key_order with one query head per key head only: with grouped heads the
// sorted order measured slower than balanced_item (coalibi_common.h), which keeps runs of key
// blocks of a head on one XCD.
inline bool key_order_used(int B, int Hq, int Hkv, int Skv) { return Hq == Hkv && key_order_fits(B, Hkv, Skv); }
template <typename T>
constexpr float order_window() {
  return (skip_log2<T>() + 8.0f) / (0.5f * kLog2eHost);
}
// Element strides of one (B, H, S, D) operand: from batch to batch, head to head and row to row.  The
// D elements of a row are consecutive; r >= D.  A model's projections leave (B, S, H, D) memory, whose
// transposed views the kernels read and write in place this way.
struct Layout {
  long long b, h;
  int r;
};
__host__ __device__ inline Layout contiguous_layout(int H, int S, int D) {
  return {static_cast<long long>(H) * S * D, static_cast<long long>(S) * D, D};
}
inline bool is_contiguous(const Layout& l, int H, int S, int D) {
  const Layout c = contiguous_layout(H, S, D);
  return l.b == c.b && l.h == c.h && l.r == c.r;
}
struct FwdArgs {
  Layout ql, kl, vl, ol;
  const void* q;
  const void* k;
  const void* v;
  const float* slopes;  // (Hq,) penalty slope per query head
  void* o;
  float* lse;          // (B*Hq, Sq) natural-log log-sum-exp, or NULL
  int* kstart;         // (B*Hq, nQB), written when not NULL (the backward's statistics)
  const float* knorm;  // (B*Hq, nKC) chunk maxima of |k|, filled before the forward; NULL: no tail skip
  int* flags;          // the statistics' header, written by work-group 0 when not NULL
  int order_flags;     // its flags word: which work orders the key-norm launch wrote
  float* rsum;         // (2, B*Hq, Sq) row sigmoid totals (hi, lo), written when not NULL
  int B, Hq, Hkv, Sq, Skv, nKC;
  float sc2;  // sm_scale * log2(e)
  bool every_key;  // the tail skip is switched off
  // Work orders (above): written by the key-norm launch when not NULL (key_order only with
  // row_order); the forward follows row_order when it is sorted (row_order_fits).
  int* row_order;
  int* key_order;
};

// Score store (16-bit types, D = 64 or 128): pass 1 writes the probabilities s and score
// gradients dS of every tile it processes, and pass 2 reduces them into dK and dV instead of
// recomputing them.  One record per (b*Hq + h, 32-key block jb, 32-row block qb) of a pair
// that can be visible: 4096 bytes, the four 16 x 32 B operands of pass 2's products in MFMA
// lane order -- s for rows 0-15, s for rows 16-31, dS for rows 0-15, dS for rows 16-31 of the
// block; in each, lane l holds the 8 rows 8*(l/32) .. +7 of key l%32.  Records are key-block
// major; causal: qb from jb to nQ32 - 1 (a row block below its key block holds no visible
// pair), otherwise every qb.  Records of skipped tiles (tail skip) are never written or read.
constexpr int kScoreRecordBytes = 4096;
// Pass 2 keeps, per query head of a key head's group, one bit per 128-row block (rounded up to
// 64 per head) of whether the forward processed its key block: at most this many 32-bit words.
constexpr int kStoreProcessedWords = 512;
inline bool score_store_fits(int Hq, int Hkv, int Sq) {
  const int wph = (Sq + kSkipRows * 64 - 1) / (kSkipRows * 64) * 2;
  return static_cast<long long>(Hq / Hkv) * wph <= kStoreProcessedWords;
}
__host__ __device__ inline size_t score_record(int jb, int qb, int nQ32, bool causal) {
  if (!causal) return static_cast<size_t>(jb) * nQ32 + qb;
  return static_cast<size_t>(jb) * nQ32 - static_cast<size_t>(jb) * (jb - 1) / 2 + (qb - jb);
}
inline size_t score_records_per_head(int Sq, int Skv, bool causal) {
  const int nQ32 = (Sq + 31) / 32, nJB = (Skv + 31) / 32;
  if (!causal) return static_cast<size_t>(nJB) * nQ32;
  const int J = nJB < nQ32 ? nJB : nQ32;
  return score_record(J, J, nQ32, true);  // records of the blocks before J
}

// Backward scratch: dsum (B*Hq, Sq) holds dO_i . O_i.  The recompute path (pass 2 recomputes s
// and dS) adds zb and cb, (B*Hq, nZB, Sq) fp32 each with nZB = ceil(Skv/32): for every 32-key
// block J, zb[J][i] = sum of sigmoid(p_ik) over the keys k >= 32J of row i and cb[J][i] = sum of
// dA_ik over the keys k < 32J, written by pass 1 for the blocks it processes.  The score-store
// path needs neither.
struct BwdArgs {
  // Other than contiguous layouts on the score-store path only.
  Layout dol, ql, kl, vl, ol, dql, dkl, dvl;
  const void* dout;
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  const float* lse;
  const float* rsum;  // (2, B*Hq, Sq): the forward's row sigmoid totals, hi and lo parts
  const float* slopes;
  void* dq;
  void* dk;
  void* dv;
  float* dsum;
  float* zb;
  float* cb;
  const int* kstart;  // (B*Hq, nQB): keys left of kstart are skipped (see above)
  const int* flags;   // the forward's flags word: which of the work orders below it wrote
  void* scores;       // score store (above), or NULL: pass 2 recomputes s and dS from zb / cb
  size_t score_head;  // records per (b, h)
  const int* row_order;  // pass 1's work order (above) when flagged, or NULL: the fixed order
  const int* key_order;  // pass 2's work order for 64-key work-groups when flagged, or NULL
  int B, Hq, Hkv, Sq, Skv, nZB;
  float sc2;
  float sm_scale;
};

// Decode: q/o (B, Hq, D); the caches k/v are (B, Hkv, cap, D) with the first L rows
// of every head valid (or the first seq_lens[b] rows of sequence b, at most L).  The
// keys of a sequence form chunks of kDecodeChunkKeys; split s of a head covers chunks
// [s*cps, (s+1)*cps), with cps from decode_cps below.  Split-K partials per (b*Hq + h, split):
// pmax / psum / psig (B*Hq, nSplits) and pout (B*Hq, nSplits, D), fp32; unused with one split,
// whose work-group writes o and lse itself.
constexpr int kDecodeChunkKeys = 128;
constexpr int kMaxDecodeGroup = 32;     // query heads per kv head (MFMA tile columns)
constexpr int kMaxDecodeChunks = 16384;  // bounds seq_kv (2^21 keys)
constexpr int kMaxDecodeSplits = 1024;   // split partials per (batch, query head); merge weights in LDS

struct DecodeArgs {
  const void* q;
  const void* k;
  const void* v;
  const float* slopes;  // (Hq,)
  void* o;
  float* lse;  // (B*Hq,) or NULL
  float* pmax;
  float* psum;
  float* psig;
  float* pout;
  const int* seq_lens;  // (B,) per-sequence cache lengths, or NULL (all L)
  int B, Hq, Hkv, G, L, cap;
  int nSplits;  // most splits of any sequence: the partials' stride
  int cps;      // chunks per split (with a plan the kernels share the chunks out)
  int slots;    // resident work-groups the splits are sized for
  int slack;    // the plan's (decode_cps)
  bool plan;    // splits sized by the lengths in seq_lens (DecodeRule::plans, coalibi_capi.hip)
  float sc2;
};

// Split-K work-groups the decode aims at per CU: one round of the two that are resident.
constexpr int kDecodeWGsPerCU = 2;

// Chunks per split of a decode over sequences with `work` chunks in all (summed over the kv heads;
// `longest` in the longest one): an equal share of `work` per resident work-group, or up to
// slack/16 more and one chunk (and at most `most`) where that brings groups(c), the work-groups that c chunks per
// split make, into one round of `slots`.  At most `max_splits` splits per sequence.  On the host
// for equal lengths, in the kernels for a length per sequence.
template <typename F>
__host__ __device__ inline int decode_cps(long long work, int longest, int slots, int max_splits, int slack, int most,
                                          const F& groups) {
  const int share = static_cast<int>((work + slots - 1) / slots), fit = (longest + max_splits - 1) / max_splits;
  const int c0 = share > fit ? (share > 1 ? share : 1) : (fit > 1 ? fit : 1);
  const int c1 = c0 + 1 + static_cast<int>(static_cast<long long>(c0) * slack / 16);
  for (int c = c0; c <= (c1 < most ? c1 : most); c += 1 + c / 16)
    if (groups(c) <= slots) return c;
  return c0;
}

// Which kernel forms a call takes, from its element bytes, head dim, 128-row blocks (batch * heads_q *
// ceil(seq_q / 128)) and the most keys a row sees (`keys`).  The split forms win where the row blocks leave
// the GPU room, and longer walks leave more of it (causal: half the work of the longest block on average,
// and the short blocks' work-groups cost their prologue and merge all the same); they lose K and V reads (four
// times as many from L2) and, in training, the tail skip's record: both backward passes walk every key of a
// split block.  `every_key`: the tail skip is switched off.
//   Types of more than 256 bytes a row (fp32 at D 128, 16 bits at D 256) have one work-group per CU in the split
// forms, two in the others, so they fill the GPU at half the blocks; their split forms do not fit LDS
// above 512 bytes.
//   Figures: us by hipGraph replay, whole-block form -> split, forward alone / forward and backward with the
// rules' choice for the other launches; f: tail skip off.
constexpr bool split_fits(int elem, int D) { return D * elem <= 512; }

// Forward.
//   fp16 D 128  n 64: 64 blocks 12.7 -> 13.1, 128 13.0 -> 15.8;  n 96: 128 15.8 -> 16.0;  n 128: 128 16.8 -> 16.3
//          n 256: 64 blocks 20.8 -> 15.6 / 52 -> 41, 128 21.0 -> 17.0 / 54 -> 49;  n 512: 128 28.6 -> 23.1 / 78 -> 68
//          n 1024: 128 blocks 44.0 -> 28.0 / 123 -> 92, 256 45.4 -> 40.8 / 133 -> 130 f 36.7 -> 35.2
//          n 2048: 128 blocks 75.6 -> 41.0 / 216 -> 146, 384 78.1 -> 60.3 / 235 -> 218 f 68.5 -> 73.2, 320 f 66.7 -> 66.3
//   fp16 D 64   n 64: 128 blocks 10.4 -> 11.7;  n 512: 128 22.6 -> 17.6 / 61 -> 46;  n 1024: 256 34.5 -> 28.2 / 105 -> 87
//          n 2048: 384 blocks 60.4 -> 41.9 / 191 -> 148 f 48.0 -> 48.1
//   fp32 D 64   n 64: 64 blocks 14.7 -> 13.0, 128 15.1 -> 16.3;  n 1024: 256 93.8 -> 76.8;  n 2048: 384 175 -> 156 / 659 -> 619
//   fp32 D 128  n 1024: 256 blocks 167 -> 144;  n 1536: 288 240 -> 205, 384 243 -> 267;  n 2048: 352 313 -> 226, 384 315 -> 329
//   fp16 D 256  n 128: 64 blocks 27.1 -> 20.1, 128 29.4 -> 32.0;  n 192: 128 30.2 -> 31.7;  n 256: 128 38.0 -> 34.8
//          n 1024: 224 blocks 91 -> 81, 256 94 -> 99 / 255 -> 269;  n 1536: 288 128 -> 118 / 345 -> 338, 384 131 -> 154 / 382 -> 422
//          n 2048: 352 blocks 159 -> 127 f 256: 142 -> 124, 320: 144 -> 159;  n 4096: 384 296 -> 183 f 272 -> 317
//   non-causal  fp16 D 128 333 x 2047: 96 blocks 89.5 -> 42.1 / 232 -> 154;  n 2048: 128 f 73 -> 48, 192 f 74 -> 74, 256 88 -> 58 f 76 -> 85
//          fp16 D 64 n 2048: 128 blocks f 46 -> 38, 160 f 47 -> 54, 256 56 -> 41 f 48 -> 67;  fp32 D 128: 192 f 304 -> 292, 224 f 308 -> 381
//          fp16 D 256 n 2048: 256 blocks 304 -> 163 f 358 -> 209 (the whole-block form spills);  1024 x 64: 128 35 -> 31
inline bool split_fwd_grid(int elem, int D, long long row_blocks, int keys, bool causal, bool every_key) {
  const bool fp32 = elem == 4, wide = D * elem > 256;
  if (wide && !fp32) {
    const int least = causal && keys < 256 ? 64 : 128;
    if (!causal) return row_blocks <= std::max(least, std::min(keys / 8, 256));
    return row_blocks <= std::max(least, std::min(keys / 5, every_key ? 256 : 352));
  }
  if (keys <= 64) return row_blocks <= (fp32 ? 64 : 0);
  const int most = causal ? (wide ? 320 : every_key && D > 64 ? 320 : 384) : every_key ? (fp32 ? 192 : 128) : 256;
  return row_blocks <= std::max(128, std::min(causal ? keys / 4 : keys / 8, most));
}

// Forward beyond those grids (causal, tail skip on): whether only the longer half of the row blocks is split.
// The flat heads' last blocks otherwise walk on alone after the rest.
//   fp16 D 128  n 1536: 576 blocks 66.7 -> 63.0, 696 68.0 -> 67.7, 768 68.2 -> 75.2 / 234 -> 243;  n 1741 (448, bf16) 70.5 -> 58.6
//          n 2048: 512 blocks 81.2 -> 68.5 / 251 -> 239, 768 83.7 -> 76.7, 1024 90.1 -> 113.4;  n 4096: 768 144 -> 118 / 451 -> 425
//   fp16 D 64   n 1536: 576 blocks 50.6 -> 44.4, 768 52.1 -> 56.9;  n 2048: 768 64.0 -> 62.4;  n 4096: 768 110 -> 93;  n 8192: 512 144 -> 149
//   fp32 D 64   n 1536: 480 blocks 137 -> 130, 576 139 -> 150;  n 2048: 512 180 -> 176, 640 180 -> 192;  n 4096: 640 342 -> 342, 704 342 -> 362
//   fp16 D 256  n 1536: 336 blocks 130 -> 105;  n 2048: 448 164 -> 136, 512 170 -> 170, 768 175 -> 205;  n 3072: 576 237 -> 186, 768 242 -> 281
//   fp32 D 128  n 1536: 360 blocks 242 -> 216, 576 248 -> 270;  n 2048: 416 316 -> 262, 512 321 -> 344;  n 3072: 576 470 -> 369, 672 475 -> 495
inline bool split_fwd_long_rows(int elem, int D, long long row_blocks, int keys) {
  if (keys < 1536 || keys > 4096) return false;
  if (D * elem > 256) return row_blocks <= std::min(keys / 5, 768);
  if (elem == 4 && D > 32) return row_blocks <= std::min(keys / 4, 640);
  return row_blocks <= std::min(keys * 2 / 5, 768);
}

// Forward, whole-block form, fp32 at D = 64: asked for one work-group per CU it takes 267 registers, for two 256.
// The roomier code is the faster one where the tail skip's uneven blocks hardly ever give a CU two.  Two per CU -> one:
//   n 512: 384 blocks 70.6 -> 71.9;  n 1024: 384 111 -> 96, 576 122 -> 113, 640 122 -> 123, 1024 176 -> 196
//   n 2048: 448 168 -> 167, 704 205 -> 180, 1024 253 -> 287;  n 4096: 768 378 -> 344, 1024 431 -> 418;  n 8192: 512 700 -> 667
//   non-causal  n 1024: 384 blocks 107 -> 97, 448 120 -> 124;  n 2048: 448 197 -> 181, 512 216 -> 212, 768 221 -> 237
//   tail skip off: 2 to 4 % slower everywhere
constexpr bool has_roomy_form(int elem, int D) { return elem == 4 && D == 64; }
inline bool roomy_fwd_grid(long long row_blocks, int keys, bool causal, bool every_key) {
  return !every_key && keys >= 896 && row_blocks <= (causal ? std::min(448 + keys / 8, 1024) : 400);
}

// Backward pass 1.  At D = 128 in 16-bit types a step waits longer for its own K, whose tile the dQ product
// reads last (and reloads spilled registers), and the limit is lower.  Both passes, pass 1 whole -> split:
//   fp16 D 64   n 64: 64 blocks 11.9 -> 12.7;  n 96: 64 15.5 -> 14.5, 128 16.1 -> 17.6;  n 128: 128 17.8 -> 17.3;  n 256: 128 25.0 -> 21.3
//          n 1024: 256 blocks 70 -> 57;  n 2048: 384 130 -> 102;  non-causal n 2048: 256 126 -> 114, f 224 134 -> 134
//   fp16 D 128  n 96: 128 blocks 21.4 -> 25.8;  n 128: 96 24.0 -> 26.6;  n 192: 96 26.0 -> 29.4;  n 256: 128 33.3 -> 32.1;  n 1024: 192 84 -> 74, 256 87 -> 84
//          n 2048: 256 blocks 149 -> 125, 320 (f) 103 -> 114 (pass 1 alone);  non-causal n 2048: 128 f 141 -> 118, 144 to 256 +13 to 18 %
//   fp16 D 256  n 128: 96 blocks 41.8 -> 52.1;  n 256: 64 55 -> 47, 128 58 -> 64;  n 512: 128 87 -> 85;  n 1024: 128 150 -> 130, 192 152 -> 151
//          n 2048: 192 blocks 274 -> 231, 256 278 -> 274, 384 284 -> 320;  non-causal n 2048: 128 294 -> 277, 192 f +6 %
//   fp32 D 64   n 32: 64 blocks 21.3 -> 23.6;  n 64: 64 26.4 -> 25.0, 128 27.4 -> 32.2;  n 1024: 256 264 -> 218;  n 2048: 384 482 -> 399
//   fp32 D 128  n 1024: 256 blocks 736 -> 658;  n 2048: 384 1435 -> 1328;  non-causal n 2048: 192 f 1404 -> 1327, 224 f 1409 -> 1458
inline bool split_dq_grid(int elem, int D, long long row_blocks, int keys, bool causal) {
  if (elem == 4) {
    if (keys <= 64) return row_blocks <= (keys <= 32 ? 0 : 64);
    return row_blocks <= std::max(128, causal ? std::min(keys / 3, 384) : std::min(keys / 4, D > 64 ? 192 : 320));
  }
  if (keys <= 64) return false;
  const int least = keys < (D > 128 ? 512 : D > 64 ? 256 : 128) ? 64 : 128;
  if (D <= 64) return row_blocks <= std::max(least, causal ? std::min(keys / 3, 384) : std::min(keys / 4, 320));
  if (!causal) return row_blocks <= least;
  return row_blocks <= std::max(least, D > 128 ? std::min(keys / 8, 224) : std::min(keys / 5, 256));
}

// Backward pass 2, recompute path: the 32-key form, for fp32 at D <= 64 and 16-bit types at D <= 32 (16-bit types at
// D >= 64 have their own kernel).  It wins where the 128-key blocks are few, and where a wavefront's walk (a tile per
// row block and query head) is long enough to carry its prologue and merge; in 16-bit types the 128-key form
// is ahead again once its work-groups fill the GPU.  Both passes, 128-key -> 32-key, by key blocks and tiles:
//   fp32 D 64   128 x 1: 52.6 -> 45.1, 192 x 1 62 -> 74, 256 x 1 65 -> 96, 256 x 2 100 -> 101 (non-causal 99 -> 111), 256 x 4 180 -> 155
//          384 x 8: 344 -> 308, 512 x 8 397 -> 414, 1024 x 8 734 -> 746, 512 x 4 248 -> 272, 640 x 16 708 -> 645, 1024 x 16 1194 -> 1153, 64 x 64 1761 -> 551
//   fp32 D 32   192 x 1: 41 -> 44, 256 x 2 64 -> 56, 512 x 8 249 -> 218, 1024 x 16 567 -> 538
//   fp16 D 32   128 x 1: 17.3 -> 14.2, 192 x 1 23 -> 29, 256 x 2 29.4 -> 28.4, 256 x 4 49 -> 40, 512 x 4 52 -> 59, 512 x 8 89 -> 83
//          640 x 16: 164 -> 129, 1024 x 16 175 -> 188, 768 x 3 51 -> 64
constexpr bool has_key_form(int elem, int D) { return D * elem <= (elem == 2 ? 64 : 256); }
inline bool use_key_form(int elem, int D, long long key_blocks, int tiles) {
  if (key_blocks <= 128) return true;
  if (key_blocks <= 256) return tiles >= (elem == 4 && D > 32 ? 3 : 2);
  return tiles >= (elem == 4 && D > 32 && key_blocks > 448 ? 12 : 8) && (elem == 4 || key_blocks <= 640);
}

// Forward; with a.knorm (the tail skip) it first launches the key-norm kernel that fills it.
template <typename T, int D, bool CAUSAL>
hipError_t launch_fwd(const FwdArgs& a, hipStream_t stream);

template <typename T, int D>
hipError_t launch_decode(const DecodeArgs& a, hipStream_t stream);

// stages: bit 0 = pass 1 (dq, dsum, and zb / cb or the score store), bit 1 = pass 2 (dk, dv; needs pass
// 1's output).
template <typename T, int D, bool CAUSAL>
hipError_t launch_bwd(const BwdArgs& a, int stages, hipStream_t stream);

}  // namespace coalibi
