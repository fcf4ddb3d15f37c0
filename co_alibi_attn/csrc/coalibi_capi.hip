// C ABI entry points: argument checks, dtype / head-dim dispatch, launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <utility>

#include "../../include/co_alibi.h"
#include "coalibi_kernels.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

size_t num_zblocks(int seq_kv) { return (static_cast<size_t>(seq_kv) + 31) / 32; }

// fp32 elements of one per-32-key-block array of the recompute path's workspace (zb or cb).
size_t block_sums_numel(int batch, int heads_q, int seq_q, int seq_kv) {
  return static_cast<size_t>(batch) * heads_q * num_zblocks(seq_kv) * seq_q;
}

// The tail skip (the library setting of co_alibi_set_tail_skip): on unless switched off.
std::atomic<int> g_tail_skip{1};

// Where the parts of the forward's statistics lie (coalibi_kernels.h).
struct StatsLayout {
  size_t kstart, knorm, row_order, key_order, rsum, total;  // offsets in 4-byte words
};
StatsLayout stats_layout(int batch, int heads_q, int seq_q, int seq_kv) {
  const size_t bh = static_cast<size_t>(batch) * heads_q;
  StatsLayout l;
  l.kstart = coalibi::kStatsHeader;
  l.knorm = l.kstart + bh * coalibi::stats_kstart_count(seq_q);
  l.row_order = l.knorm + bh * coalibi::stats_knorm_count(seq_kv);
  l.key_order = l.row_order + bh * coalibi::stats_kstart_count(seq_q);
  l.rsum = l.key_order + bh * coalibi::stats_key_block_count(seq_kv);
  l.total = l.rsum + 2 * bh * static_cast<size_t>(seq_q);
  return l;
}

size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

struct Shape {
  int B, Hq, Hkv, Sq, Skv, D;
};

int check_shape(const char* fn, int dtype, const Shape& s) {
  if (dtype != CO_ALIBI_F32 && dtype != CO_ALIBI_F16 && dtype != CO_ALIBI_BF16)
    return fail(CO_ALIBI_EUNSUPPORTED, std::string(fn) + ": dtype must be 0 (fp32), 1 (fp16) or 2 (bf16)");
  if (s.B < 1 || s.Hq < 1 || s.Hkv < 1 || s.Sq < 1 || s.Skv < 1)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": batch, heads and sequence lengths must be >= 1");
  if (s.Hq % s.Hkv != 0)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": heads_q must be a multiple of heads_kv");
  if (s.D != 16 && s.D != 32 && s.D != 64 && s.D != 128 && s.D != 256)
    return fail(CO_ALIBI_EUNSUPPORTED,
                std::string(fn) + ": head_dim must be 16, 32, 64, 128 or 256, got " + std::to_string(s.D));
  // Sequence indices are 32-bit in the kernels; grids must fit a 31-bit launch.
  const double wg = std::ceil(s.Sq / 128.0) * s.B * s.Hq;
  if (s.Sq > (1 << 30) || s.Skv > (1 << 30) || wg > 2147483647.0)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": problem too large for one launch");
  return CO_ALIBI_OK;
}

// The layout of operand `name`: contiguous without strides, else the caller's batch, head and row
// strides, which must keep every row 16-byte aligned.  A tile's byte offsets are 32-bit in the kernels
// (at most 256 rows of 4-byte elements).
constexpr long long kMaxRowStride = 1 << 20;
// K and V share a row stride: the kernels keep one set of tile offsets for both.
int check_kv_rows(const char* fn, const coalibi::Layout& k, const coalibi::Layout& v) {
  return k.r == v.r ? CO_ALIBI_OK : fail(CO_ALIBI_EINVAL, std::string(fn) + ": k and v must have the same row stride");
}
int read_layout(const char* fn, const char* name, const long long* strides, int dtype, int H, int S, int D,
                coalibi::Layout* out) {
  *out = coalibi::contiguous_layout(H, S, D);
  if (strides == nullptr) return CO_ALIBI_OK;
  const long long per16 = dtype == CO_ALIBI_F32 ? 4 : 8;
  for (int i = 0; i < 3; ++i)
    if (strides[i] < 0 || strides[i] % per16 != 0)
      return fail(CO_ALIBI_EINVAL, std::string(fn) + ": the strides of " + name + " must be >= 0 and whole 16-byte units");
  if (strides[2] < D || strides[2] > kMaxRowStride)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": the row stride of " + name + " must be in [head_dim, " +
                                     std::to_string(kMaxRowStride) + "]");
  *out = {strides[0], strides[1], static_cast<int>(strides[2])};
  return CO_ALIBI_OK;
}

// An output's rows must not overlap: different work-groups write them.  Of the dimensions longer than 1,
// in order of their strides, each must step past all that the smaller ones cover.
int check_output(const char* fn, const char* name, const coalibi::Layout& l, int B, int H, int S, int D) {
  std::array<std::pair<long long, long long>, 3> dims = {{{l.b, B}, {l.h, H}, {l.r, S}}};  // stride, length
  std::sort(dims.begin(), dims.end());
  __int128 covered = D;
  for (const auto& [stride, n] : dims) {
    if (n == 1) continue;
    if (stride < covered) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": the rows of " + name + " overlap");
    covered += static_cast<__int128>(stride) * (n - 1);
  }
  return CO_ALIBI_OK;
}

// Optional outputs may be NULL; when given they must be aligned.
int check_opt_ptr(const char* fn, const char* name, const void* p, uintptr_t align) {
  if (p != nullptr && !aligned(p, align))
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": " + name + " is not " + std::to_string(align) + "-byte aligned");
  return CO_ALIBI_OK;
}

int check_ptr(const char* fn, const char* name, const void* p, uintptr_t align) {
  if (p == nullptr) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": " + name + " is NULL");
  if (!aligned(p, align))
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": " + name + " is not " + std::to_string(align) + "-byte aligned");
  return CO_ALIBI_OK;
}

template <typename T, int D>
hipError_t fwd_dispatch_causal(const coalibi::FwdArgs& a, bool causal, hipStream_t st) {
  return causal ? coalibi::launch_fwd<T, D, true>(a, st) : coalibi::launch_fwd<T, D, false>(a, st);
}

template <typename T>
hipError_t fwd_dispatch_d(const coalibi::FwdArgs& a, int D, bool causal, hipStream_t st) {
  switch (D) {
    case 16: return fwd_dispatch_causal<T, 16>(a, causal, st);
    case 32: return fwd_dispatch_causal<T, 32>(a, causal, st);
    case 64: return fwd_dispatch_causal<T, 64>(a, causal, st);
    case 256: return fwd_dispatch_causal<T, 256>(a, causal, st);
    default: return fwd_dispatch_causal<T, 128>(a, causal, st);
  }
}

template <typename T, int D>
hipError_t bwd_dispatch_causal(const coalibi::BwdArgs& a, bool causal, int stages, hipStream_t st) {
  return causal ? coalibi::launch_bwd<T, D, true>(a, stages, st) : coalibi::launch_bwd<T, D, false>(a, stages, st);
}

template <typename T>
hipError_t bwd_dispatch_d(const coalibi::BwdArgs& a, int D, bool causal, int stages, hipStream_t st) {
  switch (D) {
    case 16: return bwd_dispatch_causal<T, 16>(a, causal, stages, st);
    case 32: return bwd_dispatch_causal<T, 32>(a, causal, stages, st);
    case 64: return bwd_dispatch_causal<T, 64>(a, causal, stages, st);
    case 256: return bwd_dispatch_causal<T, 256>(a, causal, stages, st);
    default: return bwd_dispatch_causal<T, 128>(a, causal, stages, st);
  }
}

}  // namespace

extern "C" {

size_t co_alibi_stats_numel(int batch, int heads_q, int seq_q, int seq_kv) {
  if (batch < 1 || heads_q < 1 || seq_q < 1 || seq_kv < 1) return 0;
  return stats_layout(batch, heads_q, seq_q, seq_kv).total;
}

size_t co_alibi_bwd_workspace_bytes(int batch, int heads_q, int seq_q, int seq_kv) {
  if (batch < 1 || heads_q < 1 || seq_q < 1 || seq_kv < 1) return 0;
  const size_t rows = static_cast<size_t>(batch) * heads_q * seq_q;
  return round_up(rows * sizeof(float), 256) +
         2 * round_up(block_sums_numel(batch, heads_q, seq_q, seq_kv) * sizeof(float), 256);
}

int co_alibi_attention_forms(int dtype, int batch, int heads_q, int heads_kv, int seq_q, int seq_kv, int head_dim,
                             int causal) {
  if (check_shape("co_alibi_attention_forms", dtype, {batch, heads_q, heads_kv, seq_q, seq_kv, head_dim})) return -1;
  const int elem = dtype == CO_ALIBI_F32 ? 4 : 2, row_tiles = (seq_q + coalibi::kSkipRows - 1) / coalibi::kSkipRows;
  const int keys = causal ? std::min(seq_q, seq_kv) : seq_kv;
  const long long row_blocks = static_cast<long long>(row_tiles) * batch * heads_q;
  const bool every_key = g_tail_skip.load() == 0, fits = coalibi::split_fits(elem, head_dim);
  int forms = 0;
  if (fits && coalibi::split_fwd_grid(elem, head_dim, row_blocks, keys, causal != 0, every_key))
    forms |= CO_ALIBI_FORM_FWD_SPLIT;
  else if (fits && causal && !every_key && coalibi::split_fwd_long_rows(elem, head_dim, row_blocks, keys))
    forms |= CO_ALIBI_FORM_FWD_LONG_ROWS;
  else if (coalibi::has_roomy_form(elem, head_dim) && coalibi::roomy_fwd_grid(row_blocks, keys, causal != 0, every_key))
    forms |= CO_ALIBI_FORM_FWD_ROOMY;
  if (fits && coalibi::split_dq_grid(elem, head_dim, row_blocks, keys, causal != 0)) forms |= CO_ALIBI_FORM_DQ_SPLIT;
  if (coalibi::has_key_form(elem, head_dim) &&
      coalibi::use_key_form(elem, head_dim, static_cast<long long>((seq_kv + 127) / 128) * batch * heads_kv,
                            heads_q / heads_kv * row_tiles))
    forms |= CO_ALIBI_FORM_DKDV_KEYS;
  return forms;
}

int co_alibi_set_tail_skip(int enabled) { return g_tail_skip.exchange(enabled != 0 ? 1 : 0); }

int co_alibi_tail_skip(void) { return g_tail_skip.load(); }

size_t co_alibi_bwd_score_store_workspace_bytes(int dtype, int batch, int heads_q, int heads_kv, int seq_q,
                                                int seq_kv, int head_dim, int causal) {
  if (batch < 1 || heads_q < 1 || heads_kv < 1 || heads_q % heads_kv != 0 || seq_q < 1 || seq_kv < 1) return 0;
  if ((dtype != CO_ALIBI_F16 && dtype != CO_ALIBI_BF16) || (head_dim != 64 && head_dim != 128)) return 0;
  if (!coalibi::score_store_fits(heads_q, heads_kv, seq_q)) return 0;
  const size_t rows = static_cast<size_t>(batch) * heads_q * seq_q;
  return round_up(rows * sizeof(float), 256) + static_cast<size_t>(batch) * heads_q *
                                                   coalibi::score_records_per_head(seq_q, seq_kv, causal != 0) *
                                                   coalibi::kScoreRecordBytes;
}

size_t co_alibi_fwd_inference_workspace_bytes(int batch, int heads_q, int seq_q, int seq_kv) {
  if (batch < 1 || heads_q < 1 || seq_q < 1 || seq_kv < 1) return 0;
  return round_up(static_cast<size_t>(batch) * heads_q *
                      (coalibi::stats_knorm_count(seq_kv) + coalibi::stats_kstart_count(seq_q)) * sizeof(float),
                  256);
}

}  // extern "C"

namespace {

// The forward with its statistics (lse and stats: kstart, the key norms and the work orders),
// without them (lse = stats = NULL: no tail skip), or for inference (knorm scratch only: the
// tail skip without the backward's statistics).  With the tail skip switched off
// (co_alibi_set_tail_skip) no key norms are computed and every key is processed.
// strides: of q, k, v and o (12 values), or NULL.
int fwd_impl(const char* fn, int dtype, const void* q, const void* k, const void* v, const float* slopes, void* o,
             const long long* strides, float* lse, float* stats, float* knorm_ws, int batch, int heads_q, int heads_kv, int seq_q,
             int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  const Shape s{batch, heads_q, heads_kv, seq_q, seq_kv, head_dim};
  int rc;
  if ((rc = check_shape(fn, dtype, s))) return rc;
  if ((rc = check_ptr(fn, "q", q, 16)) || (rc = check_ptr(fn, "k", k, 16)) || (rc = check_ptr(fn, "v", v, 16)) ||
      (rc = check_ptr(fn, "o", o, 16)) || (rc = check_ptr(fn, "slopes", slopes, 4)) ||
      (rc = check_opt_ptr(fn, "lse", lse, 4)) || (rc = check_opt_ptr(fn, "stats", stats, 4)))
    return rc;
  if (!std::isfinite(sm_scale)) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": sm_scale must be finite");

  coalibi::FwdArgs a{};
  const long long* const st4[4] = {strides, strides ? strides + 3 : nullptr, strides ? strides + 6 : nullptr,
                                   strides ? strides + 9 : nullptr};
  if ((rc = read_layout(fn, "q", st4[0], dtype, heads_q, seq_q, head_dim, &a.ql)) ||
      (rc = read_layout(fn, "k", st4[1], dtype, heads_kv, seq_kv, head_dim, &a.kl)) ||
      (rc = read_layout(fn, "v", st4[2], dtype, heads_kv, seq_kv, head_dim, &a.vl)) ||
      (rc = read_layout(fn, "o", st4[3], dtype, heads_q, seq_q, head_dim, &a.ol)) ||
      (rc = check_output(fn, "o", a.ol, batch, heads_q, seq_q, head_dim)) || (rc = check_kv_rows(fn, a.kl, a.vl)))
    return rc;
  a.q = q;
  a.k = k;
  a.v = v;
  a.slopes = slopes;
  a.o = o;
  a.lse = lse;
  const bool skip = g_tail_skip.load() != 0;
  a.every_key = !skip;
  if (stats != nullptr) {  // header, kstart, knorm and the work orders (coalibi_kernels.h)
    const StatsLayout l = stats_layout(batch, heads_q, seq_q, seq_kv);
    int* words = reinterpret_cast<int*>(stats);
    a.flags = words;
    a.kstart = words + l.kstart;
    a.rsum = stats + l.rsum;
    if (skip) {
      a.knorm = stats + l.knorm;
      a.row_order = words + l.row_order;
      a.key_order = words + l.key_order;
    }
  } else if (knorm_ws != nullptr && skip) {  // inference: the row order follows the norms
    a.knorm = knorm_ws;
    a.row_order = reinterpret_cast<int*>(knorm_ws + static_cast<size_t>(batch) * heads_q *
                                                        coalibi::stats_knorm_count(seq_kv));
  }
  a.B = batch;
  a.Hq = heads_q;
  a.Hkv = heads_kv;
  a.Sq = seq_q;
  a.Skv = seq_kv;
  a.nKC = coalibi::stats_knorm_count(seq_kv);
  a.sc2 = sm_scale * coalibi::kLog2eHost;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (dtype) {
    case CO_ALIBI_F16: e = fwd_dispatch_d<_Float16>(a, head_dim, causal != 0, st); break;
    case CO_ALIBI_BF16: e = fwd_dispatch_d<__bf16>(a, head_dim, causal != 0, st); break;
    default: e = fwd_dispatch_d<float>(a, head_dim, causal != 0, st); break;
  }
  if (e != hipSuccess) return fail(CO_ALIBI_ELAUNCH, std::string(fn) + ": launch failed: " + hipGetErrorString(e));
  return CO_ALIBI_OK;
}

}  // namespace

extern "C" {

int co_alibi_fwd(int dtype, const void* q, const void* k, const void* v, const float* slopes, void* o,
                 float* lse, float* stats, int batch, int heads_q, int heads_kv, int seq_q, int seq_kv,
                 int head_dim, int causal, float sm_scale, void* stream) {
  return fwd_impl("co_alibi_fwd", dtype, q, k, v, slopes, o, nullptr, lse, stats, nullptr, batch, heads_q, heads_kv, seq_q,
                  seq_kv, head_dim, causal, sm_scale, stream);
}

int co_alibi_fwd_strided(int dtype, const void* q, const void* k, const void* v, const float* slopes, void* o,
                         const long long* strides, float* lse, float* stats, void* workspace, size_t workspace_bytes,
                         int batch, int heads_q, int heads_kv, int seq_q, int seq_kv, int head_dim, int causal,
                         float sm_scale, void* stream) {
  const char* fn = "co_alibi_fwd_strided";
  int rc;
  if (stats == nullptr) {
    if ((rc = check_ptr(fn, "workspace", workspace, 256))) return rc;
    const size_t need = co_alibi_fwd_inference_workspace_bytes(batch, heads_q, seq_q, seq_kv);
    if (workspace_bytes < need)
      return fail(CO_ALIBI_EINVAL, std::string(fn) + ": workspace of " + std::to_string(workspace_bytes) +
                                       " bytes, need " + std::to_string(need));
  }
  return fwd_impl(fn, dtype, q, k, v, slopes, o, strides, lse, stats, static_cast<float*>(workspace), batch, heads_q,
                  heads_kv, seq_q, seq_kv, head_dim, causal, sm_scale, stream);
}

int co_alibi_fwd_inference(int dtype, const void* q, const void* k, const void* v, const float* slopes, void* o,
                           void* workspace, size_t workspace_bytes, int batch, int heads_q, int heads_kv, int seq_q,
                           int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  const char* fn = "co_alibi_fwd_inference";
  int rc;
  if ((rc = check_ptr(fn, "workspace", workspace, 256))) return rc;
  const size_t need = co_alibi_fwd_inference_workspace_bytes(batch, heads_q, seq_q, seq_kv);
  if (workspace_bytes < need)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": workspace of " + std::to_string(workspace_bytes) +
                                     " bytes, need " + std::to_string(need));
  return fwd_impl(fn, dtype, q, k, v, slopes, o, nullptr, nullptr, nullptr, static_cast<float*>(workspace), batch,
                  heads_q, heads_kv, seq_q, seq_kv, head_dim, causal, sm_scale, stream);
}

}  // extern "C"

namespace {

// stages: 1 = pass 1 (dq, dsum, and zb / cb or the score store), 2 = pass 2 (dk, dv), 3 = both.
// strides: of dout, q, k, v, o, dq, dk and dv (24 values; score-store path only), or NULL.
int bwd_impl(const char* fn, int stages, const long long* strides, int dtype, const void* dout, const void* q, const void* k,
             const void* v, const void* o, const float* lse, const float* stats, const float* slopes, void* dq,
             void* dk, void* dv, void* workspace, size_t workspace_bytes, int batch, int heads_q,
             int heads_kv, int seq_q, int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  const Shape s{batch, heads_q, heads_kv, seq_q, seq_kv, head_dim};
  int rc;
  if ((rc = check_shape(fn, dtype, s))) return rc;
  if ((rc = check_ptr(fn, "dout", dout, 16)) || (rc = check_ptr(fn, "q", q, 16)) ||
      (rc = check_ptr(fn, "k", k, 16)) || (rc = check_ptr(fn, "v", v, 16)) ||
      (rc = check_ptr(fn, "lse", lse, 4)) || (rc = check_ptr(fn, "stats", stats, 4)) ||
      (rc = check_ptr(fn, "slopes", slopes, 4)) || (rc = check_ptr(fn, "workspace", workspace, 256)))
    return rc;
  if ((stages & 1) && ((rc = check_ptr(fn, "o", o, 16)) || (rc = check_ptr(fn, "dq", dq, 16)))) return rc;
  if ((stages & 2) && ((rc = check_ptr(fn, "dk", dk, 16)) || (rc = check_ptr(fn, "dv", dv, 16)))) return rc;
  // A workspace that holds the score store selects that path (where it exists).
  const size_t need_store =
      co_alibi_bwd_score_store_workspace_bytes(dtype, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal);
  const bool store = need_store != 0 && workspace_bytes >= need_store;
  const size_t need = co_alibi_bwd_workspace_bytes(batch, heads_q, seq_q, seq_kv);
  if (!store && strides != nullptr)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": strided operands need the score store (a workspace of " +
                                     std::to_string(need_store) + " bytes; 0: no such path)");
  if (!store && workspace_bytes < need)
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": workspace of " + std::to_string(workspace_bytes) +
                                     " bytes, need " + std::to_string(need));
  if (!std::isfinite(sm_scale)) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": sm_scale must be finite");

  const size_t rows = static_cast<size_t>(batch) * heads_q * seq_q;
  coalibi::BwdArgs a{};
  coalibi::Layout* const layouts[8] = {&a.dol, &a.ql, &a.kl, &a.vl, &a.ol, &a.dql, &a.dkl, &a.dvl};
  const char* const names[8] = {"dout", "q", "k", "v", "o", "dq", "dk", "dv"};
  for (int i = 0; i < 8; ++i) {
    const bool kv = i == 2 || i == 3 || i >= 6;
    if ((rc = read_layout(fn, names[i], strides ? strides + 3 * i : nullptr, dtype, kv ? heads_kv : heads_q,
                          kv ? seq_kv : seq_q, head_dim, layouts[i])) ||
        (i >= 5 && (rc = check_output(fn, names[i], *layouts[i], batch, kv ? heads_kv : heads_q, kv ? seq_kv : seq_q,
                                      head_dim))))
      return rc;
  }
  if ((rc = check_kv_rows(fn, a.kl, a.vl))) return rc;
  a.dout = dout;
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.lse = lse;
  a.slopes = slopes;
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  a.dsum = static_cast<float*>(workspace);
  char* const after_dsum = static_cast<char*>(workspace) + round_up(rows * sizeof(float), 256);
  if (store) {  // the records follow dsum
    a.scores = after_dsum;
    a.score_head = coalibi::score_records_per_head(seq_q, seq_kv, causal != 0);
  } else {  // zb and cb follow dsum
    a.zb = reinterpret_cast<float*>(after_dsum);
    a.cb = reinterpret_cast<float*>(after_dsum +
                                    round_up(block_sums_numel(batch, heads_q, seq_q, seq_kv) * sizeof(float), 256));
  }
  {  // the forward's statistics: header, kstart, knorm, then the work orders it wrote (the
     // kernels follow a table only where the header's flags say it was written)
    const StatsLayout l = stats_layout(batch, heads_q, seq_q, seq_kv);
    const int* words = reinterpret_cast<const int*>(stats);
    a.flags = words;
    a.kstart = words + l.kstart;
    a.rsum = stats + l.rsum;
    a.row_order = words + l.row_order;
    a.key_order = coalibi::key_order_used(batch, heads_q, heads_kv, seq_kv) ? words + l.key_order : nullptr;
  }
  a.B = batch;
  a.Hq = heads_q;
  a.Hkv = heads_kv;
  a.Sq = seq_q;
  a.Skv = seq_kv;
  a.nZB = static_cast<int>(num_zblocks(seq_kv));
  a.sc2 = sm_scale * coalibi::kLog2eHost;
  a.sm_scale = sm_scale;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (dtype) {
    case CO_ALIBI_F16: e = bwd_dispatch_d<_Float16>(a, head_dim, causal != 0, stages, st); break;
    case CO_ALIBI_BF16: e = bwd_dispatch_d<__bf16>(a, head_dim, causal != 0, stages, st); break;
    default: e = bwd_dispatch_d<float>(a, head_dim, causal != 0, stages, st); break;
  }
  if (e != hipSuccess) return fail(CO_ALIBI_ELAUNCH, std::string(fn) + ": launch failed: " + hipGetErrorString(e));
  return CO_ALIBI_OK;
}

}  // namespace

extern "C" {

int co_alibi_bwd(int dtype, const void* dout, const void* q, const void* k, const void* v, const void* o,
                 const float* lse, const float* stats, const float* slopes, void* dq, void* dk, void* dv,
                 void* workspace, size_t workspace_bytes, int batch, int heads_q, int heads_kv, int seq_q,
                 int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  return bwd_impl("co_alibi_bwd", 3, nullptr, dtype, dout, q, k, v, o, lse, stats, slopes, dq, dk, dv, workspace,
                  workspace_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal, sm_scale, stream);
}

int co_alibi_bwd_strided(int dtype, const void* dout, const void* q, const void* k, const void* v, const void* o,
                         const float* lse, const float* stats, const float* slopes, void* dq, void* dk, void* dv,
                         const long long* strides, void* workspace, size_t workspace_bytes, int batch, int heads_q,
                         int heads_kv, int seq_q, int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  return bwd_impl("co_alibi_bwd_strided", 3, strides, dtype, dout, q, k, v, o, lse, stats, slopes, dq, dk, dv,
                  workspace, workspace_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal, sm_scale,
                  stream);
}

int co_alibi_bwd_dq(int dtype, const void* dout, const void* q, const void* k, const void* v, const void* o,
                    const float* lse, const float* stats, const float* slopes, void* dq, void* workspace,
                    size_t workspace_bytes, int batch, int heads_q, int heads_kv, int seq_q, int seq_kv,
                    int head_dim, int causal, float sm_scale, void* stream) {
  return bwd_impl("co_alibi_bwd_dq", 1, nullptr, dtype, dout, q, k, v, o, lse, stats, slopes, dq, nullptr, nullptr,
                  workspace, workspace_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal,
                  sm_scale, stream);
}

int co_alibi_bwd_dkdv(int dtype, const void* dout, const void* q, const void* k, const void* v,
                      const float* lse, const float* stats, const float* slopes, void* dk, void* dv,
                      void* workspace, size_t workspace_bytes, int batch, int heads_q, int heads_kv,
                      int seq_q, int seq_kv, int head_dim, int causal, float sm_scale, void* stream) {
  return bwd_impl("co_alibi_bwd_dkdv", 2, nullptr, dtype, dout, q, k, v, nullptr, lse, stats, slopes, nullptr, dk, dv,
                  workspace, workspace_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal,
                  sm_scale, stream);
}

}  // extern "C"

namespace {

template <typename T>
hipError_t decode_dispatch_d(const coalibi::DecodeArgs& a, int D, hipStream_t st) {
  switch (D) {
    case 32: return coalibi::launch_decode<T, 32>(a, st);
    case 64: return coalibi::launch_decode<T, 64>(a, st);
    case 256:
      if constexpr (sizeof(T) == 2) return coalibi::launch_decode<T, 256>(a, st);
      return hipErrorInvalidValue;
    default: return coalibi::launch_decode<T, 128>(a, st);
  }
}

size_t decode_chunks(int seq_kv) {
  return (static_cast<size_t>(seq_kv) + coalibi::kDecodeChunkKeys - 1) / coalibi::kDecodeChunkKeys;
}

// Upper bound of the split count of a decode over seq_kv keys (one split holds >= 1 chunk).
size_t decode_splits_max(int seq_kv) {
  return std::min(decode_chunks(seq_kv), static_cast<size_t>(coalibi::kMaxDecodeSplits));
}

// Compute units of the current device (queried once per device).
int device_cus() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// How a decode is split, by its type and by units = batch * heads_kv against the `slots` work-groups
// that the launch is sized for.  Figures: us on the GPU alone, 512 slots, more splits -> fewer.
constexpr int kDecodeRaggedSplits = 4;
struct DecodeRule {
  bool fp32;
  int head_dim, slots;
  long long units;

  // Whether a sequence of up to `chunks` chunks is one work-group's (one split, and no merge launch, which
  // costs as much as one to three more chunks of the walk).  Units 8: D 32 fp16 at 3 chunks 8.2 -> 6.8, D 64 8.8 ->
  // 8.4, D 128 bf16 at 2 10.3 -> 9.0 (at 3 10.8 -> 10.9, with lengths of 1/8 to all of the bound 10.4 -> 8.7), fp32 D 32
  // at 2 9.2 -> 7.8; D 256 at 2 13.9 -> 14.1 and fp32 D 64 11.1 -> 11.4 (at 3 14.5 -> 18.3 and 11.3 -> 15.5).  With a
  // work-group per chunk above half the slots more splits cost more: at 3 chunks, units 100, D 128 12.7 -> 10.8, D 256
  // 21.8 -> 17.9; units 192 fp32 D 64 22.7 -> 17.6 (units 128 16.8 -> 17.3; ragged, D 256 16.5 -> 18.7).  Above half
  // the slots in units two splits take two rounds: units 288, 6 chunks, D 128 29.5 -> 28.0, 5 chunks, D 256 61 -> 57
  // (8: 79 -> 84), 3 chunks, fp32 D 128 62 -> 55 (4: 64 -> 69); ragged lengths of at most 8 chunks take 5 to 30 % less
  // on average.  From 5/6 of the slots on one split loses nothing: units 432, D 128, 8 chunks 43.4 -> 38.7, 32 chunks
  // 157 -> 147 (units 384: 124 -> 135), but D 32 from 16 chunks on (units 448, 32 chunks 65.9 -> 67.6).
  bool one_split(int chunks, bool ragged) const {
    if (units >= slots) return true;
    if (units * 6 >= slots * 5LL) return head_dim > 32 || chunks <= 16;
    if (units * 2 > slots) return chunks <= (ragged ? 8 : fp32 ? 3 : head_dim <= 128 ? 6 : 5);
    if (chunks <= 3 && units * chunks * (ragged || fp32 ? 4 : 6) > slots * 3LL) return true;
    if (fp32) return chunks <= (head_dim <= 32 ? 2 : 1);
    return chunks <= (head_dim <= 64 ? 3 : head_dim > 128 ? 1 : ragged ? 3 : 2);
  }

  // Equal splits: as many per sequence as it takes to give every slot a work-group.
  int even_splits(int chunks) const {
    const long long want = (slots + units - 1) / units;
    const int most = std::min(chunks, coalibi::kMaxDecodeSplits);
    const int cps = (chunks + static_cast<int>(std::min<long long>(want, most)) - 1) /
                    static_cast<int>(std::min<long long>(want, most));
    return (chunks + cps - 1) / cps;
  }

  // Splits of every sequence of a launch bound by `chunks` chunks.  Equal lengths: where even_splits' last
  // round is nearly empty, longer splits (decode_cps): units 100, 32 chunks, D 128 48 -> 39; units 36, 100 chunks,
  // D 256 113 -> 89.  Up to half as long again from D 128 on (units 180, 125 chunks, D 128 294 -> 267; with a quarter
  // 295).  The small types gain from a quarter on few units (units 110, 32 chunks, D 64 33 -> 29), not on short
  // walks (units 100, 6 chunks, D 32 10.1 -> 11.3) or more units (units 210, 125 chunks, D 32 122 -> 133).
  int splits(int chunks, bool ragged) const {
    if (one_split(chunks, ragged)) return 1;
    const bool small = !fp32 && head_dim <= 64;
    const int even = even_splits(chunks);
    if (ragged || (small && (chunks < 4 * even || units * 4 >= slots))) return even;
    const int cps = coalibi::decode_cps(units * chunks, chunks, slots, coalibi::kMaxDecodeSplits, small ? 4 : 8, chunks - 1,
                                        [&](int c) { return units * ((chunks + c - 1) / c); });
    const int n = (chunks + cps - 1) / cps, own = (chunks + n - 1) / n;
    return (chunks + own - 1) / own;  // in equal runs
  }

  // Whether a batch with a length per sequence shares its real chunks out (the kernels' plan) rather than
  // splitting every sequence by the bound.  The plan costs the two kernels about 3.5 us together, against
  // the part of a split's walk that it saves.  Lengths of 1/8 to all of the bound, units 128: D 128 at 2 chunks per
  // split 17.7 -> 20.6, at 4 +2 %, at 6 -17 %, at 16 -8 %; D 64 at 4 +5 %, at 6 -15 %; D 32 at 4 +11 %, at 8 +2 %, at
  // 12 -12 %; D 256 at 2 +10 %, at 4 -3 %; fp32 D 64 at 2 +17 %, at 4 -9 %.
  bool plans(int chunks, int splits) const {
    return splits > 1 && (chunks + splits - 1) / splits >= (fp32 || head_dim > 128 ? 4 : head_dim > 32 ? 5 : 9);
  }
  int plan_slack() const { return !fp32 && head_dim <= 64 ? 4 : 6; }
};

// Bytes of split-K partials for `parts` (batch, query head, split) triples: the maximum, the sum
// and the sigma total (one 256-byte aligned fp32 array each), then head_dim floats of O per part.
size_t decode_partials_bytes(size_t parts, int head_dim) {
  return 3 * round_up(parts * sizeof(float), 256) + parts * head_dim * sizeof(float);
}

// Device scratch of co_alibi_decode_noalloc: the split-K partials of callers that cannot
// allocate.  Each GPU holds its own copy for the life of the process.  Host code never uses
// this name as an address: its device address, per device, comes from hipGetSymbolAddress.
constexpr size_t kDecodeScratchBytes = CO_ALIBI_DECODE_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kDecodeScratchBytes];

// The device address of `scratch` on the current device, looked up once per device (with that
// device current) and kept.
int scratch_address(const char* fn, void** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(CO_ALIBI_ELAUNCH, std::string(fn) + ": no current HIP device");
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(CO_ALIBI_ELAUNCH, std::string(fn) + ": scratch lookup failed: " + hipGetErrorString(e));
    addr[dev] = p;
  }
  *out = addr[dev];
  return CO_ALIBI_OK;
}

// co_alibi_decode and co_alibi_decode_noalloc.  The caller's workspace is laid out for the
// largest split count a decode of seq_kv keys can take (its size depends on the shape only);
// the library's scratch is laid out for this launch's split count, which fits more.
int decode_impl(const char* fn, bool scratch_ws, int dtype, const void* q, const void* k_cache,
                const void* v_cache, const float* slopes, const int* seq_lens, void* o, float* lse,
                void* workspace, size_t workspace_bytes, int batch, int heads_q, int heads_kv, int seq_kv,
                int kv_capacity, int head_dim, float sm_scale, void* stream) {
  const Shape s{batch, heads_q, heads_kv, 1, seq_kv, head_dim};
  int rc;
  if ((rc = check_shape(fn, dtype, s))) return rc;
  // The decode kernels read K in pairs of 16-element fragments; a head dim of 16 is one.  The
  // torch operator co_alibi::decode pads such heads to 32 with zero columns, which changes no
  // product.
  if (head_dim == 16)
    return fail(CO_ALIBI_EUNSUPPORTED, std::string(fn) + ": head_dim 16 has no decode kernel (pad q and the "
                                                         "caches to 32 with zeros)");
  // A wavefront's K and V tiles (32 cache rows each) of fp32 at head dim 256 take 66 KB of LDS,
  // four wavefronts more than a CU has.
  if (head_dim == 256 && dtype == CO_ALIBI_F32)
    return fail(CO_ALIBI_EUNSUPPORTED, std::string(fn) + ": decode at head_dim 256 needs fp16 or bf16");
  if (heads_q / heads_kv > coalibi::kMaxDecodeGroup)
    return fail(CO_ALIBI_EUNSUPPORTED, std::string(fn) + ": at most " + std::to_string(coalibi::kMaxDecodeGroup) +
                                           " query heads per kv head");
  if (kv_capacity < seq_kv) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": kv_capacity is below seq_kv");
  if (decode_chunks(seq_kv) > static_cast<size_t>(coalibi::kMaxDecodeChunks))
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": seq_kv above " +
                                     std::to_string(coalibi::kMaxDecodeChunks * coalibi::kDecodeChunkKeys));
  // The workspace size first: it depends on the shape only, and a decode whose partials do not fit
  // is refused before any pointer is looked at.
  const DecodeRule rule{dtype == CO_ALIBI_F32, head_dim, coalibi::kDecodeWGsPerCU * device_cus(),
                        static_cast<long long>(batch) * heads_kv};
  const int chunks = static_cast<int>(decode_chunks(seq_kv));
  int splits = rule.splits(chunks, seq_lens != nullptr);
  const size_t rows = static_cast<size_t>(batch) * heads_q;
  size_t parts = rows * (scratch_ws ? static_cast<size_t>(splits) : decode_splits_max(seq_kv));
  const size_t need = decode_partials_bytes(parts, head_dim);
  if (workspace_bytes < need) {
    if (scratch_ws)
      return fail(CO_ALIBI_EINVAL, std::string(fn) + ": the split-K partials of this decode need " +
                                       std::to_string(need) + " bytes, above the library scratch of " +
                                       std::to_string(workspace_bytes) + " bytes");
    return fail(CO_ALIBI_EINVAL, std::string(fn) + ": workspace of " + std::to_string(workspace_bytes) +
                                     " bytes, need " + std::to_string(need));
  }
  if ((rc = check_ptr(fn, "q", q, 16)) || (rc = check_ptr(fn, "k_cache", k_cache, 16)) ||
      (rc = check_ptr(fn, "v_cache", v_cache, 16)) || (rc = check_ptr(fn, "o", o, 16)) ||
      (rc = check_ptr(fn, "slopes", slopes, 4)) || (rc = check_opt_ptr(fn, "seq_lens", seq_lens, 4)) ||
      (rc = check_opt_ptr(fn, "lse", lse, 4)) || (rc = check_ptr(fn, "workspace", workspace, 256)))
    return rc;
  if (!std::isfinite(sm_scale)) return fail(CO_ALIBI_EINVAL, std::string(fn) + ": sm_scale must be finite");

  const bool plan = seq_lens != nullptr && rule.plans(chunks, splits);
  if (plan) {
    // Lengths below seq_kv leave work-groups to the longer sequences, up to kDecodeRaggedSplits
    // times as many splits each, where their partials fit.
    const size_t most = std::min(static_cast<size_t>(splits) * kDecodeRaggedSplits, decode_splits_max(seq_kv));
    for (size_t n = most; n > static_cast<size_t>(splits); n = n / 2)
      if (decode_partials_bytes(rows * n, head_dim) <= workspace_bytes) {
        splits = static_cast<int>(n);
        break;
      }
    if (scratch_ws) parts = rows * splits;
  }
  const size_t stat_bytes = round_up(parts * sizeof(float), 256);
  char* ws = static_cast<char*>(workspace);
  coalibi::DecodeArgs a{};
  a.q = q;
  a.k = k_cache;
  a.v = v_cache;
  a.slopes = slopes;
  a.o = o;
  a.lse = lse;
  a.pmax = reinterpret_cast<float*>(ws);
  a.psum = reinterpret_cast<float*>(ws + stat_bytes);
  a.psig = reinterpret_cast<float*>(ws + 2 * stat_bytes);
  a.pout = reinterpret_cast<float*>(ws + 3 * stat_bytes);
  a.seq_lens = seq_lens;
  a.B = batch;
  a.Hq = heads_q;
  a.Hkv = heads_kv;
  a.G = heads_q / heads_kv;
  a.L = seq_kv;
  a.cap = kv_capacity;
  a.nSplits = splits;
  a.cps = (chunks + splits - 1) / splits;
  a.slots = rule.slots;
  a.slack = rule.plan_slack();
  a.plan = plan;
  a.sc2 = sm_scale * coalibi::kLog2eHost;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (dtype) {
    case CO_ALIBI_F16: e = decode_dispatch_d<_Float16>(a, head_dim, st); break;
    case CO_ALIBI_BF16: e = decode_dispatch_d<__bf16>(a, head_dim, st); break;
    default: e = decode_dispatch_d<float>(a, head_dim, st); break;
  }
  if (e != hipSuccess) return fail(CO_ALIBI_ELAUNCH, std::string(fn) + ": launch failed: " + hipGetErrorString(e));
  return CO_ALIBI_OK;
}

}  // namespace

extern "C" {

size_t co_alibi_decode_workspace_bytes(int batch, int heads_q, int seq_kv, int head_dim) {
  if (batch < 1 || heads_q < 1 || seq_kv < 1 || head_dim < 1) return 0;
  return decode_partials_bytes(static_cast<size_t>(batch) * heads_q * decode_splits_max(seq_kv), head_dim);
}

int co_alibi_decode_splits(int dtype, int batch, int heads_kv, int seq_kv, int head_dim, int ragged) {
  if (batch < 1 || heads_kv < 1 || seq_kv < 1 || decode_chunks(seq_kv) > static_cast<size_t>(coalibi::kMaxDecodeChunks))
    return 0;
  const DecodeRule rule{dtype == CO_ALIBI_F32, head_dim, coalibi::kDecodeWGsPerCU * device_cus(),
                        static_cast<long long>(batch) * heads_kv};
  const int chunks = static_cast<int>(decode_chunks(seq_kv)), splits = rule.splits(chunks, ragged != 0);
  return ragged != 0 && rule.plans(chunks, splits) ? -splits : splits;
}

int co_alibi_decode(int dtype, const void* q, const void* k_cache, const void* v_cache, const float* slopes,
                    const int* seq_lens, void* o, float* lse, void* workspace, size_t workspace_bytes, int batch,
                    int heads_q, int heads_kv, int seq_kv, int kv_capacity, int head_dim, float sm_scale,
                    void* stream) {
  return decode_impl("co_alibi_decode", false, dtype, q, k_cache, v_cache, slopes, seq_lens, o, lse, workspace,
                     workspace_bytes, batch, heads_q, heads_kv, seq_kv, kv_capacity, head_dim, sm_scale, stream);
}

int co_alibi_decode_noalloc(int dtype, const void* q, const void* k_cache, const void* v_cache,
                            const float* slopes, const int* seq_lens, void* o, float* lse, int batch, int heads_q,
                            int heads_kv, int seq_kv, int kv_capacity, int head_dim, float sm_scale, void* stream) {
  const char* fn = "co_alibi_decode_noalloc";
  void* ws = nullptr;
  if (const int rc = scratch_address(fn, &ws)) return rc;
  return decode_impl(fn, true, dtype, q, k_cache, v_cache, slopes, seq_lens, o, lse, ws, kDecodeScratchBytes, batch,
                     heads_q, heads_kv, seq_kv, kv_capacity, head_dim, sm_scale, stream);
}

const char* co_alibi_last_error(void) { return g_last_error.c_str(); }

int co_alibi_abi_version(void) { return 6; }

}  // extern "C"
