// PyTorch-ROCm operators over the C ABI of libco_alibi (include/co_alibi.h).
//
//   co_alibi::fwd(q, k, v, slopes, causal, sm_scale, with_stats) -> (o, lse, stats)
//   co_alibi::bwd(do, q, k, v, o, lse, stats, slopes, causal, sm_scale) -> (dq, dk, dv)
//   co_alibi::bwd_dq(do, q, k, v, o, lse, stats, slopes, causal, sm_scale) -> dq
//   co_alibi::fwd_qkv(qkv, slopes, causal, sm_scale, with_stats) -> (o, lse, stats)
//   co_alibi::bwd_qkv(do, qkv, o, lse, stats, slopes, causal, sm_scale) -> dqkv
//   co_alibi::decode(q, k_cache, v_cache, slopes, seq_lens, max_seq_len, sm_scale, with_lse) -> (o, lse)
//
// They replace the reference's two Triton launches with their buffer set-up
// (co_alibi_attn/co_alibi_attn.py:35-57 and :83-133); decode has no counterpart there.  Each
// kernel runs on the caller's current HIP stream under a device guard of the inputs' device and
// allocates only through torch's caching allocator, so the operators can be captured in a HIP
// graph.  co_alibi::fwd carries its backward as a C++ autograd kernel: dQ alone runs backward
// pass 1 only (co_alibi::bwd_dq); any key / value gradient runs both passes (co_alibi::bwd).
// co_alibi::bwd uses the score store (pass 1 keeps s and dS, pass 2 reduces them) where the
// library has it and its workspace fits: at most CO_ALIBI_SCORE_STORE_LIMIT_MB megabytes (an
// environment variable read once; 16384 by default, 0 turns the store off) and at most half
// of the device memory that is free or cached by torch's allocator at the call.  If allocating
// it fails anyway, the backward takes the recompute path, whose workspace is O(S^2 / 32).
// The shape functions for FakeTensor / meta tracing are registered from Python.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/autograd.h>
#include <torch/library.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstdlib>
#include <tuple>

#include "../../include/co_alibi.h"

namespace {

using at::Tensor;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CO_ALIBI_F32;
    case at::kHalf: return CO_ALIBI_F16;
    case at::kBFloat16: return CO_ALIBI_BF16;
    default: TORCH_CHECK_TYPE(false, "co_alibi: q, k, v must be float32, float16 or bfloat16, got ", t);
  }
  return -1;
}

void check(int rc) {
  TORCH_CHECK(rc == CO_ALIBI_OK, "co_alibi_attn: ", co_alibi_last_error(), " (status ", rc, ")");
}

// Contiguous tensor whose data pointer is 16-byte aligned (what the kernels load).
Tensor aligned(const Tensor& t) {
  Tensor c = t.contiguous();
  if (reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 != 0) c = c.clone();
  return c;
}

// Whether the kernels can read a (B, H, S, D) operand in place (co_alibi_fwd_strided's rules), and its
// batch, head and row strides: those of dimensions of size 1 do not matter and are given as if
// contiguous, which the kernels have faster instantiations for.
struct Strides {
  long long v[3];
};
Strides strides_of(const Tensor& t) {
  const int64_t H = t.size(1), S = t.size(2), D = t.size(3);
  return {{t.size(0) == 1 ? H * S * D : t.stride(0), H == 1 ? S * D : t.stride(1), S == 1 ? D : t.stride(2)}};
}
bool readable(const Tensor& t) {
  const int64_t per16 = 16 / t.element_size();
  if (t.stride(3) != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
  const Strides s = strides_of(t);
  return s.v[0] % per16 == 0 && s.v[1] % per16 == 0 && s.v[2] % per16 == 0 && s.v[2] >= t.size(3) && s.v[2] <= 1 << 20;
}
// The operand itself where the kernels can read it in place, else a contiguous aligned copy.
Tensor in_place(const Tensor& t) { return readable(t) ? t : aligned(t); }
// An output itself where the kernels can write it in place, else a contiguous tensor to copy from (a
// packed projection's rows can be further apart than the kernels' 2^20 elements).
Tensor writable(const Tensor& t) { return readable(t) ? t : at::empty(t.sizes(), t.options()); }
// K and V, whose row strides must agree.
std::pair<Tensor, Tensor> kv_in_place(const Tensor& k, const Tensor& v) {
  if (readable(k) && readable(v) && strides_of(k).v[2] == strides_of(v).v[2]) return {k, v};
  return {aligned(k), aligned(v)};
}
template <size_t N>
std::array<long long, 3 * N> all_strides(const std::array<Tensor, N>& ts) {
  std::array<long long, 3 * N> out{};
  for (size_t i = 0; i < N; ++i) {
    const Strides s = strides_of(ts[i]);
    std::copy(s.v, s.v + 3, out.begin() + 3 * i);
  }
  return out;
}

// fp32 copy of the penalty slopes on the inputs' device (no copy when already so).
Tensor slopes_f32(const Tensor& slopes, const Tensor& like) {
  return slopes.detach().to(like.device(), at::kFloat).contiguous();
}

Tensor empty_stats(const Tensor& q) { return at::empty({0}, q.options().dtype(at::kFloat)); }

int64_t stats_numel(int64_t batch, int64_t heads_q, int64_t seq_q, int64_t seq_kv) {
  return static_cast<int64_t>(co_alibi_stats_numel(static_cast<int>(batch), static_cast<int>(heads_q),
                                                   static_cast<int>(seq_q), static_cast<int>(seq_kv)));
}

hipStream_t current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ---------------------------------------------------------------------------- forward

// The forward into o (B, Hq, Sq, D); returns lse and stats (empty for inference).
std::tuple<Tensor, Tensor> launch_fwd(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& slopes,
                                      const Tensor& o, bool causal, double sm_scale, bool with_stats) {
  const int64_t batch = q_in.size(0), heads_q = q_in.size(1), seq_q = q_in.size(2), head_dim = q_in.size(3);
  const int64_t heads_kv = k_in.size(1), seq_kv = k_in.size(2);
  c10::hip::HIPGuard guard(q_in.device().index());
  const Tensor q = in_place(q_in);
  const auto [k, v] = kv_in_place(k_in, v_in);
  const Tensor sl = slopes_f32(slopes, q);
  const auto f32 = q.options().dtype(at::kFloat);
  Tensor lse = with_stats ? at::empty({batch, heads_q, seq_q}, f32) : empty_stats(q);
  Tensor stats = with_stats ? at::empty({stats_numel(batch, heads_q, seq_q, seq_kv)}, f32) : empty_stats(q);
  // Inference: the tail skip with only its key-norm and work-order scratch.
  const size_t ws_bytes = with_stats ? 0 : co_alibi_fwd_inference_workspace_bytes(batch, heads_q, seq_q, seq_kv);
  Tensor ws;
  if (!with_stats) ws = at::empty({static_cast<int64_t>(ws_bytes)}, q.options().dtype(at::kByte));
  const Tensor out = writable(o);
  const auto strides = all_strides<4>({q, k, v, out});
  check(co_alibi_fwd_strided(dtype_code(q.scalar_type()), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                             sl.data_ptr<float>(), out.data_ptr(), strides.data(),
                             with_stats ? lse.data_ptr<float>() : nullptr,
                             with_stats ? stats.data_ptr<float>() : nullptr, with_stats ? nullptr : ws.data_ptr(),
                             ws_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal ? 1 : 0,
                             static_cast<float>(sm_scale), current_stream(q)));
  if (!out.is_same(o)) o.copy_(out);
  return {lse, stats};
}

std::tuple<Tensor, Tensor, Tensor> fwd_hip(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in,
                                           const Tensor& slopes, bool causal, double sm_scale, bool with_stats) {
  const int64_t batch = q_in.size(0), heads_q = q_in.size(1), seq_q = q_in.size(2), head_dim = q_in.size(3);
  const int64_t heads_kv = k_in.size(1), seq_kv = k_in.size(2);
  if (q_in.numel() == 0 || seq_kv == 0) {
    // Nothing to launch.  Rows that see no key get what the reference's l = 0 gives:
    // O = 0 / (0 + 1e-9) = 0 and LSE = -inf + log(1e-9) = -inf (co_alibi_fwd_kernel.py:115,120).
    Tensor o = at::zeros(q_in.sizes(), q_in.options());
    if (!with_stats) return {o, empty_stats(q_in), empty_stats(q_in)};
    Tensor lse = at::full({batch, heads_q, seq_q}, -std::numeric_limits<float>::infinity(),
                          q_in.options().dtype(at::kFloat));
    return {o, lse, at::zeros({stats_numel(batch, heads_q, seq_q, seq_kv)}, q_in.options().dtype(at::kFloat))};
  }
  Tensor o = at::empty(q_in.sizes(), q_in.options());
  auto [lse, stats] = launch_fwd(q_in, k_in, v_in, slopes, o, causal, sm_scale, with_stats);
  return {o, lse, stats};
}

// --------------------------------------------------------------------------- backward

// Largest workspace co_alibi::bwd takes for the score store (the environment's limit).
size_t score_store_limit() {
  static const size_t limit = [] {
    const char* e = std::getenv("CO_ALIBI_SCORE_STORE_LIMIT_MB");
    const long long mb = e != nullptr && *e != '\0' ? std::atoll(e) : 16384;
    return mb > 0 ? static_cast<size_t>(mb) << 20 : size_t{0};
  }();
  return limit;
}

// Device memory a new allocation can take on the current device: what the driver reports free
// plus what torch's caching allocator holds unused.
size_t device_memory_available() {
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return 0;
  const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats(c10::hip::current_device());
  const size_t agg = static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE);
  const int64_t cached = stats.reserved_bytes[agg].current - stats.allocated_bytes[agg].current;
  return free_b + static_cast<size_t>(cached > 0 ? cached : 0);
}

// Shared set-up of the backward operators; stages 1 = pass 1 only (dq), 3 = both passes, into the
// given outputs (dk and dv undefined with stages 1).  The score-store path reads and writes every
// operand in place; the recompute path takes contiguous ones.
void launch_bwd(int stages, const Tensor& do_in, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in,
                const Tensor& o_in, const Tensor& lse_in, const Tensor& stats_in, const Tensor& slopes, bool causal,
                double sm_scale, const Tensor& dq, const Tensor& dk, const Tensor& dv) {
  const int64_t batch = q_in.size(0), heads_q = q_in.size(1), seq_q = q_in.size(2), head_dim = q_in.size(3);
  const int64_t heads_kv = k_in.size(1), seq_kv = k_in.size(2);
  c10::hip::HIPGuard guard(q_in.device().index());
  const Tensor lse = lse_in.contiguous(), stats = stats_in.contiguous();
  const Tensor sl = slopes_f32(slopes, q_in);
  const int code = dtype_code(q_in.scalar_type());
  const int causal_i = causal ? 1 : 0;
  const float scale = static_cast<float>(sm_scale);
  const hipStream_t st = current_stream(q_in);
  const Tensor do_t = do_in.to(q_in.scalar_type());
  const auto bytes = q_in.options().dtype(at::kByte);
  if (stages & 2) {
    const size_t store_bytes =
        co_alibi_bwd_score_store_workspace_bytes(code, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal_i);
    Tensor ws;
    if (store_bytes != 0 && store_bytes <= score_store_limit() && store_bytes <= device_memory_available() / 2) {
      try {
        ws = at::empty({static_cast<int64_t>(store_bytes)}, bytes);
      } catch (const c10::OutOfMemoryError&) {  // the recompute path's smaller workspace below
      }
    }
    if (ws.defined()) {
      const Tensor q = in_place(q_in), o = in_place(o_in), dout = in_place(do_t);
      const auto [k, v] = kv_in_place(k_in, v_in);
      const std::array<Tensor, 3> to = {dq, dk, dv}, out = {writable(dq), writable(dk), writable(dv)};
      const auto strides = all_strides<8>({dout, q, k, v, o, out[0], out[1], out[2]});
      check(co_alibi_bwd_strided(code, dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                 lse.data_ptr<float>(), stats.data_ptr<float>(), sl.data_ptr<float>(),
                                 out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), strides.data(),
                                 ws.data_ptr(), store_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim,
                                 causal_i, scale, st));
      for (int i = 0; i < 3; ++i)
        if (!out[i].is_same(to[i])) to[i].copy_(out[i]);
      return;
    }
  }
  const Tensor q = aligned(q_in), k = aligned(k_in), v = aligned(v_in), o = aligned(o_in), dout = aligned(do_t);
  const size_t ws_bytes = co_alibi_bwd_workspace_bytes(batch, heads_q, seq_q, seq_kv);
  const Tensor ws = at::empty({static_cast<int64_t>(ws_bytes)}, bytes);
  auto dense = [](const Tensor& t) { return t.defined() && !t.is_contiguous() ? at::empty(t.sizes(), t.options()) : t; };
  const Tensor cq = dense(dq), ck = dense(dk), cv = dense(dv);
  if (stages & 2) {
    check(co_alibi_bwd(code, dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                       lse.data_ptr<float>(), stats.data_ptr<float>(), sl.data_ptr<float>(), cq.data_ptr(),
                       ck.data_ptr(), cv.data_ptr(), ws.data_ptr(), ws_bytes, batch, heads_q, heads_kv, seq_q, seq_kv,
                       head_dim, causal_i, scale, st));
  } else {
    check(co_alibi_bwd_dq(code, dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                          lse.data_ptr<float>(), stats.data_ptr<float>(), sl.data_ptr<float>(), cq.data_ptr(),
                          ws.data_ptr(), ws_bytes, batch, heads_q, heads_kv, seq_q, seq_kv, head_dim, causal_i, scale,
                          st));
  }
  for (const auto& [to, from] : {std::pair(dq, cq), std::pair(dk, ck), std::pair(dv, cv)})
    if (to.defined() && !to.is_same(from)) to.copy_(from);
}

std::tuple<Tensor, Tensor, Tensor> bwd_common(int stages, const Tensor& dout, const Tensor& q, const Tensor& k,
                                              const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& stats,
                                              const Tensor& slopes, bool causal, double sm_scale) {
  if (q.numel() == 0 || k.numel() == 0) {  // no (query, key) pair: every gradient is zero
    return {at::zeros(q.sizes(), q.options()), at::zeros(k.sizes(), k.options()), at::zeros(v.sizes(), v.options())};
  }
  Tensor dq = at::empty(q.sizes(), q.options()), dk, dv;
  if (stages & 2) {
    dk = at::empty(k.sizes(), k.options());
    dv = at::empty(v.sizes(), v.options());
  }
  launch_bwd(stages, dout, q, k, v, o, lse, stats, slopes, causal, sm_scale, dq, dk, dv);
  return {dq, dk, dv};
}

std::tuple<Tensor, Tensor, Tensor> bwd_hip(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v,
                                           const Tensor& o, const Tensor& lse, const Tensor& stats,
                                           const Tensor& slopes, bool causal, double sm_scale) {
  return bwd_common(3, dout, q, k, v, o, lse, stats, slopes, causal, sm_scale);
}

Tensor bwd_dq_hip(const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                  const Tensor& lse, const Tensor& stats, const Tensor& slopes, bool causal, double sm_scale) {
  return std::get<0>(bwd_common(1, dout, q, k, v, o, lse, stats, slopes, causal, sm_scale));
}

// ------------------------------------------------------------------------- packed QKV

// Part i (0 q, 1 k, 2 v) of a packed (B, S, 3, H, D) tensor, and any (B, S, H, D) tensor, as (B, H, S, D).
Tensor qkv_part(const Tensor& qkv, int64_t i) { return qkv.select(2, i).transpose(1, 2); }

// Attention of a fused projection's output, read in place; o is (B, S, H, D) contiguous, which the
// output projection reads without a copy.
std::tuple<Tensor, Tensor, Tensor> fwd_qkv_hip(const Tensor& qkv, const Tensor& slopes, bool causal, double sm_scale,
                                               bool with_stats) {
  const Tensor q = qkv_part(qkv, 0), k = qkv_part(qkv, 1), v = qkv_part(qkv, 2);
  const std::vector<int64_t> shape{qkv.size(0), qkv.size(1), qkv.size(3), qkv.size(4)};
  if (qkv.numel() == 0) {
    Tensor o, lse, stats;
    std::tie(o, lse, stats) = fwd_hip(q, k, v, slopes, causal, sm_scale, with_stats);
    return {at::zeros(shape, qkv.options()), lse, stats};
  }
  Tensor o = at::empty(shape, qkv.options());
  auto [lse, stats] = launch_fwd(q, k, v, slopes, o.transpose(1, 2), causal, sm_scale, with_stats);
  return {o, lse, stats};
}

// Its gradient, written into one packed tensor (no per-part gradients to zero-fill and add up).
Tensor bwd_qkv_hip(const Tensor& dout, const Tensor& qkv, const Tensor& o, const Tensor& lse, const Tensor& stats,
                   const Tensor& slopes, bool causal, double sm_scale) {
  if (qkv.numel() == 0) return at::zeros(qkv.sizes(), qkv.options());
  Tensor dqkv = at::empty(qkv.sizes(), qkv.options());
  launch_bwd(3, dout.transpose(1, 2), qkv_part(qkv, 0), qkv_part(qkv, 1), qkv_part(qkv, 2), o.transpose(1, 2), lse,
             stats, slopes, causal, sm_scale, qkv_part(dqkv, 0), qkv_part(dqkv, 1), qkv_part(dqkv, 2));
  return dqkv;
}

// ----------------------------------------------------------------------------- decode

std::tuple<Tensor, Tensor> decode_hip(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& slopes,
                                      const c10::optional<Tensor>& seq_lens, int64_t max_seq_len, double sm_scale,
                                      bool with_lse) {
  const int64_t batch = q_in.size(0), heads_q = q_in.size(1), head_dim = q_in.size(3);
  const int64_t heads_kv = k_in.size(1), capacity = k_in.size(2);
  if (q_in.numel() == 0) {  // an empty batch
    Tensor o = at::empty(q_in.sizes(), q_in.options());
    Tensor lse = with_lse ? at::empty({batch, heads_q, 1}, q_in.options().dtype(at::kFloat)) : empty_stats(q_in);
    return {o, lse};
  }
  c10::hip::HIPGuard guard(q_in.device().index());
  if (head_dim == 16) {
    // The decode kernels have no head dim of 16: run on heads padded to 32 with zero columns
    // (the products over d are unchanged, the padding columns of O come out zero) and return
    // the first 16 columns.  This copies the caches once per step.
    auto [o32, lse] = decode_hip(at::constant_pad_nd(q_in, {0, 16}), at::constant_pad_nd(k_in, {0, 16}),
                                 at::constant_pad_nd(v_in, {0, 16}), slopes, seq_lens, max_seq_len, sm_scale, with_lse);
    return {o32.narrow(3, 0, 16).contiguous(), lse};
  }
  const Tensor q = aligned(q_in), k = aligned(k_in), v = aligned(v_in);
  Tensor lens;
  if (seq_lens.has_value() && seq_lens->defined()) lens = seq_lens->to(q.device(), at::kInt).contiguous();
  const Tensor sl = slopes_f32(slopes, q);
  Tensor o = at::empty_like(q);
  Tensor lse = with_lse ? at::empty({batch, heads_q, 1}, q.options().dtype(at::kFloat)) : empty_stats(q);
  const size_t ws_bytes = co_alibi_decode_workspace_bytes(batch, heads_q, max_seq_len, head_dim);
  Tensor ws = at::empty({static_cast<int64_t>(ws_bytes)}, q.options().dtype(at::kByte));
  check(co_alibi_decode(dtype_code(q.scalar_type()), q.data_ptr(), k.data_ptr(), v.data_ptr(), sl.data_ptr<float>(),
                        lens.defined() ? lens.data_ptr<int>() : nullptr, o.data_ptr(),
                        with_lse ? lse.data_ptr<float>() : nullptr, ws.data_ptr(), ws_bytes, batch, heads_q, heads_kv,
                        max_seq_len, capacity, head_dim, static_cast<float>(sm_scale), current_stream(q)));
  return {o, lse};
}

// --------------------------------------------------------------------------- autograd

// The operators called below autograd (the forward kernel) and from the backward.
std::tuple<Tensor, Tensor, Tensor> call_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes,
                                            bool causal, double sm_scale, bool with_stats) {
  static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("co_alibi::fwd", "").typed<decltype(fwd_hip)>();
  return op.call(q, k, v, slopes, causal, sm_scale, with_stats);
}

// Autograd function of co_alibi::fwd (the role of the reference's CoALIBIAttention,
// co_alibi_attn.py:24-135): saves q, k, v, o, lse, stats and the slopes; lse and stats carry no
// gradient; slopes, causal, sm_scale and with_stats get none.
class FwdFunction : public torch::autograd::Function<FwdFunction> {
 public:
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q,
                                                const Tensor& k, const Tensor& v, const Tensor& slopes, bool causal,
                                                double sm_scale, bool with_stats) {
    Tensor o, lse, stats;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(o, lse, stats) = call_fwd(q, k, v, slopes, causal, sm_scale, with_stats);
    }
    ctx->save_for_backward({q, k, v, o, lse, stats, slopes});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["sm_scale"] = sm_scale;
    ctx->saved_data["with_stats"] = with_stats;
    ctx->mark_non_differentiable({lse, stats});
    // lse and stats never get a gradient: without this the engine would fill zero tensors for
    // them before every backward.
    ctx->set_materialize_grads(false);
    return {o, lse, stats};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    TORCH_CHECK(ctx->saved_data["with_stats"].toBool(),
                "co_alibi::fwd ran with with_stats=False (inference) and has no backward");
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4],
                 &stats = saved[5], &slopes = saved[6];
    const bool causal = ctx->saved_data["causal"].toBool();
    const double sm_scale = ctx->saved_data["sm_scale"].toDouble();
    const bool need_q = ctx->needs_input_grad(0), need_k = ctx->needs_input_grad(1), need_v = ctx->needs_input_grad(2);
    Tensor dq, dk, dv;
    const Tensor& dout = grads[0];
    if (dout.defined()) {
      if (!need_k && !need_v) {
        static const auto op_dq =
            c10::Dispatcher::singleton().findSchemaOrThrow("co_alibi::bwd_dq", "").typed<decltype(bwd_dq_hip)>();
        if (need_q) dq = op_dq.call(dout, q, k, v, o, lse, stats, slopes, causal, sm_scale);
      } else {
        static const auto op =
            c10::Dispatcher::singleton().findSchemaOrThrow("co_alibi::bwd", "").typed<decltype(bwd_hip)>();
        std::tie(dq, dk, dv) = op.call(dout, q, k, v, o, lse, stats, slopes, causal, sm_scale);
        if (!need_q) dq = Tensor();
        if (!need_k) dk = Tensor();
        if (!need_v) dv = Tensor();
      }
    }
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor, Tensor> fwd_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes,
                                                bool causal, double sm_scale, bool with_stats) {
  const auto r = FwdFunction::apply(q, k, v, slopes, causal, sm_scale, with_stats);
  return {r[0], r[1], r[2]};
}

// The packed form: as FwdFunction, with one saved tensor and one gradient for q, k and v.
class FwdQkvFunction : public torch::autograd::Function<FwdQkvFunction> {
 public:
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& qkv,
                                                const Tensor& slopes, bool causal, double sm_scale, bool with_stats) {
    static const auto op =
        c10::Dispatcher::singleton().findSchemaOrThrow("co_alibi::fwd_qkv", "").typed<decltype(fwd_qkv_hip)>();
    Tensor o, lse, stats;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(o, lse, stats) = op.call(qkv, slopes, causal, sm_scale, with_stats);
    }
    ctx->save_for_backward({qkv, o, lse, stats, slopes});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["sm_scale"] = sm_scale;
    ctx->saved_data["with_stats"] = with_stats;
    ctx->mark_non_differentiable({lse, stats});
    ctx->set_materialize_grads(false);
    return {o, lse, stats};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    TORCH_CHECK(ctx->saved_data["with_stats"].toBool(),
                "co_alibi::fwd_qkv ran with with_stats=False (inference) and has no backward");
    const auto saved = ctx->get_saved_variables();
    Tensor dqkv;
    if (grads[0].defined() && ctx->needs_input_grad(0)) {
      static const auto op =
          c10::Dispatcher::singleton().findSchemaOrThrow("co_alibi::bwd_qkv", "").typed<decltype(bwd_qkv_hip)>();
      dqkv = op.call(grads[0], saved[0], saved[1], saved[2], saved[3], saved[4], ctx->saved_data["causal"].toBool(),
                     ctx->saved_data["sm_scale"].toDouble());
    }
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor, Tensor> fwd_qkv_autograd(const Tensor& qkv, const Tensor& slopes, bool causal,
                                                    double sm_scale, bool with_stats) {
  const auto r = FwdQkvFunction::apply(qkv, slopes, causal, sm_scale, with_stats);
  return {r[0], r[1], r[2]};
}

}  // namespace

TORCH_LIBRARY(co_alibi, m) {
  m.def("fwd(Tensor q, Tensor k, Tensor v, Tensor slopes, bool causal, float sm_scale, bool with_stats) -> "
        "(Tensor, Tensor, Tensor)");
  m.def("bwd(Tensor do, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor stats, Tensor slopes, "
        "bool causal, float sm_scale) -> (Tensor, Tensor, Tensor)");
  m.def("bwd_dq(Tensor do, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor stats, Tensor slopes, "
        "bool causal, float sm_scale) -> Tensor");
  m.def("fwd_qkv(Tensor qkv, Tensor slopes, bool causal, float sm_scale, bool with_stats) -> "
        "(Tensor, Tensor, Tensor)");
  m.def("bwd_qkv(Tensor do, Tensor qkv, Tensor o, Tensor lse, Tensor stats, Tensor slopes, bool causal, "
        "float sm_scale) -> Tensor");
  m.def("decode(Tensor q, Tensor k_cache, Tensor v_cache, Tensor slopes, Tensor? seq_lens, SymInt max_seq_len, "
        "float sm_scale, bool with_lse) -> (Tensor, Tensor)");
}

TORCH_LIBRARY_IMPL(co_alibi, CUDA, m) {
  m.impl("fwd", &fwd_hip);
  m.impl("bwd", &bwd_hip);
  m.impl("bwd_dq", &bwd_dq_hip);
  m.impl("fwd_qkv", &fwd_qkv_hip);
  m.impl("bwd_qkv", &bwd_qkv_hip);
  m.impl("decode", &decode_hip);
}

TORCH_LIBRARY_IMPL(co_alibi, Autograd, m) {
  m.impl("fwd", &fwd_autograd);
  m.impl("fwd_qkv", &fwd_qkv_autograd);
}
