"""Decode step (co_alibi_decode) vs the CPU oracle and vs the native forward.  Needs an MI355X.

A decode step is the reference forward with causal=False and Sq = 1 over the
cache's first seq_len rows (co_alibi_attn.py:137-148; its top-left causal mask
would show an Sq = 1 query only key 0).  Bar: max-abs <= 1e-4 (fp32) or 2e-2
(fp16 / bf16) on O, the same on the natural-log LSE, against the oracle in fp32
on the same dtype-rounded inputs and slopes.
"""
import math

import pytest
import torch

from co_alibi_attn import _native, co_alibi_attention, co_alibi_decode
from co_alibi_attn.co_alibi_attn import _device_slopes
from oracle import co_alibi_ref as ref

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = {torch.float32: 1e-4, torch.float16: 2e-2, torch.bfloat16: 2e-2}
DTYPES = (torch.float32, torch.float16, torch.bfloat16)


def cache_inputs(B, Hq, Hkv, L, cap, D, dtype, seed=0, scale=0.5):
    """q (B,Hq,1,D) and caches (B,Hkv,cap,D); rows >= L hold large garbage that must not leak in."""
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(B, Hq, 1, D, generator=g) * scale).to(dtype)
    k = (torch.randn(B, Hkv, cap, D, generator=g) * scale).to(dtype)
    v = (torch.randn(B, Hkv, cap, D, generator=g) * scale).to(dtype)
    k[:, :, L:] = 100.0
    v[:, :, L:] = -1000.0
    return q, k, v


def oracle_decode(q, k, v, L, sm_scale=None, bias_max=8.0):
    lam = ref.slopes(q.shape[1], bias_max, dtype=q.dtype).float()
    scale = 1.0 / math.sqrt(q.shape[-1]) if sm_scale is None else sm_scale
    o, lse = ref.forward(q.float(), k[:, :, :L].float(), v[:, :, :L].float(), lam, causal=False, scale=scale)
    return o, lse


def check(label, got, want, tol):
    assert torch.isfinite(got).all(), f"{label}: non-finite values"
    err = (got.float().cpu() - want.float()).abs().max().item()
    print(f"  {label}: max-abs {err:.3e} (tol {tol:g})", flush=True)
    assert err <= tol, f"{label}: max-abs {err:.3e} > {tol:g}"


# (B, Hq, Hkv, seq_len, capacity, D)
CASES = [
    (1, 4, 4, 1, 1, 64),            # one key: O = v_0
    (2, 8, 2, 300, 512, 128),       # group of 4, capacity > seq_len, last 128-key chunk 44 keys
    (1, 6, 2, 1000, 1000, 32),      # group of 3 (not a power of two)
    (1, 32, 1, 700, 768, 64),       # group of 32 (every MFMA column)
    (2, 16, 16, 257, 300, 128),     # no grouping, one key past a chunk
    (1, 32, 8, 4113, 4113, 128),    # Llama-style 4:1 grouping, ragged tail
    (2, 8, 2, 700, 1024, 16),       # head dim 16 (the operator pads the heads to 32)
]
# Head dim 256 (fp16 / bf16 only).
CASES_D256 = [
    (2, 8, 2, 1300, 1536, 256),
]


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16), ids=("float16", "bfloat16"))
@pytest.mark.parametrize("case", CASES_D256, ids=lambda c: "B{}_Hq{}_Hkv{}_L{}_cap{}_D{}".format(*c))
def test_decode_head_dim_256(case, dtype):
    B, Hq, Hkv, L, cap, D = case
    q, k, v = cache_inputs(B, Hq, Hkv, L, cap, D, dtype, seed=L)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=L, return_lse=True)
    torch.cuda.synchronize()
    ro, rlse = oracle_decode(q, k, v, L)
    check("o", o, ro, TOL[dtype])
    check("lse", lse, rlse, TOL[dtype])


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}_Hq{}_Hkv{}_L{}_cap{}_D{}".format(*c))
def test_decode_matches_oracle(case, dtype):
    B, Hq, Hkv, L, cap, D = case
    q, k, v = cache_inputs(B, Hq, Hkv, L, cap, D, dtype, seed=L)
    print(f"decode {case} {dtype}", flush=True)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=L, return_lse=True)
    torch.cuda.synchronize()
    ro, rlse = oracle_decode(q, k, v, L)
    check("o", o, ro, TOL[dtype])
    check("lse", lse, rlse, TOL[dtype])
    if L == 1:  # a single visible key: the softmax weight is exactly 1
        check("o == v_0", o, v[:, :, :1].float().repeat_interleave(Hq // Hkv, dim=1), TOL[dtype])


def test_decode_long_cache_merges_many_chunks():
    """70000 keys = 547 chunks of 128 in 183 splits of 3 chunks (on 256 CUs): every split walks several
    chunks, carrying sigma across them, and the last one is partial."""
    B, Hq, Hkv, L, D = 1, 8, 2, 70000, 128
    q, k, v = cache_inputs(B, Hq, Hkv, L, L, D, torch.float16, seed=7)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True)
    torch.cuda.synchronize()
    ro, rlse = oracle_decode(q, k, v, L)
    check("o", o, ro, TOL[torch.float16])
    check("lse", lse, rlse, TOL[torch.float16])


def test_decode_maximum_length():
    """seq_len = 2^21, the largest accepted: 16384 chunks in 512 splits (on 256 CUs), so the merge's
    suffix scan of the split sigma totals crosses its 256-split step."""
    B, Hq, Hkv, L, D = 1, 2, 1, 1 << 21, 64
    q, k, v = cache_inputs(B, Hq, Hkv, L, L, D, torch.bfloat16, seed=11)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True)
    torch.cuda.synchronize()
    ro, rlse = oracle_decode(q, k, v, L)
    check("o", o, ro, TOL[torch.bfloat16])
    check("lse", lse, rlse, TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_decode_equals_forward_non_causal(dtype):
    """Same inputs through co_alibi_attention(causal=False) with Sq = 1 (the native forward kernel)."""
    B, Hq, Hkv, L, D = 2, 12, 4, 1500, 64
    q, k, v = cache_inputs(B, Hq, Hkv, L, L, D, dtype, seed=3)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    with torch.no_grad():
        want = co_alibi_attention(qd, kd, vd, causal=False)
    got = co_alibi_decode(qd, kd, vd)
    torch.cuda.synchronize()
    check("decode vs forward", got, want.cpu(), TOL[dtype])


def test_decode_after_prefill_is_the_last_causal_row():
    """The last row of a causal prefill over L positions sees all L keys: it is the decode step."""
    B, Hq, Hkv, L, D = 1, 16, 8, 777, 128
    g = torch.Generator().manual_seed(5)
    q = (torch.randn(B, Hq, L, D, generator=g) * 0.5).half().to(DEV)
    k = (torch.randn(B, Hkv, L, D, generator=g) * 0.5).half().to(DEV)
    v = (torch.randn(B, Hkv, L, D, generator=g) * 0.5).half().to(DEV)
    with torch.no_grad():
        prefill = co_alibi_attention(q, k, v, causal=True)
    step = co_alibi_decode(q[:, :, -1:], k, v)
    torch.cuda.synchronize()
    check("decode vs last prefill row", step, prefill[:, :, -1:].cpu(), TOL[torch.float16])


def test_decode_is_deterministic_and_lse_optional():
    B, Hq, Hkv, L, D = 1, 8, 2, 5000, 128
    q, k, v = (t.to(DEV) for t in cache_inputs(B, Hq, Hkv, L, L, D, torch.float16, seed=9))
    a, lse = co_alibi_decode(q, k, v, return_lse=True)
    b = co_alibi_decode(q, k, v)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert lse.shape == (B, Hq, 1) and lse.dtype == torch.float32


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_decode_per_sequence_lengths(dtype):
    """A serving batch: each sequence against its own filled prefix of the cache (lengths 1 .. capacity, and 0)."""
    B, Hq, Hkv, cap, D = 5, 16, 4, 1500, 128
    lens = [700, 1, 1500, 0, 257]
    q, k, v = cache_inputs(B, Hq, Hkv, cap, cap, D, dtype, seed=21)
    for b, n in enumerate(lens):  # rows past each sequence's length hold garbage that must not leak in
        k[b, :, n:] = 100.0
        v[b, :, n:] = -1000.0
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=seq, return_lse=True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.equal(o[b].float().cpu(), torch.zeros(Hq, 1, D)), "empty sequence: O must be 0"
            assert torch.isneginf(lse[b]).all(), "empty sequence: LSE must be -inf"
            continue
        ro, rlse = oracle_decode(q[b:b + 1], k[b:b + 1], v[b:b + 1], n)
        check(f"o[{b}] (len {n})", o[b:b + 1], ro, TOL[dtype])
        check(f"lse[{b}] (len {n})", lse[b:b + 1], rlse, TOL[dtype])


def test_decode_lengths_are_clamped_to_the_bound():
    """Per-sequence lengths past max_seq_len count as max_seq_len (the kernel clamps device data)."""
    B, Hq, Hkv, cap, D = 2, 8, 2, 2048, 64
    q, k, v = (t.to(DEV) for t in cache_inputs(B, Hq, Hkv, cap, cap, D, torch.float16, seed=4))
    seq = torch.tensor([5000, 1000], dtype=torch.int32, device=DEV)
    got = co_alibi_decode(q, k, v, seq_len=seq, max_seq_len=1000)
    want = co_alibi_decode(q, k, v, seq_len=1000)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def _random_decode_cases(n=10, seed=99):
    """Seeded serving batches: 1-4 sequences of random lengths (0 included) over caches of
    random capacity, 1-8 kv heads with 1-8 query heads each, every head dim and dtype."""
    g = torch.Generator().manual_seed(seed)
    pick = lambda seq: seq[int(torch.randint(len(seq), (1,), generator=g))]  # noqa: E731
    cases = []
    for i in range(n):
        D = pick([32, 64, 128, 256])
        dtype = pick([torch.float16, torch.bfloat16] + ([torch.float32] if D != 256 else []))
        Hkv = pick([1, 2, 3, 8])
        grp = pick([1, 2, 4, 5, 8])
        B = pick([1, 2, 3, 4])
        cap = int(torch.randint(1, 5000, (1,), generator=g))
        lens = [int(torch.randint(0, cap + 1, (1,), generator=g)) for _ in range(B)]
        cases.append((B, Hkv * grp, Hkv, cap, D, dtype, tuple(lens), i))
    return cases


@pytest.mark.parametrize("case", _random_decode_cases(),
                         ids=lambda c: "{}-B{}_Hq{}_Hkv{}_cap{}_D{}-{}".format(c[7], *c[:5], str(c[5])[6:]))
def test_decode_random_batches(case):
    B, Hq, Hkv, cap, D, dtype, lens, i = case
    print(f"case {case}", flush=True)
    q, k, v = cache_inputs(B, Hq, Hkv, cap, cap, D, dtype, seed=100 + i)
    for b, n in enumerate(lens):
        k[b, :, n:] = 100.0
        v[b, :, n:] = -1000.0
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=seq, return_lse=True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.equal(o[b].float().cpu(), torch.zeros(Hq, 1, D)), "empty sequence: O must be 0"
            assert torch.isneginf(lse[b]).all(), "empty sequence: LSE must be -inf"
            continue
        ro, rlse = oracle_decode(q[b:b + 1], k[b:b + 1], v[b:b + 1], n)
        check(f"o[{b}] (len {n})", o[b:b + 1], ro, TOL[dtype])
        check(f"lse[{b}] (len {n})", lse[b:b + 1], rlse, TOL[dtype])


# Ragged batches at the edges of the split plan: more sequences than a wavefront's lanes, empty ones
# first and last, one long sequence among empty ones (its splits are capped), lengths around the
# chunk of 128, and batches with a work-group per head (one split, no merge launch).
PLAN_CASES = [
    ("B70", [0] + [130 * i % 1500 for i in range(68)] + [0], 8, 2, 1500, 64),
    ("one_long", [0, 0, 20000, 0, 0], 8, 2, 20000, 64),
    ("chunk_edges", [127, 128, 129, 255, 256, 257, 384, 385], 6, 3, 2000, 32),
    ("all_empty", [0, 0, 0], 4, 4, 1000, 64),
    ("direct", [384, 1, 0, 129, 383], 16, 4, 384, 128),
    ("head_each", [700, 0, 1, 900], 128, 128, 900, 32),
]


@pytest.mark.parametrize("case", PLAN_CASES, ids=lambda c: c[0])
def test_decode_split_plan(case):
    _, lens, Hq, Hkv, cap, D = case
    print(f"case {case[0]}", flush=True)
    q, k, v = cache_inputs(len(lens), Hq, Hkv, cap, cap, D, torch.float16, seed=31)
    for b, n in enumerate(lens):
        k[b, :, n:] = 100.0
        v[b, :, n:] = -1000.0
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=seq, return_lse=True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        if n == 0:
            assert not o[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rlse = oracle_decode(q[b:b + 1], k[b:b + 1], v[b:b + 1], n)
        check(f"o[{b}] (len {n})", o[b:b + 1], ro, TOL[torch.float16])
        check(f"lse[{b}] (len {n})", lse[b:b + 1], rlse, TOL[torch.float16])


@pytest.mark.parametrize("L", [384, 385, 1100, 8200])
def test_decode_equal_lengths_split_alike(L):
    """A batch of equal lengths gives the same bits with and without a length tensor."""
    q, k, v = (t.to(DEV) for t in cache_inputs(3, 8, 2, L, L, 64, torch.bfloat16, seed=7))
    seq = torch.full((3,), L, dtype=torch.int64, device=DEV)
    assert torch.equal(co_alibi_decode(q, k, v, seq_len=seq), co_alibi_decode(q, k, v))


# (lens, Hq, Hkv, bound, D, dtype, plan): lengths far below the bound, splits sized by the bound (those past a
# length hold no key) and by the lengths.
BOUND_CASES = [
    ([0, 1, 128, 129, 1000, 4000], 8, 2, 4000, 128, torch.bfloat16, False),
    ([130, 0, 900], 6, 3, 900, 256, torch.float16, False),
    ([500, 0, 20, 4000], 16, 16, 4000, 64, torch.float32, True),
    ([2600, 100, 0] * 6, 8, 8, 2600, 64, torch.float16, True),
]


@pytest.mark.parametrize("case", BOUND_CASES, ids=lambda c: "D{}-{}-{}".format(c[4], str(c[5])[6:], c[6]))
def test_decode_bound_and_plan(case):
    lens, Hq, Hkv, L, D, dtype, plan = case
    print(f"case {case}", flush=True)
    code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
    n = _native.lib().co_alibi_decode_splits(code, len(lens), Hkv, L, D, 1)
    assert n < -1 if plan else n > 1
    q, k, v = cache_inputs(len(lens), Hq, Hkv, L, L, D, dtype, seed=41)
    for b, m in enumerate(lens):
        k[b, :, m:] = 100.0
        v[b, :, m:] = -1000.0
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=seq, return_lse=True)
    torch.cuda.synchronize()
    for b, m in enumerate(lens[:6]):
        if m == 0:
            assert not o[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rlse = oracle_decode(q[b:b + 1], k[b:b + 1], v[b:b + 1], m)
        check(f"o[{b}] (len {m})", o[b:b + 1], ro, TOL[dtype])
        check(f"lse[{b}] (len {m})", lse[b:b + 1], rlse, TOL[dtype])


def test_decode_noalloc_plan_past_the_scratch():
    """A plan whose longest sequences may take four times the even split count (16 of 4096 heads at
    D 128: 34.3 MB of partials) does not fit the 32 MiB scratch of co_alibi_decode_noalloc and takes half
    as many."""
    B, Hq, Hkv, L, D, dtype = 16, 256, 8, 2560, 128, torch.bfloat16
    lib = _native.lib()
    assert lib.co_alibi_decode_splits(2, B, Hkv, L, D, 1) == -4
    lens = [L, 300] + [L - 150 * b for b in range(B - 2)]
    q, k, v = (t.to(DEV) for t in cache_inputs(B, Hq, Hkv, L, L, D, dtype, seed=43))
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    slopes = _device_slopes(Hq, 8.0, dtype, DEV)
    o = torch.full((B, Hq, D), float("nan"), dtype=dtype, device=DEV)
    print("noalloc", flush=True)
    rc = lib.co_alibi_decode_noalloc(2, q.data_ptr(), k.data_ptr(), v.data_ptr(), slopes.data_ptr(), seq.data_ptr(),
                                     o.data_ptr(), 0, B, Hq, Hkv, L, L, D, 1 / math.sqrt(D),
                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.co_alibi_last_error()
    whole = co_alibi_decode(q, k, v, seq_len=seq)
    torch.cuda.synchronize()
    check("all heads vs the allocating call", o, whole[:, :, 0].cpu(), TOL[dtype])
    lam = slopes[:32].cpu()
    for b in (0, 1, 15):
        ro, _ = ref.forward(q[b:b + 1, :32].float().cpu(), k[b:b + 1, :1, :lens[b]].float().cpu(),
                            v[b:b + 1, :1, :lens[b]].float().cpu(), lam, causal=False, scale=1 / math.sqrt(D))
        check(f"o[{b}]", o[b:b + 1, :32].unsqueeze(2), ro, TOL[dtype])


# The split plan's edges at bounds where it decides (asserted): as PLAN_CASES, (name, lens, Hq, Hkv, cap, D).
LONG_PLAN_CASES = [
    ("B70", [0] + [170 * i % 2500 for i in range(68)] + [0], 8, 2, 2500, 64),
    ("one_long", [0, 0, 34000, 0, 0], 8, 2, 34000, 64),
    ("chunk_edges", [127, 128, 129, 255, 256, 257, 384, 385], 6, 3, 26000, 32),
    ("all_empty", [0, 0, 0], 4, 4, 28000, 64),
    ("equal", [2304, 2304, 2304], 128, 64, 2304, 64),
    ("past_the_bound", [5000, 2560, 1, -3], 256, 64, 2560, 32),
]


@pytest.mark.parametrize("case", LONG_PLAN_CASES, ids=lambda c: c[0])
def test_decode_length_plan(case):
    name, lens, Hq, Hkv, cap, D = case
    assert _native.lib().co_alibi_decode_splits(1, len(lens), Hkv, cap, D, 1) < -1
    print(f"case {name}", flush=True)
    q, k, v = cache_inputs(len(lens), Hq, Hkv, cap, cap, D, torch.float16, seed=37)
    held = [min(max(n, 0), cap) for n in lens]
    for b, n in enumerate(held):
        k[b, :, n:] = 100.0
        v[b, :, n:] = -1000.0
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = co_alibi_decode(q.to(DEV), k.to(DEV), v.to(DEV), seq_len=seq, return_lse=True)
    torch.cuda.synchronize()
    for b, n in enumerate(held):
        if n == 0:
            assert not o[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rlse = oracle_decode(q[b:b + 1], k[b:b + 1], v[b:b + 1], n)
        check(f"o[{b}] (len {n})", o[b:b + 1], ro, TOL[torch.float16])
        check(f"lse[{b}] (len {n})", lse[b:b + 1], rlse, TOL[torch.float16])
