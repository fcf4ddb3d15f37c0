"""The split form of small grids (a row block's 32-row parts on work-groups of their own, their key
tiles on the work-group's wavefronts) vs the CPU oracle, at the edges of its tiles: rows and keys
around 32, around a step of 128 keys and around the 128-row block, more keys than rows and the
reverse, steep heads (whole-block form beside split ones in one launch) and flat ones, with the
tail skip on and off.  Which form a case takes is asserted through co_alibi_attention_forms; the split
pass 1 is also held to the whole-block form's bits.  Needs an MI355X.
"""
import math

import pytest
import torch

from co_alibi_attn import _native, ops
from co_alibi_attn.co_alibi_attn import CoALIBIAttention
from oracle import co_alibi_ref as ref
from tests.test_gpu_parity import DEV, TOL, assert_parity, rand_inputs

pytestmark = pytest.mark.gpu

# (B, Hq, Hkv, Sq, Skv, D, causal)
CASES = [
    (1, 2, 1, 31, 33, 64, False),
    (1, 2, 2, 33, 31, 64, True),
    (2, 2, 2, 32, 128, 128, False),
    (1, 4, 2, 129, 129, 128, True),
    (1, 2, 2, 161, 513, 32, False),
    (1, 4, 4, 640, 640, 64, True),
    (1, 2, 2, 385, 257, 16, True),
    (1, 2, 1, 97, 640, 256, False),
    (1, 1, 1, 1, 1, 128, True),
]


@pytest.mark.parametrize("skip", [True, False], ids=["skip", "full"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}/{}S{}x{}D{}{}".format(*c[:6], "c" if c[6] else "n"))
def test_split_edges(case, dtype, skip):
    B, Hq, Hkv, Sq, Skv, D, causal = case
    print(f"case {case} {dtype} skip={skip}", flush=True)
    q, k, v, do = rand_inputs(B, Hq, Hkv, Sq, Skv, D, dtype, seed=3)
    do = do * 0.25  # steep heads gather many rows' dO on few keys: keeps |dV| where the bar is unscaled
    lam = torch.tensor([4.0, 0.0, 0.02, 1.0][:Hq]).to(dtype).float()
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd = (t.to(DEV).requires_grad_() for t in (q, k, v))
    with _native.tail_skip(skip):
        o = CoALIBIAttention.apply(qd, kd, vd, lam.to(DEV), causal, scale)
        o.backward(do.to(DEV))
    torch.cuda.synchronize()
    got = tuple(t.detach().float().cpu() for t in (o, qd.grad, kd.grad, vd.grad))
    qf, kf, vf, dof = (t.float() for t in (q, k, v, do))
    ro, _ = ref.forward(qf, kf, vf, lam, causal=causal, scale=scale)
    want = (ro, *ref.backward(dof, qf, kf, vf, lam, causal=causal, scale=scale))
    assert_parity(got, want, TOL[dtype], f"{case}", dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
def test_key_form_many_query_heads(dtype):
    """Pass 2's 32-key form with more query heads per key head than its LDS bits of processed row
    blocks hold (600 heads, a word each): the bits are read from the forward's record instead."""
    q, k, v, do = rand_inputs(1, 600, 1, 70, 40, 16, dtype, seed=5)
    do = do * 0.05
    lam = torch.linspace(0.001, 2.0, 600).to(dtype).float()
    qd, kd, vd = (t.to(DEV).requires_grad_() for t in (q, k, v))
    o = CoALIBIAttention.apply(qd, kd, vd, lam.to(DEV), True, 0.25)
    o.backward(do.to(DEV))
    torch.cuda.synchronize()
    got = tuple(t.detach().float().cpu() for t in (o, qd.grad, kd.grad, vd.grad))
    qf, kf, vf, dof = (t.float() for t in (q, k, v, do))
    ro, _ = ref.forward(qf, kf, vf, lam, causal=True, scale=0.25)
    want = (ro, *ref.backward(dof, qf, kf, vf, lam, causal=True, scale=0.25))
    assert_parity(got, want, TOL[dtype], "600 heads", dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
def test_longer_half_split(dtype):
    """A grid past the small ones (25 heads x 16 row blocks): the longer half of the flat heads' row
    blocks is split, the rest and the steep heads run whole, in one launch; four heads checked."""
    H, S, D = 25, 1937, 32
    q, k, v, do = rand_inputs(1, H, H, S, S, D, dtype, seed=9)
    do = do * 0.25
    lam = torch.tensor([2.0, 0.05, 0.01, 0.0] + [0.3] * (H - 4)).to(dtype).float()
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd = (t.to(DEV).requires_grad_() for t in (q, k, v))
    o = CoALIBIAttention.apply(qd, kd, vd, lam.to(DEV), True, scale)
    o.backward(do.to(DEV))
    torch.cuda.synchronize()
    got = tuple(t.detach()[:, :4].float().cpu() for t in (o, qd.grad, kd.grad, vd.grad))
    qf, kf, vf, dof = (t[:, :4].float() for t in (q, k, v, do))
    ro, _ = ref.forward(qf, kf, vf, lam[:4], causal=True, scale=scale)
    want = (ro, *ref.backward(dof, qf, kf, vf, lam[:4], causal=True, scale=scale))
    assert_parity(got, want, TOL[dtype], "longer half", dtype)


# More keys than one tile, at the smallest sizes that are split (the forms are asserted): (B, Hq, Hkv, Sq, Skv, D, causal)
SMALLEST = [
    (1, 2, 1, 31, 65, 64, False),
    (1, 2, 2, 66, 97, 64, True),
    (2, 2, 2, 97, 66, 32, True),
    (1, 1, 1, 1, 96, 128, False),
    (1, 4, 2, 70, 129, 128, False),
    (1, 2, 2, 65, 65, 256, True),
]


@pytest.mark.parametrize("skip", [True, False], ids=["skip", "full"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("case", SMALLEST, ids=lambda c: "B{}H{}/{}S{}x{}D{}{}".format(*c[:6], "c" if c[6] else "n"))
def test_smallest_split(case, dtype, skip):
    B, Hq, Hkv, Sq, Skv, D, causal = case
    forms = _native.lib().co_alibi_attention_forms(_native.DTYPE_CODES[dtype], *case[:6], int(causal))
    if D * dtype.itemsize <= 512:
        assert forms & 5 == 5, forms
    test_split_edges(case, dtype, skip)


def test_forms_of_the_cases_above():
    """The edge cases with more than one tile of keys are split in the forward and in pass 1, and the grid of
    test_longer_half_split is a middle one."""
    forms = _native.lib().co_alibi_attention_forms
    for *shape, causal in CASES:
        if min(shape[3], shape[4]) > 64 and not (shape[5] == 256):
            assert forms(1, *shape, int(causal)) & 5 == 5 and forms(0, *shape, int(causal)) & 5 == 5, shape
    for dtype in (0, 1):
        assert forms(dtype, 1, 25, 25, 1937, 1937, 32, 1) & 3 == 2
        assert forms(dtype, 1, 600, 1, 70, 40, 16, 1) & 8


@pytest.mark.parametrize("slope,split", [(1.0, False), (0.02, True)], ids=["steep", "flat"])
def test_forward_record_shows_the_form(slope, split):
    """A split row block records that it processed every key; a steep head's blocks run whole beside it in the
    same launch, stop early and record where."""
    lam = torch.tensor([slope, 0.02])
    q, k, v, _ = (t.to(DEV) for t in rand_inputs(1, 2, 2, 1024, 1024, 64, torch.float16, seed=2))
    assert _native.lib().co_alibi_attention_forms(1, 1, 2, 2, 1024, 1024, 64, 1) & 1
    _, _, stats = ops.fwd(q, k, v, lam.to(DEV), True, 0.125, True)
    kstart = stats.view(torch.int32)[4:4 + 16].view(2, 8).cpu()
    assert not kstart[1].any()
    assert kstart[0].any() != split, kstart


@pytest.mark.parametrize("H,S,causal", [(36, 1000, True), (20, 900, False)], ids=["causal", "full"])
def test_roomy_fp32_forward(H, S, causal):
    """The fp32 forward at head dim 64 under the register budget of one work-group per CU; four heads checked, and
    the backward that follows its record."""
    assert _native.lib().co_alibi_attention_forms(0, 1, H, H, S, S, 64, int(causal)) & 19 == 16
    q, k, v, do = rand_inputs(1, H, H, S, S, 64, torch.float32, seed=17)
    do = do * 0.25
    lam = torch.tensor([2.0, 0.05, 0.01, 0.0] + [0.3] * (H - 4))
    qd, kd, vd = (t.to(DEV).requires_grad_() for t in (q, k, v))
    o = CoALIBIAttention.apply(qd, kd, vd, lam.to(DEV), causal, 0.125)
    o.backward(do.to(DEV))
    torch.cuda.synchronize()
    got = tuple(t.detach()[:, :4].float().cpu() for t in (o, qd.grad, kd.grad, vd.grad))
    ins = [t[:, :4] for t in (q, k, v)]
    ro, _ = ref.forward(*ins, lam[:4], causal=causal, scale=0.125)
    want = (ro, *ref.backward(do[:, :4], *ins, lam[:4], causal=causal, scale=0.125))
    assert_parity(got, want, TOL[torch.float32], "roomy", torch.float32)


# (Hq, S, D, dtype, causal): a batch of 17 of these takes the whole-block pass 1, one of them alone the split form.
PASS1_CASES = [
    (4, 250, 64, torch.float16, True),
    (4, 250, 64, torch.bfloat16, False),
    (4, 250, 128, torch.bfloat16, True),
    (4, 250, 32, torch.float16, True),
    (4, 250, 64, torch.float32, True),
    (4, 250, 64, torch.float32, False),
]


@pytest.mark.parametrize("case", PASS1_CASES, ids=lambda c: "D{}-{}-{}".format(c[2], str(c[3])[6:], "c" if c[4] else "n"))
def test_split_pass1_writes_the_same_bits(case):
    """The workspace of backward pass 1 (dO.O, and the score records or zb and cb) is the same bit for bit from
    the split form (one sequence) and the whole-block form (the same sequence in a batch of 17), from the
    same forward results; dQ is summed in another order."""
    H, S, D, dtype, causal = case
    B = 17
    lib, code = _native.lib(), _native.DTYPE_CODES[dtype]
    assert not lib.co_alibi_attention_forms(code, B, H, H, S, S, D, int(causal)) & 4
    assert lib.co_alibi_attention_forms(code, 1, H, H, S, S, D, int(causal)) & 4
    q, k, v, do = (t.to(DEV) for t in rand_inputs(B, H, H, S, S, D, dtype, seed=13))
    lam = torch.tensor([2.0, 0.3, 0.02, 0.0], device=DEV)
    scale = 1.0 / math.sqrt(D)
    o, lse, stats = ops.fwd(q, k, v, lam, causal, scale, True)
    nqb, nkb = -(-S // 128), -(-S // 64)
    words = lambda b: (4, b * H * nqb, b * H, b * H * nqb, b * H * nkb, b * H * S, b * H * S)  # noqa: E731
    parts = [p.view(n, -1) if i else p for i, (p, n) in enumerate(zip(stats.split(words(B)), (4,) + (B * H,) * 6))]
    alone = torch.cat([torch.zeros(4, device=DEV)] + [p[:H].reshape(-1) for p in parts[1:]])
    assert alone.numel() == lib.co_alibi_stats_numel(1, H, S, S)
    store = dtype != torch.float32 and D in (64, 128)
    nq32 = -(-S // 32)
    out = []
    for b, st in ((B, stats), (1, alone)):
        size = (lib.co_alibi_bwd_score_store_workspace_bytes(code, b, H, H, S, S, D, int(causal)) if store
                else lib.co_alibi_bwd_workspace_bytes(b, H, S, S))
        ws, dq = torch.zeros(size, dtype=torch.uint8, device=DEV), torch.zeros_like(q[:b])
        print(f"case {case} batch {b}", flush=True)
        _native.check(lib.co_alibi_bwd_dq(code, do.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                          lse.data_ptr(), st.data_ptr(), lam.data_ptr(), dq.data_ptr(), ws.data_ptr(),
                                          size, b, H, H, S, S, D, int(causal), scale,
                                          torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        pad = lambda n: -(-n // 256) * 256  # noqa: E731
        dsum = ws[:4 * b * H * S].view(torch.int32).view(b * H, S)[:H]
        rest = ws[pad(4 * b * H * S):]
        if store:
            out.append((dsum, rest.view(b * H, -1)[:H], dq[0]))
            continue
        n = 4 * b * H * nq32 * S  # a row's value for every 32-key block
        zb, cb = (rest[i * pad(n): i * pad(n) + n].view(torch.int32).view(b * H, nq32, S)[:H] for i in (0, 1))
        out.append((dsum, torch.stack((zb, cb)), dq[0]))
    (dsum, rest, dq), (dsum1, rest1, dq1) = out
    assert torch.equal(dsum, dsum1) and rest1.any()
    assert torch.equal(rest, rest1)
    err = (dq - dq1).abs().max().item()
    print(f"dq max-abs {err:.2e}", flush=True)
    assert err <= TOL[dtype] / 10
