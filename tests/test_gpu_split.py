"""The split form of small grids (a row block's 32-row parts on work-groups of their own, their key
tiles on the work-group's wavefronts) vs the CPU oracle, at the edges of its tiles: rows and keys
around 32, around a step of 128 keys and around the 128-row block, more keys than rows and the
reverse, steep heads (whole-block form beside split ones in one launch) and flat ones, with the
tail skip on and off.  Needs an MI355X.
"""
import math

import pytest
import torch

from co_alibi_attn import _native
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
