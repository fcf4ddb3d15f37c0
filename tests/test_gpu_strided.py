"""Operands in other layouts: the forward and the score-store backward read and write (B, S, H, D)
memory and parts of a packed QKV tensor in place.  Every result must equal that on contiguous
copies bit for bit, at ragged sizes and tile edges, in the small-grid and the whole-block forms;
layouts the kernels do not take are copied by the operators and refused by the C ABI.  Needs an
MI355X.
"""
import ctypes
import math

import pytest
import torch

from co_alibi_attn import _native, co_alibi_attention, ops
from co_alibi_attn.co_alibi_attn import _device_slopes, co_alibi_attention_qkv

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# (B, S, H, D, dtype, causal)
QKV_CASES = [
    (2, 129, 3, 64, torch.bfloat16, True),
    (1, 33, 2, 128, torch.float16, False),
    (1, 1, 2, 64, torch.float16, True),
    (3, 700, 40, 64, torch.float16, True),   # whole-block forms
    (2, 300, 64, 128, torch.bfloat16, True),
    (2, 200, 4, 32, torch.float16, True),    # no score store: the backward copies
    (1, 200, 4, 64, torch.float32, False),
    (1, 150, 2, 256, torch.bfloat16, True),
]


@pytest.mark.parametrize("case", QKV_CASES, ids=lambda c: "B{}S{}H{}D{}-{}-{}".format(*c[:4], str(c[4])[6:], c[5]))
def test_packed_qkv_equals_contiguous(case):
    B, S, H, D, dtype, causal = case
    print(f"case {case}", flush=True)
    g = torch.Generator().manual_seed(11)
    qkv = (torch.randn(B, S, 3, H, D, generator=g) * 0.5).to(dtype).to(DEV).requires_grad_()
    do = torch.randn(B, S, H, D, generator=g).to(dtype).to(DEV)
    o = co_alibi_attention_qkv(qkv, causal=causal)
    (dqkv,) = torch.autograd.grad(o, qkv, do)
    parts = [qkv.detach()[:, :, i].transpose(1, 2).contiguous().requires_grad_() for i in range(3)]
    want = co_alibi_attention(*parts, causal=causal)
    grads = torch.autograd.grad(want, parts, do.transpose(1, 2).contiguous())
    torch.cuda.synchronize()
    assert o.shape == (B, S, H, D) and o.is_contiguous()
    assert torch.equal(o, want.transpose(1, 2))
    for i in range(3):
        assert torch.equal(dqkv[:, :, i], grads[i].transpose(1, 2)), "qkv"[i]
    with torch.no_grad():
        assert torch.equal(co_alibi_attention_qkv(qkv, causal=causal), o)


@pytest.mark.parametrize("case", [(1, 3, 4200, 256, torch.bfloat16), (2, 2, 2800, 128, torch.float16)],
                         ids=["output", "gradient"])
def test_packed_rows_past_the_stride_limit(case):
    """Packed rows of more elements than the kernels' largest row stride (2^20): the output's (4200 heads of
    256) or only the gradient's (2800 of 128) are then written through a copy."""
    B, S, H, D, dtype = case
    assert 3 * H * D > 1 << 20
    test_packed_qkv_equals_contiguous((B, S, H, D, dtype, True))


def layouts(x):
    """The values of contiguous (B, H, S, D) x in layouts that are read in place, then in ones that are copied."""
    B, H, S, D = x.shape
    bshd = x.transpose(1, 2).contiguous().transpose(1, 2)
    wide = torch.empty(B, S, H, D + 16, dtype=x.dtype, device=x.device)[..., :D].transpose(1, 2)
    wide.copy_(x)
    odd = torch.empty(B, H, S, D + 1, dtype=x.dtype, device=x.device)[..., :D]  # rows not 16-byte aligned
    odd.copy_(x)
    shifted = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view_as(x)  # base not aligned
    shifted.copy_(x)
    cols = x.transpose(2, 3).contiguous().transpose(2, 3)  # elements of a row apart
    return [bshd, wide, odd, shifted, cols]


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16), (64, torch.float32)],
                         ids=["d64", "d128", "fp32"])
def test_operator_layouts(D, dtype):
    """Each operand in turn in another layout: the operators' results do not change by a bit."""
    B, Hq, Hkv, Sq, Skv = 2, 4, 2, 161, 200
    g = torch.Generator().manual_seed(2)
    mk = lambda h, s: (torch.randn(B, h, s, D, generator=g) * 0.5).to(dtype).to(DEV)  # noqa: E731
    q, k, v, do = mk(Hq, Sq), mk(Hkv, Skv), mk(Hkv, Skv), mk(Hq, Sq)
    sl = _device_slopes(Hq, 8.0, dtype, DEV)
    args = (sl, True, D ** -0.5)
    o, lse, stats = ops.fwd(q, k, v, *args, True)
    want = ops.bwd(do, q, k, v, o, lse, stats, *args)
    for n, i in ((n, i) for n in range(5) for i in range(5)):
        t = [q, k, v, do, o]
        t[i] = layouts(t[i])[n]
        if i < 3:
            got_o, got_lse, _ = ops.fwd(*t[:3], *args, True)
            assert torch.equal(got_o, o) and torch.equal(got_lse, lse) and got_o.is_contiguous(), (n, i)
            assert torch.equal(ops.fwd(*t[:3], *args, False)[0], o), (n, i)
        got = ops.bwd(t[3], *t[:3], t[4], lse, stats, *args)
        assert all(torch.equal(a, b) and a.is_contiguous() for a, b in zip(got, want)), (n, i)
    # an expanded key head (stride 0 over heads)
    k1, v1 = k[:, :1].expand(B, Hkv, Skv, D), v[:, :1].expand(B, Hkv, Skv, D)
    assert torch.equal(ops.fwd(q, k1, v1, *args, False)[0],
                       ops.fwd(q, k1.contiguous(), v1.contiguous(), *args, False)[0])
    torch.cuda.synchronize()


def test_c_abi_refuses_bad_strides():
    lib = _native.lib()
    q = torch.zeros(1, 2, 64, 64, dtype=torch.float16, device=DEV)
    ws = torch.zeros(1 << 16, dtype=torch.uint8, device=DEV)
    sl = torch.ones(2, device=DEV)
    good = [8192, 4096, 64]

    def call(strides):
        arr = (ctypes.c_longlong * 12)(*strides)
        return lib.co_alibi_fwd_strided(1, q.data_ptr(), q.data_ptr(), q.data_ptr(), sl.data_ptr(), ws.data_ptr(), arr,
                                        0, 0, ws.data_ptr(), 1, 1, 2, 2, 64, 64, 64, 1, 1 / math.sqrt(64), 0)

    for bad, msg in (([8192, 4096, 60], b"16-byte"), ([8192, 4096, 56], b"row stride"), ([8192, -8, 64], b">= 0"),
                     ([8192, 4096, (1 << 20) + 8], b"row stride"), ([8192, 4096, 72], b"same row stride")):
        strides = good + bad + good + good if b"same" in msg else bad + good * 3
        # refused before anything is launched (the workspace of 1 byte is refused first, so give a whole one)
        arr = (ctypes.c_longlong * 12)(*strides)
        rc = lib.co_alibi_fwd_strided(1, q.data_ptr(), q.data_ptr(), q.data_ptr(), sl.data_ptr(), ws.data_ptr(), arr,
                                      0, 0, ws.data_ptr(), ws.numel(), 1, 2, 2, 64, 64, 64, 1, 0.125, 0)
        assert rc == 1 and msg in lib.co_alibi_last_error(), (bad, lib.co_alibi_last_error())
    assert call(good * 4) == 1 and b"workspace" in lib.co_alibi_last_error()


def test_opcheck_packed():
    """Shape functions and autograd registration of the packed operators."""
    g = torch.Generator().manual_seed(4)
    qkv = (torch.randn(1, 70, 3, 2, 64, generator=g) * 0.5).half().to(DEV).requires_grad_()
    sl = _device_slopes(2, 8.0, torch.float16, DEV)
    torch.library.opcheck(torch.ops.co_alibi.fwd_qkv.default, (qkv, sl, True, 0.125, True))
    with torch.no_grad():
        o, lse, stats = ops.fwd_qkv(qkv, sl, True, 0.125, True)
        torch.library.opcheck(torch.ops.co_alibi.bwd_qkv.default, (o, qkv.detach(), o, lse, stats, sl, True, 0.125))
