"""Which kernel forms the host's rules choose, at shapes on both sides of their lines (measured at
256 CUs, the figures stand beside the rules).  The rules are host code: no GPU is needed."""
import pytest

from co_alibi_attn import _native

F32, F16, BF16 = 0, 1, 2


# (dtype, batch, heads_kv, seq_kv, head_dim, lengths per sequence, splits; negative: the lengths decide)
DECODE = [
    # short caches: one split, where the type's chunk walk is cheaper than a merge launch
    (F16, 1, 8, 300, 32, False, 1),
    (BF16, 1, 8, 200, 128, False, 1),
    (BF16, 1, 8, 300, 128, False, 3),
    (BF16, 1, 8, 300, 128, True, 1),
    (BF16, 1, 8, 300, 256, False, 3),
    (F32, 1, 8, 300, 64, False, 3),
    (F32, 1, 8, 200, 64, True, 2),
    (BF16, 10, 10, 300, 256, False, 1),  # more work-groups than half the slots
    (BF16, 16, 8, 300, 256, True, 3),
    # short walks with lengths: the plan would cost more than it shares out
    (BF16, 1, 8, 500, 128, True, 4),
    (BF16, 1, 8, 4000, 128, True, 32),
    (BF16, 8, 8, 1000, 128, True, 8),
    (BF16, 16, 8, 1000, 128, True, 4),
    (F16, 16, 8, 1000, 64, True, 4),
    (F16, 8, 8, 4000, 32, True, 8),
    (F32, 32, 8, 700, 64, True, 2),
    # long ones: it pays
    (BF16, 16, 8, 8192, 128, True, -4),
    (F16, 16, 8, 8192, 64, True, -4),
    (F16, 32, 8, 4000, 32, True, -2),
    (F32, 16, 8, 4000, 64, True, -4),
    # between half the slots and all of them: two splits unless the walk is short
    (BF16, 12, 24, 700, 128, False, 1),
    (BF16, 12, 24, 1000, 128, False, 2),
    (F32, 12, 24, 500, 64, False, 2),
    (BF16, 12, 24, 1000, 256, False, 2),
    (F16, 44, 8, 12780, 64, False, 2),
    (BF16, 48, 8, 4076, 128, False, 2),
    (BF16, 48, 8, 1000, 128, True, 1),
    (BF16, 54, 8, 4000, 128, False, 1),
    (F16, 63, 8, 16000, 32, False, 2),
    (BF16, 64, 8, 100000, 128, True, 1),
    # one sequence: a split per slot, or a chunk per split
    (BF16, 1, 8, 8192, 128, False, 64),
    (F16, 10, 10, 700, 32, False, 6),
    (F16, 11, 10, 4076, 64, False, 4),
    (F16, 21, 10, 16000, 32, False, 3),
    (BF16, 18, 10, 16000, 128, False, 2),
    (F32, 10, 10, 300, 64, False, 3),
    (F32, 18, 10, 300, 64, False, 1),
]


@pytest.mark.parametrize("case", DECODE, ids=str)
def test_decode_splits(case):
    assert _native.lib().co_alibi_decode_splits(*case[:5], int(case[5])) == case[6]


def test_decode_splits_bounds():
    """Every split holds a chunk, at most 1024 of them, for any batch and length; what the scratch of
    co_alibi_decode_noalloc has to hold (the splits of all units) stays under a round and a rest."""
    lib = _native.lib()
    for dtype, D in ((F32, 64), (F16, 32), (F16, 64), (BF16, 128), (BF16, 256)):
        for units in (1, 2, 7, 36, 100, 128, 210, 256, 257, 384, 426, 427, 448, 511, 512, 513, 4096):
            for chunks in (1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 100, 1024, 1025, 16384):
                for ragged in (0, 1):
                    n = lib.co_alibi_decode_splits(dtype, units, 1, chunks * 128, D, ragged)
                    assert 1 <= abs(n) <= min(chunks, 1024), (dtype, D, units, chunks, ragged, n)
                    assert n > 0 or ragged
                    assert abs(n) * units < 512 + units, (dtype, D, units, chunks, ragged, n)
    assert lib.co_alibi_decode_splits(F16, 0, 1, 128, 64, 0) == 0
    assert lib.co_alibi_decode_splits(F16, 1, 1, (1 << 21) + 1, 64, 0) == 0


SPLIT, LONG, DQ, KEYS = 1, 2, 4, 8


def _forms(dtype, H, n, m, D, causal, B=1, group=1):
    return _native.lib().co_alibi_attention_forms(dtype, B, H * group, H, n, m, D, int(causal))


# (dtype, heads, seq_q, seq_kv, head_dim, causal, forms with the tail skip, forward's without it)
ATTENTION = [
    # the longest walk is one tile: nothing to split
    (F16, 128, 64, 64, 64, True, 0, 0),
    (F16, 2, 33, 31, 64, True, 0, 0),
    (F16, 16, 1024, 64, 128, False, 0, 0),
    (F32, 64, 64, 64, 64, True, SPLIT | DQ | KEYS, SPLIT),
    (F32, 128, 64, 64, 64, True, KEYS, 0),
    (F32, 64, 32, 32, 64, True, SPLIT | KEYS, SPLIT),
    (BF16, 64, 64, 64, 256, True, SPLIT, SPLIT),
    # short walks
    (F16, 128, 128, 128, 128, True, SPLIT, SPLIT),
    (F16, 64, 128, 128, 128, True, SPLIT | DQ, SPLIT),
    (F16, 128, 128, 128, 64, True, SPLIT | DQ, SPLIT),
    (F16, 128, 96, 96, 64, True, SPLIT, SPLIT),
    (F16, 128, 128, 128, 256, True, 0, 0),
    (F16, 64, 128, 128, 256, True, SPLIT | DQ, SPLIT),
    (F16, 64, 256, 256, 256, True, SPLIT, SPLIT),
    (F16, 64, 256, 256, 128, True, SPLIT | DQ, SPLIT),
    # one work-group per CU: 16 bits at D 256 and fp32 at D 128
    (F16, 24, 1024, 1024, 256, True, SPLIT, SPLIT),
    (F16, 32, 1024, 1024, 256, True, 0, 0),
    (BF16, 32, 1024, 1024, 256, True, 0, 0),
    (F16, 32, 1536, 1536, 256, True, 0, 0),
    (F16, 24, 1536, 1536, 256, True, SPLIT, 0),
    (F16, 22, 2048, 2048, 256, True, SPLIT, 0),
    (F16, 24, 2048, 2048, 256, True, LONG, 0),
    (F16, 48, 2048, 2048, 256, True, 0, 0),
    (F32, 32, 1024, 1024, 128, True, SPLIT | DQ, SPLIT),
    (F32, 32, 1536, 1536, 128, True, DQ, 0),
    (F32, 24, 2048, 2048, 128, True, LONG | DQ, 0),
    (F32, 32, 2048, 2048, 128, True, 0, 0),
    (F32, 16, 2048, 2048, 128, False, SPLIT, 0),
    (F32, 12, 2048, 2048, 128, False, SPLIT | DQ, SPLIT),
    # two per CU
    (F16, 32, 1024, 1024, 128, True, SPLIT, SPLIT),
    (F16, 24, 2048, 2048, 128, True, SPLIT, 0),
    (F16, 24, 2048, 2048, 64, True, SPLIT | DQ, SPLIT),
    (F16, 16, 2048, 2048, 64, False, SPLIT | DQ, 0),
    (F16, 8, 2048, 2048, 64, False, SPLIT | DQ, SPLIT),
    (F16, 16, 2048, 2048, 128, False, SPLIT, 0),
    (F32, 16, 2048, 2048, 64, False, SPLIT | DQ | KEYS, 0),
    # middle grids
    (F16, 64, 1536, 1536, 128, True, 0, 0),
    (F16, 48, 1536, 1536, 128, True, LONG, 0),
    (F16, 48, 2048, 2048, 64, True, LONG, 0),
    (F32, 48, 1536, 1536, 64, True, KEYS, 0),
    (F32, 32, 2048, 2048, 64, True, LONG | KEYS, 0),
    (F32, 40, 2048, 2048, 64, True, KEYS, 0),
    (F16, 64, 2048, 2048, 128, True, 0, 0),
    (F16, 8, 8192, 8192, 64, True, 0, 0),
    # causal rows see at most seq_q keys, however many there are
    (F16, 32, 1024, 8192, 128, True, SPLIT, SPLIT),
    (F16, 40, 1024, 8192, 128, True, 0, 0),
    # pass 2 of the recompute path
    (F32, 192, 128, 128, 64, True, 0, 0),
    (F32, 128, 256, 256, 64, False, 0, 0),
    (F16, 256, 128, 128, 32, True, 0, 0),
    (F16, 128, 128, 128, 32, True, SPLIT | DQ | KEYS, SPLIT),
    (F16, 128, 512, 512, 32, True, 0, 0),
    (F32, 64, 1024, 1024, 64, True, 0, 0),
    (F32, 48, 1024, 1024, 64, True, KEYS | 16, 0),
    # nothing is split where the tiles do not fit LDS
    (F32, 1, 512, 512, 256, True, 0, 0),
]


@pytest.mark.parametrize("case", ATTENTION, ids=str)
def test_attention_forms(case):
    *shape, want, fwd_full = case
    assert _forms(*shape) & (31 if want & 16 else SPLIT | LONG | DQ | KEYS) == want
    with _native.tail_skip(False):
        assert _forms(*shape) & (SPLIT | LONG) == fwd_full


def test_attention_forms_grouped_heads_and_errors():
    """Query heads count in the row blocks, key heads in pass 2's key blocks and the group in its tiles."""
    assert _forms(BF16, 8, 1741, 1741, 128, True, group=4) == LONG
    assert _forms(F32, 8, 1024, 1024, 64, True, B=4, group=4) & KEYS
    assert not _forms(F32, 32, 1024, 1024, 64, True, B=4) & (SPLIT | LONG | DQ)
    lib = _native.lib()
    assert lib.co_alibi_attention_forms(3, 1, 1, 1, 1, 1, 64, 1) == -1
    assert lib.co_alibi_attention_forms(F16, 1, 3, 2, 1, 1, 64, 1) == -1
    assert lib.co_alibi_attention_forms(F16, 1, 1, 1, 1, 1, 80, 1) == -1


def test_roomy_forward():
    """fp32 at head dim 64: the register budget of one work-group per CU on grids that give a CU one."""
    for H, n, causal, B, want in ((36, 1024, True, 2, 16), (40, 1024, True, 2, 0), (22, 2048, True, 2, 16),
                                  (32, 2048, True, 2, 0), (24, 1024, False, 2, 16), (32, 1024, False, 2, 0),
                                  (48, 512, True, 2, 0), (16, 1024, True, 2, 0)):
        assert _forms(F32, H, n, n, 64, causal, B=B) & 16 == want, (H, n, causal)
        assert not _forms(F16, H, n, n, 64, causal, B=B) & 16 and not _forms(F32, H, n, n, 32, causal, B=B) & 16
        with _native.tail_skip(False):
            assert not _forms(F32, H, n, n, 64, causal, B=B) & 16
