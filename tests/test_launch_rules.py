"""Host rules that choose a launch, read from the workspace sizes they imply (no GPU).

Phase 3 of ``g4_workspace_bytes`` is more than phase 0 exactly when the forward
would split its keys.
"""

import ctypes

import pytest

from gemma4_fa4_amd import _lib


def _bytes(phase, **kw):
    p = _lib.G4Problem(**kw)
    p.total_q = kw.get("total_q", kw["num_seqs"] * kw["seqlen_q"])
    p.total_k = kw.get("total_k", kw["num_seqs"] * kw["seqlen_k"])
    return _lib.load().g4_workspace_bytes(ctypes.byref(p), phase)


def _splits(lq, lk, hq=32, hkv=4):
    kw = dict(num_seqs=1, seqlen_q=lq, seqlen_k=lk, num_q_heads=hq, num_kv_heads=hkv, head_dim=512)
    return _bytes(3, **kw) > _bytes(0, **kw)


@pytest.mark.parametrize("lq,lk,split", [
    # a few new tokens: one 128-row tile per KV head, so from about 300 keys on the split pays
    (5, 105, False), (5, 200, False), (5, 384, True), (16, 512, True), (48, 600, True),
    # a chunk of a prompt after a short and after a long prefix
    (100, 200, False), (300, 1500, True), (500, 12500, True),
    # tiles enough for every CU
    (1024, 1124, False), (2048, 2048, False),
])
def test_wide_forward_splits_where_its_tiles_leave_cus_idle(lq, lk, split):
    assert _splits(lq, lk) is split


def _dkdv_splits(lengths, vision=False):
    total, most = sum(lengths), max(lengths)
    kw = dict(num_seqs=len(lengths), seqlen_q=most, seqlen_k=most, num_q_heads=32, num_kv_heads=16,
              head_dim=256, window=1024, total_q=total, total_k=total, cu_seqlens_q=256,
              cu_seqlens_k=256, bidirectional_vision=int(vision))
    if vision:
        kw["vision_ids"] = 256
    return _bytes(2, **kw) > _bytes(1, **kw)


@pytest.mark.parametrize("lengths,vision,split", [
    # measured whole / split us: alike in average work, unlike in what shares a CU
    ([300] * 8, False, True), ([300] * 12, False, False),        # 80 / 62, 103 / 125
    ([256] * 12, False, False), ([448] * 16, False, True),       # 83 / 97, 265 / 210
    ([777] * 3, False, False), ([1000] * 3, False, True),        # 115 / 134, 225 / 182
    # one long sequence and short ones; lengths that differ
    ([2000, 100, 100, 100], False, False), ([1151, 348], False, True),  # 165 / 180, 140 / 93
    # images lengthen tiles
    ([384] * 8, True, False), ([3000] * 2, True, True),          # 124 / 150, 735 / 585
    ([2000, 100, 100, 100], True, True),                         # 272 / 232
    ([1], False, False), ([1, 1], False, False), ([5] * 64, False, False),
])
def test_dkdv_of_several_sequences_splits_where_its_schedule_is_shorter(lengths, vision, split):
    assert _dkdv_splits(lengths, vision) is split
