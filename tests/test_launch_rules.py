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
