"""Head-dim 256 forward with the keys of a query tile shared by two groups of waves.

Taken up to 256 query tiles (128 queries of one head each) from 257 reachable
keys on.  Cases: an odd and an even number of 32-key tiles, a last tile of one
key, tiles whose rows reach one key tile only (the second group has none), the
last problem below and the first above each line of the rule, several packed
sequences, a query tile of one row, small windows, vision blocks across the
groups, and document IDs.  Each against the fp64 oracle, outputs NaN before the
call, and bitwise repeatable.
"""

import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (hq, hkv, lq, lk, packed, window, vision, documents)
    (32, 16, [257], [257], False, 1024, False, False),
    (32, 16, [256], [256], False, 1024, False, False),  # the old path
    (16, 8, [1], [289], False, 1024, False, False),
    (16, 8, [129], [1153], True, 1024, False, False),
    (32, 16, [1000], [1000], False, 1024, False, False),
    (32, 16, [1025], [1025], False, 1024, False, False),  # the old path: 288 tiles
    (8, 4, [500], [2050], True, None, False, False),
    (4, 4, [300, 33, 700], [300, 500, 700], True, 200, False, False),
    (16, 8, [777], [777], False, 1024, True, False),
    (8, 4, [300, 600], [300, 900], True, 300, True, False),
    (8, 4, [700], [700], False, 1024, False, True),
]


@pytest.mark.parametrize("hq,hkv,lq,lk,packed,window,vision,documents", CASES)
def test_key_groups_match_the_oracle(hq, hkv, lq, lk, packed, window, vision, documents):
    from gemma4_fa4_amd import ops

    label = f"key groups hq={hq} hkv={hkv} lq={lq} lk={lk} window={window} vision={vision}"
    print(label, flush=True)
    q, k, v, _do, _dl = qkv(4410 + sum(lk), sum(lq), sum(lk), hq, hkv, 256)
    cq, ck = cu(lq), cu(lk)
    vid = doc = None
    pos = torch.arange(k.shape[0])
    if vision:  # blocks of 150 keys, 50 keys of text between them
        vid = torch.where(pos % 200 < 150, pos // 200, -1).to(torch.int32)
    if documents:
        doc = (pos // 333).to(torch.int32)
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq, num_kv_heads=hkv,
        head_dim=256, window=window, cu_q=cq.to(DEV) if packed else None,
        cu_k=ck.to(DEV) if packed else None, total_q=q.shape[0], total_k=k.shape[0],
        vision=vid.to(DEV) if vision else None, documents=doc.to(DEV) if documents else None)
    args = [t.to(DEV) for t in (q, k, v)]
    if not packed:
        args = [t.view(len(lq), t.shape[0] // len(lq), *t.shape[1:]) for t in args]
    st = ops.Stages(plan, *args, args[0], forward_only=True)
    runs = []
    for _ in range(2):
        for t in (st.o, st.lse):
            t.view(torch.uint8).fill_(0xFF)
        st.forward()
        runs.append((st.o.clone(), st.lse.clone()))
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])
    o = runs[0][0].cpu().reshape(-1, hq, 256)
    lse = runs[0][1].cpu()
    if not packed:
        lse = lse.permute(1, 0, 2).reshape(hq, -1)
    o_ref, l_ref, *_ = attention_fwd_bwd(
        q.to(DEV), k.to(DEV), v.to(DEV), cq.tolist(), ck.tolist(), sliding_window=window,
        vision_block_ids=vid.to(DEV) if vision else None,
        document_ids=doc.to(DEV) if documents else None, allow_vision_bidirectional=vision,
        compute_dtype=torch.float64)
    check_forward(o, lse, o_ref.cpu(), l_ref.cpu(), local=True, label=label)
