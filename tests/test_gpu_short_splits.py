"""Head-dim 512 forward of few new tokens over a few hundred keys: chunks of two key tiles.

Each chunk holds as little as two key tiles (shorter sequences of a packed batch
have chunks with one, or none).  Against the fp64 oracle, with the workspace and
the outputs NaN before the call.
"""

import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (hq, hkv, lq, lk)
    (32, 4, [5], [320]),
    (32, 4, [16], [517]),
    (32, 4, [33], [641]),
    (32, 4, [9, 30, 5], [700, 64, 31]),
    (16, 4, [40, 9], [600, 100]),
    (8, 8, [70], [500]),
]


@pytest.mark.parametrize("hq,hkv,lq,lk", CASES)
def test_short_splits_match_the_oracle(hq, hkv, lq, lk):
    from gemma4_fa4_amd import ops

    label = f"short split hq={hq} hkv={hkv} lq={lq} lk={lk}"
    print(label, flush=True)
    q, k, v, _, _ = qkv(90 + sum(lk), sum(lq), sum(lk), hq, hkv, 512)
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq, num_kv_heads=hkv,
        head_dim=512, window=None, cu_q=cu(lq).to(DEV), cu_k=cu(lk).to(DEV), total_q=sum(lq),
        total_k=sum(lk))
    assert plan.workspace_bytes(3) > plan.workspace_bytes(0), "the problem is not split"
    args = [t.to(DEV) for t in (q, k, v)]
    st = ops.Stages(plan, *args, args[0], forward_only=True)
    st.ws = torch.empty(plan.workspace_bytes(3), dtype=torch.uint8, device=DEV)
    for t in (st.ws, st.o, st.lse):
        t.view(torch.uint8).fill_(0xFF)
    st.forward()
    o_ref, l_ref, *_ = attention_fwd_bwd(*args, cu(lq).tolist(), cu(lk).tolist(),
                                         compute_dtype=torch.float64)
    check_forward(st.o, st.lse, o_ref.cpu(), l_ref.cpu(), local=False, label=label)
