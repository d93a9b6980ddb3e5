"""Decode at head dim 512 with equal parts of every sequence's key tiles.

The parts cut the (sequence, KV head) segments' key tiles laid end to end, so a
part may end one segment, cover short ones whole and begin another.  Cases:
one long cache, ragged batches with one-key and Q-empty sequences, more
sequences than a wave has lanes, more parts than tiles, several queries, GQA
ratios, a window; each with the workspace the forward needs (chunks by the
longest sequence) and with phase 3 of ``g4_workspace_bytes`` (equal parts).
Against the fp64 oracle, workspace and outputs NaN before the call.
"""

import numpy as np
import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

_R = np.random.default_rng(3)
CASES = [
    # (d, hq, hkv, window, lq, lk, packed)
    (512, 32, 4, None, [1], [8192], False),
    (512, 16, 4, None, [1, 0, 1, 1, 4], [3000, 50, 1, 700, 33], True),
    (512, 8, 8, None, [1, 1, 1], [2000, 2000, 2000], False),
    (512, 8, 2, None, [1] * 70, [int(x) for x in _R.integers(1, 600, 70)], True),
    (512, 8, 1, None, [2], [4100], True),
    (512, 8, 4, 1500, [1, 2], [300, 4000], True),
]


@pytest.mark.parametrize("d,hq,hkv,window,lq,lk,packed", CASES)
def test_decode_parts_match_the_oracle(d, hq, hkv, window, lq, lk, packed):
    from gemma4_fa4_amd import ops

    label = f"decode parts d{d} hq={hq} hkv={hkv} n={len(lq)} lk={max(lk)} packed={packed}"
    print(label, flush=True)
    q, k, v, _do, _dl = qkv(9980 + d + sum(lk), sum(lq), sum(lk), hq, hkv, d)
    cq, ck = cu(lq), cu(lk)
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq, num_kv_heads=hkv,
        head_dim=d, window=window, cu_q=cq.to(DEV) if packed else None,
        cu_k=ck.to(DEV) if packed else None, total_q=q.shape[0], total_k=k.shape[0])
    args = [t.to(DEV) for t in (q, k, v)]
    if not packed:
        args = [t.view(len(lq), t.shape[0] // len(lq), *t.shape[1:]) for t in args]
    o_ref, l_ref, *_ = attention_fwd_bwd(q.to(DEV), k.to(DEV), v.to(DEV), cq.tolist(),
                                         ck.tolist(), sliding_window=window,
                                         compute_dtype=torch.float64)
    least, most = plan.workspace_bytes(0), plan.workspace_bytes(3)
    assert least < most, "the problem does not take equal parts"
    st = ops.Stages(plan, *args, args[0], forward_only=True)
    for nbytes in (least, most):
        st.ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        for t in (st.ws, st.o, st.lse):
            t.view(torch.uint8).fill_(0xFF)
        st.forward()
        torch.cuda.synchronize()
        o = st.o.cpu().reshape(-1, hq, d)
        lse = st.lse.cpu() if packed else st.lse.cpu().permute(1, 0, 2).reshape(hq, -1)
        check_forward(o, lse, o_ref.cpu(), l_ref.cpu(), local=window is not None,
                      label=f"{label} workspace {nbytes}")
