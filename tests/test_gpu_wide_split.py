"""Head-dim 512 forward with its keys split: a chunk of new tokens after a cached prefix.

Given the workspace of ``g4_workspace_bytes`` phase 3 (the adapters' choice),
the wide forward cuts each 128-row tile's keys into chunks and merges them.
Cases: one tile, a tile with one query of its last row group, several tiles and
sequences, sequences shorter than the split was chosen for (chunks without
keys), GQA ratios, a window, and score jumps between chunks and within one (the
rescaling pass).  Each against the fp64 oracle, with every byte of the
workspace and the outputs NaN before the call, and bitwise repeatable.
"""

import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (hq, hkv, lq, lk, packed, window, jumps)
    (32, 4, [16], [3000], False, None, False),
    (32, 4, [5], [2048], True, None, False),
    (32, 4, [97], [5001], False, None, False),
    (32, 4, [20, 7, 130], [2500, 40, 4000], True, None, False),
    (32, 4, [33, 33], [2600, 2600], False, None, False),
    (16, 4, [40], [2100], True, None, False),
    (4, 4, [200], [3100], True, None, False),
    (16, 8, [70], [3000], True, 900, False),
    (32, 4, [33], [2600], True, None, True),
]


@pytest.mark.parametrize("hq,hkv,lq,lk,packed,window,jumps", CASES)
def test_split_wide_forward_matches_the_oracle(hq, hkv, lq, lk, packed, window, jumps):
    from gemma4_fa4_amd import ops

    label = f"wide split hq={hq} hkv={hkv} lq={lq} lk={lk} packed={packed} window={window}"
    print(label, flush=True)
    q, k, v, _do, _dl = qkv(9970 + sum(lk), sum(lq), sum(lk), hq, hkv, 512, unit_logits=not jumps)
    cq, ck = cu(lq), cu(lk)
    if jumps:  # tiny keys first: later tiles exceed the rows' first maxima by over 2^48
        k[:40] = (k[:40].float() / 64).to(torch.bfloat16)
        k[1000:1100] = (k[1000:1100].float() / 64).to(torch.bfloat16)
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq, num_kv_heads=hkv,
        head_dim=512, window=window, cu_q=cq.to(DEV) if packed else None,
        cu_k=ck.to(DEV) if packed else None, total_q=q.shape[0], total_k=k.shape[0])
    need = plan.workspace_bytes(3)
    assert need > plan.workspace_bytes(0), "the problem is not split"
    args = [t.to(DEV) for t in (q, k, v)]
    if not packed:
        args = [t.view(len(lq), t.shape[0] // len(lq), *t.shape[1:]) for t in args]
    st = ops.Stages(plan, *args, args[0], forward_only=True)
    st.ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    runs = []
    for fill in (0xFF, 0x7F):
        for t in (st.ws, st.o, st.lse):
            t.view(torch.uint8).fill_(fill)
        st.forward()
        runs.append((st.o.clone(), st.lse.clone()))
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])
    nq32 = (max(lq) + 31) // 32
    flags = st.ws[: 4 * len(lq) * nq32 * hq].view(torch.int32).view(len(lq), nq32, hq)
    flagged = sum(int(flags[s, : (n + 31) // 32].sum()) for s, n in enumerate(lq))
    assert (flagged > 0) == jumps
    o = runs[0][0].cpu().reshape(-1, hq, 512)
    lse = runs[0][1].cpu()
    if not packed:
        lse = lse.permute(1, 0, 2).reshape(hq, -1)
    o_ref, l_ref, *_ = attention_fwd_bwd(q.to(DEV), k.to(DEV), v.to(DEV), cq.tolist(),
                                         ck.tolist(), sliding_window=window,
                                         compute_dtype=torch.float64)
    check_forward(o, lse, o_ref.cpu(), l_ref.cpu(), local=False, label=label)


@pytest.mark.parametrize("lq,lk,hq,hkv", [([2048], [2048], 8, 2), ([16], [4096], 32, 4),
                                          ([1, 1], [3000, 900], 32, 4)])
def test_forward_in_a_backward_workspace_is_not_split(lq, lk, hq, hkv):
    """O and LSE of a forward given the backward's buffer do not follow its dS budget.

    Such a buffer's room past the forward's needs is dS; with 16 GiB of budget, with
    none and with the partial dK / dV tiles behind it, the forward is the one of the
    smallest workspace to the bit, and phase 3 still splits.
    """
    from gemma4_fa4_amd import ops

    print(f"forward in a backward workspace lq={lq} lk={lk} hq={hq}", flush=True)
    q, k, v, _do, _dl = qkv(9990, sum(lq), sum(lk), hq, hkv, 512)
    q, k, v = (t.to(DEV) for t in (q, k, v))
    got = {}
    for phase, budget in ((0, 0), (3, 0), (1, 0), (1, -1), (2, 0)):
        plan = ops.make_plan(
            num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq,
            num_kv_heads=hkv, head_dim=512, window=None, cu_q=cu(lq).to(DEV), cu_k=cu(lk).to(DEV),
            total_q=sum(lq), total_k=sum(lk))
        plan.ds_budget = budget
        st = ops.Stages(plan, q, k, v, q, forward_only=True)
        st.ws = torch.empty(plan.workspace_bytes(phase), dtype=torch.uint8, device=DEV).fill_(0xFF)
        st.forward()
        got[phase, budget] = st.o, st.lse
    o, lse = got.pop((0, 0))
    split = got.pop((3, 0))
    assert not torch.equal(split[0], o)
    for key, (o2, lse2) in got.items():
        assert torch.equal(o2, o) and torch.equal(lse2, lse), key
