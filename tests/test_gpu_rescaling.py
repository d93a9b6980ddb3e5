"""Rescaling pass of the head-dim 512 forward: which rows take it, and its share over workgroups.

The wide kernel keeps a row's first maximum; rows whose scores rise by more than
2^48 (in exp2 terms) after it are marked per head, and the rescaling pass
recomputes the marked heads' 64-query tiles.  Here one coordinate of the keys
rises along each sequence and single rows, heads or all queries point along it.
Checked: only the marked heads are recomputed (the others keep their bits), the
cost follows the number of marked tiles, and every pattern of marks (more items
than workgroups, more flags than one step reads, GQA ratios, split keys) against
the fp64 oracle, with every byte of the workspace and the outputs set before.
"""

import numpy as np
import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(seed, lq, lk, hq, hkv, hot, rise=160):
    """q, k, v on the GPU; hot(sequence, length) -> (query rows, heads) whose scores rise by `rise`."""
    q, k, v, _, _ = qkv(seed, sum(lq), sum(lk), hq, hkv, 512)
    q[:, :, 7] = 0
    q0 = k0 = 0
    for s, (nq, nk) in enumerate(zip(lq, lk)):
        k[k0:k0 + nk, :, 7] = (torch.arange(nk) * (16.0 / nk))[:, None].to(torch.bfloat16)
        rows, heads = hot(s, nq)
        for h in heads:
            q[[q0 + r for r in rows], h, 7] = rise / 16
        q0, k0 = q0 + nq, k0 + nk
    return [t.to(DEV) for t in (q, k, v)]


def _stages(q, k, v, lq, lk, phase=0):
    from gemma4_fa4_amd import ops

    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=q.shape[1],
        num_kv_heads=k.shape[1], head_dim=512, window=None, cu_q=cu(lq).to(DEV),
        cu_k=cu(lk).to(DEV), total_q=q.shape[0], total_k=k.shape[0])
    st = ops.Stages(plan, q, k, v, q, forward_only=True)
    st.ws = torch.empty(plan.workspace_bytes(phase), dtype=torch.uint8, device=DEV)
    return st


def _run(st):
    for t in (st.ws, st.o, st.lse):
        t.view(torch.uint8).fill_(0xFF)
    st.forward()
    torch.cuda.synchronize()
    return st.o.clone(), st.lse.clone()


def _flags(st, s, group):
    """Raise flags of sequence s's 32-query group: (KV head, wave of the group's rows)."""
    p = st.plan
    nq32 = (p.seqlen_q + 31) // 32
    flags = st.ws[: 4 * p.num_seqs * nq32 * p.num_q_heads].view(torch.int32)
    return flags.view(p.num_seqs, nq32, p.num_kv_heads, -1)[s, group].cpu()


@pytest.mark.parametrize("hq,hkv,head", [(32, 4, 13), (16, 8, 15), (4, 4, 2), (8, 2, 0)])
def test_a_marked_row_recomputes_its_head_alone(hq, hkv, head):
    lq = lk = [700, 300]
    grp = hq // hkv
    marked = _inputs(41, lq, lk, hq, hkv, lambda s, n: ([n - 5] if s == 0 else [], [head]))
    plain = _inputs(41, lq, lk, hq, hkv, lambda s, n: ([], []))
    a, b = _stages(*marked, lq, lk), _stages(*plain, lq, lk)
    (o, lse), (o0, lse0) = _run(a), _run(b)
    group = (700 - 5) // 32
    per_kv = _flags(a, 0, group)
    seen = [int(np.bitwise_or.reduce(x.numpy())) for x in per_kv]
    assert seen == [1 << head % grp if h == head // grp else 0 for h in range(hkv)]
    assert all(not _flags(a, 0, g).any() for g in range(group))
    others = [h for h in range(hq) if h != head]
    assert torch.equal(o[:, others], o0[:, others]) and torch.equal(lse[others], lse0[others])
    tile = 700 - 5 - (700 - 5) % 64
    assert torch.equal(o[:tile, head], o0[:tile, head]) and torch.equal(o[700:], o0[700:])
    assert not torch.equal(o[695, head], o0[695, head])


_R = np.random.default_rng(5)
_MANY = [int(x) for x in _R.integers(60, 101, 300)]
CASES = [
    # (hq, hkv, lq, lk, hot, phase): hot = rows and heads of a sequence
    (32, 4, [1500], [1500], "head", 0),
    (32, 4, [1500], [1500], "row of each head", 0),
    (32, 4, [1111, 64, 65, 700], None, "all", 0),
    (16, 4, [513, 900], None, "all", 0),
    (16, 8, [640, 33], None, "head", 0),
    (6, 6, [300, 129], None, "all", 0),
    (32, 4, _MANY, None, "all", 0),  # several steps of flags, many rounds of items
    (32, 4, _MANY, None, "some", 0),
    (32, 4, [70], [3000], "head", 3),
    (16, 8, [40, 9], [3000, 2500], "row of each head", 3),
]


@pytest.mark.parametrize("hq,hkv,lq,lk,hot,phase", CASES)
def test_rescaling_patterns_match_the_oracle(hq, hkv, lq, lk, hot, phase):
    lk = lk or lq
    label = f"rescaling hq={hq} hkv={hkv} n={len(lq)} lq={max(lq)} lk={max(lk)} {hot}"
    print(label, flush=True)
    pick = {
        "head": lambda s, n: (range(n), [hq - 2]),
        "row of each head": lambda s, n: ([n - 1], range(hq)),
        "all": lambda s, n: (range(n), range(hq)),
        "some": lambda s, n: (range(n) if s % 7 == 3 else [], range(s % 5, hq, 5)),
    }[hot]
    # (split: over 33.3 = 48 ln 2 within each of at most a dozen chunks of the keys)
    q, k, v = _inputs(50 + len(lq), lq, lk, hq, hkv, pick, rise=960 if phase else 160)
    st = _stages(q, k, v, lq, lk, phase)
    if phase:
        assert st.ws.numel() > st.plan.workspace_bytes(0), "the problem is not split"
    (o, lse), (o2, lse2) = _run(st), _run(st)
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    assert any(bool(_flags(st, s, (n - 1) // 32).any()) for s, n in enumerate(lq))
    o_ref, l_ref, *_ = attention_fwd_bwd(q, k, v, cu(lq).tolist(), cu(lk).tolist(),
                                         compute_dtype=torch.float64)
    check_forward(o, lse, o_ref.cpu(), l_ref.cpu(), local=False, label=label)


def _time(st, n=10):
    for _ in range(3):
        st.forward()
    best = float("inf")
    for _ in range(3):
        e0, e1 = torch.cuda.Event(True), torch.cuda.Event(True)
        e0.record()
        for _ in range(n):
            st.forward()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / n)
    return best


def test_rescaling_cost_follows_the_marked_tiles():
    # One marked row per sequence is one 64-query tile of one head of each of 32
    # sequences: about 1.1 times the forward without marks.  (With every head of
    # the group recomputed, and a workgroup's items all of one head, 2.9 times.)
    lens = [1024] * 32
    plain = _stages(*_inputs(7, lens, lens, 32, 4, lambda s, n: ([], [])), lens, lens)
    marked = _stages(*_inputs(7, lens, lens, 32, 4, lambda s, n: ([n - 5], [13])), lens, lens)
    assert _time(marked) < 1.6 * _time(plain)
