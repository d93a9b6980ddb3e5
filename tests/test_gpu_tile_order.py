"""Head-dim 512 forward of equal sequences: the order of its tiles.

One sequence, or several of one length, is dealt to the XCDs by (sequence, KV
head) segment and from the last tile to the first.  Cases: segments that divide
the 8 XCDs, are a multiple of them, are neither, fewer tiles than XCDs, lengths
that end inside a tile; each against the fp64 oracle with the outputs NaN before
the call (a tile left out shows).  And the cost of a length whose tiles do not
come out even is no more than that of the next one that does.
"""

import pytest
import torch

from g4_testutil import check_forward, cu, qkv
from oracle.attention import attention_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (hq, hkv, sequences, length, packed)
    (32, 4, 1, 700, True),
    (32, 4, 1, 41, False),
    (8, 1, 1, 333, True),
    (24, 3, 1, 450, False),
    (12, 6, 2, 300, False),
    (32, 4, 3, 210, False),
    (5, 5, 1, 520, True),
    (16, 16, 1, 385, False),
    (24, 12, 2, 130, False),
    (32, 4, 4, 70, False),
    # several segments in a set: up to four tiles each, remainders of 2 and 3, two batches
    (6, 6, 8, 300, False),
    (16, 16, 3, 650, False),
    (3, 3, 6, 1300, False),
    (16, 16, 8, 900, False),
]


def _stages(seed, hq, hkv, n, length, packed):
    from gemma4_fa4_amd import ops

    q, k, v, _, _ = qkv(seed, n * length, n * length, hq, hkv, 512)
    c = cu([length] * n)
    plan = ops.make_plan(
        num_seqs=n, seqlen_q=length, seqlen_k=length, num_q_heads=hq, num_kv_heads=hkv,
        head_dim=512, window=None, cu_q=c.to(DEV) if packed else None,
        cu_k=c.to(DEV) if packed else None, total_q=n * length, total_k=n * length)
    args = [t.to(DEV) for t in (q, k, v)]
    if not packed:
        args = [t.view(n, length, *t.shape[1:]) for t in args]
    st = ops.Stages(plan, *args, args[0], forward_only=True)
    st.ws = torch.empty(plan.workspace_bytes(0), dtype=torch.uint8, device=DEV)
    return st, (q, k, v, c)


@pytest.mark.parametrize("hq,hkv,n,length,packed", CASES)
def test_equal_sequences_match_the_oracle(hq, hkv, n, length, packed):
    label = f"tile order hq={hq} hkv={hkv} {n} x {length} packed={packed}"
    print(label, flush=True)
    st, (q, k, v, c) = _stages(60 + length, hq, hkv, n, length, packed)
    for t in (st.ws, st.o, st.lse):
        t.view(torch.uint8).fill_(0xFF)
    st.forward()
    torch.cuda.synchronize()
    o = st.o.cpu().reshape(-1, hq, 512)
    lse = st.lse.cpu() if packed else st.lse.cpu().permute(1, 0, 2).reshape(hq, -1)
    o_ref, l_ref, *_ = attention_fwd_bwd(q.to(DEV), k.to(DEV), v.to(DEV), c.tolist(), c.tolist(),
                                         compute_dtype=torch.float64)
    check_forward(o, lse, o_ref.cpu(), l_ref.cpu(), local=False, label=label)


def _time(st, n=20):
    for _ in range(5):
        st.forward()
    best = float("inf")
    for _ in range(4):
        e0, e1 = torch.cuda.Event(True), torch.cuda.Event(True)
        e0.record()
        for _ in range(n):
            st.forward()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / n)
    return best


@pytest.mark.parametrize("length,even", [(1200, 1408), (2000, 2048), (3500, 3584), (5000, 5120)])
def test_uneven_lengths_cost_no_more_than_even_ones(length, even):
    # (in zigzag order 1.25, 1.37, 1.3 and 1.13 times the even length, or more)
    a, _ = _stages(1, 32, 4, 1, length, True)
    b, _ = _stages(2, 32, 4, 1, even, True)
    assert _time(a) < 1.08 * _time(b)
