"""Split dK/dV launch: the steps of a problem with few key tiles cut into equal parts.

A backward given the larger workspace of ``g4_workspace_bytes`` phase 2 (the
adapters' choice) runs the dK/dV stage as equal runs of steps over the CUs and
adds the fp32 partials of the key tiles that a cut falls into.  Cases sit where
the cuts can go wrong: one tile cut many times, tiles that lie whole inside a
part, a last tile of one key, keys without queries, keys before the first query,
windows that end inside the sequence, vision spans that lengthen a tile's run
beyond the cost model's, documents.  Each is checked against the fp64 oracle,
against the launch by whole tiles (the same sums in another order; dQ from the
same dS tiles, so to the bit) and against itself on a used workspace.
"""

import pytest
import torch

from g4_testutil import check_forward, check_gradients, cu, qkv, vision_blocks
from oracle.attention import attention_fwd_bwd, bf16_baseline_fwd_bwd

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # (d, hq, hkv, lq, lk, packed, vision, docs)
    (512, 32, 4, [1000], [1000], False, False, False),
    (512, 32, 4, [193], [193], True, False, False),  # four tiles, the last of one key
    (512, 32, 4, [700, 0, 517, 96], [700, 40, 600, 96], True, False, False),
    (512, 8, 1, [450], [1500], False, False, False),  # keys before the first query
    (512, 16, 8, [640, 640], [640, 640], False, False, False),  # fixed batch, GQA 2
    (256, 32, 16, [777], [777], False, True, False),
    (256, 32, 16, [1025], [1025], True, False, False),  # a last tile of one key
    (256, 16, 2, [2600], [2600], True, True, False),  # the window ends inside, GQA 8
    (256, 8, 4, [900, 0, 1300, 64], [1100, 50, 1300, 64], True, True, True),
    (256, 8, 4, [900], [3000], False, False, False),  # keys outside every window
]


@pytest.mark.parametrize("d,hq,hkv,lq,lk,packed,with_vision,with_docs", CASES)
def test_split_dkdv_matches_whole_tiles_and_the_oracle(d, hq, hkv, lq, lk, packed, with_vision,
                                                       with_docs):
    from gemma4_fa4_amd import ops

    label = f"split dK/dV d{d} hq={hq} hkv={hkv} lq={lq} lk={lk} packed={packed}"
    print(label, flush=True)
    q, k, v, do, dlse = qkv(9950 + d + sum(lk), sum(lq), sum(lk), hq, hkv, d)
    cq, ck = cu(lq), cu(lk)
    window = 1024 if d == 256 else None
    vis = vision_blocks(78, sum(lk), 3, 100, 700) if with_vision else None
    docs = None
    if with_docs:
        docs = torch.zeros(sum(lk), dtype=torch.int32)
        docs[500:] = 1
        docs[1900:] = 2
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(lq), seqlen_k=max(lk), num_q_heads=hq, num_kv_heads=hkv,
        head_dim=d, window=window, vision=None if vis is None else vis.to(DEV),
        documents=None if docs is None else docs.to(DEV), cu_q=cq.to(DEV) if packed else None,
        cu_k=ck.to(DEV) if packed else None, total_q=q.shape[0], total_k=k.shape[0])
    assert plan.workspace_bytes(2) > plan.workspace_bytes(1), "the problem is not split"
    if packed:
        args = [t.to(DEV) for t in (q, k, v, do)]
        dl = dlse.to(DEV)
    else:
        b = len(lq)
        args = [t.view(b, t.shape[0] // b, *t.shape[1:]).to(DEV) for t in (q, k, v, do)]
        dl = dlse.view(hq, b, -1).permute(1, 0, 2).contiguous().to(DEV)
    st = ops.Stages(plan, *args, dl)
    st.forward()
    st.backward()
    whole = [t.clone() for t in (st.dq, st.dk, st.dv)]
    # NaN bytes everywhere: a partial or an output read before it is written shows
    st.ws = torch.empty(plan.workspace_bytes(2), dtype=torch.uint8, device=DEV).fill_(0xFF)
    runs = []
    for _ in range(2):
        for t in (st.dq, st.dk, st.dv):
            t.fill_(float("nan"))
        st.backward()
        runs.append([t.clone() for t in (st.dq, st.dk, st.dv)])
    for a, b in zip(*runs):
        assert torch.equal(a, b), "the split launch is not repeatable"
    assert torch.equal(runs[0][0], whole[0]), "dQ differs from the launch by whole tiles"
    for got, ref in zip(runs[0][1:], whole[1:]):
        # one rounding to bf16 of sums in another order
        assert (got.double() - ref.double()).norm() <= 2e-3 * ref.double().norm()
    flat = (lambda t: t.cpu()) if packed else (lambda t: t.reshape(-1, *t.shape[2:]).cpu())
    kw = dict(sliding_window=window, vision_block_ids=None if vis is None else vis.to(DEV),
              document_ids=None if docs is None else docs.to(DEV),
              allow_vision_bidirectional=vis is not None)
    ref = attention_fwd_bwd(q.to(DEV), k.to(DEV), v.to(DEV), cq.tolist(), ck.tolist(),
                            do=do.to(DEV), dlse=dlse.to(DEV), compute_dtype=torch.float64, **kw)
    _, *bf = bf16_baseline_fwd_bwd(q.to(DEV), k.to(DEV), v.to(DEV), cq.tolist(), ck.tolist(),
                                   do=do.to(DEV), dlse=dlse.to(DEV), **kw)
    check_gradients([flat(t) for t in runs[0]], [t.cpu() for t in ref[2:]],
                    [t.cpu() for t in bf], label=label)
    for n, k0, nk in zip(lq, ck.tolist(), lk):
        if n == 0:  # keys without queries get exact zeros
            assert not flat(runs[0][1])[k0:k0 + nk].any()
            assert not flat(runs[0][2])[k0:k0 + nk].any()
