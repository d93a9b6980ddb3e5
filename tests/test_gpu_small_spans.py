"""Vision spans of few K tokens: one workgroup instead of the six passes.

One sequence takes it up to 4096 tokens, several up to 3584 in the backward's
form (the key tiles' ranges too, as here) and 2560 in the forward's.

The same sequences are scheduled alone (one workgroup, table in LDS) and with a
text sequence appended that takes the batch past the limit (the passes over the
whole stream); the ranges of the shared sequences must agree in both
directions, and so must those at the limit itself.  IDs that repeat with gaps,
that cross documents, blocks of one token, queries that are a suffix, sequences
without queries or keys, and more sequences than the one workgroup takes.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ranges(lq, lk, vis, docs):
    from gemma4_fa4_amd import ops

    cq, ck = ([0, *np.cumsum(x).tolist()] for x in (lq, lk))
    dev = lambda x: torch.tensor(np.asarray(x), dtype=torch.int32, device=DEV)  # noqa: E731
    plan = ops.make_plan(
        num_seqs=len(lq), seqlen_q=max(max(lq), 1), seqlen_k=max(lk), num_q_heads=2,
        num_kv_heads=1, head_dim=256, window=1024, vision=dev(vis),
        documents=None if docs is None else dev(docs), cu_q=dev(cq), cu_k=dev(ck),
        total_q=cq[-1], total_k=ck[-1])
    return [ops.tile_ranges(plan, direction, 32, DEV).cpu() for direction in (0, 1)]


@pytest.mark.parametrize("seed,lq,lk,with_docs", [
    (0, [777], [777], False),
    (1, [500, 0, 64, 1000], [900, 40, 64, 1000], True),
    (2, [4096], [4096], True),
    (3, [1, 1300], [1, 2500], False),
    (4, [9] * 256, [16] * 256, True),
    (6, [9] * 256, [14] * 256, True),
    (7, [500, 700], [1000, 2584], True), (8, [500, 700], [1000, 2585], True),
    (5, [5] * 300, [5] * 300, False),  # too many sequences: the passes either way
])
def test_small_spans_match_the_passes(seed, lq, lk, with_docs):
    rng = np.random.default_rng(seed)
    tk = sum(lk)
    vis = np.full(tk, -1)
    for b in range(max(3, tk // 150)):  # few IDs: they repeat, with gaps
        a = int(rng.integers(0, tk))
        vis[a:a + int(rng.choice([1, 7, 40, 300]))] = b % 5
    docs = np.sort(rng.integers(0, 4, size=tk)) if with_docs else None
    print(f"small spans seed {seed} n={len(lk)} tk={tk}", flush=True)
    alone = _ranges(lq, lk, vis, docs)
    extra = 4200  # a text sequence past the limit
    more = _ranges([*lq, extra], [*lk, extra], np.concatenate([vis, np.full(extra, -1)]),
                   None if docs is None else np.concatenate([docs, np.full(extra, 9)]))
    for direction, (a, b) in enumerate(zip(alone, more)):
        # (the batches differ in tiles per sequence; the extra ones are empty)
        for s, n in enumerate(lk if direction else lq):
            tiles = (n + 31) // 32
            assert torch.equal(a[s, :tiles], b[s, :tiles]), (direction, s)
