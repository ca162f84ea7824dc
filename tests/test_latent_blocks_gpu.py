"""Latent attention over few long and many short portions, where rows of a multiple of 8 blocks are launched with one block more: against plain attention."""

import math

import pytest
import torch

from test_milozen_gpu import DEV, attend_plain, close, dev, ints, paged_rows, rnd

pytestmark = pytest.mark.gpu


# (heads, (context after the step, tokens of the step) ...): 8 blocks of 128 pairs beside single tokens; 16, exactly half of all rows' room, and a row
# beyond half, which keeps the 16; blocks that are no multiple of 8; a request without keys or tokens among them
@pytest.mark.parametrize("heads,lengths", [(32, [(150, 1), (97, 1), (64, 32)]), (16, [(70, 64), (300, 64), (33, 1), (33, 1), (40, 30)]),
                                           (32, [(64, 64), (200, 1)]), (32, [(64, 64), (200, 64), (33, 1)]), (128, [(9, 8), (500, 1), (20, 2), (31, 1)]),
                                           (32, [(80, 36), (400, 1), (17, 1)]), (32, [(40, 32), (0, 0), (0, 6), (90, 1)])])
@pytest.mark.parametrize("splits,window", [(1, None), (3, None), (2, 50)])
def test_short_portions_beside_a_long_one(heads, lengths, splits, window):
    from llmserve.ops import library as ops

    r, dr, bs, dt = 48, 16, 16, torch.bfloat16
    scale = 0.5 / math.sqrt(r + dr)
    pools, tables, qs, refs, at = [], [], [], [], 0
    for b, (ctx, count) in enumerate(lengths):
        q, rows = rnd(max(ctx, count), heads, r + dr, seed=10 + b), rnd(max(ctx, 1), r + dr, seed=40 + b)
        qs.append(q[q.shape[0] - count:].reshape(count, heads * (r + dr)))
        refs.append(attend_plain(q.to(dt).double(), rows.to(dt).double(), r, window, scale)[ctx - count:] if ctx else None)
        pool, table = paged_rows(rows, bs, dt, seed=b)
        tables.append(table[0] + at)
        pools.append(pool)
        at += pool.shape[0]
    table = torch.zeros((len(lengths), max(len(t) for t in tables)), dtype=torch.int32)
    for b, t in enumerate(tables):
        table[b, : len(t)] = t
    counts = [c for _, c in lengths]
    cu = [sum(counts[:i]) for i in range(len(counts) + 1)]
    out = torch.full((cu[-1], heads * r), float("nan"), dtype=dt, device=DEV)
    ops.attend_latent_mfma(out, dev(torch.cat(qs), dt), torch.cat(pools), table.to(DEV), ints(cu), ints([c for c, _ in lengths]), n_seqs=len(counts),
                           max_count=max(counts), heads=heads, r=r, dr=dr, block_size=bs, window=window or 0, scale=scale, splits=splits)
    for b, ref in enumerate(refs):
        got = out[cu[b]: cu[b + 1]].view(-1, heads, r)
        if ref is None:
            assert (got == 0).all()
        else:
            close(got, ref, dt, f"request {b}")
