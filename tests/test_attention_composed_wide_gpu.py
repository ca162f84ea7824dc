"""The composed attention whose columns meet the values before heads are mixed, against the plain implementation in float64
(tests/plain_dibepel.py), at the edges of its steps of 32 keys, its shares and its blocks of tokens.

Tolerance as for the kernel that mixes weights (test_dibepel_gpu.close): operands and results rounded to bfloat16 once."""
import pytest
import torch

import plain_dibepel as pd
from test_dibepel_gpu import DEV, F64, attend_mfma, close, rnd, rounded

pytestmark = pytest.mark.gpu


# (context, first new row): one token at the edges of tiles, steps and shares; then portions of prompts
REQUESTS = [(1, 0), (16, 15), (17, 16), (33, 32), (200, 199), (90, 0), (58, 33), (40, 38), (131, 64)]


def run(seqs, bs, shares=1, **kw):
    from llmserve.ops import library as ops

    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, "attend_composed_mfma", ops.attend_composed_wide)
        return attend_mfma(seqs, bs, shares=shares, **kw)


TALK = [  # heads, kv_heads, dk, dv, chunk, block size
    (32, 4, 64, 64, 128, 16),
    (4, 2, 64, 32, 20, 16),
    (3, 1, 128, 128, None, 32),  # 5 tokens a unit, a padded column, heads not a multiple of 4
    (16, 1, 64, 64, 48, 16),  # a unit is one token
    (8, 8, 128, 32, None, 48),  # pages that are no power of two
    (12, 2, 64, 128, 64, 16),
    (8, 8, 64, 32, 100, 32),  # eight waves on one turn of values
]


@pytest.mark.parametrize("heads,kv,dk,dv,chunk,bs", TALK)
def test_mixed_heads(heads, kv, dk, dv, chunk, bs, monkeypatch):
    from llmserve.ops import library as ops

    dt = torch.bfloat16
    talk = torch.eye(heads, dtype=F64) + rnd(heads, heads, seed=33, scale=0.3 / heads ** 0.5)
    slopes = pd.distance_slopes(heads)
    seqs, refs = [], []
    for i, (t, first) in enumerate(REQUESTS):
        q, k, v = (rounded(x, dt) for x in (rnd(t, heads, dk, seed=60 + i), rnd(t, kv, dk, seed=70 + i), rnd(t, kv, dv, seed=80 + i)))
        ref = pd.talking_heads(q, k, v, pd.visible_chunk(t, chunk), 0.1, slopes, talk)
        refs.append(ref.reshape(t, -1)[first:])
        seqs.append((q, k, v, first, t - first))
    can_share = kv >= 4 and kv * dv == 256 and dk == 64
    for shares, units, shared in ((1, 1, False), (3, 2 if kv * dv <= 128 else 1, False), (16, 1, can_share)):
        monkeypatch.setattr(ops, "wide_prompt_units", lambda *a: units)
        monkeypatch.setattr(ops, "wide_prompt_shared", lambda *a: shared)
        got = run(seqs, bs, shares=shares, heads=heads, kv_heads=kv, chunk=chunk or 0, scale=0.1, slopes=slopes.float().to(DEV),
                  talk=talk.float().to(DEV))
        for i, (g, r) in enumerate(zip(got, refs)):
            close(g, r, dt, f"request {i}, {shares} shares, {units} units")


MAPS = [  # heads, kv_heads, maps, dk, dv, window, keep_first, block size
    (16, 2, 2, 64, 128, 33, 20, 16),
    (3, 1, 2, 128, 64, 48, 0, 16),
    (4, 4, 2, 64, 64, None, 0, 32),
    (10, 5, 2, 64, 128, 100, 16, 16),  # ten score heads: three workgroups of up to four
]


@pytest.mark.parametrize("heads,kv,maps,dk,dv,window,keep,bs", MAPS)
def test_two_maps(heads, kv, maps, dk, dv, window, keep, bs, monkeypatch):
    from llmserve.ops import library as ops

    dt = torch.bfloat16
    lam, diff, eps, scale = 0.83, 0.3, 1e-5, 0.1
    seqs, refs = [], []
    for i, (t, first) in enumerate(REQUESTS):
        q, k, v = (rounded(x, dt) for x in (rnd(t, heads, 2, dk, seed=60 + i), rnd(t, kv, 2, dk, seed=70 + i), rnd(t, kv, dv, seed=80 + i)))
        ref = pd.differential_heads(q, k, v, pd.visible_window(t, window, keep), scale, lam, diff, eps)
        refs.append(ref.reshape(t, -1)[first:])
        seqs.append((q.reshape(t, heads * 2, dk), k.reshape(t, kv * 2, dk), v, first, t - first))
    for shares, units in ((1, 1), (2, 2), (16, 1)):
        monkeypatch.setattr(ops, "wide_prompt_units", lambda *a: units)
        got = run(seqs, bs, shares=shares, heads=heads, kv_heads=kv, maps=2, window=window or 0, keep_first=keep, scale=scale, lam=lam,
                  head_norm=True, eps=eps, out_scale=1 - diff)
        for i, (g, r) in enumerate(zip(got, refs)):
            close(g, r, dt, f"request {i}, {shares} shares, {units} units")


@pytest.mark.parametrize("sink", [False, True])
def test_one_map_with_a_sink_as_the_other_kernel(sink):
    """One map without a mixture: the same results as the kernel that takes any size, in bfloat16 (two roundings apart)."""
    heads, kv, dk, dv, bs = 8, 2, 64, 64, 16
    seqs = []
    for i, (t, first) in enumerate(REQUESTS):
        q, k, v = (rounded(x, torch.bfloat16) for x in (rnd(t, heads, dk, seed=1 + i), rnd(t, kv, dk, seed=20 + i), rnd(t, kv, dv, seed=40 + i)))
        seqs.append((q, k, v, first, t - first))
    kw = dict(heads=heads, kv_heads=kv, scale=0.1, chunk=64, slopes=pd.distance_slopes(heads).float().to(DEV), sink=sink)
    for i, (g, r) in enumerate(zip(run(seqs, bs, shares=4, **kw), attend_mfma(seqs, bs, **kw))):
        close(g, r.double().cpu(), torch.bfloat16, f"request {i}")


@pytest.mark.parametrize("heads,kv,dv,maps,shared", [(8, 2, 64, 1, False), (32, 4, 64, 1, False), (32, 4, 64, 1, True), (8, 8, 32, 1, True),
                                                      (4, 2, 64, 2, False)])
def test_values_behind_the_end_and_pages_of_other_requests_are_not_seen(heads, kv, dv, maps, shared, monkeypatch):
    """NaN in every place of the pools that the request does not own: to the bit the result of pools with zeros there."""
    from llmserve.ops import library as ops

    d, bs, t = 64, 16, 37
    monkeypatch.setattr(ops, "wide_prompt_shared", lambda *a: shared)
    g = torch.Generator().manual_seed(3)
    k_pool = torch.full((6, kv * maps, bs, d), float("nan"), dtype=torch.bfloat16)
    v_pool = torch.full((6, kv, dv, bs), float("nan"), dtype=torch.bfloat16)
    for j in range(t):
        k_pool[j // bs, :, j % bs] = torch.randn(kv * maps, d, generator=g).bfloat16()
        v_pool[j // bs, :, :, j % bs] = torch.randn(kv, dv, generator=g).bfloat16()
    talk = (torch.eye(heads) + 0.1 * torch.randn(heads, heads, generator=g)).to(DEV) if maps == 1 else None
    table = torch.tensor([[0, 1, 2, 5]], dtype=torch.int32, device=DEV)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    for new in (1, 7, 37):
        q = torch.randn(new, heads * maps * d, generator=g).bfloat16().to(DEV)
        got = []
        for k, v in ((k_pool, v_pool), (k_pool.nan_to_num(0.0), v_pool.nan_to_num(0.0))):
            out = torch.empty(new, heads * dv, dtype=torch.bfloat16, device=DEV)
            got.append(ops.attend_composed_wide(out, q, k.to(DEV), v.to(DEV), table, i32(0, new), i32(t), 0, 1, new, heads=heads,
                                                kv_heads=kv, maps=maps, dk=d, dv=dv, block_size=bs, scale=0.1, talk=talk, lam=0.5, shares=2))
        assert torch.isfinite(got[0].float()).all() and torch.equal(*got)


def _relative_error(got, want):
    got, want = torch.cat([g.double().cpu().flatten() for g in got]), torch.cat([w.flatten() for w in want])
    return float((got - want).norm() / want.norm())


@pytest.mark.parametrize("scale", [1.0, 0.3, 0.1, 0.03])  # of the queries: the flatter the weights, the more of them cancels
@pytest.mark.parametrize("heads,kv,dk,dv", [(32, 4, 64, 64), (8, 8, 64, 32), (8, 1, 128, 128)])
def test_heads_that_are_subtracted_from_one_another(heads, kv, dk, dv, scale, monkeypatch):
    """A head minus the next one, and minus the mean of all: what is left is small beside the heads' own results.  In the norm the
    result is as near as where the mixed weights are rounded: two roundings to 8 bits, of a weight and of the result, each at most
    2^-8 / sqrt(3) of the norm when they fall evenly (3.2e-3 together)."""
    from llmserve.ops import library as ops

    subtracting = (torch.eye(heads, dtype=F64) - torch.eye(heads, dtype=F64).roll(1, 1), torch.eye(heads, dtype=F64) - 1.0 / heads)
    for talk in subtracting:
        seqs, refs = [], []
        for i, (t, first) in enumerate(REQUESTS[3:]):
            q, k, v = (rounded(s * x, torch.bfloat16) for s, x in ((scale, rnd(t, heads, dk, seed=60 + i)), (1, rnd(t, kv, dk, seed=70 + i)),
                                                                   (1, rnd(t, kv, dv, seed=80 + i))))
            ref = pd.talking_heads(q, k, v, pd.visible_chunk(t, None), dk ** -0.5, torch.zeros(heads, dtype=F64), talk.float().double())
            refs.append(ref.reshape(t, -1)[first:])
            seqs.append((q, k, v, first, t - first))
        kw = dict(heads=heads, kv_heads=kv, chunk=0, scale=dk ** -0.5, talk=talk.float().to(DEV))
        for shared in {False, kv >= 4 and kv * dv == 256 and dk == 64}:
            monkeypatch.setattr(ops, "wide_prompt_shared", lambda *a: shared)
            assert _relative_error(run(seqs, 16, shares=3, **kw), refs) <= 2.0 ** -8
        assert _relative_error(attend_mfma(seqs, 16, **kw), refs) <= 2.0 ** -8


@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("counts", [[2], [1, 40], [0, 33, 2], [70, 1, 0, 5, 31, 2, 64, 1], [3, 0, 50, 1, 2, 9, 0, 17, 4], [1 + i % 4 for i in range(70)]])
def test_portions_of_ragged_lengths(counts, maps, monkeypatch):
    """Which workgroup takes which block of which request (one request, up to 8, more, and more than a wave's lanes; requests without
    rows and without keys between them) changes no result: each request's rows are the same numbers as in a launch of its own."""
    from llmserve.ops import library as ops

    monkeypatch.setattr(ops, "wide_prompt_units", lambda *a: 1 if maps == 1 else 2)
    monkeypatch.setattr(ops, "wide_prompt_shared", lambda *a: False)
    heads, kv, dk, dv, bs = (8, 2, 64, 32, 16) if maps == 1 else (4, 2, 64, 64, 16)
    dt, gen = torch.bfloat16, torch.Generator().manual_seed(len(counts))
    rows, n = sum(counts), len(counts)
    ends = [c + 7 * (i % 5) if c else (11 if i % 2 else 0) for i, c in enumerate(counts)]
    if n > 3:
        ends[3] = 0  # padding: left alone
    width = -(-max(ends) // bs)
    q = torch.randn(rows, heads * maps * dk, generator=gen).to(dt).to(DEV)
    pages = n * width
    k_pool = torch.randn(pages, kv * maps, bs, dk, generator=gen).to(dt).to(DEV)
    v_pool = torch.randn(pages, kv, dv, bs, generator=gen).to(dt).to(DEV)
    table = torch.randperm(pages, generator=gen).int().view(n, width).to(DEV)
    cu = [0]
    for c in counts:
        cu.append(cu[-1] + c)
    cu_d, ends_d = torch.tensor(cu, dtype=torch.int32, device=DEV), torch.tensor(ends, dtype=torch.int32, device=DEV)
    kw = dict(heads=heads, kv_heads=kv, dk=dk, dv=dv, block_size=bs, scale=0.1, maps=maps)
    if maps == 1:
        kw["talk"] = (torch.eye(heads) + 0.1 * torch.randn(heads, heads, generator=gen)).to(DEV)
    else:
        kw.update(lam=0.8, head_norm=True, eps=1e-5, out_scale=0.5)
    out = torch.full((rows, heads * dv), 7.0, dtype=dt, device=DEV)
    ops.attend_composed_wide(out, q, k_pool, v_pool, table, cu_d, ends_d, 0, n, max(2, max(counts)), **kw)
    alone = torch.full_like(out, 7.0)
    for s in range(n):
        ops.attend_composed_wide(alone, q, k_pool, v_pool, table, cu_d, ends_d, s, 1, max(2, counts[s]), **kw)
    assert torch.equal(out, alone)
    seen = [s for s in range(n) if ends[s] > 0 and counts[s]]
    for s in range(n):
        part = out[cu[s]:cu[s + 1]]
        assert bool((part != 7.0).any(1).all()) if s in seen else bool((part == 7.0).all())


@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("counts", [[33] * 9, [7 + 5 * (i % 6) for i in range(16)], [150] + [3] * 20, [0, 90, 1] * 8, [40] * 63, [2 + i for i in range(64)],
                                    [0] * 30 + [40, 0, 77] + [1] * 31])
def test_portions_of_many_requests(counts, maps, monkeypatch):
    """More than 8 requests and up to a wave's lanes, whose blocks go by their keys where the chip does not take them all at once: alike, ragged,
    one long, some without rows, a wave full."""
    test_portions_of_ragged_lengths(counts, maps, monkeypatch)
