"""A step's first launch: rows of the embedding, angles and block table entries, beside the operations that do each alone."""

import pytest
import torch

DEV = "cuda:0"


def ops():
    from llmserve.ops import library

    return library


@pytest.mark.gpu
@pytest.mark.parametrize("n,hidden,half,tables", [(1, 8, 0, 0), (8, 2048, 32, 1), (5, 2052, 3, 2), (17, 36, 64, 8), (300, 4096, 16, 1), (3, 7, 1, 3), (2, 1032, 2, 1)])  # (a row of 1,032: 1,024 in one turn of the threads)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("scale", [None, 3.5])
def test_step_start(n, hidden, half, tables, dtype, scale):
    g = torch.Generator().manual_seed(n)
    table = torch.randn(50, hidden, generator=g).to(dtype).to(DEV)
    ids = torch.randint(0, 50, (n,), generator=g, dtype=torch.int32)
    ids[n // 2] = 50  # outside the vocabulary
    positions = torch.randint(0, 5000, (n,), generator=g, dtype=torch.int32).to(DEV)
    freq = torch.rand(half, generator=g).to(DEV)
    scatters, want = [], []
    for t in range(tables):
        dst = torch.randint(0, 99, (7, 300), generator=g, dtype=torch.int32).to(DEV)
        count = [n, 1, 257, 600][t % 4]
        index = torch.randperm(2100, generator=g)[:count].to(torch.int32)
        index[::3] = -1
        value = torch.randint(100, 999, (count,), generator=g, dtype=torch.int32)
        kept = dst.clone()
        ops().scatter_i32(kept, index.to(DEV), value.to(DEV))
        scatters.append((dst, index.to(DEV), value.to(DEV)))
        want.append(kept)
    out = torch.full((n, hidden), 7.0, dtype=dtype if scale is None else torch.float32, device=DEV)
    turned = ops().step_start(out, table, ids.to(DEV), scale=scale, angles=(positions, freq) if half else None, scatters=scatters)
    rows = table[ids.long().clamp(max=49).to(DEV)]
    if scale is None:
        rows[n // 2] = float("nan")
    else:
        rows = rows.float() * scale
    assert torch.equal(out.nan_to_num(nan=1e9), rows.nan_to_num(nan=1e9))
    assert (turned is None) == (half == 0)
    if half:
        assert torch.equal(turned, ops().rotary_angles(positions, freq))
    assert all(torch.equal(dst, kept) for (dst, _, _), kept in zip(scatters, want))
