"""Steps whose spare places for single tokens take tokens of a portion: the same tokens at the same places, fewer rows."""

import random

import pytest

from llmserve.cache.manager import StepLayout
from llmserve.engine.runner import ModelRunner


def step_of(rng, n_single, counts):
    counts = [1] * n_single + counts
    starts = [rng.randrange(1, 500) if c == 1 else rng.choice([0, 17, 300]) for c in counts]
    total, names = sum(counts), [f"r{i}" for i in range(len(counts))]
    slots = {g: rng.sample(range(10 * total), total) for g in (0, 1)}
    layout = StepLayout(seq_ids=names, counts=counts, starts=starts, state_slots=rng.sample(range(200), len(counts)),
                        fresh_slots=[1], slots=slots, table_updates={0: [(1, 2, 3)], 1: []})
    tokens, t = [], 0
    for c in counts:
        tokens.append(list(range(t, t + c)))
        t += c
    return layout, tokens, rng.sample(range(total), min(total, 5))


def rows_of(layout, tokens):
    """Per row: (request, state slot, position, token, cache slots)."""
    out, row = [], 0
    for name, count, start, state, own in zip(layout.seq_ids, layout.counts, layout.starts, layout.state_slots, tokens):
        assert len(own) == count
        for i in range(count):
            out.append((name, state, start + i, own[i], tuple(layout.slots[g][row] for g in sorted(layout.slots))))
            row += 1
    return out


@pytest.mark.parametrize("n_single", [0, 1, 2, 3, 5, 6, 8, 9, 17, 31, 33])
@pytest.mark.parametrize("counts", [[2], [3], [509], [507], [200, 309], [16, 2, 480], [500, 5, 5], [80], [1000], []])
def test_rows_are_the_same(n_single, counts):
    rng = random.Random(n_single * 1000 + sum(counts))
    layout, tokens, wanted = step_of(rng, n_single, counts)
    if not layout.counts:
        return
    filled, own, rows = ModelRunner._spare_rows_filled(layout, tokens, wanted)
    before, after = rows_of(layout, tokens), rows_of(filled, own)
    assert sorted(before) == sorted(after)
    assert [after[r] for r in rows] == [before[r] for r in wanted]
    n_dec = next((i for i, c in enumerate(filled.counts) if c != 1), len(filled.counts))
    assert all(c > 1 for c in filled.counts[n_dec:]) and len(filled.counts) - n_dec == len(counts)
    assert (filled.table_updates, filled.fresh_slots) == (layout.table_updates, layout.fresh_slots)
    if counts:
        def rows_run(singles, tokens):
            shape = ModelRunner._step_shape(singles, 1, tokens, 1, 1)
            return shape[0] + shape[2]

        moved = n_dec - n_single
        assert rows_run(n_dec, sum(counts) - moved) <= rows_run(n_single, sum(counts))
        assert moved == 0 or rows_run(n_dec, sum(counts) - moved) < rows_run(n_single, sum(counts))


def test_512_tokens_are_512_rows():
    for n_single in (1, 2, 3, 5, 12, 23, 33, 60):
        layout, tokens, wanted = step_of(random.Random(1), n_single, [512 - n_single])
        filled, _, _ = ModelRunner._spare_rows_filled(layout, tokens, wanted)
        n_dec = sum(c == 1 for c in filled.counts)
        shape = ModelRunner._step_shape(n_dec, 1, 512 - n_dec, 1, 1)
        assert shape[0] + shape[2] == 512
