"""What a step of portions beside single tokens is padded to, and which of its tokens fill the places of single tokens (no GPU)."""

import random

import pytest
import torch

from llmserve.cache.manager import StepLayout
from llmserve.engine.runner import ModelRunner


def step_of(n_single, counts, start=0):
    counts = [1] * n_single + counts
    total = sum(counts)
    layout = StepLayout(seq_ids=[f"r{i}" for i in range(len(counts))], counts=counts, starts=[start] * len(counts), state_slots=list(range(len(counts))),
                        fresh_slots=[], slots={0: list(range(total))}, table_updates={0: []})
    return layout, [list(range(c)) for c in counts], [total - 1]


def moved(n_single, counts, start=0, **kw):
    filled, _, _ = ModelRunner._spare_rows_filled(*step_of(n_single, counts, start), **kw)
    return next(i for i, c in enumerate(filled.counts) if c != 1) - n_single


@pytest.mark.parametrize("n_single,portion,want", [
    (3, 509, 1), (33, 479, 31),  # 512 tokens: all spare places, to 512 rows
    (33, 467, 19), (40, 460, 12), (33, 450, 2),  # fewer tokens: as few as get the step to 512 rows
    (33, 400, 0), (9, 131, 0), (5, 195, 0), (33, 667, 0),  # no line between the rows without and with
    (65, 368, 0), (65, 447, 63), (3, 1021, 1)])
def test_as_few_tokens_as_get_a_step_under_a_line(n_single, portion, want):
    assert moved(n_single, [portion]) == want
    assert moved(n_single, [portion], pays=lambda tokens, start: False) == 0
    seen = []
    moved(n_single, [portion], 700, pays=lambda tokens, start: seen.append((tokens, start)) or True)
    assert seen == ([(want, 700)] if want else [])


def runner(key_bytes, elements):
    r = ModelRunner.__new__(ModelRunner)
    r._key_bytes, r._elements_per_token = key_bytes, elements
    return r


def test_keys_read_alone_are_weighed():
    """One layer of the 1.1B shape, of the 7B shape, and of a small one whose query heads all have keys of their own."""
    small = runner(4 * 4 * 64, 44e6)
    assert small._keys_alone_pay(1, 30000) and small._keys_alone_pay(31, 1500) and small._keys_alone_pay(58, 900) and not small._keys_alone_pay(63, 1500)
    large = runner(4 * 32 * 128, 202e6)
    assert large._keys_alone_pay(3, 1500) and large._keys_alone_pay(15, 1500) and not large._keys_alone_pay(31, 1500)
    assert not runner(4 * 16 * 64, 12e6)._keys_alone_pay(15, 1500)


def test_which_models_steps_are_filled():
    """Those of plain attention in every layer: latent and composed attention and layers with a state take single tokens dearly or not at all."""
    from llmserve.config import preset
    from llmserve.config.registry import architecture_of
    from llmserve.parts.model import Model
    from llmserve.parts.registry import BuildContext

    for name, may in (("tinyllama-1.1b", True), ("llama2-7b", True), ("milozen-1b", False), ("zotunex-1b", False), ("dibepel-1b", False),
                      ("ramolix-1b", False), ("felavik-1b", False), ("nolavik-1b", False)):
        cfg = dict(preset(name))
        arch = architecture_of(cfg)
        model = Model(arch.build_spec(arch.config_class.from_dict(cfg)), BuildContext(torch.bfloat16, torch.device("cpu")))
        assert all(block.mixer.takes_tokens_of_portions for block in model.blocks) == may


def test_portions_have_few_sizes():
    """Beside any number of single tokens the rows of portions are `_row_bucket`'s, but for the one size that ends at a line."""
    rng = random.Random(5)
    for n_single in (0, 1, 3, 9, 20, 33, 60, 100):
        decode = 1 << (n_single - 1).bit_length() if n_single else 0
        for tokens in {2, 511, 512, 513, 1024} | {rng.randrange(2, 1100) for _ in range(300)}:
            rows = ModelRunner._step_shape(n_single, 1, tokens, 1, 1)[2]
            alone = ModelRunner._row_bucket(tokens)
            assert tokens <= rows <= alone and (rows == alone or (decode + rows) % 512 == 0)
            assert (decode + rows - 1) // 512 == (decode + tokens - 1) // 512 or rows == alone
