"""What a step of portions beside single tokens is padded to (no GPU)."""

import random

from llmserve.engine.runner import ModelRunner


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
