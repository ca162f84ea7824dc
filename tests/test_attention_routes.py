"""Which launches a step's attention becomes: rules by sizes alone (no GPU)."""
import pytest


def step_in_one(nh, nkv, d, n_decode, n_portions, max_new, window=0, splits=1, waves=8, counters=1 << 14, prompt_splits=1):
    from llmserve.ops import library

    return library.load("attention_mfma").llms_attention_mfma_step_in_one(nh, nkv, d, window, n_decode, splits, waves, counters, n_portions,
                                                                           max_new, prompt_splits)


@pytest.mark.parametrize("way,args,options", [
    (2, (32, 4, 64, 8, 1, 2048), {}), (1, (32, 4, 64, 8, 1, 512), {}), (2, (64, 8, 128, 1, 1, 512), {}), (1, (32, 4, 16, 1, 1, 600), dict(splits=16)),
    (0, (32, 4, 64, 8, 1, 16), {}),                                                                    # no twins for so few workgroups
    (0, (32, 4, 64, 8, 1, 2048), dict(window=90)), (0, (32, 4, 144, 8, 1, 2048), {}), (0, (32, 4, 64, 8, 1, 2048), dict(waves=4)),
    (0, (32, 4, 64, 8, 1, 2048), dict(splits=17)), (0, (32, 4, 64, 8, 1, 2048), dict(splits=4, counters=0)),
    (2, (32, 4, 64, 8, 1, 2048), dict(counters=0)), (0, (32, 4, 64, 8, 1, 2048), dict(prompt_splits=2)),
    (2, (32, 4, 64, 64, 1, 2048), dict(splits=4, counters=256)), (0, (32, 4, 64, 65, 1, 2048), dict(splits=4, counters=256))])
def test_single_tokens_and_portions_in_one_launch(way, args, options):
    """Column groups a wave of the portions, or 0: two launches."""
    assert step_in_one(*args, **options) == way


def test_one_launch_has_fewer_threads_than_a_dimension_takes():
    """It counts workgroups of 512 threads in one dimension, which holds 2^32 - 1 threads; the portions' own launch has three.  A step of one
    long portion among a thousand short ones has a place in the launch for each of all their blocks."""
    blocks = 65536 // 128  # 128 tokens a block: 4 waves with two groups of 16 tokens
    portions = (1 << 23) // (32 * blocks)
    assert step_in_one(32, 32, 64, 1, portions - 1, 65536) == 2
    assert step_in_one(32, 32, 64, 1, portions, 65536) == 0
    assert step_in_one(32, 32, 64, 32 * blocks // 32 - 1, portions - 1, 65536) == 2
    assert step_in_one(32, 32, 64, 32 * blocks // 32, portions - 1, 65536) == 0
