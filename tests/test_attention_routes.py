"""Which launches a step's attention becomes: rules by sizes alone (no GPU)."""
import pytest
import torch


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


@pytest.mark.parametrize("nkv,g,d,n,keys,micros", [  # microseconds by workgroups a request
    (4, 8, 64, 8, 900, {1: 8.7, 4: 7.9}), (8, 2, 80, 4, 640, {1: 7.2, 4: 8.2}), (8, 2, 80, 8, 900, {1: 12.5, 4: 10.9}),
    (8, 2, 96, 4, 520, {1: 7.5, 4: 8.2}), (8, 2, 96, 4, 900, {1: 11.3, 4: 9.3}), (8, 2, 112, 8, 760, {1: 13.8, 4: 12.0}),
    (8, 4, 128, 4, 520, {1: 9.8, 4: 9.3}), (8, 4, 128, 8, 900, {1: 17.1, 4: 13.3}),
    (4, 4, 64, 1, 16000, {4: 30.0, 8: 19.3, 16: 15.2}), (8, 4, 64, 1, 8000, {4: 18.6, 8: 13.7, 16: 12.9}),
    (8, 4, 64, 2, 8000, {4: 19.8, 8: 15.7, 16: 16.6}), (4, 4, 64, 4, 8000, {4: 19.5, 8: 15.6, 16: 16.5}),
    (8, 4, 64, 4, 8000, {4: 21.6, 8: 19.4, 16: 26.0}), (4, 8, 64, 32, 580, {1: 8.5, 2: 8.6}), (4, 8, 64, 20, 800, {1: 9.3, 3: 10.1}),
    (2, 4, 64, 4, 16000, {4: 30.5, 8: 20.2, 16: 17.0})])
def test_workgroups_that_share_a_requests_keys(nkv, g, d, n, keys, micros):
    from llmserve.parts.attention import decode_arrangement

    shares, waves = decode_arrangement(g * nkv, nkv, d, None, n, keys)
    assert waves == 8 and micros[shares] <= 1.03 * min(micros.values())


def test_the_kernel_shares_keys_out_from_the_line_of_the_rule():
    """The rule's line in tiles of 32 keys a wave is the kernel's too, so that what is planned for one workgroup is not shared out by a longer
    request beside it (`alone` in attn_decode, the same in a launch with portions beside it: the bits are tested on the GPU)."""
    from llmserve.parts.attention import decode_arrangement

    for d, tiles in ((16, 3), (64, 3), (80, 3), (96, 3), (112, 2), (128, 2)):
        assert decode_arrangement(8, 2, d, None, 2, 32 * 8 * tiles) == (1, 8)
        assert decode_arrangement(8, 2, d, None, 2, 32 * 8 * tiles + 1) == (4, 8)


def test_counters_made_inside_a_step_can_be_zeroed_outside_one(monkeypatch):
    """A step runs in inference mode, and the first one whose attention shares keys out makes the counters; a runner that is built later
    zeroes them, outside."""
    from llmserve.ops import library

    monkeypatch.setattr(library, "_ARRIVAL_COUNTERS", {})
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with torch.inference_mode():
        counters = library._arrival_counters(torch.device("cpu"))
        counters[3] = 7
    library.reset_arrival_counters()
    assert library.arrival_counters_are_zero() and int(counters.sum()) == 0
