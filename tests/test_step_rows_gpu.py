"""A step whose spare places take tokens of a portion gives the rows of the step without: the same sums in another order."""

from dataclasses import replace

import pytest
import torch

pytestmark = pytest.mark.gpu

CONFIG = dict(architectures=["LlamaForCausalLM"], model_type="llama", vocab_size=320, hidden_size=256, intermediate_size=512, num_hidden_layers=3,
              num_attention_heads=8, num_key_value_heads=2, max_position_embeddings=2048, rope_theta=10000.0, rms_norm_eps=1e-5,
              tie_word_embeddings=False)


def runner(dtype, window):
    from llmserve.config import EngineConfig
    from llmserve.config.registry import architecture_of
    from llmserve.engine.runner import ModelRunner
    from llmserve.ops import library as ops
    from llmserve.parts.model import Model
    from llmserve.parts.registry import BuildContext
    from llmserve.weights.random import random_tensors

    arch = architecture_of(CONFIG)
    config, device = arch.config_class.from_dict(CONFIG), torch.device("cuda:0")
    spec = arch.build_spec(config)
    mixers = [replace(layer.mixer, params={**layer.mixer.params, "window": window if i % 2 else None}) for i, layer in enumerate(spec.layers)]
    spec = replace(spec, layers=tuple(replace(layer, parts={**layer.parts, "mixer": mixer}) for layer, mixer in zip(spec.layers, mixers)))
    model = Model(spec, BuildContext({"float32": torch.float32, "bfloat16": torch.bfloat16}[dtype], device))
    ops.ensure_built(dtype, extra=model.libraries(dtype))
    model.load(random_tensors(model.param_infos(), 3, model.ctx.dtype, device))
    made = ModelRunner(model, config, EngineConfig(dtype=dtype, block_size=16, num_blocks=400, max_num_seqs=48, max_num_batched_tokens=2048), device)
    made.storage.poison()
    return made


def run(dtype, window, singles, behind, fill, monkeypatch):
    """Logits of two steps of 512 tokens beside `singles` decoding requests, the second by replay or capture; the rows they ran."""
    from llmserve.engine.runner import ModelRunner, StepEntry

    made = runner(dtype, window)
    made._key_bytes = 1 if fill else 0  # (also in 32-bit, where the engine does not)
    gen = torch.Generator().manual_seed(11)
    ids = lambda n: torch.randint(0, 320, (n,), generator=gen).tolist()  # noqa: E731
    out = []
    for i in range(singles):
        made.add_sequence(i)
        made.step([StepEntry(i, ids(20 + 3 * i), [0])])
    for p in ("p", "o"):
        made.add_sequence(p)
    made.step([StepEntry("p", ids(behind), [0]), StepEntry("o", ids(9), [0])])
    rows = made.rows_run
    for _ in range(2):
        n = 512 - singles - 40
        entries = [StepEntry(i, ids(1), [0]) for i in range(singles)]
        out.append(made.step([StepEntry("o", ids(40), [0, 39]), *entries, StepEntry("p", ids(n), [0, 1, 2, 30, 31, n - 1])]).float().cpu())
        made.manager.check_invariants()
    return torch.cat(out), made.rows_run - rows


@pytest.mark.parametrize("window", [None, 70])
@pytest.mark.parametrize("singles,behind", [(3, 30), (33, 150)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_filled_steps_give_the_same_rows(dtype, singles, behind, window, monkeypatch):
    """32-bit: sums of at most 512 products in another order, through three layers.  bfloat16: a rounding of 2^-9 that falls otherwise, of the
    result of each of some ten roundings a layer; a wrong key, place or page moves a row by its own size."""
    (got, rows), (want, unfilled) = (run(dtype, window, singles, behind, fill, monkeypatch) for fill in (True, False))
    assert rows == 1024 and unfilled > rows
    off = ((got - want).norm(dim=1) / want.norm(dim=1)).max()
    assert float(off) <= (1e-5 if dtype == "float32" else 2 * (3 * 10) ** 0.5 * 2.0 ** -9)
