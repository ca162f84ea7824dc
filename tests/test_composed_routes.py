"""Which kernel of the composed attention a step's requests go to (a rule on sizes alone; no GPU)."""
from types import SimpleNamespace

import pytest

from llmserve.ops import library as ops
from llmserve.parts.attention_composed import ComposedAttention


def route(monkeypatch, heads, kv, new, context, n=1, n_dec=0, chunk=None, talking=True, maps=1, dk=64, dv=32, **params):
    """(kernel, first request, requests, most new tokens, shares) of every launch."""
    calls = []
    for name in ("attend_composed_wide", "attend_composed_mfma"):
        monkeypatch.setattr(ops, name, lambda *a, name=name, **kw: calls.append((name, *a[7:10], kw.get("shares"))))
    for name in ("attend_composed_wide_supported", "attend_composed_mfma_supported"):
        monkeypatch.setattr(ops, name, lambda *a: True)
    monkeypatch.setattr(ops, "compute_units", lambda device: 256)
    monkeypatch.setattr(ops, "attend_composed_mfma_tokens", lambda *a: 16)
    part = ComposedAttention({"hidden": 64, "num_heads": heads, "num_kv_heads": kv, "head_dim": dk, "value_dim": dv, "chunk": chunk,
                              "talking_heads": talking, "differential": maps == 2, **params}, None)
    batch = SimpleNamespace(num_decode=n_dec, num_seqs=n + n_dec, max_count=new, max_context=context, max_decode_context=context,
                            state_slots=None, cu_seqlens=None, context_lens=None, num_tokens=n * new + n_dec)
    part.attend(None, SimpleNamespace(dtype=None, device=None), SimpleNamespace(k_pool=None, v_pool=None, block_size=16),
                SimpleNamespace(block_tables=None), batch)
    return calls


@pytest.mark.parametrize("heads,kv,new,context,chunk,dv,kernel", [
    (8, 8, 8, 4000, None, 32, "mfma"), (8, 8, 16, 16000, None, 32, "mfma"), (16, 8, 8, 4000, None, 32, "mfma"),
    (4, 4, 8, 4000, None, 64, "mfma"), (16, 4, 2, 4000, None, 64, "mfma"),
    (8, 8, 8, 1000, None, 32, "wide"),      # few keys
    (8, 8, 8, 4000, 1024, 32, "wide"),      # (its own chunk's)
    (8, 8, 32, 4000, None, 32, "wide"),     # more than one unit of columns
    (16, 8, 16, 4000, None, 32, "wide"),
    (64, 8, 2, 4000, None, 32, "wide"),     # many heads to mix
    (4, 2, 8, 16000, None, 64, "wide"),     # few key/value heads
])
def test_short_portions_behind_many_keys_share_them(heads, kv, new, context, chunk, dv, kernel, monkeypatch):
    (call,) = route(monkeypatch, heads, kv, new, context, chunk=chunk, dv=dv)
    assert call[:4] == (f"attend_composed_{kernel}", 0, 1, new)
    assert kernel == "wide" or call[4] == 4


def test_single_tokens_beside_them_do_not_change(monkeypatch):
    decode, portion = route(monkeypatch, 8, 8, 8, 4000, n=2, n_dec=3)
    assert decode[:4] == ("attend_composed_wide", 0, 3, 1) and portion[:4] == ("attend_composed_mfma", 3, 2, 8)


@pytest.mark.parametrize("heads,kv,maps,dk,new,context,params,kernel", [
    (16, 4, 1, 64, 4, 1000, {}, "mfma"), (8, 8, 1, 64, 16, 500, {}, "mfma"), (8, 8, 1, 64, 16, 4000, {"window": 512}, "mfma"),
    (32, 8, 1, 128, 4, 4000, {}, "mfma"), (4, 4, 2, 64, 16, 4000, {}, "mfma"),
    (16, 4, 1, 64, 4, 300, {}, "wide"),     # few keys
    (16, 4, 1, 64, 4, 4000, {"chunk": 256}, "wide"), (16, 4, 1, 64, 4, 4000, {"window": 100}, "wide"),
    (16, 4, 1, 64, 5, 4000, {}, "wide"),    # more than one unit of columns
    (32, 8, 1, 128, 4, 800, {}, "wide"), (4, 4, 2, 64, 16, 1000, {}, "wide"), (8, 8, 2, 128, 8, 16000, {}, "wide"),
])
def test_without_mixing_too(heads, kv, maps, dk, new, context, params, kernel, monkeypatch):
    (call,) = route(monkeypatch, heads, kv, new, context, talking=False, maps=maps, dk=dk, dv=64, distance_slope_base=8, **params)
    assert call[:4] == (f"attend_composed_{kernel}", 0, 1, new)


def test_nothing_but_single_tokens_is_one_launch(monkeypatch):
    (call,) = route(monkeypatch, 8, 8, 1, 4000, n=0, n_dec=5)
    assert call[:4] == ("attend_composed_wide", 0, 5, 1)


@pytest.mark.parametrize("heads,kv,dk,dv,maps,counts,one,two", [  # microseconds with one unit a wave and with two
    (8, 4, 128, 128, 2, [512], 17.6, 25.4), (8, 4, 128, 128, 2, [1000], 39.1, 43.8), (8, 4, 128, 128, 2, [2048], 144.5, 98.6),
    (8, 4, 128, 128, 2, [512] * 4, 42.0, 31.8), (8, 4, 128, 128, 2, [256] * 8, 25.2, 20.4), (8, 4, 128, 128, 2, [128] * 16, 16.3, 13.8),
    (8, 2, 128, 64, 2, [1100], 39.9, 43.7), (8, 2, 128, 64, 2, [2048], 105.0, 89.3), (8, 2, 128, 64, 2, [256] * 8, 19.9, 18.0),
    (32, 8, 128, 128, 1, [512], 22.3, 24.8), (32, 8, 128, 128, 1, [850], 44.8, 39.0), (32, 8, 128, 128, 1, [128] * 16, 26.2, 21.5),
    (16, 2, 64, 128, 2, [1100], 44.7, 53.1), (16, 2, 64, 128, 2, [1500], 70.6, 67.3), (16, 2, 64, 128, 2, [811, 890, 150, 197], 53.8, 43.0),
    (16, 4, 64, 64, 2, [1100], 41.6, 47.2), (16, 4, 64, 64, 2, [700, 700], 33.0, 31.5), (16, 4, 64, 64, 2, [1500], 62.8, 57.3),
    (8, 8, 64, 64, 2, [2048], 75.1, 82.5), (8, 8, 64, 64, 2, [512] * 4, 23.6, 26.3), (8, 8, 64, 64, 2, [3000], 121.3, 113.7),
    (16, 4, 64, 64, 1, [2048], 64.9, 70.1), (16, 8, 64, 64, 1, [2048], 75.1, 70.1), (16, 8, 64, 64, 1, [1500], 38.3, 52.1),
    (32, 4, 64, 128, 1, [850], 29.6, 36.3), (32, 4, 64, 128, 1, [1500], 73.5, 67.7), (32, 2, 128, 64, 1, [1000], 47.8, 40.9)])
def test_units_of_a_wave_over_portions(heads, kv, dk, dv, maps, counts, one, two):
    """As many columns a wave as is the faster: a line by the waves, the keys' length and the maps."""
    from llmserve.ops.library import wide_prompt_units

    assert wide_prompt_units(heads, kv, dk, dv, maps, False, len(counts), max(counts), sum(counts)) == (1 if one < two else 2)
    assert wide_prompt_units(heads, kv, dk, dv, maps, True, len(counts), max(counts), sum(counts)) == 1
