"""Prompts of one and two tokens run as layers-only resident launches, one after
the other without a wait between them: each storage type, at the start, over a
cache, across the context whose attention chunks change and at the capacity,
bit for bit against a step per token on the stream kernels. And the layer
counts around which a range of layers changes kernels."""
import os

import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

LAYERS, VOCAB, CAPACITY = 4, 1024, 1100


@pytest.fixture(scope="module", params=["f32", "bf16", "f16"])
def pair(request):
    engines = []
    for resident in ("1", "0"):
        os.environ["QD_RESIDENT"] = resident
        try:
            engines.append(qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=CAPACITY, max_batch=2,
                                     decoder_dtype=request.param))
        finally:
            del os.environ["QD_RESIDENT"]
        engines[-1].load_synthetic(8)
    assert engines[0].resident_grid() > 0 and engines[1].resident_grid() == 0
    yield engines
    for eng in engines:
        eng.close()


def fill_cache(engines, slot, rows):
    for layer in range(LAYERS):
        k, v = (qo.fill_normal(max(rows, 1) * 128, 9, 0x500000 + 2 * layer + i, 0.0, 1.0).reshape(-1, 128)[:rows]
                for i in range(2))
        for eng in engines:
            if rows:
                eng.write_kv(slot, layer, 0, k, v)


def all_equal(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("start", [0, 1, 62, 63, 1022, 1023, CAPACITY - 2])
@pytest.mark.parametrize("rows", [1, 2])
def test_short_prompt_equals_steps(pair, start, rows):
    print(f"prompt of {rows} at {start}, {pair[0].config.decoder_dtype}", flush=True)
    res, stream = pair
    fill_cache(pair, 1, start)
    tokens = qo.fill_tokens(rows, 5, 0x300000, VOCAB)
    for eng in pair:
        eng.kv_reset(1, start)
    token, _, logits = res.prefill(1, tokens)
    for t in tokens.tolist():
        want_token, _, want = stream.step(1, t)
    assert token == want_token and np.array_equal(logits, want)
    for layer in range(LAYERS):
        assert all_equal(res.read_kv(1, layer, start, rows), stream.read_kv(1, layer, start, rows)), layer
    assert res.decode_state(1).token_position == start + rows


@pytest.mark.parametrize("count", [2, 3, 4])
@pytest.mark.parametrize("keys", [1, 64, 65])
def test_layer_ranges_agree(pair, count, keys):
    print(f"{count} layers at {keys} keys, {pair[0].config.decoder_dtype}", flush=True)
    fill_cache(pair, 0, keys)
    got = []
    for eng in pair:
        eng.load_hidden(0, qo.fill_normal(896, 4, 0x600000, 0.0, 1.0))
        eng.layer_decode(0, LAYERS - count, count, keys)
        got.append([eng.read_activation(0, which) for which in range(4)] + list(eng.read_kv(0, LAYERS - 1, 0, keys)))
    assert all_equal(*got)
