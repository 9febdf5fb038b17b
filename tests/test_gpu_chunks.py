"""Attention chunks of the batch-1 decode: one engine of a large capacity at
contexts around the edges of a 64-position block and of the last context whose
chunks are single blocks (16 x 64 = 1,024). The resident kernel and the stream
kernels agree bit for bit, and both match the oracle."""
import os

import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

LAYERS, VOCAB, CAPACITY, STEPS = 2, 1024, 1536, 3


@pytest.fixture(scope="module")
def pair():
    res = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=CAPACITY)
    os.environ["QD_RESIDENT"] = "0"
    try:
        stream = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=CAPACITY)
    finally:
        del os.environ["QD_RESIDENT"]
    model = qo.Model(qo.ModelShape(layers=LAYERS, vocab=VOCAB))
    model.fill_synthetic(6)
    for eng in (res, stream):
        eng.load_synthetic(6)
    yield res, stream, model
    res.close()
    stream.close()
    model.close()


@pytest.mark.parametrize("context", [0, 1, 62, 63, 127, 700, 959, 1022, 1023, 1039, 1279])
def test_resident_stream_and_oracle_agree(pair, context):
    print(f"decode chunks at context {context}", flush=True)
    res, stream, model = pair
    assert res.resident_grid() > 0 and stream.resident_grid() == 0
    cache = qo.Cache(model, CAPACITY)
    for layer in range(LAYERS):
        k = qo.fill_normal(max(context, 1) * 128, 9, 0x500000 + 2 * layer, 0.0, 1.0).reshape(-1, 128)[:context]
        v = qo.fill_normal(max(context, 1) * 128, 9, 0x500001 + 2 * layer, 0.0, 1.0).reshape(-1, 128)[:context]
        for eng in (res, stream):
            if context:
                eng.write_kv(0, layer, 0, k, v)
        cache.layer(layer, False)[:context] = k
        cache.layer(layer, True)[:context] = v
    for eng in (res, stream):
        eng.kv_reset(0, context)
    toks, _, logits = res.generate(0, 17, STEPS, want_logits=True)
    toks2, _, logits2 = stream.generate(0, 17, STEPS, want_logits=True)
    assert toks.tolist() == toks2.tolist()
    assert np.array_equal(logits, logits2)
    res.kv_reset(0, context)
    assert np.array_equal(res.step(0, 17)[2], logits[0])
    feed = 17
    for i, t in enumerate(toks.tolist()):
        _, _, ref = cache.decode_step(feed, context + i)
        # The FP32 bar of the other oracle tests.
        assert np.abs(logits[i] - ref).max() <= 1e-4 * np.abs(ref).max(), i
        feed = t
    cache.close()


@pytest.mark.parametrize("first,count", [(0, 2), (0, 3), (2, 3), (0, 6), (5, 1)])
@pytest.mark.parametrize("keys", [1, 64, 1024, 1025])
def test_layer_ranges_agree(first, count, keys):
    """A range of layers by one layers-only resident launch (from three layers
    on) and by the stream kernels: the hidden vector, the last layer's query,
    attention output and activation, the K/V rows, then the tail."""
    print(f"layers [{first}, {first + count}) at {keys} keys", flush=True)
    engines = []
    for resident in ("1", "0"):
        os.environ["QD_RESIDENT"] = resident
        try:
            engines.append(qd.Engine(layers=6, vocab=VOCAB, capacity=1100, max_batch=2))
        finally:
            del os.environ["QD_RESIDENT"]
    h = qo.fill_normal(896, 4, 0x600000, 0.0, 1.0)
    got = []
    for eng in engines:
        eng.load_synthetic(8)
        for layer in range(first, first + count):
            k = qo.fill_normal(keys * 128, 9, 0x500000 + 2 * layer, 0.0, 1.0).reshape(-1, 128)
            v = qo.fill_normal(keys * 128, 9, 0x500001 + 2 * layer, 0.0, 1.0).reshape(-1, 128)
            eng.write_kv(1, layer, 0, k, v)
        eng.load_hidden(1, h)
        eng.layer_decode(1, first, count, keys)
        out = [eng.read_activation(1, which) for which in range(4)]
        for layer in range(first, first + count):
            out += eng.read_kv(1, layer, 0, keys)
        token, _, logits = eng.tail(1)
        state = eng.decode_state(1)
        got.append(out + [logits, np.array([token, state.token_position, state.generated_tokens, state.stop_reason])])
        eng.close()
    assert all(np.array_equal(a, b) for a, b in zip(*got))


def test_failed_layers_launch_surfaces_at_the_next_call_that_waits():
    print("layers-only launch with a spin limit of 1", flush=True)
    os.environ["QD_RESIDENT_SPIN_LIMIT"] = "1"
    try:
        eng = qd.Engine(layers=6, vocab=VOCAB, capacity=64)
    finally:
        del os.environ["QD_RESIDENT_SPIN_LIMIT"]
    eng.load_synthetic(8)
    eng.load_hidden(0, np.ones(896, np.float32))
    eng.layer_decode(0, 0, 6, 1)
    eng.layer_decode(0, 0, 2, 1)  # stream kernels: the error of the launch before stays
    with pytest.raises(qd.QdError) as err:
        eng.sync()
    assert err.value.status == qd.DEVICE_FAULT
    eng.sync()
    eng.load_hidden(0, np.ones(896, np.float32))
    eng.layer_decode(0, 0, 2, 1)
    assert np.isfinite(eng.read_activation(0, 0)).all()
    eng.close()
