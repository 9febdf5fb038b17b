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
