"""Batched steps at the edges of the row tile and of the LM head's share per
wave (vocabularies of fewer tiles than waves, of one tile more, ragged), against
the oracle."""
import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

LAYERS, CAPACITY, SLOTS = 2, 48, 16
WAVES = 256 * 8  # of the LM head; one 16-row vocabulary tile each at a time
# Largest difference over the largest value. Sums of up to 4,864 FP32 products
# rounded in any order: about sqrt(4864) 2^-24 = 4e-6.
RTOL = 1e-5


def rel_err(a, b):
    return float(np.abs(a.astype(np.float64) - b).max() / np.abs(b).max())


@pytest.fixture(scope="module", params=[16, 1003, 16 * WAVES - 1, 16 * WAVES + 5])
def pair(request):
    eng = qd.Engine(layers=LAYERS, vocab=request.param, capacity=CAPACITY, max_batch=SLOTS)
    eng.load_synthetic(3)
    model = qo.Model(qo.ModelShape(layers=LAYERS, vocab=request.param))
    model.fill_synthetic(3)
    prompts = [qo.fill_tokens(1 + (7 * s) % 41, 3, 0x500000 + s, request.param) for s in range(SLOTS)]
    # The oracle's step of each slot's last token over the rows before it.
    want = []
    for p in prompts:
        cache = qo.Cache(model, CAPACITY)
        if len(p) > 1:
            cache.prefill(p[:-1], want_logits=False)
        tok, _, logits = cache.decode_step(int(p[-1]), len(p) - 1)
        want.append((logits, cache.layer(LAYERS - 1, False)[len(p) - 1].copy(), cache.layer(LAYERS - 1, True)[len(p) - 1].copy()))
        cache.close()
    yield eng, prompts, want
    eng.close()
    model.close()


@pytest.mark.parametrize("rows", [1, 2, 7, 15, 16])
def test_batch_rows_match_oracle(pair, rows):
    eng, prompts, want = pair
    print(f"batch of {rows}, vocabulary {eng.config.vocab}", flush=True)
    slots = [(5 * i + rows) % SLOTS for i in range(rows)]  # not in slot order
    for s in slots:
        eng.kv_reset(s, 0)
        if len(prompts[s]) > 1:
            eng.prefill(s, prompts[s][:-1], want_logits=False)
    greedy, logits = eng.step_batch(slots, [int(prompts[s][-1]) for s in slots])
    for i, s in enumerate(slots):
        ref, k, v = want[s]
        assert rel_err(logits[i], ref) <= RTOL
        assert int(greedy[i]) == int(np.argmax(logits[i]))
        gk, gv = eng.read_kv(s, LAYERS - 1, len(prompts[s]) - 1, 1)
        assert rel_err(gk[0], k) <= RTOL and rel_err(gv[0], v) <= RTOL


def test_batch_attention_chunk_edges():
    """Contexts at the edges of a wave's 16 positions, a chunk's 128 and the
    longest split into chunks of 128 (2,048), each against the batch-1 step."""
    lengths = [1, 15, 16, 17, 127, 128, 129, 143, 144, 255, 257, 1025, 2047, 2048, 2049, 2299]
    eng = qd.Engine(layers=LAYERS, vocab=1003, capacity=2300, max_batch=len(lengths))
    eng.load_synthetic(3)
    prompt = qo.fill_tokens(2300, 3, 0x600000, 1003)
    slots = list(range(len(lengths)))
    for s, n in zip(slots, lengths):
        eng.kv_reset(s, 0)
        eng.prefill(s, prompt[:n], want_logits=False)
    print("batch over", lengths, flush=True)
    _, logits = eng.step_batch(slots, [int(prompt[n]) for n in lengths])
    for s, n in zip(slots, lengths):
        eng.kv_reset(s, n)
        _, _, single = eng.step(s, int(prompt[n]))
        assert rel_err(logits[s], single) <= RTOL, n
    eng.close()
