"""The prompt GEMMs at the edges of their tile shapes (32, 64 and 128 rows, one
row more and less, chunks of 2,048 rows) for each storage type of the decoder
matrices, against the oracle, and their values outside the BF16 range."""
import os

import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

LAYERS, VOCAB, LONGEST = 2, 1024, 2090
MATRICES = (2, 3, 4, 8, 9, 10, 11)
SIZES = [896, 896, 896 * 896, 128 * 896, 128 * 896, 896, 128, 128, 896 * 896, 4864 * 896, 4864 * 896, 896 * 4864]
# Largest difference over the largest value. Sums of up to 4,864 FP32 products
# rounded in any order: about sqrt(4864) 2^-24 = 4e-6.
RTOL = 1e-5


def bf16_round(x):
    u = x.view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


ROUND = {"f32": lambda x: x, "bf16": bf16_round, "f16": lambda x: x.astype(np.float16).astype(np.float32)}


def rel_err(a, b):
    return float(np.abs(a.astype(np.float64) - b).max() / np.abs(b).max())


@pytest.fixture(scope="module", params=["f32", "bf16", "f16"])
def pair(request):
    """An engine of one storage type and the K/V rows of the oracle on its weights."""
    eng = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=LONGEST, decoder_dtype=request.param)
    eng.load_synthetic(3)
    model = qo.Model(qo.ModelShape(layers=LAYERS, vocab=VOCAB))
    model.fill_synthetic(3)
    for layer in range(LAYERS):
        for kind in MATRICES:
            t = model.tensor(layer, kind)
            t[:] = ROUND[request.param](np.ascontiguousarray(t).reshape(-1)).reshape(t.shape)
    prompt = qo.fill_tokens(LONGEST, 3, 0x300000, VOCAB)
    cache = qo.Cache(model, LONGEST)
    cache.prefill(prompt, want_logits=False)
    yield eng, prompt, cache
    eng.close()
    cache.close()
    model.close()


@pytest.mark.parametrize("rows", [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 511, 1024, 1025, 2047, 2048, 2049, LONGEST])
def test_rows_match_oracle(pair, rows):
    eng, prompt, cache = pair
    print(f"prefill {eng.config.decoder_dtype} {rows} rows", flush=True)
    eng.kv_reset(0, 0)
    eng.prefill(0, prompt[:rows], want_logits=False)
    # The last layer's K/V rows depend on all of the layer before.
    k, v = eng.read_kv(0, LAYERS - 1, 0, rows)
    assert rel_err(k, cache.layer(LAYERS - 1, False)[:rows]) <= RTOL
    assert rel_err(v, cache.layer(LAYERS - 1, True)[:rows]) <= RTOL


@pytest.mark.parametrize("rows", [192, 193, 256, 288, 289, 385, 481, 576, 577])
def test_rows_match_oracle_at_the_96_row_tiles(pair, rows):
    test_rows_match_oracle(pair, rows)


@pytest.mark.parametrize("rows", [1, 2, 33, 513, 2048, 2049, LONGEST])
def test_last_row_matches_a_step_after_the_rows_before(pair, rows):
    """The last layer runs for the prompt's last row alone."""
    eng, prompt, _ = pair
    print(f"prefill {eng.config.decoder_dtype} {rows} rows, last row", flush=True)
    eng.kv_reset(0, 0)
    _, _, logits = eng.prefill(0, prompt[:rows])
    eng.kv_reset(0, rows - 1)
    _, _, step = eng.step(0, int(prompt[rows - 1]))
    assert rel_err(logits, step) <= RTOL


def write_bundle(directory, layers, tail):
    for i, tensors in enumerate(layers):
        d = os.path.join(directory, f"layer_{i}")
        os.makedirs(d)
        qd.bundle_write_layer(os.path.join(d, "weights.json"), "weights.bin", [64, 896, 14, 2, 64, 4864], 1e6,
                              np.concatenate(tensors))
    os.makedirs(os.path.join(directory, "model_tail"))
    emb, norm = tail
    qd.bundle_write_tail(os.path.join(directory, "model_tail", "weights.json"), "weights.bin", 896, VOCAB,
                         np.arange(VOCAB), emb, norm, emb)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_narrow_prefill_equals_fp32_prefill_of_the_rounded_weights(dtype, tmp_path):
    print(f"{dtype} prefill against an FP32 engine on the rounded weights", flush=True)
    e16 = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=256, decoder_dtype=dtype)
    e32 = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=256)
    e16.load_synthetic(3)
    layers = [[e16.read_weight(layer, k, n) for k, n in enumerate(SIZES)] for layer in range(LAYERS)]
    write_bundle(str(tmp_path), layers, (e16.read_weight(0, qd.EMBED, VOCAB * 896), e16.read_weight(0, qd.FINAL_NORM, 896)))
    e32.load_bundle(str(tmp_path))
    for rows in (20, 200):
        prompt = qo.fill_tokens(rows, 5, 0x300000, VOCAB)
        got = []
        for eng in (e16, e32):
            eng.kv_reset(0, 0)
            logits = eng.prefill(0, prompt)[2]
            got.append((logits, *eng.read_kv(0, LAYERS - 1, 0, rows)))
        assert all(np.array_equal(a, b) for a, b in zip(*got)), rows
    e16.close()
    e32.close()


@pytest.mark.parametrize("value", [3.395e38, np.inf])
def test_weights_beyond_bf16_range_give_fp32_results(value, tmp_path):
    """A finite weight that rounds to infinity in BF16, and an infinite one:
    the prompt path gives what the step kernels' FP32 arithmetic gives."""
    print(f"prefill with an up weight of {value}", flush=True)
    layers = [[qo.fill_normal(n, 11 + i, 0x400000 + j, 0.0, 0.02) for j, n in enumerate(SIZES)] for i in range(LAYERS)]
    for t in layers:
        t[0][:] = 1.0
        t[1][:] = 1.0
    # Layer 0: activation 7 becomes about 1e36, its down weights bring it back.
    layers[0][1][5] = 0.01
    layers[0][10][7 * 896 + 5] = value
    layers[0][11].reshape(896, 4864)[:, 7] = 1e-36
    write_bundle(str(tmp_path), layers, (qo.fill_normal(VOCAB * 896, 13, 0x7FFF00, 0.0, 0.02), np.ones(896, np.float32)))
    eng = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=64, max_batch=2)
    eng.load_bundle(str(tmp_path))
    prompt = qo.fill_tokens(40, 5, 0x300000, VOCAB)
    eng.kv_reset(0, 0)
    eng.kv_reset(1, 0)
    got = eng.prefill(0, prompt)[2]
    for t in prompt.tolist():
        want = eng.step(1, t)[2]
    k0, k1 = eng.read_kv(0, 1, 0, 40)[0], eng.read_kv(1, 1, 0, 40)[0]
    eng.close()
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and np.array_equal(np.isfinite(k0), np.isfinite(k1))
    assert np.isfinite(want).all() == np.isfinite(value)
    if np.isfinite(value):
        assert rel_err(k0, k1) <= RTOL and rel_err(got, want) <= RTOL


@pytest.mark.parametrize("start,rows", [(1, 1), (15, 17), (47, 17), (63, 2), (64, 64), (100, 16), (1000, 37), (1500, 590)])
def test_continued_prompts_match_oracle(pair, start, rows):
    """Row blocks of 16 and key blocks of 64 at positions that are not their
    multiples, with one and with several key splits per row block."""
    eng, prompt, cache = pair
    print(f"prefill {eng.config.decoder_dtype} {start} + {rows} rows", flush=True)
    eng.kv_reset(0, 0)
    eng.prefill(0, prompt[:start], want_logits=False)
    eng.prefill(0, prompt[start:start + rows], want_logits=False)
    k, v = eng.read_kv(0, LAYERS - 1, start, rows)
    assert rel_err(k, cache.layer(LAYERS - 1, False)[start:start + rows]) <= RTOL
    assert rel_err(v, cache.layer(LAYERS - 1, True)[start:start + rows]) <= RTOL


@pytest.mark.parametrize("k_value,v_value", [(3.395e38, 1.0), (-np.inf, 1.0), (np.inf, 1.0), (1.0, 3.395e38), (1.0, np.inf)])
def test_cache_rows_beyond_bf16_range_give_fp32_results(k_value, v_value):
    """Cached K / V values that round to infinity in BF16 or are infinite:
    attention gives what the step kernels' FP32 arithmetic gives."""
    print(f"prefill over cached K {k_value}, V {v_value}", flush=True)
    eng = qd.Engine(layers=LAYERS, vocab=VOCAB, capacity=128, max_batch=2)
    eng.load_synthetic(3)
    k = qo.fill_normal(80 * 128, 3, 0x200000, 0.0, 1.0).reshape(80, 128)
    v = qo.fill_normal(80 * 128, 3, 0x200001, 0.0, 1.0).reshape(80, 128)
    k[70, 3] *= np.float32(k_value)
    v[70, 9] *= np.float32(v_value)
    k[np.abs(k) > 3.4e38] = k_value
    v[np.abs(v) > 3.4e38] = v_value
    for seq in range(2):
        for layer in range(LAYERS):
            eng.write_kv(seq, layer, 0, k, v)
        eng.kv_reset(seq, 80)
    prompt = qo.fill_tokens(20, 5, 0x300000, VOCAB)
    got = eng.prefill(0, prompt)[2]
    for t in prompt.tolist():
        want = eng.step(1, t)[2]
    k0, k1 = (eng.read_kv(seq, 1, 80, 20)[0] for seq in range(2))
    eng.close()
    fine = np.isfinite(k1)
    assert np.array_equal(np.isfinite(k0), fine) and np.array_equal(np.isfinite(got), np.isfinite(want))
    if fine.any():
        assert np.abs(k0[fine] - k1[fine]).max() <= RTOL * np.abs(k1[fine]).max()
