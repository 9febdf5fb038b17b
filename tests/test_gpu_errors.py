"""Failure handling of the engine on the GPU, forced from the host.

* A resident hand-off wait that exhausts its spin limit ends the launch with
  QD_ERROR_DEVICE_FAULT and a message that says so; every workgroup exits
  (the call returns) and the engine keeps working. The give-up is forced
  with QD_RESIDENT_SPIN_LIMIT=1 at engine creation: waits then give up after
  a few polls, long before any producer publishes.
* A prompt or a batched step whose workspace the device has no room for fails
  and can be tried again (QD_DEVICE_BYTES_LIMIT refuses the allocation); long prompts make do
  with the workspace of a short one.
* NaN payloads never survive a load: K/V rows written through qd_write_kv,
  hidden vectors of qd_load_hidden and qd_layer_step and weights loaded from a
  bundle hold only the canonical NaN 0x7FC00000,
  so a NaN whose bits equal the resident kernel's empty-slot pattern
  (0xFFFFFFFF) cannot stall a hand-off; a NaN model decodes to NaN logits on
  the resident path without waiting.
"""
import os

import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

SMALL = dict(layers=2, vocab=4096, capacity=64, max_batch=1)
CANONICAL = 0x7FC00000


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)


def test_resident_wait_give_up_reports_device_fault(monkeypatch):
    say("resident wait give-up: QD_RESIDENT_SPIN_LIMIT=1")
    monkeypatch.setenv("QD_RESIDENT_SPIN_LIMIT", "1")
    eng = qd.Engine(**SMALL)
    monkeypatch.delenv("QD_RESIDENT_SPIN_LIMIT")
    ref = qd.Engine(**SMALL)
    try:
        assert eng.resident_grid() > 0
        for e in (eng, ref):
            e.load_synthetic(5)
        prompt = qo.fill_tokens(4, 5, 0x300000, SMALL["vocab"])
        eng.kv_reset(0, 0)
        first, _, _ = eng.prefill(0, prompt, want_logits=False)
        with pytest.raises(qd.QdError) as err:
            eng.generate(0, first, 4)
        assert err.value.status == qd.DEVICE_FAULT
        assert "gave up" in str(err.value)
        # The position did not move, and the device is healthy: a stream step
        # (the graph replay of the step kernels) from the same state equals
        # the step on an untouched engine (the resident kernel's one-token
        # launch, as qd_step runs it there).
        assert eng.decode_state(0).token_position == len(prompt)
        ref.kv_reset(0, 0)
        ref.prefill(0, prompt, want_logits=False)
        tok, _, logits = eng.step_graph(0, first)
        tok2, _, logits2 = ref.step(0, first)
        assert tok == tok2 and np.array_equal(logits, logits2)
        # And the untouched engine's resident path still completes.
        toks, reason, _ = ref.generate(0, tok2, 3)
        assert reason == qd.STOP_MAXIMUM_TOKENS and len(toks) == 3
    finally:
        eng.close()
        ref.close()


def state_of(eng):
    s = eng.decode_state(0)
    return {name: getattr(s, name) for name, *_ in s._fields_}


@pytest.mark.parametrize("call", ["prefill 1", "prefill 2", "tail"])
def test_failed_layers_leave_the_slot_where_it_was(monkeypatch, call):
    say(f"layers-only launch gives up under {call}")
    config = dict(SMALL, layers=6)
    monkeypatch.setenv("QD_RESIDENT_SPIN_LIMIT", "1")
    eng = qd.Engine(**config)
    monkeypatch.delenv("QD_RESIDENT_SPIN_LIMIT")
    ref = qd.Engine(**config)
    try:
        prompt = qo.fill_tokens(7, 5, 0x300000, SMALL["vocab"])
        for e in (eng, ref):
            e.load_synthetic(5)
            e.prefill(0, prompt[:5], want_logits=False)
            assert e.resident_grid() > 0
        if call == "tail":
            eng.embed_hidden(0, int(prompt[5]))
            eng.layer_decode(0, 0, 6, 6)
        before = None if call == "tail" else state_of(eng)
        with pytest.raises(qd.QdError) as err:
            if call == "tail":
                eng.tail(0)
            else:
                eng.prefill(0, prompt[5:5 + int(call[-1])])
        assert err.value.status == qd.DEVICE_FAULT
        if before:
            assert state_of(eng) == before
        assert eng.decode_state(0).token_position == 5
        # Its next step writes and attends over the rows that the reference's does.
        tok, _, logits = eng.step_graph(0, int(prompt[5]))
        tok2, _, logits2 = ref.step_graph(0, int(prompt[5]))
        assert tok == tok2 and np.array_equal(logits, logits2)
        for layer in range(6):
            for a, b in zip(eng.read_kv(0, layer, 0, 6), ref.read_kv(0, layer, 0, 6)):
                assert np.array_equal(a, b)
    finally:
        eng.close()
        ref.close()


@pytest.mark.parametrize("call", ["step_graph", "step_batch", "step_batch_noalloc", "kv_reset"])
def test_failed_layers_of_another_slot_leave_the_slot_where_it_was(monkeypatch, call):
    say(f"layers-only launch of slot 1 gives up, {call} of slot 0 reports it")
    config = dict(SMALL, layers=6, max_batch=2)
    monkeypatch.setenv("QD_RESIDENT_SPIN_LIMIT", "1")
    eng = qd.Engine(**config)
    monkeypatch.delenv("QD_RESIDENT_SPIN_LIMIT")
    try:
        eng.load_synthetic(5)
        eng.prefill(0, qo.fill_tokens(5, 5, 0x300000, SMALL["vocab"]), want_logits=False)
        before = state_of(eng)
        assert before["token_position"] == 5
        eng.embed_hidden(1, 3)
        eng.layer_decode(1, 0, 6, 1)
        with pytest.raises(qd.QdError) as err:
            if call.startswith("step_batch"):
                getattr(eng, call)([0], [7])
            elif call == "kv_reset":
                eng.kv_reset(0, 3)
            else:
                eng.step_graph(0, 7)
        assert err.value.status == qd.DEVICE_FAULT
        assert state_of(eng) == before
        eng.step_graph(0, 7)  # the error was that launch's, and has been reported
        assert eng.decode_state(0).token_position == 6
    finally:
        eng.close()


def test_prompt_without_room_for_its_workspace(monkeypatch):
    say("prompt workspace allocations refused by QD_DEVICE_BYTES_LIMIT")
    config = dict(SMALL, capacity=700)
    prompt = qo.fill_tokens(600, 5, 0x300000, SMALL["vocab"])
    engines = []

    def engine(limit=None):
        if limit:
            monkeypatch.setenv("QD_DEVICE_BYTES_LIMIT", str(limit))
        engines.append(qd.Engine(**config))
        monkeypatch.delenv("QD_DEVICE_BYTES_LIMIT", raising=False)
        engines[-1].load_synthetic(5)
        return engines[-1]

    try:
        ref = engine()
        base = ref.device_bytes()
        _, _, want = ref.prefill(0, prompt[:3])
        short = ref.device_bytes() - base
        ref.prefill(0, prompt[3:600])
        full = ref.device_bytes() - base  # the short one is given back
        say(f"workspace bytes: {short} for 3 tokens, {full} for 597")
        assert 0 < short < full
        # No room at all: an error each time, nothing kept, and steps still run.
        none = engine(base + short // 2)
        for _ in range(2):
            with pytest.raises(qd.QdError) as err:
                none.prefill(0, prompt[:3])
            assert err.value.status == qd.RUNTIME and none.device_bytes() == base
            assert none.decode_state(0).token_position == 0
        for t in prompt[:3].tolist():
            _, _, got = none.step(0, t)
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
        # Room for the short one: a long prompt runs in its chunks.
        some = engine(base + short)
        some.kv_reset(0, 0)
        _, _, got = some.prefill(0, prompt)
        assert some.device_bytes() == base + short
        ref.kv_reset(0, 0)
        ref.prefill(0, prompt[:512], want_logits=False)
        _, _, want = ref.prefill(0, prompt[512:])
        assert np.array_equal(got, want)
        for layer in range(SMALL["layers"]):
            for a, b in zip(some.read_kv(0, layer, 0, 600), ref.read_kv(0, layer, 0, 600)):
                assert np.array_equal(a, b)
    finally:
        for e in engines:
            e.close()


def test_batch_without_room_for_its_workspace(monkeypatch):
    say("batch workspace allocation refused by QD_DEVICE_BYTES_LIMIT")
    config = dict(SMALL, max_batch=2)
    ref = qd.Engine(**config)
    base = ref.device_bytes()
    monkeypatch.setenv("QD_DEVICE_BYTES_LIMIT", str(base + (1 << 20)))
    eng = qd.Engine(**config)
    monkeypatch.delenv("QD_DEVICE_BYTES_LIMIT")
    try:
        for e in (ref, eng):
            e.load_synthetic(5)
        for _ in range(2):
            with pytest.raises(qd.QdError) as err:
                eng.step_batch([0, 1], [3, 4])
            assert err.value.status == qd.RUNTIME and eng.device_bytes() == base  # nothing kept
        assert [eng.decode_state(s).token_position for s in range(2)] == [0, 0]
        got = eng.step_batch_noalloc([0, 1], [3, 4])
        want = ref.step_batch([0, 1], [3, 4])
        assert ref.device_bytes() > base + (1 << 20)
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
    finally:
        ref.close()
        eng.close()


def nan_bits(*patterns):
    return np.array(patterns, np.uint32).view(np.float32)


def test_write_kv_canonicalises_nan():
    say("write_kv NaN payloads")
    eng = qd.Engine(**SMALL)
    try:
        k = qo.fill_normal(8 * 128, 3, 0x200000, 0.0, 1.0).reshape(8, 128)
        v = qo.fill_normal(8 * 128, 3, 0x200001, 0.0, 1.0).reshape(8, 128)
        k[1, 5], k[7, 127] = nan_bits(0xFFFFFFFF, 0x7FFFFFFF)
        v[0, 0], v[3, 64] = nan_bits(0xFFC00001, 0x7F800001)
        eng.write_kv(0, 1, 10, k, v)
        gk, gv = eng.read_kv(0, 1, 10, 8)
        for got, want in ((gk, k), (gv, v)):
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(got), nan)
            assert (got.view(np.uint32)[nan] == CANONICAL).all()
            assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])
    finally:
        eng.close()


def hidden_with_nans():
    h = qo.fill_normal(896, 3, 0x600000, 0.0, 1.0)
    h[0], h[7], h[500], h[895] = nan_bits(0xFFFFFFFF, 0x7FFFFFFF, 0xFFC00001, 0x7F800001)
    return h


def test_load_hidden_canonicalises_nan():
    say("load_hidden NaN payloads, then six layers from the vector")
    eng = qd.Engine(**dict(SMALL, layers=6))
    try:
        eng.load_synthetic(5)
        h = hidden_with_nans()
        eng.load_hidden(0, h)
        got, nan = eng.read_activation(0, 0), np.isnan(h)
        assert np.array_equal(np.isnan(got), nan) and (got.view(np.uint32)[nan] == CANONICAL).all()
        assert np.array_equal(got[~nan], h[~nan])
        # The resident kernel reads the vector: NaN everywhere, and no wait
        # for a slot that only looks empty.
        assert eng.resident_grid() > 0
        eng.layer_decode(0, 0, 6, 1)
        assert np.isnan(eng.read_activation(0, 0)).all()
    finally:
        eng.close()


def test_layer_step_canonicalises_nan():
    say("layer_step NaN payloads: hidden vector and the K/V row derived from it")
    eng = qd.Engine(**SMALL)
    try:
        eng.load_synthetic(5)
        out = eng.layer_step(0, 1, hidden_with_nans())
        k, v = eng.read_kv(0, 1, 0, 1)
        for got in (out, k, v):
            bits = np.ascontiguousarray(got).view(np.uint32)
            assert np.isnan(got).all() and not (bits == 0xFFFFFFFF).any() and not (bits == 0x7FFFFFFF).any()
    finally:
        eng.close()


def test_bundle_nan_weights_are_canonical_and_resident_decode_returns(tmp_path):
    say("bundle with NaN payloads: load, canonical NaN, resident decode returns")
    h, i, q, kv, vocab = 896, 4864, 896, 128, 1024
    sizes = [h, h, q * h, kv * h, kv * h, q, kv, kv, h * q, i * h, i * h, h * i]
    tensors = [qo.fill_normal(n, 9, 0x400000 + j, 0.0, 0.02) for j, n in enumerate(sizes)]
    tensors[0][:] = 1.0
    tensors[1][:] = 1.0
    tensors[2][0] = nan_bits(0xFFFFFFFF)[0]   # q weight
    tensors[9][5] = nan_bits(0x7FFFFFFF)[0]   # gate weight
    tensors[11][-1] = nan_bits(0xFFC00001)[0]  # down weight
    layer_dir = tmp_path / "layer_0"
    layer_dir.mkdir()
    qd.bundle_write_layer(str(layer_dir / "weights.json"), "weights.bin", [1, h, 14, 2, 64, i], 1e6,
                          np.concatenate(tensors))
    emb = qo.fill_normal(vocab * h, 9, 0x500000, 0.0, 0.02)
    emb[3] = nan_bits(0xFFFFFFFF)[0]
    tail_dir = tmp_path / "model_tail"
    tail_dir.mkdir()
    qd.bundle_write_tail(str(tail_dir / "weights.json"), "weights.bin", h, vocab, np.arange(vocab),
                         emb, np.ones(h, np.float32), emb)
    eng = qd.Engine(layers=1, vocab=vocab, capacity=32, max_batch=1)
    try:
        eng.load_bundle(str(tmp_path))
        for kind, idx in ((qo.Q_W, 0), (qo.GATE_W, 5), (qo.DOWN_W, sizes[11] - 1)):
            got = eng.read_weight(0, kind, sizes[kind])
            assert got.view(np.uint32)[idx] == CANONICAL, kind
            assert np.isnan(got).sum() == 1, kind
        assert eng.read_weight(0, qd.EMBED, vocab * h).view(np.uint32)[3] == CANONICAL
        # Every hidden state is NaN from the first layer on (the NaN query
        # weight reaches every head through the O projection): the resident
        # launch must still run to its end and report a NaN argmax.
        assert eng.resident_grid() > 0
        eng.kv_reset(0, 0)
        toks, reason, logits = eng.generate(0, 7, 3, want_logits=True)
        assert toks.tolist() == [0xFFFFFFFF] and reason == qd.STOP_NONE
        assert np.isnan(logits).all()
    finally:
        eng.close()
