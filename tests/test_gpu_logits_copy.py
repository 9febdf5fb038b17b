"""Logits rows on their way to the caller: in pieces through pinned memory for
pageable buffers, directly for pinned ones, for rows below and above the size
that takes the pieces, whole pieces and a remainder, more rows than one export
holds. Every route returns the same bytes, and only the rows asked for."""
import ctypes as C

import numpy as np
import pytest

import qwen_decode as qd
import qwen_oracle as qo

pytestmark = pytest.mark.gpu

PIECE, EXPORT_BYTES, SLOTS = 4096, 256 * 1024, 18


def pinned_rows(n, vocab):
    """Pinned memory of the HIP runtime the library runs on, for the process."""
    hip = C.CDLL(None)
    if not hasattr(hip, "hipHostMalloc"):
        hip = C.CDLL("libamdhip64.so.7")
    ptr = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(ptr), C.c_size_t(n * vocab * 4), C.c_uint(0)) == 0
    return np.ctypeslib.as_array(C.cast(ptr, C.POINTER(C.c_float)), (n, vocab))


@pytest.mark.parametrize("vocab", [1003, EXPORT_BYTES // 4 - 1, EXPORT_BYTES // 4, 20 * PIECE, 20 * PIECE + 7])
def test_every_route_returns_the_same_logits(vocab):
    print(f"logits of vocabulary {vocab}", flush=True)
    eng = qd.Engine(layers=1, vocab=vocab, capacity=8, max_batch=SLOTS)
    eng.load_synthetic(3)
    slots = [(7 * i + 3) % SLOTS for i in range(SLOTS)]
    tokens = [int(t) for t in qo.fill_tokens(SLOTS, 3, 0x700000, vocab)]
    for n in (SLOTS, 16, 5, 1):
        for s in slots:
            eng.kv_reset(s, 0)
        _, logits = eng.step_batch(slots[:n], tokens[:n])
        # The row whose end the copy could overrun, in a larger buffer.
        guarded = np.full(vocab + 2 * PIECE, 7.0, np.float32)
        for i, s in enumerate(slots[:n]):
            assert np.array_equal(eng.read_logits(s), logits[i])
            out = guarded[PIECE:PIECE + vocab]
            qd._check(qd.lib().qd_read_logits(eng.handle, s, out.ctypes.data_as(C.POINTER(C.c_float)), vocab))
            assert np.array_equal(out, logits[i])
            assert (guarded[:PIECE] == 7).all() and (guarded[PIECE + vocab:] == 7).all()
        pinned = pinned_rows(n, vocab)
        for s in slots:
            eng.kv_reset(s, 0)
        ids, toks = np.array(slots[:n], np.uint32), np.array(tokens[:n], np.uint32)
        greedy = np.empty(n, np.uint32)
        qd._check(qd.lib().qd_step_batch(eng.handle, n, qd._u(ids), qd._u(toks), qd._f(pinned), qd._u(greedy)))
        assert np.array_equal(pinned, logits)
        assert np.array_equal(greedy, np.argmax(logits, axis=1))
    eng.close()


@pytest.mark.parametrize("vocab", [EXPORT_BYTES // 4 - 1, EXPORT_BYTES // 4, 20 * PIECE + 7])
def test_a_step_writes_its_row_and_nothing_beside_it(vocab):
    print(f"a step's logits of vocabulary {vocab} into a larger buffer", flush=True)
    eng = qd.Engine(layers=1, vocab=vocab, capacity=8, max_batch=2)
    eng.load_synthetic(3)
    guarded = np.full(vocab + 2 * PIECE, 7.0, np.float32)
    out = guarded[PIECE:PIECE + vocab]
    qd._check(qd.lib().qd_step(eng.handle, 1, 5, qd._f(out), None, None))
    assert np.array_equal(out, eng.read_logits(1))
    assert (guarded[:PIECE] == 7).all() and (guarded[PIECE + vocab:] == 7).all()
    eng.close()
