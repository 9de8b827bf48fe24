"""Results as kernels give them to the host (shares with a flag each, segments of
the staging), against the device's own copy of the logits."""
import os
import time

import numpy as np
import pytest

from conftest import TINY

pytestmark = pytest.mark.gpu


def _model(lm, vocab, B, S):
    cfg = lm.make_config(**dict(TINY, vocab_size=vocab))
    return lm.Model.create(cfg, lm.synth_weights_f16(cfg, 97, 0.02, True), True, B, S)


@pytest.mark.parametrize("vocab", [1, 3, 301, 1023, 1024, 1025, 40001])
@pytest.mark.parametrize("B", [1, 2, 7, 64])
def test_step_results_equal_device_logits(lm, vocab, B):
    """The same values bit for bit, ids the first maximum; changing inputs, so
    that a result of the call before would show."""
    with _model(lm, vocab, B, 16) as m:
        rng = np.random.default_rng(vocab + B)
        for p in range(4):
            tk = rng.integers(0, vocab, B).astype(np.int32)
            lg, am = m.forward_batch(tk, np.full(B, p, np.int32))
            assert np.array_equal(lg, m.read_logits(0, B))
            assert np.array_equal(am, lg.argmax(1))
            none, am2 = m.forward_batch(tk, np.full(B, p, np.int32), want_logits=False)
            assert none is None and np.array_equal(am, am2)
        one = m.forward(int(tk[0]), 3)
        assert np.array_equal(one, m.read_logits(0, 1)[0])


@pytest.mark.parametrize("vocab,n,S", [(301, 3, 5), (32000, 1, 40), (32001, 2, 33), (9001, 5, 47)])
def test_prompt_logits_equal_device_logits(lm, vocab, n, S):
    """Several segments (more than 2 MiB), the last ragged, into fresh and
    reused host memory."""
    with _model(lm, vocab, n, S) as m:
        rng = np.random.default_rng(S)
        for _ in range(3):
            toks = rng.integers(0, vocab, (n, S)).astype(np.int32)
            lg = m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL)
            assert np.array_equal(lg, m.read_logits(0, n * S))
            loss, lg2 = m.prefill_loss(toks, want_logits=True) if vocab % 4 == 0 else (None, lg)
            assert np.array_equal(lg, lg2)
            last = m.prefill_batch(toks, mode=lm.LM_LOGITS_LAST)
            assert np.array_equal(last, m.read_logits(0, n))


@pytest.mark.parametrize("B,steps", [(1, 1), (1, 16), (3, 33), (64, 50)])
def test_greedy_ids_equal_single_steps(lm, B, steps):
    """A run of the device loop against its steps one call at a time."""
    with _model(lm, 2, B, 64) as m:
        first = (np.arange(B) % 2).astype(np.int32)
        ids = m.generate_greedy(first, np.zeros(B, np.int32), steps)
        tk = first
        for t in range(steps):
            tk = m.forward_batch(tk, np.full(B, t, np.int32), want_logits=False)[1]
            assert np.array_equal(ids[t], tk), t


@pytest.mark.parametrize("B", [1, 3, 5, 64])
def test_first_step_equals_its_replays(lm, B):
    """A handle's first step of a batch and kind is launched directly and captured
    behind that launch; its second replays the capture: the same bits, also
    with other work of the handle between them."""
    rng = np.random.default_rng(B)
    tk = rng.integers(0, 301, B).astype(np.int32)
    pos = np.full(B, 2, np.int32)
    rows = rng.integers(0, 301, (B, 2)).astype(np.int32)
    with _model(lm, 301, B, 64) as m:
        m.prefill_batch(rows, mode=lm.LM_LOGITS_LAST, want_logits=False)
        first = m.forward_batch(tk, pos)
        ids = m.forward_batch(tk, pos, want_logits=False)[1]
        for _ in range(3):
            lg, am = m.forward_batch(tk, pos)
            assert np.array_equal(lg, first[0]) and np.array_equal(am, first[1])
            assert np.array_equal(m.forward_batch(tk, pos, want_logits=False)[1], ids)
            m.prefill_batch(rows, mode=lm.LM_LOGITS_LAST)
        assert np.array_equal(ids, first[1])
        runs = [m.generate_greedy(first[1], pos + 1, 37) for _ in range(3)]
        m.set_option(lm.LM_OPT_USE_GRAPH, 0)
        runs.append(m.generate_greedy(first[1], pos + 1, 37))
        assert all(np.array_equal(r, runs[0]) for r in runs)


@pytest.mark.parametrize("n,S", [(1, 5), (3, 33), (2, 150)])
def test_prompt_calls_equal_their_replays(lm, n, S):
    """A prompt shape's first call launches directly, its second captures behind
    its launch, later ones replay: the same bits, for new tokens too, and with
    more shapes between them than are kept."""
    rng = np.random.default_rng(S)
    a, b = rng.integers(0, 300, (2, n, S)).astype(np.int32)
    with _model(lm, 300, n, 256) as m:
        for mode in (lm.LM_LOGITS_LAST, lm.LM_LOGITS_ALL):
            m.set_option(lm.LM_OPT_USE_GRAPH, 0)
            want = [m.prefill_batch(t, mode=mode) for t in (a, b)]
            m.set_option(lm.LM_OPT_USE_GRAPH, 1)
            for k in (0, 1, 0, 1, 1, 0):
                assert np.array_equal(m.prefill_batch((a, b)[k], mode=mode), want[k]), k
            for L in range(2, 8):
                for _ in range(2):
                    m.prefill_batch(a[:, :L] if L < S else b, mode=mode)
            for k in (0, 1, 0):
                assert np.array_equal(m.prefill_batch((a, b)[k], mode=mode), want[k]), k


def test_large_results_wait_on_one_thread(lm):
    """A call with megabytes of results waits for the device on one thread: the
    copying threads sleep until results land, and between calls (four spinning
    threads: four times the wall time).  They end with the handle."""
    cfg = lm.make_config(2048, 5632, 4, 16, 8, 500, 1900)
    w16 = lm.synth_weights_f16(cfg, 97, 0.02, True)
    toks = np.random.default_rng(97).integers(0, 500, (1, 1900)).astype(np.int32)
    before = None
    for _ in range(3):
        with lm.Model.create(cfg, w16, True, 1, 1900) as m:
            for _ in range(3):
                first = m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL)
            wall, cpu = time.perf_counter(), time.process_time()
            for _ in range(15):
                m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL)
            wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
            assert np.array_equal(m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL), first)
        assert cpu < 2.5 * wall, (cpu, wall)
        n = len(os.listdir("/proc/self/task"))
        assert before is None or n <= before
        before = n
