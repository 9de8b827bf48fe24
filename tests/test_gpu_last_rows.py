"""LM_LOGITS_LAST: the last layer after its K and V runs on the sequences' last
rows alone.  Against the last rows of LM_LOGITS_ALL, and the cache both leave."""
import numpy as np
import pytest

from conftest import TINY, TINY_GQA, TINY_HD128

pytestmark = pytest.mark.gpu

ONE = dict(TINY_GQA, n_layers=1)


@pytest.mark.parametrize("d,n,S", [(TINY, 1, 2), (TINY_GQA, 3, 33), (TINY_HD128, 2, 150), (ONE, 5, 17),
                                   (TINY, 70, 3), (TINY_GQA, 130, 2), (TINY, 7, 1), (TINY, 40, 64)])
@pytest.mark.parametrize("kv32", [False, True])
def test_last_rows_match_all_rows(lm, d, n, S, kv32):
    """The last row's attention runs in fp32 instead of fp16 operands, the rest
    on other tiles: the logit bound of the fp16 path.  K and V of every row are
    the same bits, so a decode step behind either prefill is the same."""
    cfg = lm.make_config(**d)
    w16 = lm.synth_weights_f16(cfg, 83, 0.02, True)
    toks = np.random.default_rng(83).integers(0, d["vocab_size"], (n, S)).astype(np.int32)
    nxt = np.arange(n, dtype=np.int32) % d["vocab_size"]
    nb = min(n, 64)
    with lm.Model.create(cfg, w16, True, n, S + 2) as m:
        m.set_option(lm.LM_OPT_KV_F32, int(kv32))
        full = m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL).reshape(n, S, -1)
        step_full = m.forward_batch(nxt[:nb], np.full(nb, S, np.int32))[0]
        for graph in (1, 0, 1):
            m.set_option(lm.LM_OPT_USE_GRAPH, graph)
            last = m.prefill_batch(toks, mode=lm.LM_LOGITS_LAST)
            assert np.array_equal(m.read_logits(0, 1)[0], last[n - 1 - (n - 1) % max(1, min(n, 2048 // S))])
            np.testing.assert_allclose(last, full[:, -1], rtol=1e-2, atol=2e-2)
            assert np.abs(last - full[:, -1]).mean() < 2e-3
        step_last = m.forward_batch(nxt[:nb], np.full(nb, S, np.int32))[0]
        assert np.array_equal(step_full, step_last)
