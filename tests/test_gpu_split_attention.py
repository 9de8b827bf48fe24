"""Decode attention over long contexts: a head's positions split over several
work-groups (batch 1-4 chain), around the context lengths where the split
changes, against the unsplit launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HD64 = dict(dim=256, hidden_dim=512, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=500, seq_len=4700)
HD128 = dict(dim=512, hidden_dim=1024, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=500, seq_len=4700)
CTX = 4608
EDGES = [256, 511, 512, 513, 544, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4097, 4600]


def _model(lm, d, B, kv32):
    cfg = lm.make_config(**d)
    m = lm.Model.create(cfg, lm.synth_weights_f16(cfg, 71, 0.05, True), True, B, d["seq_len"])
    m.set_option(lm.LM_OPT_KV_F32, int(kv32))
    toks = np.random.default_rng(71).integers(0, d["vocab_size"], (B, CTX)).astype(np.int32)
    for b in range(B):
        m.prefill(toks[b], slot=b, want_logits=False)
    return m, toks


@pytest.mark.parametrize("d", [HD64, HD128], ids=["hd64", "hd128"])
@pytest.mark.parametrize("kv32", [False, True])
@pytest.mark.parametrize("B", [1, 3])
def test_split_heads_match_one_work_group_per_head(lm, d, kv32, B):
    """Levels 2 and 3 (split) against level 0 (one work-group per head): fp32
    throughout, only the order of the softmax sums differs, over up to 4600
    positions: 1e-4 of a logit (a binary16 cache may round a K or V element
    of the step differently: 1e-3)."""
    m, toks = _model(lm, d, B, kv32)
    tol = 1e-4 if kv32 else 1e-3
    for p in EDGES:
        pos = np.array([p, max(p - 700, 3), 40][:B], np.int32)
        tk = toks[np.arange(B), pos]
        out = {}
        for level in (0, 2, 3):
            m.set_option(lm.LM_OPT_FUSE_QKV_ATTN, level)
            out[level] = m.forward_batch(tk, pos)[0]
        np.testing.assert_allclose(out[2], out[0], rtol=tol, atol=tol, err_msg=f"pos {p}")
        np.testing.assert_allclose(out[3], out[0], rtol=tol, atol=tol, err_msg=f"pos {p}")
    m.close()


def test_greedy_run_across_split_changes(lm):
    """Greedy runs whose steps cross from one work-group per head to four and
    from four to eight: graphs of both kinds against direct launches, the same ids."""
    m, toks = _model(lm, HD64, 1, True)
    runs = []
    for graph in (1, 0, 1):
        m.set_option(lm.LM_OPT_USE_GRAPH, graph)
        runs.append(np.concatenate([m.generate_greedy(toks[:1, p], np.array([p], np.int32), 40)
                                    for p in (490, 1010)]))
    assert np.array_equal(runs[0], runs[1]) and np.array_equal(runs[0], runs[2])
    m.close()


@pytest.mark.parametrize("d", [HD64, HD128], ids=["hd64", "hd128"])
@pytest.mark.parametrize("B,level", [(1, 3), (1, 2), (3, 2)])
def test_abort_ends_split_heads(lm, d, B, level):
    """The give-up flag raised from the host before a call whose heads are split:
    the work-groups that merge end their waits at once, the call and a greedy
    run report LM_ERR_HIP, and the calls after them give the bits of before."""
    m, toks = _model(lm, d, B, True)
    m.set_option(lm.LM_OPT_FUSE_QKV_ATTN, level)
    for p in (600, 1100, 4600):
        pos = np.array([p, max(p - 700, 3), 40][:B], np.int32)
        tk = toks[np.arange(B), pos]
        want = m.forward_batch(tk, pos)[0]
        m.set_option(lm.LM_OPT_HANDOFF_ABORT, 1)
        with pytest.raises(lm.LMError) as ei:
            m.forward_batch(tk, pos)
        assert ei.value.status == lm.LM_ERR_HIP
        assert np.array_equal(m.forward_batch(tk, pos)[0], want)
        m.set_option(lm.LM_OPT_HANDOFF_ABORT, 1)
        with pytest.raises(lm.LMError) as ei:
            m.generate_greedy(tk, pos, 18)
        assert ei.value.status == lm.LM_ERR_HIP
        assert np.array_equal(m.forward_batch(tk, pos)[0], want)
    m.close()
