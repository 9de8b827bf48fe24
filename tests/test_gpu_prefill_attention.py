"""The prefill attention kernels at the edges of their query blocks (32, 64, 128)
and key tiles (64), on both sides of the choice between them, against the same
prompt in 32-row pieces (whose attention is held to the oracle elsewhere)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HD64 = dict(dim=1024, hidden_dim=512, n_layers=1, n_heads=16, n_kv_heads=4, vocab_size=300, seq_len=2100)
HD128 = dict(dim=2048, hidden_dim=512, n_layers=1, n_heads=16, n_kv_heads=16, vocab_size=300, seq_len=2100)
H12 = dict(dim=768, hidden_dim=512, n_layers=1, n_heads=12, n_kv_heads=12, vocab_size=300, seq_len=2100)


@pytest.mark.parametrize("d", [HD64, HD128, H12], ids=["hd64", "hd128", "h12"])
@pytest.mark.parametrize("n,S", [(1, 63), (1, 65), (1, 129), (1, 1000), (1, 1281), (1, 1937), (2, 896),
                                 (9, 127), (10, 128), (9, 130), (3, 640)])
@pytest.mark.parametrize("kv32", [False, True])
def test_blocks_match_small_pieces(lm, d, n, S, kv32):
    """fp16 q, K, V and probabilities in either kernel, other orders of the key
    tiles: the logit bound of the fp16 path, and its mean."""
    cfg = lm.make_config(**d)
    w16 = lm.synth_weights_f16(cfg, 101, 0.03, True)
    toks = np.random.default_rng(S + n).integers(0, 300, (n, S)).astype(np.int32)
    with lm.Model.create(cfg, w16, True, n, S) as m:
        m.set_option(lm.LM_OPT_KV_F32, int(kv32))
        got = m.prefill_batch(toks, mode=lm.LM_LOGITS_ALL).reshape(n, S, -1)
        for i in sorted({0, n - 1}):
            ref = np.concatenate([m.prefill(toks[i, p:p + 32], slot=i, pos0=p) for p in range(0, S, 32)])
            np.testing.assert_allclose(got[i], ref, rtol=1e-2, atol=2e-2)
            assert np.abs(got[i] - ref).mean() < 2e-3


@pytest.mark.parametrize("d", [HD64, HD128], ids=["hd64", "hd128"])
@pytest.mark.parametrize("pos0,S", [(1, 1300), (10, 1200), (40, 1200), (63, 1300), (100, 1200),
                                    (1, 1900), (40, 1850), (63, 1937),
                                    (1, 64), (10, 100), (40, 41), (63, 65), (100, 160)])
@pytest.mark.parametrize("kv32", [False, True])
def test_offsets_that_straddle_a_key_tile(lm, d, pos0, S, kv32):
    """Prompts behind pos0 cached positions, pos0 no multiple of 32: a group of 32
    queries then holds some that see none of a wave's first key tile beside
    some that do.  The bound of the test above (pieces at multiples of 32 have
    no such group)."""
    cfg = lm.make_config(**d)
    w16 = lm.synth_weights_f16(cfg, 103, 0.03, True)
    toks = np.random.default_rng(S + pos0).integers(0, 300, pos0 + S).astype(np.int32)
    with lm.Model.create(cfg, w16, True, 1, pos0 + S) as m:
        m.set_option(lm.LM_OPT_KV_F32, int(kv32))
        ref = np.concatenate([m.prefill(toks[p:p + 32], pos0=p) for p in range(0, pos0 + S, 32)])[pos0:]
        got = m.prefill(toks[pos0:], pos0=pos0)
    assert np.all(np.isfinite(got)), np.unique(np.argwhere(~np.isfinite(got))[:, 0])[:8]
    np.testing.assert_allclose(got, ref, rtol=1e-2, atol=2e-2)
    assert np.abs(got - ref).mean() < 2e-3
