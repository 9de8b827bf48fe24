"""Up to 64 rows of models up to 1024 wide: the projections of k_rows.hip (norm,
RoPE and cache append, residual, gate in the launch), at the edges of their
16-row tiles and of the columns per work-group, against the oracle."""
import numpy as np
import pytest

from conftest import TINY_GQA, TINY_HD128, cfg7

pytestmark = pytest.mark.gpu

W768 = dict(dim=768, hidden_dim=2048, n_layers=2, n_heads=12, n_kv_heads=12, vocab_size=300, seq_len=72)
W1024 = dict(dim=1024, hidden_dim=2048, n_layers=2, n_heads=8, n_kv_heads=2, vocab_size=300, seq_len=72)


@pytest.mark.parametrize("d", [TINY_GQA, TINY_HD128, W768, W1024], ids=["256", "512", "768", "1024"])
@pytest.mark.parametrize("S", [2, 15, 16, 17, 33, 48, 49, 64])
@pytest.mark.parametrize("kv32", [False, True])
def test_short_prompt_and_batch_match_oracle(lm, orc, d, S, kv32):
    """S rows as one prompt (all logits), then S rows as a decode batch of S
    sequences: fp16 operands, fp32 sums, the logit bound of that path."""
    cfg = lm.make_config(**d)
    w16 = lm.synth_weights_f16(cfg, 91, 0.02, True)
    w32 = lm.f16_to_f32(w16)
    rng = np.random.default_rng(S)
    toks = rng.integers(0, d["vocab_size"], S).astype(np.int32)
    with lm.Model.create(cfg, w16, True, S, 72) as m:
        m.set_option(lm.LM_OPT_KV_F32, int(kv32))
        got = m.prefill(toks, slot=S - 1)
        ref = orc.Oracle(cfg7(d), w32, True, 72, kv_f16=not kv32).forward_full(toks)
        np.testing.assert_allclose(got, ref, rtol=1e-2, atol=2e-2)
        assert np.abs(got - ref).mean() < 2e-3
        if S < 5:
            return
        # row b continues a prompt of 3 tokens of its own in slot b
        p3 = rng.integers(0, d["vocab_size"], (S, 4)).astype(np.int32)
        m.prefill_batch(p3[:, :3], mode=lm.LM_LOGITS_LAST, want_logits=False)
        lg = m.forward_batch(p3[:, 3], np.full(S, 3, np.int32))[0]
        for b in (0, S // 2, S - 1):
            o = orc.Oracle(cfg7(d), w32, True, 72, kv_f16=not kv32)
            ref = o.forward_full(p3[b])[-1]
            np.testing.assert_allclose(lg[b], ref, rtol=1e-2, atol=2e-2)
