"""The prefill GEMM tiles that pick_tile chooses beyond 64 rows (64x64, 64x128,
128x128 of eight waves, 256x128), at shapes whose last row and column tiles are
ragged, and their fused epilogues inside a prefill."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ab(M, N, K):
    rng = np.random.default_rng(M + 3 * N + 11 * K)
    return (rng.standard_normal((M, K)).astype(np.float16),
            (0.02 * rng.standard_normal((N, K))).astype(np.float16))


@pytest.mark.parametrize("M,N,K", [(65, 40, 64), (300, 11200, 256),      # 64x64, 64x128
                                   (1030, 2000, 1024), (1900, 2050, 512),  # 64x128, 128x128
                                   (101, 32000, 768), (1025, 4001, 2048),  # 128x128
                                   (2047, 4070, 768)])                      # 256x128
def test_store_tiles_match_numpy(lm, M, N, K):
    """fp32 sums of exact products: 1e-5 of each row's absolute products."""
    A, W = _ab(M, N, K)
    C, pv, pi = lm.selftest_gemm(A.view(np.uint16), W.view(np.uint16), want_parts=True)
    Af, Wf = A.astype(np.float32), W.astype(np.float32)
    ref, scale = Af @ Wf.T, np.abs(Af) @ np.abs(Wf).T
    # the float32 reference adds its own rounding, of the same bound
    assert np.all(np.abs(C - ref) <= 2e-5 * scale + 1e-6)
    for b in range(0, (N + 31) // 32, 7):
        blk = C[:, b * 32:min(N, b * 32 + 32)]
        assert np.array_equal(pi[:, b], b * 32 + np.argmax(blk, axis=1))


@pytest.mark.parametrize("M,N,K", [(300, 11264, 256), (1000, 4096, 1024), (1025, 11264, 512)])
def test_gate_tiles_match_numpy(lm, M, N, K):
    """fp16 result of an fp32 gate: half an ulp (4.9e-4) and the sums' rounding."""
    A, W = _ab(M, N, K)
    g = lm.selftest_gemm_gate(A.view(np.uint16), W.view(np.uint16)).view(np.float16).astype(np.float64)
    h = (A.astype(np.float32) @ W.astype(np.float32).T).astype(np.float64)
    i = np.arange(N // 2)
    h1, h3 = h[:, 32 * (i // 16) + i % 16], h[:, 32 * (i // 16) + 16 + i % 16]
    ref = h1 / (1.0 + np.exp(-h1)) * h3
    assert np.all(np.abs(g - ref) <= 2e-3 * np.abs(ref) + 2e-5)


WIDE = dict(dim=2048, hidden_dim=5632, n_layers=2, n_heads=16, n_kv_heads=8, vocab_size=512, seq_len=2048)
MID = dict(dim=1024, hidden_dim=2048, n_layers=2, n_heads=16, n_kv_heads=8, vocab_size=512, seq_len=2048)


@pytest.mark.parametrize("d,S,fold,kv32", [(WIDE, 1030, 1, False), (WIDE, 1900, 1, True),
                                           (WIDE, 1900, 0, False), (MID, 2047, 1, False),
                                           (MID, 515, 1, False)])
def test_long_prompt_equals_its_64_row_chunks(lm, d, S, fold, kv32):
    """One prompt in one chunk (the tiles of its row count, QKV, residual and
    gate epilogues with and without the row scale) against the same prompt 64
    rows at a time (the decode-row tiles, held to the oracle elsewhere).  Both
    round the same operands to fp16, in other places where the norm is folded:
    the logit bound of the fp16 path, and its mean."""
    cfg = lm.make_config(**d)
    w16 = lm.synth_weights_f16(cfg, 61, 0.02, True)
    toks = np.random.default_rng(S).integers(0, d["vocab_size"], S).astype(np.int32)
    with lm.Model.create(cfg, w16, True, 1, S) as m:
        m.set_option(lm.LM_OPT_KV_F32, int(kv32))
        m.set_option(lm.LM_OPT_PREFILL_FOLD, fold)
        got = m.prefill(toks)
        got2 = m.prefill(toks)
        ref = np.concatenate([m.prefill(toks[p:p + 64], pos0=p) for p in range(0, S, 64)])
    assert np.array_equal(got, got2)
    np.testing.assert_allclose(got, ref, rtol=1e-2, atol=2e-2)
    assert np.abs(got - ref).mean() < 2e-3
