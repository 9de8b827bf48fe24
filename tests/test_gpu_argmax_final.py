"""The greedy pick's last reduction (k_argmax_final: four partials a thread and
pass, the row's last partial repeated past the end) at partial counts around its
256 threads and 1024 partials a pass: ids must be the lowest column of each
row's maximum, with the maximum in the last column, in the first, and tied."""
import numpy as np
import pytest

from test_zz_no_alloc import _Dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblk", [1, 255, 256, 257, 1023, 1024, 1025, 2050])
def test_ids_at_partial_counts(lm, nblk):
    assert lm.init() == 0
    M, K, N = 4, 64, nblk * 32 - 5   # (a ragged last block)
    rng = np.random.default_rng(nblk)
    A = rng.standard_normal((M, K)).astype(np.float16)
    W = (0.02 * rng.standard_normal((N, K))).astype(np.float16)
    hit = (0.5 * A.astype(np.float32)).astype(np.float16)
    W[N - 1], W[0] = hit[0], hit[1]
    W[N // 2] = W[N - 2] = hit[2]
    dev = _Dev()
    try:
        dA, dW = dev.put(A.view(np.uint16)), dev.put(W.view(np.uint16))
        dC, dI = dev.alloc(M * N * 4), dev.alloc(M * 4)
        assert lm.gemm_argmax_noalloc(M, N, K, dA, dW, dC, dI) == 0
        dev.sync()
        C, ids = dev.get(dC, (M, N), np.float32), dev.get(dI, M, np.int32)
    finally:
        dev.free()
    assert np.array_equal(ids, np.argmax(C, axis=1))
    assert list(ids[:3]) == [N - 1, 0, N // 2]
