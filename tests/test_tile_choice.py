"""The prefill GEMM's choice of tile (CPU only) against times of all four tiles,
measured with their real epilogues (us; None: not built)."""
import pytest

STORE, GATE, QKV, RESNORM = 0, 2, 3, 5

# (epilogue, M, N, K, (64x64, 64x128, 128x128, 256x128))
MEASURED = [
    (QKV, 1118, 2304, 768, (13.2, None, 15.4, 21.2)),
    (QKV, 1500, 2304, 768, (17.3, None, 14.7, 21.4)),
    (GATE, 1118, 4096, 768, (17.1, 18.2, 19.9, 17.3)),
    (GATE, 1500, 4096, 768, (20.2, 18.8, 20.0, 17.8)),
    (RESNORM, 1500, 768, 2048, (16.1, 17.3, 20.2, 34.8)),
    (GATE, 640, 2048, 1024, (9.3, 9.8, 11.8, 18.4)),
    (RESNORM, 1118, 1024, 1024, (10.7, 11.9, 13.8, 22.1)),
    (STORE, 1118, 1024, 1024, (8.5, 9.2, 10.8, 17.1)),
    (RESNORM, 1280, 1024, 1024, (11.0, 12.0, 13.8, 22.5)),
    (QKV, 1500, 2048, 1024, (15.5, None, 16.9, 23.7)),
    (QKV, 2048, 2048, 1024, (22.4, None, 17.8, 23.9)),
    (GATE, 2048, 2048, 1024, (20.0, 15.0, 14.2, 19.7)),
    (GATE, 320, 11264, 2048, (30.1, 24.6, 38.8, 35.5)),
    (QKV, 640, 6144, 2048, (33.0, None, 26.9, 39.0)),
    (GATE, 640, 11264, 2048, (49.0, 44.6, 41.4, 64.9)),
    (RESNORM, 640, 2048, 5632, (31.6, 33.6, 41.2, 75.5)),
    (QKV, 1118, 6144, 2048, (52.7, None, 45.9, 42.3)),
    (RESNORM, 1118, 2048, 5632, (56.0, 51.9, 43.3, 76.1)),
    (RESNORM, 1500, 2048, 5632, (67.5, 59.2, 49.2, 78.0)),
    (QKV, 2048, 6144, 2048, (117.4, None, 73.1, 76.4)),
    (RESNORM, 2048, 2048, 2048, (40.0, 29.3, 26.8, 37.3)),
    (RESNORM, 2048, 768, 768, (10.9, 11.2, 12.6, 20.4)),
    (QKV, 2048, 4096, 2048, (75.0, None, 50.0, 44.1)),
    (GATE, 2048, 2048, 512, (11.0, 9.3, 9.3, 12.6)),
    (STORE, 128, 32000, 768, (14.8, 19.3, 13.5, 17.9)),
    (STORE, 1024, 32000, 2048, (257.5, 219.5, 184.0, 149.0)),
]


@pytest.mark.parametrize("epi,M,N,K,us", MEASURED)
def test_choice_is_near_the_fastest_tile(lm, epi, M, N, K, us):
    k = lm.lib().lmk_pick_tile(M, N, K, epi)
    assert us[k] is not None
    assert us[k] <= 1.05 * min(t for t in us if t is not None), (k, us)


def test_every_tile_is_chosen_somewhere(lm):
    assert {lm.lib().lmk_pick_tile(M, N, K, epi) for epi, M, N, K, _ in MEASURED} == {0, 1, 2, 3}
