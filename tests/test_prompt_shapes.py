"""Which prompt shapes are kept as captured graphs (CPU only): recurring ones
replay, no rotation of more shapes than graphs captures at each call."""
import ctypes

import pytest

DIRECT, CAPTURE, REPLAY = 0, 1, 2
GRAPHS = 4


@pytest.fixture()
def use(lm):
    f = lm.lib().lmh_shape_use
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    table, slot = ctypes.create_string_buffer(4096), ctypes.c_int()
    held = {}

    def call(R, S=None, all_=0):
        key = (R, S or R, all_)
        how = f(table, *key, ctypes.byref(slot))
        if how == CAPTURE:
            assert 0 <= slot.value < GRAPHS
            held[slot.value] = key
        if how == REPLAY:
            assert held[slot.value] == key      # the graph of this very shape
        return how
    return call


def test_second_use_captures_and_later_ones_replay(use):
    assert [use(40) for _ in range(4)] == [DIRECT, CAPTURE, REPLAY, REPLAY]
    assert use(40, 20) == DIRECT and use(40, 40, 1) == DIRECT     # other shapes of as many rows


@pytest.mark.parametrize("n", [1, 4, 5, 6, 12, 16, 17, 40])
def test_rotation_captures_no_more_often_than_it_keeps(use, n):
    how = [[use(10 + i) for i in range(n)] for _ in range(12)]
    assert all(h == DIRECT for h in how[0])
    flat = [h for r in how for h in r]
    assert flat.count(CAPTURE) <= GRAPHS
    if n <= 16:      # as many as are remembered: the graphs stay in use
        for r in how[2:]:
            assert r.count(REPLAY) == min(n, GRAPHS) and r.count(CAPTURE) == 0


def test_new_lengths_throw_out_no_graph(use):
    for _ in range(2):
        use(7), use(8)
    assert all(use(100 + i) == DIRECT for i in range(50))
    assert use(7) == REPLAY and use(8) == REPLAY


def test_new_working_set_replaces_an_old_one(use):
    for _ in range(3):
        for i in range(GRAPHS):
            use(10 + i)
    for i in range(GRAPHS):
        assert [use(50 + i) for _ in range(3)] == [DIRECT, CAPTURE, REPLAY]
    assert [use(50 + i) for i in range(GRAPHS)] == [REPLAY] * GRAPHS
    assert use(10) == DIRECT
