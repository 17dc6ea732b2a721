"""Every tuning entry of the repeated-row classes is read by the requests it is measured on (host-side
layout calls of the C ABI, no device): under the tile entry the tuner sets, the blocks and waves
entries of a class change the partial slots of its requests, and where a request runs at another
class's side by the built-in choice, that class's entries decide."""
import ctypes

import pytest

from thewalrus_amd import _native, tune

REPS = {1: [9, 8, 8, 7], 3: [6, 6, 5, 5, 5], 2: [4, 4, 4, 4, 4, 3, 3]}  # edge multiplicities, cut to h = 16


def request(T, loop, real):
    E = len(REPS[T])
    r = _native.WhRequest()
    r.E, r.glynn, r.real, r.a_off = E, 1, int(real), 0
    r.d_off, r.v_off = (4 * E * E if loop else -1), -1
    left = 16
    for i, e in enumerate(REPS[T]):
        r.edge_reps[i] = max(1, min(e, left - (E - 1 - i)))
        left -= r.edge_reps[i]
    return r


def slots(r):
    out = ctypes.c_int64()
    assert _native.load().wh_request_partials(ctypes.byref(r), 0, ctypes.byref(out)) == 0
    return out.value


@pytest.fixture
def table():
    L = _native.load()
    before = tune.current(), tune.current_waves(), tune.current_tiles()
    for k in before[0]:
        L.wh_tune_set(*k, 0)
        if k[0] != 1:
            L.wh_tune_set_waves(*k, 0)
            L.wh_tune_set_tile(*k, 0)
    yield L
    for k, v in before[0].items():
        L.wh_tune_set(*k, v)
    for k, v in before[1].items():
        L.wh_tune_set_waves(*k, v)
    for k, v in before[2].items():
        L.wh_tune_set_tile(*k, v)


@pytest.mark.parametrize("loop", [0, 1])
@pytest.mark.parametrize("T", [1, 3, 2])
def test_entries_reach_their_requests(T, loop, table):
    r = request(T, loop, real=False)
    assert table.wh_tune_set_tile(2, T, loop, tune.forced_tile(2, T)) == 0
    seen = []
    for blocks in (1, 2):
        assert table.wh_tune_set(2, T, loop, blocks) == 0
        seen.append(slots(r))
    assert seen[0] < seen[1]
    w = request(T, loop, real=T == 2)  # (the symmetric powers choose their waves themselves)
    assert table.wh_tune_set(2, T, loop, 4096) == 0
    seen = []
    for waves in (4, 1):
        assert table.wh_tune_set_waves(2, T, loop, waves) == 0
        seen.append(slots(w))
    assert seen[0] < seen[1]


@pytest.mark.parametrize("loop", [0, 1])
def test_built_in_choice_of_the_smallest_class(loop, table):
    """2E <= 8 runs at side 3 unless the table asks for side 1."""
    r = request(1, loop, real=False)
    base = slots(r)
    assert table.wh_tune_set(2, 1, loop, 1) == 0 and slots(r) == base
    assert table.wh_tune_set(2, 3, loop, 1) == 0
    assert slots(r) < base
    assert table.wh_tune_set_tile(2, 1, loop, 1) == 0 and table.wh_tune_set(2, 1, loop, 0) == 0
    own = slots(r)
    assert table.wh_tune_set(2, 1, loop, 1) == 0 and slots(r) < own


@pytest.mark.parametrize("loop", [0, 1])
def test_own_sides_are_accepted(loop, table):
    for T in (1, 2):
        assert table.wh_tune_set_tile(2, T, loop, T) == 0 and table.wh_tune_get_tile(2, T, loop) == T
    # and the other refusals stand
    for args in ((2, 3, loop, 3), (2, 3, loop, 1), (2, 2, loop, 3), (2, 2, loop, 1), (2, 1, loop, 4)):
        assert table.wh_tune_set_tile(*args) != 0


def test_flops_count_the_products_formed():
    """The four-terms-per-wave kernel forms symmetric powers: m (m + 1) / 2 entries of m products each."""
    r = request(3, 0, real=False)
    L = _native.load()
    b = ctypes.c_void_p()
    assert L.wh_batch_create(ctypes.byref(r), 1, 0, ctypes.byref(b)) == 0
    terms, flops = ctypes.c_int64(), ctypes.c_double()
    assert L.wh_batch_info(b, None, None, ctypes.byref(terms), ctypes.byref(flops)) == 0
    L.wh_batch_destroy(b)
    m, powers = 10, 7  # h = 16: powers 2 .. 8
    assert flops.value == terms.value * 8.0 * (m * (m + 1) / 2) * m * powers
