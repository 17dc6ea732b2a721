"""The symmetric-power kernel for any multiplicities (sieve_sym.hip) against the oracle's
double-double truth and the general kernel, at the edges of its tiles and of its coefficient
routes.  Bar: relative error <= 1e-10, or twice the reference algorithm's own FP64 error where
that is larger; the two kernels, each within the bar of the truth, within twice of each other."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import random_symmetric, relerr

TOL = 1e-10


def cases():
    """(name, modes, rpt, loop, real, glynn): sides 2E (2E + 2 for odd N) at 8T - 2, 8T and past
    it, h = N / 2 at 16 and 17, 32 and 33 (the coefficient routes), self-paired modes, delta = 0
    in every digit, one edge, and odd N with the unpaired mode also repeated."""
    out = []
    for n in (5, 7, 9, 11, 13, 15, 17, 19):  # odd all-ones: sides 6, 8, 10 .. 20
        out.append(("odd_ones", n, [1] * n, True, n % 4 == 1, True))
    out += [
        ("one_edge", 2, [17, 17], False, False, True),
        ("one_edge_loop", 1, [37], True, False, True),
        ("self_pairs", 3, [12, 1, 2], True, False, True),
        ("odd_self", 3, [13, 2, 2], True, False, True),
        ("odd_mode_repeated", 4, [3, 3, 3, 2], True, False, True),
        ("zero_modes", 6, [2, 0, 3, 0, 2, 2], True, False, True),
        ("inclexcl_ones", 10, [1] * 10, False, False, False),
        ("inclexcl_ones_real", 12, [1] * 12, False, True, False),
        ("inclexcl_rep_h17", 4, [9, 9, 8, 8], True, False, False),
        ("h17", 3, [12, 12, 10], True, False, True),
        ("h32", 2, [32, 32], True, False, True),
        ("h33", 2, [33, 33], True, False, True),
        ("h64", 2, [64, 64], False, True, True),
        ("odd_127", 2, [64, 63], True, False, True),
        ("side_18", 18, [1] * 16 + [2, 2], True, False, True),
        ("side_18_plain", 18, [1] * 16 + [2, 2], False, True, True),
        ("side_24_odd", 23, [1] * 20 + [2, 0, 1], True, False, True),
    ]
    # four terms per wave (2E <= 12, 2E <= 10 for odd N): every side, h = 8 | 9 and 16 | 17, and the
    # sides past it
    for rpt in ([3], [4, 1], [3, 2, 2], [5, 4, 4, 2], [3, 3, 3, 3, 3], [2, 2, 2, 2, 2, 1], [2] * 8 + [1], [2] * 5 + [1],
                [9, 8], [6, 6, 5], [11, 10, 10], [11, 11, 11], [17, 16], [3, 2, 2, 2, 2, 2, 2, 2], [3, 3, 2, 2, 2, 2, 2, 2]):
        out.append(("four_terms_odd%d" % (sum(rpt) % 2), len(rpt), rpt, True, len(rpt) % 3 == 0, True))
    for rpt in ([2, 2], [4, 4, 2], [2] * 5 + [0], [2] * 6, [2] * 7, [2] * 8, [8, 8], [9, 9], [16, 16], [6] * 5 + [2]):
        out.append(("four_terms_plain", len(rpt), rpt, False, len(rpt) % 2 == 0, True))
        out.append(("four_terms_inclexcl", len(rpt), rpt, True, len(rpt) % 2 == 1, False))
    return out



def make(name, modes, real, seed=0):
    rng = np.random.default_rng([modes, seed, len(name)])
    A = random_symmetric(rng, modes, complex_=not real, scale=1.0 / np.sqrt(modes))
    mu = rng.normal(size=modes) if real else rng.normal(size=modes) + 1j * rng.normal(size=modes)
    return A, mu


@pytest.mark.gpu
@pytest.mark.parametrize("name,modes,rpt,loop,real,glynn", cases(), ids=lambda v: str(v)[:24])
def test_against_truth_and_general_kernel(name, modes, rpt, loop, real, glynn):
    from thewalrus_amd.batch import DeviceBatch, prepare_repeated

    A, mu = make(name, modes, real)
    p = prepare_repeated(A, rpt, mu=mu if loop else None, loop=loop, glynn=glynn)
    got = DeviceBatch([p])
    got.run()
    ref = DeviceBatch([p], force_generic=True)
    ref.run()
    v, g = got.results()[0], ref.results()[0]
    kw = dict(loop=loop, rpt=rpt, mu=mu if loop else None, glynn=glynn)
    truth = O.hafnian_sieve(A, precision="dd", **kw)
    bar = max(TOL, 2 * relerr(O.hafnian_sieve(A, precision="double", **kw), truth))
    assert relerr(v, truth) < bar, (name, v, truth)
    assert relerr(v, g) < 2 * bar, (name, v, g)
    if real:
        assert v.imag == 0.0 or abs(v.imag) < bar * abs(v)


@pytest.mark.gpu
@pytest.mark.parametrize("E,odd", [(13, False), (16, True), (19, True), (20, False), (23, True), (24, False)])
def test_large_sides_against_general_kernel(E, odd):
    """Tile sides 4 to 6, a few terms each: most edges carry no photon (multiplicity 0)."""
    import ctypes

    from thewalrus_amd import _native
    from thewalrus_amd.batch import PackedJob, layout_packed
    import torch

    rng = np.random.default_rng(E)
    A = random_symmetric(rng, 2 * E, scale=1.0 / np.sqrt(2 * E))
    D = rng.normal(size=2 * E) + 1j * rng.normal(size=2 * E)
    V = rng.normal(size=2 * E) + 1j * rng.normal(size=2 * E)
    vals = []
    for options in (0, 1):
        r = _native.WhRequest()
        r.E, r.glynn, r.options, r.a_off, r.d_off = E, 1, options, 0, 4 * E * E
        r.v_off = 4 * E * E + 2 * E if odd else -1
        if odd:
            r.oddloop[0], r.oddloop[1] = 0.3, -0.2
        for i in range(E):
            r.edge_reps[i] = (0, 2, 1)[i % 3] if i < 18 else 0
        payload = np.concatenate([A.ravel(), D, V] if odd else [A.ravel(), D])
        reqs, pool = layout_packed([PackedJob(payload, r)], np.empty(payload.size, dtype=np.complex128))
        L = _native.load()
        d = torch.from_numpy(pool.view(np.float64).copy()).cuda()
        out = torch.zeros(2, dtype=torch.float64, device="cuda")
        plan = ctypes.c_void_p()
        _native.check(L.wh_plan_create(reqs, 1, 0, ctypes.byref(plan)))
        _native.check(L.wh_plan_run(plan, d.data_ptr(), out.data_ptr(), None))
        torch.cuda.synchronize()
        L.wh_plan_destroy(plan)
        vals.append(complex(*out.cpu().tolist()))
    assert relerr(vals[0], vals[1]) < TOL, vals


def test_layout_keeps_within_the_general_kernels_slots():
    """Partial-sum slots never exceed the general kernel's, so whatever fitted an arena or the
    static scratch still does; tile and wave options stay refused for these requests."""
    import ctypes

    from thewalrus_amd import _native

    L = _native.load()
    rng = np.random.default_rng(5)
    for _ in range(200):
        E = int(rng.integers(1, 25))
        odd = bool(rng.integers(0, 2))
        r = _native.WhRequest()
        r.E, r.glynn, r.a_off, r.d_off, r.v_off = E, 1, 0, 0, 0 if odd else -1
        budget = 60
        for i in range(E):
            r.edge_reps[i] = int(min(rng.integers(1, 5), budget // 2, 4 if i < 12 else 1))
            budget -= r.edge_reps[i]
        slots = []
        for options in (0, 1):
            r.options = options
            n = ctypes.c_int64()
            _native.check(L.wh_request_partials(ctypes.byref(r), 0, ctypes.byref(n)))
            slots.append(n.value)
        if odd:  # even requests may have a kernel class of their own
            assert slots[0] <= slots[1], (E, list(r.edge_reps), slots)
            for options in (2 << 8, 2 << 12):
                r.options = options
                assert L.wh_request_partials(ctypes.byref(r), 0, ctypes.byref(n)) == -1
        elif E <= 8 and sum(r.edge_reps[:E]) <= 16:  # the repeated-row class: its vector kernel's slots
            r.options = (1 if E <= 4 else 2) << 8
            if any(e != 1 for e in r.edge_reps[:E]):
                _native.check(L.wh_request_partials(ctypes.byref(r), 0, ctypes.byref(n)))
                assert slots[0] <= n.value, (E, list(r.edge_reps), slots, n.value)


@pytest.mark.gpu
@pytest.mark.parametrize("modes,fixed,cutoff", [
    (1, [], 1), (1, [], 0), (1, [], 9),          # no fixed edge; no power at all
    (2, [1], 2), (3, [2, 1], 3),                 # tile side 1, odd variant
    (2, [26], 12), (2, [27], 13),                # three series of up to 64 orders side by side or in turn
    (2, [40], 24), (2, [41], 24),                # exactly 64 orders and one more
    (2, [60], 30), (2, [61], 60),                # by rows (more than 64 orders)
    (9, [1] * 8, 4), (10, [1] * 9, 3),           # sides 10 and 12
    (13, [1] * 12, 2), (16, [1] * 15, 2),        # sides 14 and 18
])
def test_loop_hafnian_batch_series_and_tiles(modes, fixed, cutoff):
    from thewalrus_amd.loop_hafnian_batch import loop_hafnian_batch

    rng = np.random.default_rng([modes, cutoff])
    A = random_symmetric(rng, modes, scale=0.5 / np.sqrt(modes))
    D = 0.4 * (rng.normal(size=modes) + 1j * rng.normal(size=modes))
    got = loop_hafnian_batch(A, D, fixed, cutoff)
    truth = O.loop_hafnian_batch(A, D, fixed, cutoff, precision="dd")
    ref = O.loop_hafnian_batch(A, D, fixed, cutoff, precision="double")
    assert got.shape == truth.shape
    for g, t, r in zip(got, truth, ref):
        assert relerr(g, t) < max(TOL, 2 * relerr(r, t)), (modes, fixed, cutoff)


@pytest.mark.gpu
@pytest.mark.parametrize("modes,clicks", [(26, 25), (36, 35), (48, 46)])
def test_loop_hafnian_batch_large_sides(modes, clicks):
    """Tile sides 4 to 6 with few terms: pairs of modes carry no photon but two of them."""
    from thewalrus_amd import _native

    E = modes // 2
    rng = np.random.default_rng(modes)
    A = random_symmetric(rng, 2 * E, scale=0.5 / np.sqrt(modes))
    D = 0.4 * (rng.normal(size=(3, 2 * E)) + 1j * rng.normal(size=(3, 2 * E)))
    reps = [0] * (E - 1)
    reps[2], reps[5], reps[-1] = 2, 1, 1
    got = _native.loop_hafnian_batch(A, D, reps, 2, 1, 0)
    # the empty edges' rows take part in nothing: the same request without them
    keep = [0, 3, 6, E - 1]
    idx = keep + [k + E for k in keep]
    want = _native.loop_hafnian_batch(A[np.ix_(idx, idx)], D[:, idx], [2, 1, 1], 2, 1, 0)
    assert np.all(np.abs(got - want) <= TOL * np.abs(want))
