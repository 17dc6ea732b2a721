"""The other routes of calls whose larger buffers are not to be had (wh_debug_fail_allocations): the
montrealer's subset sum instead of its walk sums, a Hermite tensor without its device array or
without the pinned ring of its copy; and the subset sum as plans and batches run it."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import random_symmetric, relerr
from thewalrus_amd import _native, lmtl, mtl
from thewalrus_amd._hermite_multidimensional import hafnian_batched

pytestmark = pytest.mark.gpu


@pytest.fixture
def refused():
    L = _native.load()
    yield L.wh_debug_fail_allocations
    L.wh_debug_fail_allocations(0)


def test_montrealer_without_room_for_its_layers(refused):
    """19 modes (layers past 64 MiB): the subset sum cancels up to 19 / 2 digits of 16, the walk sums none."""
    rng = np.random.default_rng(19)
    A = random_symmetric(rng, 38, scale=0.2)
    z = rng.normal(size=38) + 1j * rng.normal(size=38)
    want = mtl(A), lmtl(A, z)
    for f, args, w in ((mtl, (A,), want[0]), (lmtl, (A, z), want[1])):
        refused(1)
        got = f(*args)
        assert refused(-1) == 0
        assert relerr(got, w) < 1e-6
        assert f(*args) == w  # the next call has its room again


def test_tensor_without_its_device_array(refused):
    A, mu = np.diag([0.1, 0.2]), np.array([0.3, 0.4])
    refused(1)
    with pytest.raises(Exception, match="device tensor"):
        hafnian_batched(A, (2100, 2100), mu=mu, renorm=True)
    assert refused(-1) == 0
    assert hafnian_batched(A, (2, 2), mu=mu, renorm=True)[1, 1] == pytest.approx(0.12)


@pytest.mark.parametrize("cutoffs", [(3, 4), (300, 301)])
def test_tensor_without_pinned_memory(refused, cutoffs):
    rng = np.random.default_rng(3)
    A = random_symmetric(rng, 2, scale=0.2)
    mu = 0.3 * (rng.normal(size=2) + 1j * rng.normal(size=2))
    want = hafnian_batched(A, cutoffs, mu=mu, renorm=True)
    refused(1)
    got = hafnian_batched(A, cutoffs, mu=mu, renorm=True)
    assert refused(-1) == 0
    assert np.isfinite(want).all() and np.array_equal(got, want)


@pytest.mark.parametrize("n", [2, 3, 5, 8, 9, 12])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("loop", [False, True])
def test_subset_sum_plans(n, real, loop):
    """WH_OPT_MONTREALER: A = X Sigma, D = X zeta, V its conjugate."""
    import torch

    from thewalrus_amd.batch import PackedJob, layout_packed

    rng = np.random.default_rng([n, real, loop])
    S = rng.normal(size=(2 * n, 2 * n)) + (0 if real else 1j * rng.normal(size=(2 * n, 2 * n)))
    z = rng.normal(size=2 * n) + (0 if real else 1j * rng.normal(size=2 * n))
    swap = np.r_[n:2 * n, :n]
    r = _native.WhRequest()
    r.E, r.glynn, r.options, r.real, r.a_off = n, 1, 4, int(real), 0
    r.d_off, r.v_off = (4 * n * n, 4 * n * n + 2 * n) if loop else (-1, -1)
    for i in range(n):
        r.edge_reps[i] = 1
    parts = [S[swap].ravel()] + ([z[swap], z[swap].conj()] if loop else [])
    payload = np.concatenate(parts).astype(np.complex128)
    reqs, pool = layout_packed([PackedJob(payload, r)], np.empty(payload.size, dtype=np.complex128))
    L = _native.load()
    d = torch.from_numpy(pool.view(np.float64).copy()).cuda()
    out = torch.zeros(2, dtype=torch.float64, device="cuda")
    plan = ctypes.c_void_p()
    _native.check(L.wh_plan_create(reqs, 1, 0, ctypes.byref(plan)))
    _native.check(L.wh_plan_run(plan, d.data_ptr(), out.data_ptr(), None))
    torch.cuda.synchronize()
    got = complex(*out.cpu().numpy())
    L.wh_plan_destroy(plan)
    truth = O.montrealer(S, z if loop else None, precision="dd")
    ref = relerr(O.montrealer(S, z if loop else None, precision="double"), truth)
    assert relerr(got, truth) < max(1e-10, 2 * ref)
