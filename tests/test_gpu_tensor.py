"""Hermite tensors at the edges of their launch and copy forms: innermost positions in LDS or not
(6144 entries), one workgroup or a launch per slice (strides of 8192 entries), one copy chunk, a
ragged last chunk, and more than the pinned ring holds (32 MiB, in parts).  An entry depends on
entries with smaller indices only, by the same operations whatever the cutoffs, so a tensor's
corner is bit for bit the tensor of smaller cutoffs that took another form."""
import numpy as np
import pytest

from tests.conftest import random_symmetric
from thewalrus_amd._hermite_multidimensional import hafnian_batched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cutoffs,smaller", [
    ((70001,), (6145,)), ((6145,), (6144,)), ((6144,), (1,)),
    ((3, 8193), (3, 8192)), ((3, 8192), (2, 3000)), ((2, 79, 78), (2, 78, 78)), ((2, 78, 78), (2, 70, 70)),
    ((257, 257), (91, 91)), ((91, 91), (60, 60)), ((37, 41, 53), (3, 9, 53)), ((1500, 1501), (257, 256)),
    ((9, 8, 7, 6, 5, 4), (3, 8, 2, 6, 5, 1)),
])
@pytest.mark.parametrize("renorm", [False, True])
def test_corner_equals_smaller_tensor(cutoffs, smaller, renorm):
    n = len(cutoffs)
    rng = np.random.default_rng([n, cutoffs[0]])
    A = random_symmetric(rng, n, scale=0.3 / np.sqrt(n))
    mu = 0.3 * (rng.normal(size=n) + 1j * rng.normal(size=n))
    big = hafnian_batched(A, cutoffs, mu=mu, renorm=renorm)
    small = hafnian_batched(A, smaller, mu=mu, renorm=renorm)
    assert big.shape == tuple(cutoffs) and big.flags.owndata and small.shape == tuple(smaller)
    corner = big[tuple(slice(0, c) for c in smaller)]
    assert np.array_equal(corner, small, equal_nan=True)


def test_waiting_threads_sleep():
    """A tensor whose recursion is one long chain (400000 steps in one workgroup, some tenths of a
    second) before the first chunk of its copy: the copying threads must not poll all that while.
    CPU time is that of the calling thread and the runtime's own, at most three cores, where five
    polling helpers make it six and more."""
    import time

    A = np.array([[0.1, 0.02], [0.02, 0.1]])
    mu = np.array([0.01, 0.02])
    hafnian_batched(A, (2, 5000), mu=mu, renorm=True)
    wall, cpu = time.perf_counter(), time.process_time()
    hafnian_batched(A, (2, 400000), mu=mu, renorm=True)
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.05, "the recursion is too short to tell"
    assert cpu < 3.0 * wall, (cpu, wall)


def host_tensor(A, mu, cutoffs):
    """The renormalised recursion of two modes on the host: G[v, :] from the rows v - 1 and v - 2."""
    m, n = cutoffs
    sq = np.sqrt(np.arange(max(m, n)))
    G = np.zeros((m, n), dtype=np.complex128)
    G[0, 0] = 1.0
    for k in range(1, n):
        G[0, k] = (mu[1] * G[0, k - 1] + (A[1, 1] * sq[k - 1] * G[0, k - 2] if k > 1 else 0.0)) / sq[k]
    for v in range(1, m):
        row = mu[0] * G[v - 1]
        if v > 1:
            row = row + A[0, 0] * sq[v - 1] * G[v - 2]
        row[1:] += A[0, 1] * sq[1:n] * G[v - 1, :-1]
        G[v] = row / sq[v]
    return G


@pytest.mark.parametrize("cutoffs", [(257, 257), (1500, 1501), (1448, 1449), (2048, 1024), (2048, 1025)])
def test_every_chunk_of_the_copy(cutoffs):
    """Whole tensors against the host's recursion: ragged last chunks, exactly 32 MiB, and past it.
    With these values every entry lies between 1e-6 and 1 and hardly cancels, so both sides round each of
    its up to 3100 steps a few times: 1e-12 of the entry."""
    A = np.array([[0.99, 0.005], [0.005, 0.99]])
    mu = np.array([0.05 + 0.02j, -0.03j])
    want = host_tensor(A, mu, cutoffs)
    got = hafnian_batched(A, cutoffs, mu=mu, renorm=True)
    assert 1e-6 < np.abs(want).min() and np.abs(want).max() <= 1.0
    assert (np.abs(got - want) < 1e-10 * np.abs(want)).all()
