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
