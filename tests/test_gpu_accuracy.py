"""Rounding errors of the symmetric-power kernels in the mean over many inputs: the geometric mean
of the relative errors against double-double values is no larger than that of the reference's own
algorithm in double precision (the oracle) on the same inputs.  Single results scatter by factors
of ten, so a sum or product of lower quality shows only in such a mean."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import random_symmetric
from thewalrus_amd.batch import DeviceBatch, prepare_repeated

pytestmark = pytest.mark.gpu


def cases():
    """(modes, least and most photons or None for one each, loop, real, glynn, count): odd N with one term
    per wave and with four, plain repeated rows, even loops, inclusion-exclusion."""
    return [(7, None, True, False, True, 400), (11, None, True, False, True, 400), (15, None, True, False, True, 300),
            (6, (11, 17), True, False, True, 400), (12, (19, 23), True, False, True, 300),
            (6, (12, 16), True, False, True, 400), (12, (18, 22), False, False, True, 300),
            (12, (18, 22), True, True, True, 200),
            (10, None, False, False, False, 400), (16, None, False, False, False, 400)]


@pytest.mark.parametrize("modes,photons,loop,real,glynn,count", cases())
def test_mean_error_no_larger_than_the_reference_algorithms(modes, photons, loop, real, glynn, count):
    rng = np.random.default_rng([modes, count, loop, real])
    jobs = []
    for k in range(count):
        A = random_symmetric(rng, modes, complex_=not real, scale=1.0 / np.sqrt(modes))
        mu = rng.normal(size=modes) + (0 if real else 1j * rng.normal(size=modes))
        rpt = [1] * modes
        if photons:
            n = photons[0] + 2 * (k % ((photons[1] - photons[0]) // 2 + 1))
            rpt = [int(x) for x in rng.multinomial(n, [1.0 / modes] * modes)]
        jobs.append((A, rpt, mu if loop else None))
    b = DeviceBatch([prepare_repeated(A, rpt, mu=mu, loop=loop, glynn=glynn) for A, rpt, mu in jobs])
    b.run()
    logs = []
    for got, (A, rpt, mu) in zip(b.results(), jobs):
        kw = dict(loop=loop, rpt=rpt, mu=mu, glynn=glynn)
        truth = O.hafnian_sieve(A, precision="dd", **kw)
        ours, ref = (abs(x - truth) / abs(truth) + 1e-17 for x in (got, O.hafnian_sieve(A, precision="double", **kw)))
        logs.append(np.log(ours) - np.log(ref))
    assert np.exp(np.mean(logs)) <= 1.0
