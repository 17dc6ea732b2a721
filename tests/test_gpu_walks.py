"""The montrealer's walk sums (montrealer.hip) at the edges of their forms: one workgroup up to 8
modes, layer launches above, layer buffers of their own from 17 modes on; matrices that are not
symmetric (directions matter) against the enumeration of walks.  The walk sums cancel nothing, so
the closed forms hold to 1e-12: (n + 1) n roundings of a few 1e-16 per walk."""
import numpy as np
import pytest
from scipy.special import factorial2

from oracle import oracle as O
from tests.conftest import relerr
from thewalrus_amd import lmtl, mtl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 8, 9, 10, 15, 16, 17, 18])
def test_all_ones_closed_forms(n):
    J = np.ones((2 * n, 2 * n))
    want = float(factorial2(2 * n - 2))
    assert relerr(mtl(J), want) < 1e-12
    assert relerr(lmtl(J, np.ones(2 * n)), (n + 1) * want) < 1e-12


@pytest.mark.parametrize("n", [2, 3, 4, 5])
def test_nonsymmetric_matrix_against_enumerated_walks(n):
    rng = np.random.default_rng(90 + n)
    A = rng.normal(size=(2 * n, 2 * n)) + 1j * rng.normal(size=(2 * n, 2 * n))
    z = rng.normal(size=2 * n) + 1j * rng.normal(size=2 * n)
    assert relerr(mtl(A), O.mtl_walks(A)) < 1e-12
    assert relerr(lmtl(A, z), O.mtl_walks(A, z)) < 1e-12


def test_sizes_in_turn_reuse_the_buffers():
    """Growing and shrinking sizes, and other calls of the context in between."""
    import thewalrus_amd as tw

    rng = np.random.default_rng(7)
    B = rng.normal(size=(12, 12)) + 1j * rng.normal(size=(12, 12))
    H = (B + B.T) / 2
    first = {}
    for rnd in range(2):
        for n in (9, 3, 14, 17, 8, 11):
            M = np.random.default_rng(n).normal(size=(2 * n, 2 * n))
            v = (mtl(M), tw.hafnian(H), lmtl(M, np.ones(2 * n)))
            if rnd == 0:
                first[n] = v
            assert v == first[n]


@pytest.mark.parametrize("n", [2, 5, 8, 9, 11])
@pytest.mark.parametrize("bad", [np.nan, np.inf, 1j * np.nan])
def test_entries_that_are_not_finite_reach_the_value(n, bad):
    """Also the entries between a mode's own two copies, which no walk takes: the reference's traces
    of Sigma_S^n hold them, and NaN or an infinity there leaves no finite value."""
    from thewalrus_amd._montrealer import lmontrealer, montrealer

    for i, j in [(0, 0), (0, n), (n, 0), (n + 1, 1), (2 * n - 1, 2 * n - 1), (0, 1)]:
        S = np.random.default_rng(n).normal(size=(2 * n, 2 * n)) * (1 + 0j)
        S[i, j] = bad
        assert not np.isfinite(montrealer(S)), (i, j)
        assert not np.isfinite(lmontrealer(S, np.ones(2 * n) * (1 + 0j))), (i, j)
