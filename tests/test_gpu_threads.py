"""Per-call entry points from several threads at once: they share one context (staging blocks, pinned
answer, flag, tensor ring) under its lock, and every answer is its own call's."""
import threading

import numpy as np
import pytest

import thewalrus_amd as tw
from tests.conftest import random_symmetric
from thewalrus_amd._hermite_multidimensional import hafnian_batched
from thewalrus_amd.loop_hafnian_batch import loop_hafnian_batch

pytestmark = pytest.mark.gpu


def test_calls_of_every_kind_side_by_side():
    rng = np.random.default_rng(5)
    H = [random_symmetric(rng, n, scale=0.4) for n in (8, 20, 13, 26)]
    T = 0.3 * random_symmetric(rng, 3)
    mu = 0.3 * rng.normal(size=3)
    work = [lambda: tw.hafnian(H[0], loop=True), lambda: tw.hafnian(H[1]), lambda: tw.hafnian(H[2], loop=True),
            lambda: tw.hafnian(H[3]), lambda: tw.mtl(H[3]), lambda: tw.lmtl(H[1], np.diag(H[1])),
            lambda: loop_hafnian_batch(H[0], np.diag(H[0]), [1, 2, 0, 1, 1, 2, 1], 4),
            lambda: hafnian_batched(T, (60, 41, 53), mu=mu, renorm=True)]
    want = [f() for f in work]
    bad = []

    def loop(k):
        for r in range(12):
            i = (k + r) % len(work)
            try:
                same = np.array_equal(work[i](), want[i])
            except Exception as e:  # pragma: no cover - reported below
                same = e
            if same is not True:
                bad.append((k, i, same))

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
