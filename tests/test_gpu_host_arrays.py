"""The host-array entry points' staging and scratch memory: matrices on both sides of one staging chunk and of several,
calls of changing sizes from one thread, and calls from several threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spd(n, seed):
    """A symmetric matrix with eigenvalues in [1, 6]."""
    g = np.random.default_rng(seed).standard_normal((n, n))
    return g @ g.T / n + np.eye(n)


def check(rsd, n, seed):
    A = spd(n, seed)
    X, info = rsd.matrev(A)
    assert info == 0
    ref = np.linalg.inv(A)
    # forward error of an inverse by Cholesky: a few n eps cond(A), cond <= 6
    assert np.max(np.abs(X - ref)) <= 4 * 6.0 * n * np.finfo(float).eps * np.max(np.abs(ref))


# a chunk holds 524288 doubles: one chunk up to n = 724, two from 725, an odd last chunk at 1500
@pytest.mark.parametrize("n", [1, 63, 724, 725, 1500])
def test_matrev_across_the_staging_chunks(rsd, n):
    check(rsd, n, n)


def test_calls_of_changing_sizes(rsd):
    for k, n in enumerate([40, 900, 64, 1300, 1299, 10]):
        check(rsd, n, 100 + k)


def test_calls_from_several_threads(rsd):
    errors = []

    def work(seed):
        try:
            for n in (130, 640, 77):
                check(rsd, n, seed + n)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(1000 * t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
