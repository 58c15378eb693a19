"""The device memory that the host-array entry points keep between a thread's calls: given back after a run of calls
that need much less of it, and all of it when the thread ends."""
import threading
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MIB = 2 ** 20


def free_bytes():
    return torch.cuda.mem_get_info()[0]


def test_memory_is_given_back(rsd):
    small, large = np.eye(10), np.eye(3000)  # rsd_matrev(3000) takes three matrices of 69 MiB
    seen = {}

    def work():
        rsd.matrev(large)
        rsd.matrev(small)
        seen["large"] = free_bytes()
        for _ in range(40):
            rsd.matrev(small)
        seen["small"] = free_bytes()

    t = threading.Thread(target=work)
    t.start()
    t.join()
    # the three matrices but for what the small calls need and the driver's granularity
    assert seen["small"] - seen["large"] >= 180 * MIB, seen


def test_a_thread_that_ends_keeps_nothing(rsd):
    A = np.eye(3000)
    rsd.matrev(np.eye(10))
    start = free_bytes()
    for _ in range(3):
        t = threading.Thread(target=rsd.matrev, args=(A,))
        t.start()
        t.join()
    # (the last destructors run shortly after join() returns; an order of 3000 takes 86 MiB of workspace)
    for _ in range(100):
        if start - free_bytes() <= 16 * MIB:
            break
        time.sleep(0.05)
    assert start - free_bytes() <= 16 * MIB, (start, free_bytes())


def test_sizes_around_a_shrink(rsd):
    """Small calls until the block shrinks, and larger ones straight after: results as ever."""
    def spd(n):
        g = np.random.default_rng(n).standard_normal((n, n))
        return g @ g.T / n + np.eye(n)

    errors = []

    def work():
        try:
            for n in [700] + [20] * 35 + [700, 33, 1200] + [65] * 20 + [900]:
                A = spd(n)
                X, info = rsd.matrev(A)
                assert info == 0
                # forward error of an inverse by Cholesky: a few n eps cond(A), cond <= 6
                ref = np.linalg.inv(A)
                assert np.max(np.abs(X - ref)) <= 4 * 6.0 * n * np.finfo(float).eps * np.max(np.abs(ref)), n
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert not errors, errors
