"""The dataflow Cholesky's order of tasks, played through on the CPU: every tile is one task's, and every order finishes
with the workgroups that the kernel's text and its launches count on."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def dag(tmp_path_factory):
    out = tmp_path_factory.mktemp("dag") / "libdag.so"
    src = os.path.join(ROOT, "tests", "host", "dag_host.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", src, "-o", str(out)], check=True)
    return C.CDLL(str(out))


# (single tiles below 136 block columns, macro tasks from there on; 172, 242 and 705: 11N of N = 997, 1400 and 4096)
SIZES = list(range(1, 33)) + [58, 88, 110, 135, 136, 137, 138, 141, 172, 242, 705]


def trailing(nt):
    """First block columns of X = inv(L_S): none, the last one, that of a 6N Schur complement in 11N, and all."""
    return sorted({-1, nt - 1, (5 * nt + 10) // 11 if nt > 1 else 0, 0})


@pytest.mark.parametrize("nt", SIZES)
def test_every_tile_is_one_tasks(dag, nt):
    assert dag.dag_covers(nt, 0) == 0
    assert nt < dag.dag_macro_tiles() or dag.dag_covers(nt, 1) == 0
    assert dag.dag_x_covers(nt) == 0


@pytest.mark.parametrize("nt", SIZES)
@pytest.mark.parametrize("cus", [256, 32])
def test_launches_have_the_workgroups_that_they_need(dag, nt, cus):
    macro = int(nt >= dag.dag_macro_tiles())
    for s0 in trailing(nt):
        total, need = dag.dag_total(nt, macro, s0), 1 + dag.dag_beside()
        n = dag.dag_launch(nt, macro, s0, cus)
        assert min(total, need) <= n <= min(total, cus)
        # no more than the stated number resident, whatever the launch asked for
        if nt <= 242:
            assert dag.dag_play(nt, macro, s0, min(n, need)) == 0


def test_the_bound_is_the_least(dag):
    """With one workgroup fewer the macro order stops for good, so a change of the order that needs more shows here."""
    nt = dag.dag_macro_tiles()
    assert dag.dag_play(nt, 1, -1, dag.dag_beside()) > 0
    assert dag.dag_play(nt, 1, -1, dag.dag_beside() + 1) == 0
