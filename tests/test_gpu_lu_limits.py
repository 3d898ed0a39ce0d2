"""The LU's paths that depend on how many workgroups may factor a panel together, at small
orders with that number set by the caller.

A factorization whose workgroups have given up waiting for each other (its status word
starts negative) does nothing more with what the panel should have left behind: every kernel
ends, and the call factors its matrix again on one workgroup per panel, or reports it where
that is left out. Factorizations that together want more workgroups than the GPU has wait for
each other."""
import threading

import numpy as np
import pytest

from hornsculpt_amd import bem

pytestmark = pytest.mark.gpu


def _system(n, nrhs, seed=0):
    rng = np.random.default_rng(n + seed)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return A, rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))


def _check(A, X, B):
    # the bar of the other LU tests: 4 n eps |A| |X|
    residual = np.max(np.abs(A @ X - B)) / (np.linalg.norm(A, np.inf) * np.max(np.abs(X)))
    assert residual <= 4 * len(A) * np.finfo(float).eps


@pytest.mark.parametrize("n,groups", [(64, 0), (129, 0), (321, 0), (321, 1), (1089, 0), (1089, 2)])
def test_given_up_panel_is_reported(n, groups):
    A, B = _system(n, 2)
    with pytest.raises(RuntimeError, match="resident"):
        bem.dense_lu_solve(A, B, limits=bem.LuLimits(panel_groups=groups, status=-1, once=1))
    _check(A, bem.dense_lu_solve(A, B), B)


@pytest.mark.parametrize("n", [64, 129, 321, 1089])
def test_given_up_panel_is_factored_again(n):
    A, B = _system(n, 3)
    _check(A, bem.dense_lu_solve(A, B, limits=bem.LuLimits(status=-1)), B)


def test_concurrent_factorizations():
    # 10 streams at once, 40 panel workgroups each: more than the GPU has compute units
    A, B = _system(4099, 1)
    out = [None] * 10

    def work(i):
        out[i] = bem.dense_lu_solve(A, B * (i + 1), bem.Context())

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(out))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    _check(A, out[0], B)
    for i, x in enumerate(out):
        # the same system up to the order of the sums: a random matrix of this order has a condition below 1e6
        assert np.linalg.norm(x - out[0] * (i + 1)) <= 1e-9 * np.linalg.norm(x)


# one workgroup takes panels of more than 128 rows a limit's workgroup: 4 columns at a time, pairs of 32
# columns, until few enough rows are left (the hand-over to 64-column panels at k0 > 0), and the
# interchanges of the right-hand sides go through memory
@pytest.mark.parametrize("n,nrhs,groups", [(129, 1, 1), (193, 2, 1), (257, 3, 1), (257, 1, 2), (321, 9, 1), (449, 2, 2),
                                           (513, 1, 1), (513, 4, 2), (1091, 5, 3), (2113, 1, 7)])
@pytest.mark.parametrize("pivoted", [True, False])
def test_panels_beyond_the_limit(n, nrhs, groups, pivoted):
    A, B = _system(n, nrhs)
    if not pivoted:
        A += 4 * n * np.eye(n)
    X = bem.dense_lu_solve(A, B, limits=bem.LuLimits(panel_groups=groups, permute_rows=1))
    _check(A, X, B)
    _check(A, bem.dense_lu_solve(A, B, limits=bem.LuLimits(panel_groups=groups)), B)


@pytest.mark.parametrize("groups", [0, 1, 2])
@pytest.mark.parametrize("column", [0, 3, 130, 300])
def test_zero_pivot_beyond_the_limit(groups, column):
    A, B = _system(301, 1)
    A[:, column] = 0
    with pytest.raises(RuntimeError, match=f"pivot {column + 1}$"):
        bem.dense_lu_solve(A, B, limits=bem.LuLimits(panel_groups=groups))


def test_many_panel_workgroups():
    # 73 workgroups of one panel, an odd tail
    A, B = _system(9217, 1)
    _check(A, bem.dense_lu_solve(A, B), B)
