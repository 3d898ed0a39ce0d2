"""The LU's paths that depend on how many workgroups may factor a panel together, at small
orders with that number set by the caller.

A factorization whose workgroups have given up waiting for each other (its status word
starts negative) does nothing more with what the panel should have left behind: every kernel
ends, the call reports it and the next one is not affected."""
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
        bem.dense_lu_solve(A, B, limits=bem.LuLimits(panel_groups=groups, status=-1))
    _check(A, bem.dense_lu_solve(A, B), B)
