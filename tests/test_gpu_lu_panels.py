"""The LU's panels at the edges of their 64 columns and of the 128 rows per workgroup: one
workgroup (no exchange), two and several, tails of the last panel, matrices that interchange
rows at almost every column and matrices that never do."""
import numpy as np
import pytest

from hornsculpt_amd import bem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs", [(2, 1), (63, 5), (127, 1), (128, 4), (130, 3), (192, 1), (193, 2), (256, 9), (257, 1),
                                    (513, 1), (1089, 6), (2113, 1)])
@pytest.mark.parametrize("pivoted", [True, False])
def test_lu_solution_at_panel_edges(n, nrhs, pivoted):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    if not pivoted:
        A += 4 * n * np.eye(n)
    B = rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))
    X = bem.dense_lu_solve(A, B)
    # partial pivoting: the residual is within a small multiple of sqrt(n) eps of |A||X| for
    # random matrices (growth about n^(2/3)); 4 n eps leaves room for any order of the sums
    residual = np.max(np.abs(A @ X - B)) / (np.linalg.norm(A, np.inf) * np.max(np.abs(X)))
    assert residual <= 4 * n * np.finfo(float).eps
