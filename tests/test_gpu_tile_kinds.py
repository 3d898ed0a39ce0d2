"""Kinds of panel-pair tiles against each other.

Tiles of separated panels against general ones: with a near tolerance of 4e-5 the plan has
no tile of separated panels (the degree 4 rule is outside its budget), and above k h = .5
every separated pair takes degree 6 either way, so that entries of distant nodes are the same
sums. They are sums of some thousand terms of alternating sign: at the median the two may
differ by 16 units in the last place, in FP64 and in FP32, on a mesh of any size.

Flux columns of the mixed form against the FP64 ones: no further off than with the normal
projections formed in every sample, 2.46e-8 on this sphere.

The matrix of the mixed form against the FP64 one: its largest entries are sums of some forty
touching pairs, the smaller terms first, so that few roundings are those of the whole sum: one
and a quarter units of FP32 in the Frobenius norm."""
import math

import numpy as np
import pytest

from hornsculpt_amd import bem, meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e-4])
@pytest.mark.parametrize("precision,eps", [(bem.PRECISION_FP64, 2.0**-52), (bem.PRECISION_MIXED, 2.0**-23)])
def test_separated_tiles_match_general_ones(precision, eps, scale):
    mesh = meshes.icosphere(4, 0.1 * scale)
    k = 2 * math.pi * 4000.0 / 343.0 / scale
    V, T = np.asarray(mesh.vertices), np.asarray(mesh.triangles, np.int64)
    edges = np.linalg.norm(V[T] - V[np.roll(T, 1, axis=1)], axis=2)
    assert 0.5 < k * edges.max(axis=1).min() and k * edges.max() < 2
    solver = bem.HipBemSolver(mesh)
    A, _ = solver.assemble(bem.BemNumerics(precision=precision), k, k)
    G, _ = solver.assemble(bem.BemNumerics(precision=precision, near_relative_tolerance=4e-5), k, k)
    distant = np.linalg.norm(V[:, None] - V[None], axis=2) > 0.1 * scale
    difference = np.abs(A - G)[distant] / np.abs(G)[distant]
    print(f"median {np.median(difference):.1e}, 99% {np.quantile(difference, .99):.1e}")
    assert np.median(difference) <= 16 * eps


def test_mixed_flux_columns():
    solver = bem.HipBemSolver(meshes.octa_sphere(3))
    k = 2 * math.pi * 1000.0 / 343.0
    _, B = solver.assemble(bem.BemNumerics(), k, k)
    _, B32 = solver.assemble(bem.BemNumerics(precision=bem.PRECISION_MIXED), k, k)
    error = np.linalg.norm(B32 - B) / np.linalg.norm(B)
    print(f"flux columns {error:.2e}")
    assert error <= 2.5e-8


def test_mixed_matrix():
    solver = bem.HipBemSolver(meshes.icosphere(3))
    k = 2 * math.pi * 500.0 / 343.0
    A, _ = solver.assemble(bem.BemNumerics(), k, k)
    A32, _ = solver.assemble(bem.BemNumerics(precision=bem.PRECISION_MIXED), k, k)
    error = np.linalg.norm(A32 - A) / np.linalg.norm(A)
    print(f"matrix {error:.2e}")
    assert error <= 1.25 * 2.0**-23
