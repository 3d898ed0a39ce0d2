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
and a quarter units of FP32 in the Frobenius norm.

Tiles of every kind against the FP64 oracle: pairs of degree 4, 6, 8 and 14 sorted within general
tiles, tiles of separated panels below, around and above k h = .5, small meshes whose tiles are
split over several workgroups, near patches of degree 8 and 14 gathered per cluster pair. FP64
entries differ by the order of up to a few hundred additions (1e-12 of the matrix norm), FP32 ones
by FP32 rounding of the same sums (24 bits over some tens of terms: 2e-6)."""
import math

import numpy as np
import pytest

import oracle_bind as ob
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


def _slab(gap):
    """A box of 20 mm by 20 mm by gap, two triangles a side: its faces are near each other."""
    V = np.array([(x, y, z) for z in (0, gap) for y in (0, 0.02) for x in (0, 0.02)], float)
    quads = [(0, 2, 3, 1), (4, 5, 7, 6), (0, 1, 5, 4), (2, 6, 7, 3), (0, 4, 6, 2), (1, 3, 7, 5)]
    T = [t for a, b, c, d in quads for t in ((a, b, c), (a, c, d))]
    return bem.SurfaceMesh(V, np.array(T, np.uint32), np.arange(12, dtype=np.uint32), np.ones(12, np.uint8))


# (mesh, frequency, near tolerance, near patches of degree 14, pairs of degree 14 among the regular ones)
@pytest.mark.parametrize("mesh,frequency,tolerance,near14,whole14",
                         [(meshes.octa_sphere(2), 300.0, 1e-4, False, False), (meshes.octa_sphere(2), 300.0, 1e-6, False, True),
                          (meshes.icosphere(3), 300.0, 1e-4, False, False), (meshes.icosphere(3), 1700.0, 1e-4, False, False),
                          (meshes.icosphere(3), 2500.0, 1e-4, False, False), (_slab(0.002), 1000.0, 1e-4, True, False),
                          (meshes.exponential_horn(0.03), 900.0, 1e-4, True, False)])
def test_tile_kinds_match_oracle(mesh, frequency, tolerance, near14, whole14):
    k, num = 2 * math.pi * frequency / 343.0, bem.BemNumerics(near_relative_tolerance=tolerance)
    plan = bem.interaction_plan(mesh, num, k)
    patches = plan["patches"]
    assert np.any((patches[:, 19] == 14) & (patches[:, 20] == 0)) == near14
    assert (len(plan["whole"]) > 0 and np.any(np.asarray(plan["whole"]) == 14)) == whole14
    A, B = ob.oracle_assemble(mesh, plan, k, tolerance=tolerance)
    solver = bem.HipBemSolver(mesh)
    for precision, bar in ((bem.PRECISION_FP64, 1e-12), (bem.PRECISION_MIXED, 2e-6)):
        got, flux = solver.assemble(bem.BemNumerics(near_relative_tolerance=tolerance, precision=precision), k, k)
        err, errb = (np.linalg.norm(g - w) / np.linalg.norm(w) for g, w in ((got, A), (flux, B)))
        print(f"{len(mesh.triangles)} panels {frequency} Hz precision {precision}: A {err:.1e} B {errb:.1e}")
        assert err <= bar and errb <= bar
