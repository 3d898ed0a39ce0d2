"""The fused Arnoldi step at the edges of its tiles: orders around one lane block (64
rows), around the change of rows per workgroup (4096 | 16384), restarts beyond the 256
coefficients held on chip, and several systems in one step. A is twice the identity plus a
cyclic shift (or the shift alone, on which GMRES makes its progress late), so
|A^-1| <= 1 and |A| <= 3: a relative residual t bounds the error of x by 3 t."""
import numpy as np
import pytest

from hornsculpt_amd import bem, meshes

pytestmark = pytest.mark.gpu


def _shift(n, diagonal):
    A = np.zeros((n, n), dtype=np.complex128, order="F")
    A[np.arange(n), np.arange(n)] += diagonal
    A[(np.arange(n) + 1) % n, np.arange(n)] += 1.0
    return A


@pytest.mark.parametrize("graph", ["0", "1"])
@pytest.mark.parametrize("n,restart,diagonal", [(1, 2, 2), (2, 1, 2), (63, 9, 2), (64, 50, 2), (65, 7, 2), (290, 300, 0),
                                                (4096, 20, 2), (4097, 50, 2), (16385, 50, 2)])
def test_arnoldi_step_solves(monkeypatch, n, restart, diagonal, graph):
    if n > 16384 and graph == "0":
        pytest.skip("one run at this order: the host-driven cycle launches the same kernels")
    monkeypatch.setenv("HSBEM_GMRES_GRAPH", graph)
    rng = np.random.default_rng(n)
    A = _shift(n, diagonal)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    b = diagonal * x + np.roll(x, 1)  # A x
    got, residual, iterations = bem.dense_gmres(A, b, restart, 2000, 1e-11)
    err = np.linalg.norm(got - x) / np.linalg.norm(x)
    print(f"n={n} restart={restart}: {iterations} iterations, residual {residual:.1e}, error {err:.1e}")
    assert residual <= 1e-11 and err <= 3.1e-11
    if diagonal == 0:
        assert iterations > 256


@pytest.mark.parametrize("count", [2, 5])
def test_systems_of_one_step(count):
    # each system drives its own part of the sphere, so they stop at different steps
    sphere = meshes.icosphere(2, 0.1)
    nt = len(sphere.triangles)
    mesh = meshes.SurfaceMesh(sphere.vertices, sphere.triangles, (1 + np.arange(nt) * count // nt).astype(np.uint32),
                              sphere.boundary)
    faces = [bem.BemExcitation(f"e{i}", [bem.FaceVelocity(f, 1.0) for f in range(1, i + 2)]) for i in range(count)]
    out = {}
    for solver in (bem.SOLVER_LU, bem.SOLVER_GMRES):
        req = bem.BemRequest(medium=bem.AcousticMedium(1.205, 343.0), frequencies=[600.0], excitations=faces,
                             numerics=bem.BemNumerics(solver=solver, relative_residual_tolerance=1e-11, gmres_restart=30))
        out[solver] = bem.HipBemSolver(mesh).solve(req).frequencies[0].excitations
    for a, b in zip(out[bem.SOLVER_LU], out[bem.SOLVER_GMRES]):
        p, q = np.asarray(a.boundary.pressure_trace), np.asarray(b.boundary.pressure_trace)
        # residual 1e-11 times the condition of this system, which is below 100
        assert np.linalg.norm(p - q) <= 1e-9 * np.linalg.norm(p)
