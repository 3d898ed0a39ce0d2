"""64 x 64 block-Jacobi inverses whose last block is short by one row or holds two rows,
against numpy solves with the same blocks of the near matrix in tree order (1e-10, the
bar of the other block widths: FP64 rounding times the condition of a block)."""
import dataclasses
import math

import numpy as np
import pytest

from hornsculpt_amd import bem, meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh,tail,frequency", [(meshes.exponential_horn(0.02), 63, 200.0), (meshes.icosphere(3), 2, 600.0),
                                                 (meshes.exponential_horn(0.02), 63, 2500.0)])
def test_block_inverses(mesh, tail, frequency):
    n, k = len(mesh.vertices), 2 * math.pi * frequency / 343.0
    assert n % 64 == tail
    num = dataclasses.replace(bem.BemNumerics(), fmm_block_width=64)
    solver = bem.HipBemSolver(mesh)
    near = solver.near_operator(num, k, k, [1], leaf_capacity=32)
    N = np.zeros((n, n), complex)
    N[np.repeat(np.arange(n), np.diff(near["row_offsets"])), near["columns"]] = near["values"]
    shifted = bem.SurfaceMesh(mesh.vertices - mesh.vertices[0], mesh.triangles, mesh.face_ids, mesh.boundary)
    order = bem.parse_support_tree(bem.support_tree(shifted, leaf_capacity=32))["pressure_order"]
    op = solver.fmm_operator(num, k, k, leaf_capacity=32)
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    z = op.precondition(v)
    for b0 in range(0, n, 64):
        idx = order[b0:b0 + 64]
        want = np.linalg.solve(N[np.ix_(idx, idx)], v[idx])
        assert np.linalg.norm(z[idx] - want) <= 1e-10 * np.linalg.norm(want)
    op.close()
