"""Translations on matrix tiles at the edges of their sizes: degrees whose blocks end
within, at and beyond one to four row tiles (every degree up to orders 24 to 30), chunks of
one to sixteen links, deep trees whose levels have different source and target orders. The operator against the dense device
matrix to the accuracy of the multipole form (2e-6), its FP32 form against the FP64 one to
FP32 rounding of the expansions (1e-5)."""
import math

import numpy as np
import pytest

from hornsculpt_amd import bem, meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge,frequency,leaf_capacity", [(0.02, 100.0, 8), (0.02, 2500.0, 16), (0.012, 1500.0, 12),
                                                          (0.012, 8000.0, 48), (0.012, 8000.0, 200)])
def test_translations_match_dense(edge, frequency, leaf_capacity):
    mesh = meshes.exponential_horn(edge)
    k = 2 * math.pi * frequency / 343.0
    solver = bem.HipBemSolver(mesh)
    A, _ = solver.assemble(bem.BemNumerics(), k, k)
    op = solver.fmm_operator(bem.BemNumerics(), k, k, leaf_capacity=leaf_capacity)
    st = op.statistics()
    rng = np.random.default_rng(5)
    x = rng.standard_normal(A.shape[0]) + 1j * rng.standard_normal(A.shape[0])
    y = op.apply(x)
    err = np.linalg.norm(y - A @ x) / np.linalg.norm(A @ x)
    err32 = np.linalg.norm(op.apply_fp32(x) - y) / np.linalg.norm(y) if max(st["level_orders"]) <= 48 and not \
        st["plane_wave_levels"] else 0.0
    print(f"orders {st['level_orders']} m2l {st['m2l_links']}: {err:.2e}, FP32 {err32:.2e}")
    assert st["m2l_links"] > 0 and err <= 2e-6 and err32 <= 1e-5
    op.close()
