"""Residual norms of per-column operators against the oracle's matrices: one to seven columns (chunks of
four, the last one not full) and a mesh with long seam rows.

Tolerance: each residual is a rounded sum of about thirty products of values up to 1 (relative 1e-14 of
the right-hand side's scale) and the residuals are of that scale: 1e-11 as for the other norms."""
import numpy as np
import pytest

import oracle
from helpers import icosphere_system, mass_matrix, stiffness_matrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("columns", [1, 3, 4, 7])
def test_weighted_residual_norms(columns):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, H, S = icosphere_system(300, 4, 3, max_cols=columns)
    L0 = oracle.level_from_product(H, S, 0)
    M, stiff = mass_matrix(H, L0), stiffness_matrix(H, L0)
    rng = np.random.default_rng(columns)
    x, b = rng.standard_normal((columns, L0.N)), rng.standard_normal((columns, L0.N))
    w = np.stack([rng.uniform(0.5, 2, columns), 10.0 ** rng.uniform(-4, -2, columns)], 1)
    r, bn = S.weighted_residual_norms(torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda(), w)
    want = [np.linalg.norm(b[c] - w[c, 0] * (M @ x[c]) - w[c, 1] * (stiff @ x[c])) for c in range(columns)]
    assert np.allclose(r, want, rtol=1e-11, atol=0)
    assert np.allclose(bn, np.linalg.norm(b, axis=1), rtol=1e-12, atol=0)
    again, _ = S.weighted_residual_norms(torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda(), w)
    assert np.array_equal(r, again)
