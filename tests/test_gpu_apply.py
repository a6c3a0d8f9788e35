"""Operator application, residual, residual norms and restriction against the oracle where their forms
differ: one to seven columns (chunks of three, last one not full) on a mesh with long seam rows.

Tolerance: the rows' terms are added in the oracle's order; deep rows are a chain of nine fused
multiply-adds against nine rounded ones: 1e-13 of the largest value."""
import numpy as np
import pytest

import oracle
from helpers import icosphere_system, mass_matrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("columns", [1, 2, 4, 7])
def test_apply_residual_norms_restrict(columns):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, H, S = icosphere_system(300, 4, 3, max_cols=columns)
    L = [oracle.level_from_product(H, S, l) for l in range(2)]
    A, M = oracle.full_matrix(L[0]), mass_matrix(H, L[0])
    rng = np.random.default_rng(columns)
    x, b = rng.random((columns, L[0].N)), 1e-4 * rng.random((columns, L[0].N))
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    rel = lambda got, want: np.abs(got.cpu().numpy() - want).max() / np.abs(want).max()  # noqa: E731
    out = torch.full((columns, L[0].N), float("nan"), dtype=torch.float64, device="cuda")
    S.apply(1, dev(x), out)
    assert rel(out, (M @ x.T).T) < 1e-13
    S.residual(dev(x), dev(b), out)
    want = b - (A @ x.T).T
    assert rel(out, want) < 1e-13
    _, r, bn = S.residual_norms(dev(x), dev(b))
    assert np.allclose(r, np.linalg.norm(want, axis=1), rtol=1e-12) and np.allclose(bn, np.linalg.norm(b, axis=1), rtol=1e-12)
    coarse = torch.full((columns, L[1].N), float("nan"), dtype=torch.float64, device="cuda")
    S.restrict(0, dev(want), coarse)
    assert rel(coarse, oracle.restrict(L[0], L[1], want)) < 1e-13
