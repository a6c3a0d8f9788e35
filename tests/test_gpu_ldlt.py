"""The staged LDL^T solves on the GPU against SuperLU, at sizes that take each form of them.

Tolerances as for the other exact solves (sliver-support texels make A ill-conditioned, so two exact
solvers agree to cond(A) eps in the plain norm only): relative residual 1e-11, energy norm 1e-10."""
import numpy as np
import pytest
import scipy.sparse.linalg as spla

import oracle
from helpers import cube_system, icosphere_system

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def check(A, solve, n, columns, seed):
    rhs = np.random.default_rng(seed).standard_normal((columns, n))
    b = torch.from_numpy(rhs).cuda()
    x = torch.full_like(b, float("nan"))
    solve(b, x)
    got = x.cpu().numpy()
    res = np.linalg.norm(rhs - (A @ got.T).T, axis=1) / np.linalg.norm(rhs, axis=1)
    want = spla.splu(A.tocsc()).solve(np.ascontiguousarray(rhs.T)).T
    e = got - want
    energy = np.sqrt(np.einsum("ij,ij->i", e, (A @ e.T).T) / np.einsum("ij,ij->i", want, (A @ want.T).T))
    print(f"[ldlt] n={n} columns={columns}: residual {res.max():.1e}, energy {energy.max():.1e}", flush=True)
    assert res.max() < 1e-11 and energy.max() < 1e-10
    solve(b, b)  # in place: the rows are read before any is written
    assert torch.equal(b, x)


# boundary rows: the top alone (1536 and 768 rows), one workgroup per subtree and the top (7680), two such
# stages and the top (43,150 rows)
@pytest.mark.parametrize("make, width, columns", [(cube_system, 128, 1), (cube_system, 512, 4), (icosphere_system, 1024, 5)])
def test_boundary_solve_stages(make, width, columns):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, H, S = make(width, levels=3, max_cols=columns) if make is cube_system else make(width, 5, 3, max_cols=columns)
    for level in range(H.levels - 1):
        L = oracle.level_from_product(H, S, level)
        check(L.bb.scipy(), lambda b, x: S.boundary_solve(level, b, x), L.B, columns, level)


# the full level-0 matrix: a stage of components larger than a workgroup's below the top
@pytest.mark.parametrize("columns", [2, 9])
def test_direct_solve_wide_stage(columns):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, H, S = cube_system(256, 3, max_cols=columns)
    A = oracle.full_matrix(oracle.level_from_product(H, S, 0))
    check(A, lambda b, x: S.direct_solve(x, b), A.shape[0], columns, 5)
