"""A direct solve whose solution takes the right-hand side's place: the same solution and the same relative
residual as into another array, by factorisation and, above 2^20 texels, by V-cycles."""
import numpy as np
import pytest

import gradientdomaintextureprocessing_amd as g

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("width, levels, method", [(128, 3, 0), (1400, 7, 1)])
def test_in_place(width, levels, method):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    H = g.InitializeHierarchy(g.TexturedMesh.cube(16, width, width), width, width, levels)
    S = g.UpdateLinearSystem(H, 1e-3, 1.0, max_cols=2)
    n = H.level_info(0)["texels"]
    assert (n > 1 << 20) == (method == 1)
    b = torch.from_numpy(np.random.default_rng(1).standard_normal((2, n))).cuda()
    x = torch.empty_like(b)
    want, by = S.direct_solve(x, b)
    got, by_in_place = S.direct_solve(b, b)
    assert by == by_in_place == method
    assert torch.equal(x, b) and np.array_equal(got, want) and (want < 1e-10).all()
