"""The weighted operator gives a workgroup as many columns as leave eight workgroups per CU: a column's
iterate is the same bits in a group of several columns, a last group that is not full, or alone."""
import numpy as np
import pytest

from gradientdomaintextureprocessing_amd._lib import GdtpError
from helpers import icosphere_system

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("columns", [7, 9])  # 690 blocks of deep rows: two columns a group, three
def test_groups_of_columns(columns):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, H, S = icosphere_system(512, 4, 4, max_cols=columns)
    deep = (H.level_info(0)["deep"] + 255) // 256
    assert 1 < deep * columns // 2048 < columns
    rng = np.random.default_rng(columns)
    b = torch.from_numpy(rng.standard_normal((columns, H.level_info(0)["texels"]))).cuda()
    weights = [[1.0, 10.0 ** rng.uniform(-4, -2)] for _ in range(columns)]

    def two_steps(b, weights):
        x = torch.zeros_like(b)
        with pytest.raises(GdtpError) as e:  # a fixed number of steps
            S.solve_weighted(x, b, weights, tol=1e-300, max_iters=2)
        assert e.value.code == 3
        return x

    together = two_steps(b, weights)
    assert bool(torch.isfinite(together).all()) and float(together.abs().max()) > 0
    for c in (0, 1, columns - 1):
        assert torch.equal(two_steps(b[c:c + 1].contiguous(), weights[c:c + 1])[0], together[c]), c
