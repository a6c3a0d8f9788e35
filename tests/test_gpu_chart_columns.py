"""Levels swept one chart per workgroup: after a fixed number of refinement steps a column's iterate is the
same bits alone and with others, with both smoother stencils, for one texel of each colour per thread
and for two."""
import numpy as np
import pytest

import gradientdomaintextureprocessing_amd as g
from gradientdomaintextureprocessing_amd._lib import GdtpError

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("kind, width, height", [("cube", 300, 333), ("icosphere", 301, 277)])
def test_columns_alone_and_together(kind, width, height, half, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if not half:
        monkeypatch.setenv("GDTP_FP16_RATIO_LIMIT", "1e-9")  # the FP32 smoother stencil
    m = g.TexturedMesh.cube(16, width, height) if kind == "cube" else g.TexturedMesh.icosphere(4, width, height, 0.05, 3)
    H = g.InitializeHierarchy(m, width, height, 4)
    planes = [max(((w + 1) // 2) * ((h + 1) // 2) for w, h in H.array(l, "charts").reshape(-1, 9)[:, :2]) for l in range(3)]
    assert 1024 < max(planes) <= 2048 and min(planes) <= 1024, planes  # two texels of a colour per thread, and one
    S = g.UpdateLinearSystem(H, 1e-3, 1.0, max_cols=5)
    b = torch.from_numpy(1e-4 * np.random.default_rng(1).standard_normal((5, H.level_info(0)["texels"]))).cuda()

    def two_steps(b):
        x = torch.zeros_like(b)
        with pytest.raises(GdtpError) as e:  # a fixed number of steps
            S.solve(x, b, tol=1e-300, max_iters=2)
        assert e.value.code == 3
        return x

    together = two_steps(b)
    assert bool(torch.isfinite(together).all()) and float(together.abs().max()) > 0
    for c in range(5):
        assert torch.equal(two_steps(b[c:c + 1].contiguous())[0], together[c]), c
