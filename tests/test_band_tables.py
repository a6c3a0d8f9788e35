"""The tables that the GPU band kernel runs on, rebuilt from the band tasks' segments: per block the chart
rows of its deep rows and one either side, every deep texel of the block once, in its segments' order and
paired with its right neighbour; places, spans and limits as the kernel reads them."""
import os

import numpy as np
import pytest

import gradientdomaintextureprocessing_amd as g


def mesh(name):
    if name == "icosphere":
        return g.TexturedMesh.icosphere(4, 512, 512, 0.05, 7), 512, 512
    if name == "torus":
        return g.TexturedMesh.torus(64, 32, 4, 2, 401, 355, 1.0, 0.35, 0.05, 5), 401, 355
    d = np.load(os.path.join(os.path.dirname(__file__), "golden", "julius_mesh.npz"))
    return g.TexturedMesh.from_arrays(d["vertices"], d["triangles"], d["corner_uv"]), 1024, 1024


@pytest.mark.parametrize("name", ["icosphere", "torus", "julius"])
def test_band_tables_restate_the_segments(name):
    m, width, height = mesh(name)
    H = g.InitializeHierarchy(m, width, height, 2)
    odd = gaps = 0
    for level in range(H.levels):
        n = H.level_info(level)["texels"]
        A = lambda k: H.array(level, "tasks." + k).astype(np.int64)  # noqa: E731
        seg, line_ptr, line_row = A("segments").reshape(-1, 5), A("linePtr"), A("lineRow")
        begin, deep_end = A("blockBegin"), A("blockDeepEnd")
        block_row, rows, pairs = A("bandBlockRow"), A("bandRows").reshape(-1, 4), A("bandPairs").reshape(-1, 4)
        assert block_row[0] == 0 and len(block_row) == len(begin) + 1 and block_row[-1] == len(rows)
        assert rows[:, 3].sum() == len(pairs) and np.array_equal(rows[:, 2], np.cumsum(rows[:, 3]) - rows[:, 3])
        assert rows[:, 3].max() <= 64 and rows[:, 1].max() + 2 <= 136
        assert (rows[:, 0] >= 0).all() and (rows[:, 0] + rows[:, 1] <= n).all()
        for b in range(len(begin)):
            R = rows[block_row[b]:block_row[b + 1]]
            lines = range(begin[b], deep_end[b])
            top = line_row[begin[b]] if len(lines) else 0
            assert len(R) == (line_row[deep_end[b] - 1] - top + 1 if len(lines) else 0) + 2
            own = {line_row[l] - top + 1: l for l in lines}
            assert len(own) == len(lines)
            gaps += len(R) - 2 - len(own)
            for r, (base, length, first, count) in enumerate(R):
                want = []
                if r in own:
                    for s in seg[line_ptr[own[r]]:line_ptr[own[r] + 1]]:
                        size = s[1] - s[0] + 1
                        odd += size % 2
                        for o in range(0, size, 2):
                            want.append((s[0] + o, s[4] + o, s[0] + o - base, s[2] + o - 1 - R[r - 1][0], s[3] + o - 1 - R[r + 1][0],
                                         (1 if o == 0 else 0) | (2 if o + 1 < size else 0)))
                got = [(t, d, p & 255, p >> 8 & 255, p >> 16, f) for t, d, p, f in pairs[first:first + count]]
                assert got == [tuple(int(v) for v in w) for w in want], (level, b, r)
                for _, _, at, above, below, flags in got:  # all that the kernel uses lies in the rows' spans
                    last = 1 if flags & 2 else 0
                    assert 1 <= at and at + last + 1 < length
                    assert 0 <= above and above + last + 2 < R[r - 1][1] and 0 <= below and below + last + 2 < R[r + 1][1]
    assert odd > 0 or name == "torus"  # (its charts are rectangles)
    assert gaps > 0 or name != "julius"
    print(f"[band tables {name}] segments of odd length {odd}, rows without deep texels {gaps}")
