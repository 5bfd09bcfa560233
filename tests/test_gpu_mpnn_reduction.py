"""The parameter gradient's reduction over tiles of 64 nodes (mpnn.hip,
grad_chunk: up to 24 tiles in one stage, chunks of 24 up to 576 tiles, of the
square root of the tile count above) at the edges of its chunks: the output
gradient lives on one tile, the last or one on either side of a chunk's end,
so a tile left out or taken twice shows in full. Against the oracle with the
device's BF16 rounding, with the bounds of test_gpu_mpnn.py (FP32 accumulation
order): cosine 0.9995 and 1 % in norm for every parameter block."""
import numpy as np
import pytest

import cfdx_dev_amd as cx
import mpnn_oracle as M

pytestmark = pytest.mark.gpu

TILE = 64
BLOCKS = [(0, 64)] + [(64 + 2080 * l, 64 + 2080 * (l + 1)) for l in range(4)] + [(M.OFF_WOUT, M.NPARAMS)]


def _chunk(tiles):
    c = 24
    while c * c < tiles:
        c += 1
    return c


@pytest.mark.parametrize("n", [24 * TILE, 24 * TILE + 1, 576 * TILE - 1, 576 * TILE + 1, 626 * TILE])
def test_gradient_of_one_tile(n):
    rows = np.arange(n)
    cols = np.stack([rows - 1, rows, rows + 1], 1)
    vals = np.stack([np.full(n, -1.0), 2.1 + 0.3 * np.sin(rows), np.full(n, -1.0)], 1)
    ok = (cols >= 0) & (cols < n)
    rowp = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.uint32)
    cols, vals = cols[ok].astype(np.uint32), vals[ok]
    h = cx.NativeAMGPreconditioner(precision="fp32", smoother_fp32="chebyshev")
    assert h.setup(n, rowp, cols, vals), h.last_error()
    rng = np.random.default_rng(n)
    p = (M.init_params(3, out_scale=1.0) + 0.05 * rng.standard_normal(M.NPARAMS)).astype(np.float32)
    net = cx.LearnedStage(params=p)
    g = M.Graph(rowp, cols, vals)
    r = rng.standard_normal(n)
    tiles = (n + TILE - 1) // TILE
    c = _chunk(tiles)
    for t in sorted({0, min(c, tiles) - 1, min(c, tiles - 1), tiles - 1}):
        ge = np.zeros(n)
        ge[t * TILE:(t + 1) * TILE] = rng.standard_normal(len(ge[t * TILE:(t + 1) * TILE]))
        gg = net.vjp(h, r, ge).astype(np.float64)
        go = M.vjp(g, p, r, ge, emulate_bf16=True)
        for a, b in BLOCKS:
            x, y = gg[a:b], go[a:b]
            cos = x @ y / (np.linalg.norm(x) * np.linalg.norm(y))
            assert cos >= 0.9995 and abs(np.linalg.norm(x) / np.linalg.norm(y) - 1) <= 0.01, (t, a, cos)
