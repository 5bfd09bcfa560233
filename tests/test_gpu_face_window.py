"""The cell window of the face-list operators (fv.hip, accumulate_faces) at
its edges: chunk remainders, owners that span exactly the window and one cell
more, neighbours inside and far outside it, an ungrouped list, boundary faces
only, and an out-of-range index in the last chunk. Against the oracle's
ordered sums, to 1e-12 of the field (the FP64 atomics arrive in no order; a
cell here sums at most a few dozen terms)."""
import numpy as np
import pytest

import cfdx_dev_amd as cx
from hipmem import DeviceArray
from oracle import face_divergence, face_gradient_gauss
from test_gpu_face_ops import _close, _gpu_divergence, _gpu_gradient

pytestmark = pytest.mark.gpu

CHUNK, W3, W1 = 2048, 1280, 4096


def _lists():
    rng = np.random.default_rng(8)
    for nf in (1, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK + 77):
        own = np.sort(rng.integers(0, max(1, nf // 3), nf))
        yield f"grouped_{nf}", own, own + rng.choice([1, 30, 900, 50000], nf), 60000
    for span in (W3, W3 + 1, W1, W1 + 1):
        own = np.sort(np.concatenate([[0, span - 1], rng.integers(0, span, CHUNK - 2)]))
        yield f"span_{span}", own, (own + 1) % span, span
    own = rng.integers(0, 70000, 9001)
    yield "ungrouped", own, rng.permutation(own), 70000
    own = np.sort(rng.integers(500, 900, 5000))
    yield "boundary", own, np.full(5000, -1), 901


@pytest.mark.parametrize("name,own,nei,nc", list(_lists()), ids=[c[0] for c in _lists()])
def test_window_edges(name, own, nei, nc):
    rng = np.random.default_rng(5)
    nf = len(own)
    owner, neighbour = own.astype(np.uint32), nei.astype(np.int64)
    neighbour[rng.random(nf) < 0.1] = -1
    s = rng.normal(size=(3, nf))
    phi, vol = rng.normal(size=nc), rng.uniform(0.5, 2.0, nc)
    vol[0] = 0.0
    args = (phi, *s, owner, neighbour, vol)
    _close(_gpu_gradient(*args), face_gradient_gauss(*args))
    _close(_gpu_divergence(s[0], owner, neighbour, nc), face_divergence(s[0], owner, neighbour, nc))


def test_bad_index_is_reported():
    nf, nc = 2 * CHUNK + 5, 400
    owner = np.sort(np.arange(nf, dtype=np.uint32) % nc)
    owner[-1] = nc
    neighbour = np.full(nf, -1, np.int64)
    d = [DeviceArray(a) for a in (np.ones(nf), owner, neighbour, np.zeros(nc))]
    with pytest.raises(RuntimeError):
        cx.divergence_device(d[0].ptr, d[1].ptr, d[2].ptr, nf, nc, d[3].ptr)
    assert d[3].download().sum() == nf - 1
