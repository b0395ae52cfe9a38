"""GPU: quads over few, many and very many tiles (entries by the quad's lane,
through the item's table, straight from the bins' cursors, and ranges too wide
to pack), alone and mixed in one binning item, with all items kept and with
one.  Bit for bit against the oracle's sequential fold."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R

pytestmark = pytest.mark.gpu


def _bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


# quads about `tiles` 16-pixel tiles wide: 4 | 5 around the lane's limit, 15 | 16 around the packed
# range, 64 | 65 around the table's, 0: of any width up to the image's 75 tiles
@pytest.mark.parametrize("keep", [None, "1"])
@pytest.mark.parametrize("tiles", [1, 4, 5, 15, 16, 64, 65, 0])
def test_ranges(torch_cuda, monkeypatch, tiles, keep):
    torch = torch_cuda
    if keep:
        monkeypatch.setenv("RVS_KEEP_ITEMS", keep)
    print("case bin ranges %d tiles keep %s" % (tiles, keep), flush=True)
    rng = np.random.default_rng(tiles)
    w, h, ih, iw = 1203, 45, 11, 70
    gy, gx = np.mgrid[0:ih, 0:iw]
    span = rng.uniform(1, 1200, gx.shape) if tiles == 0 else np.full(gx.shape, 16.0 * tiles - 8.0)
    left = rng.uniform(4, 20, (ih, 1))
    u = left + np.where(gx % 2 == 1, span, 0.0) + rng.normal(0, 1, gx.shape)
    v = gy * 4.3 + rng.normal(0, 0.3, gx.shape) + 0.7
    if tiles == 0:   # small quads among the wide ones
        small = rng.random(gx.shape) < 0.5
        u[small] = (left + gx * 3.0)[small]
    uv = np.stack([u, v], -1).astype(np.float32)
    depth = rng.uniform(1.0, 9.0, (ih, iw)).astype(np.float32)
    col = rng.random((ih, iw, 3)).astype(np.float32)
    ref = ob.transform_triangles(col, depth, uv, w, h, 0)
    out = [torch.empty((h, w) + s, dtype=torch.float32, device="cuda") for s in ((3,), (), ())]
    R.raster(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (col, depth, uv)), w, h, 0, 1.0, *out)
    for a, b in zip(out, ref):
        assert _bits(a.cpu().numpy(), b), (tiles, keep)
