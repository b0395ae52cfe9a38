"""GPU: meshes whose pixels lie on shared edges and under repeated quads, so
that candidates tie exactly (the first in traversal order wins) or nearly (the
replay decides), for small and wide triangles, up to four and more sources.
Bit for bit against the oracle's sequential fold."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R
import workloads as W

pytestmark = pytest.mark.gpu


def _bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


def _ulps(x, n):
    return (np.ascontiguousarray(x, np.float32).view(np.int32) + np.asarray(n, np.int32)).view(np.float32)


# cell: 1 px shares every centre, 2 px every other one; 12 and 40 px are wide triangles
@pytest.mark.parametrize("near", [0, 1, 3])
@pytest.mark.parametrize("cell,off", [(1.0, 0.5), (1.0, 0.25), (2.0, 0.5), (12.0, 0.5), (40.0, 0.5)])
def test_aligned_mesh(torch_cuda, cell, off, near):
    torch = torch_cuda
    print("case ties cell %g off %g near %d" % (cell, off, near), flush=True)
    rng = np.random.default_rng(int(cell * 4 + near))
    w, h = 75, 53
    iw, ih = int(w / cell) + 3, int(h / cell) + 3
    gy, gx = np.mgrid[0:2 * ih, 0:iw]
    gy = gy % ih   # the mesh twice: every quad has an exact copy later on
    uv = np.stack([gx * cell + off, gy * cell + 0.5], -1).astype(np.float32)
    depth = np.full(gx.shape, 3.0, np.float32)
    depth[:, iw // 2:] = 2.0
    # some vertices a few ulps off: near ties beside the exact ones
    depth = _ulps(depth, np.where(rng.random(gx.shape) < 0.1, rng.integers(-near, near + 1, gx.shape), 0))
    col = rng.random(gx.shape + (3,)).astype(np.float32)
    ref = ob.transform_triangles(col, depth, uv, w, h, 0)
    out = [torch.empty((h, w) + s, dtype=torch.float32, device="cuda") for s in ((3,), (), ())]
    R.raster(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (col, depth, uv)), w, h, 0, 1.0, *out)
    for a, b in zip(out, ref):
        assert _bits(a.cpu().numpy(), b), (cell, off, near)


@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("ns", [2, 5])
def test_aligned_cameras(torch_cuda, ns, tile):
    """Unrotated cameras on a line looking at a plane and a box before it."""
    print("case ties %d cameras tile %d" % (ns, tile), flush=True)
    rng = np.random.default_rng(ns)
    w, h, f = 98, 66, 80.0
    c, srcs, refs = R.cam(0, w, h, f=(f, f), p=(w / 2.0, h / 2.0)), [], []
    for k in range(ns):
        raw = np.full((h, w), 6000, np.uint16)
        raw[20:45, 30 + 2 * k:60 + 2 * k] = 30000
        planes = [rng.integers(0, 256, s).astype(np.uint8) for s in ((h, w), (h // 2, w // 2), (h // 2, w // 2))]
        pos = [0.0, 0.05 * (k - ns / 2), 0.0]
        srcs.append(R.DeviceSource(c, pos, [0.0] * 3, 8, 16, 1.0, 10.0, planes + [raw]))
        refs.append(dict(cam=c, pos=pos, rot=[0.0] * 3, bd_color=8, bd_depth=16, znear=1.0, zfar=10.0))
    t = R.make_target(c, [0.0, 0.013, 0.0], [0.0] * 3, 8, 1.0, R.scale_of(8), R.scale_of(16), tile=tile)
    rg = dict(sources=refs, target=dict(cam=c, pos=[0.0, 0.013, 0.0], rot=[0.0] * 3, bitdepth=8, blending_exp=1.0))
    planes = [[p.cpu().numpy().view(np.uint16) if p.dtype.itemsize == 2 else p.cpu().numpy() for p in s.planes]
              for s in srcs]
    out = R.Synthesizer(srcs, t).run()
    ref = ob.synthesize(W.oracle_sources(rg, planes, ob), W.oracle_cam(c, ob), t.pos, t.rot, 8, 1.0)
    for k in ("y", "u", "v"):
        assert np.array_equal(out[k].cpu().numpy(), ref[k]), k
    for k in ("color", "depth", "quality", "validity"):
        assert _bits(out[k].cpu().numpy(), ref[k]), k
