"""GPU: triangles with many pixels in a tile (shared by a wave's lanes in the
raster), at box sizes around the limit, the tile edges and the queue's
capacity.  Bit for bit against the oracle's sequential fold."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R
import workloads as W

pytestmark = pytest.mark.gpu


def _bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


def _stage(torch, uv, depth, w, h, tag):
    print("case wide raster %s" % tag, flush=True)
    col = np.random.default_rng(1).random(depth.shape + (3,)).astype(np.float32)
    ref = ob.transform_triangles(col, depth, uv, w, h, 0)
    out = [torch.empty((h, w) + s, dtype=torch.float32, device="cuda") for s in ((3,), (), ())]
    R.raster(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (col, depth, uv)), w, h, 0, 1.0, *out)
    for a, b in zip(out, ref):
        assert _bits(a.cpu().numpy(), b), tag


# cells of 8 px fill the 64-pixel limit exactly, 8.4 px exceed it; 16 and 40 px span tiles
@pytest.mark.parametrize("cell", [7.3, 8.0, 8.4, 13.0, 16.0, 40.0])
def test_magnified_mesh(torch_cuda, cell):
    rng = np.random.default_rng(int(cell * 10))
    h, w = 150, 203
    ih, iw = int(h / cell) + 3, int(w / cell) + 3
    gy, gx = np.mgrid[0:ih, 0:iw]
    for jitter in (0.0, 0.2):
        uv = np.stack([0.1 + (gx + rng.normal(0, jitter, gx.shape)) * cell,
                       0.1 + (gy + rng.normal(0, jitter, gx.shape)) * cell], -1).astype(np.float32)
        depth = rng.uniform(1.0, 9.0, (ih, iw)).astype(np.float32)
        _stage(torch_cuda, uv, depth, w, h, "cell %g jitter %g" % (cell, jitter))


def test_more_wide_triangles_than_the_queue_holds(torch_cuda):
    """Hundreds of wide triangles over every tile, small ones between them, and
    a few non-finite vertices."""
    rng = np.random.default_rng(5)
    ih, iw = 36, 44
    gy, gx = np.mgrid[0:ih, 0:iw]
    uv = np.stack([gx % 7 * 9.0 + rng.normal(5, 3, gx.shape), gy % 5 * 11.0 + rng.normal(5, 3, gx.shape)],
                  -1).astype(np.float32)
    small = rng.random((ih, iw)) < 0.3
    uv[small] = uv[small].round() * 0.25 + 10
    depth = rng.uniform(0.5, 20, (ih, iw)).astype(np.float32)
    depth[rng.random((ih, iw)) < 0.01] = np.nan
    uv[rng.random((ih, iw)) < 0.01] = np.inf
    _stage(torch_cuda, uv, depth, 70, 61, "queue overflow")


@pytest.mark.parametrize("rig,tile", [("erp4_1080p", 16), ("erp4_1080p", 32), ("persp11_2048", 16),
                                      ("persp11_2048", 32)])
def test_telephoto_views(torch_cuda, rig, tile):
    """Fused views through a narrow field of view: one source quad covers 5 to
    40 pixels a side, up to four and more than four sources."""
    print("case telephoto %s tile %d" % (rig, tile), flush=True)
    rg = W.rig(rig, scale=16)
    planes = W.render_sources(rg)
    srcs = W.device_sources(rg, planes)
    w, h = 226, 150
    for f in (500.0, 3000.0):
        rg["target"] = dict(rg["target"], cam=R.cam(0, w, h, f=(f, f), p=(w / 2, h / 2)), pos=[0.02, 0.01, -0.03],
                            rot=[4.0, 2.0, 1.0])
        t = rg["target"]
        out = R.Synthesizer(srcs, W.device_target(rg), tile=tile).run()
        ref = ob.synthesize(W.oracle_sources(rg, planes, ob), W.oracle_cam(t["cam"], ob), t["pos"], t["rot"],
                            t["bitdepth"], t["blending_exp"])
        for k in ("y", "u", "v"):
            assert np.array_equal(out[k].cpu().numpy().view(np.uint16), ref[k]), (f, k)
        for k in ("color", "depth", "quality", "validity"):
            assert _bits(out[k].cpu().numpy(), ref[k]), (f, k)
