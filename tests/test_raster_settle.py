"""GPU: exact ties settled by the fused raster (aligned cameras, up to four
sources): magnified meshes whose edges lie on pixel centres, of one depth and
of depth codes a step or two apart (candidates that differ by an ulp or by
less than the raster tells apart, left to the replay), with triangles shared by
a wave's lanes and more of them in a tile than their queue holds.  Bit for bit
against the oracle's sequential fold."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R
import workloads as W

pytestmark = pytest.mark.gpu

SW, SH, F = 80, 36, 10.0


def _codes(kind, rng):
    """16-bit inverse-depth codes and the depth range (near, far)."""
    if kind == "plane":
        return np.full((SH, SW), 30000), (1.0, 1.05)
    if kind == "near":   # depths 7e-7 apart
        return 30000 + np.kron(rng.integers(-2, 3, (SH // 2, SW // 2)), np.ones((2, 2), int)), (1.0, 1.05)
    # columns in turn near and far: quads stretched across many others
    return np.broadcast_to(np.where(np.arange(SW) % 2, 60000, 20000), (SH, SW)), (1.0, 10.0)


def _wide(srcs, t, tile):
    """Most triangles with more than 64 pixels of a tile in their boxes, over the tiles."""
    w, h = t.cam.w, t.cam.h
    n = np.zeros((-(-h // tile), -(-w // tile)), int)
    for s, raw in srcs:
        d = ob.decode_depth(raw, 16, s.znear, s.zfar, True)
        Rm, tr = ob.relative_pose(s.pos, s.rot, list(t.pos), list(t.rot))
        uv = ob.reproject(W.oracle_cam(s.cam, ob), W.oracle_cam(t.cam, ob), Rm, tr, d)[0]
        a, b, c, e = uv[:-1, :-1], uv[:-1, 1:], uv[1:, :-1], uv[1:, 1:]
        for p, q, r in ((a, b, c), (e, c, b)):
            den = (q[..., 1] - r[..., 1]) * (p[..., 0] - r[..., 0]) + (r[..., 0] - q[..., 0]) * (p[..., 1] - r[..., 1])
            lo, hi = np.minimum(np.minimum(p, q), r)[den > 0], np.maximum(np.maximum(p, q), r)[den > 0]
            for ty in range(n.shape[0]):
                for tx in range(n.shape[1]):
                    x = np.minimum(hi[:, 0], tx * tile + tile) - np.maximum(lo[:, 0], tx * tile)
                    y = np.minimum(hi[:, 1], ty * tile + tile) - np.maximum(lo[:, 1], ty * tile)
                    n[ty, tx] += int(((x > 1) & (y > 1) & ((x - 1) * (y - 1) > 64)).sum())
    return n.max()


# cells of 8 px fill the 64-pixel limit of a lane's own triangle, 10, 12 and 40 px exceed it
@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("kind,cell,ns,axis", [
    ("plane", 2, 2, 1), ("near", 2, 3, 1), ("plane", 8, 1, 1), ("near", 8, 2, 2), ("plane", 10, 3, 1),
    ("near", 10, 4, 1), ("plane", 12, 4, 2), ("near", 12, 2, 1), ("plane", 40, 2, 1), ("near", 40, 4, 2),
    ("columns", 6, 4, 1), ("columns", 6, 1, 1)])
def test_settled(torch_cuda, kind, cell, ns, axis, tile):
    print("case settle %s cell %d sources %d axis %d tile %d" % (kind, cell, ns, axis, tile), flush=True)
    rng = np.random.default_rng(cell * 8 + ns)
    w, h, ft = 150, 118, F * cell
    sc = R.cam(0, SW, SH, f=(F, F), p=(SW / 2.0, SH / 2.0))
    tc = R.cam(0, w, h, f=(ft, ft), p=(w / 2 + 0.5, h / 2 + 0.5))   # edges on pixel centres
    codes, (near, far) = _codes(kind, rng)
    base = 1.2 if kind == "columns" else 3.0 / ft    # across the columns' shift; of a few pixels
    srcs, refs, raws = [], [], []
    for k in range(ns):
        raw = codes.astype(np.uint16)
        planes = [rng.integers(0, 256, s).astype(np.uint8) for s in ((SH, SW), (SH // 2, SW // 2), (SH // 2, SW // 2))]
        pos = [0.0, 0.0, 0.0]
        pos[axis] = base * (k + 1)
        srcs.append(R.DeviceSource(sc, pos, [0.0] * 3, 8, 16, near, far, planes + [raw]))
        refs.append(dict(cam=sc, pos=pos, rot=[0.0] * 3, bd_color=8, bd_depth=16, znear=near, zfar=far))
        raws.append(planes + [raw])
    t = R.make_target(tc, [0.0] * 3, [0.0] * 3, 8, 1.0, R.scale_of(8), R.scale_of(16), tile=tile)
    if kind == "columns" and ns == 4:
        assert _wide([(s, p[3]) for s, p in zip(srcs, raws)], t, tile) > 100 * (tile // 16) ** 2
    rg = dict(sources=refs, target=dict(cam=tc, pos=[0.0] * 3, rot=[0.0] * 3, bitdepth=8, blending_exp=1.0))
    out = R.Synthesizer(srcs, t).run()
    ref = ob.synthesize(W.oracle_sources(rg, raws, ob), W.oracle_cam(tc, ob), t.pos, t.rot, 8, 1.0)
    for k in ("y", "u", "v"):
        assert np.array_equal(out[k].cpu().numpy(), ref[k]), k
    for k in ("color", "depth", "quality", "validity"):
        assert np.array_equal(out[k].cpu().numpy().view(np.uint32), ref[k].view(np.uint32)), k
