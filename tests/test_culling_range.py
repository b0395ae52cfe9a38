"""GPU: perspective culling with depths so large that the sum of a point's
coordinates overflows while each of them is finite: such points belong to
their item's bounding box, and the item is not dropped.  Bit for bit against
the oracle, with a resident culling table and with one built by the call."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prepared", [False, True])
def test_coordinates_whose_sum_overflows(torch_cuda, prepared):
    print("case culling of huge points, prepared %d" % prepared, flush=True)
    rng = np.random.default_rng(3)
    sw, sh = 64, 48
    # (Y, Z) = (0.57..1.55, 0.5..1.24) X with X about 1.8e38: X + Y + Z > 3.7e38 everywhere
    sc = R.cam(0, sw, sh, f=(64.0, 64.0), p=(100.0, 80.0))
    raw = rng.integers(62000, 65536, (sh, sw)).astype(np.uint16)
    planes = [rng.integers(0, 256, s).astype(np.uint8) for s in ((sh, sw), (sh // 2, sw // 2), (sh // 2, sw // 2))]
    # a focal length of one pixel: the whole source lies around the centre of pixel (10, 8)
    tc = R.cam(0, 20, 18, f=(1.0, 1.0), p=(10.5 + 1.06, 8.5 + 0.87))
    s = R.DeviceSource(sc, [0.0] * 3, [0.0] * 3, 8, 16, 1.8e38, 1e4, planes + [raw])
    if prepared:
        s.prepare(R.scale_of(16))
    ref = dict(cam=sc, pos=[0.0] * 3, rot=[0.0] * 3, bd_color=8, bd_depth=16, znear=1.8e38, zfar=1e4)
    rg = dict(sources=[ref], target=dict(cam=tc))
    t = R.make_target(tc, [0.0] * 3, [0.0] * 3, 8, 1.0, R.scale_of(8), R.scale_of(16))
    ref = ob.synthesize(W.oracle_sources(rg, [planes + [raw]], ob), W.oracle_cam(tc, ob), t.pos, t.rot, 8, 1.0)
    assert ref["quality"][8, 10] > 0 and np.isfinite(ref["depth"][8, 10])   # the source is seen
    out = R.Synthesizer([s], t).run()
    for k in ("y", "u", "v"):
        assert np.array_equal(out[k].cpu().numpy(), ref[k]), k
    for k in ("color", "depth", "quality", "validity"):
        assert np.array_equal(out[k].cpu().numpy().view(np.uint32), ref[k].view(np.uint32)), k
