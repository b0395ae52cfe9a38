"""GPU: decoded colour and depth, and the resident colour plane, at sizes
around the four-pixel, two-row threads (even sizes, remainders of two columns)
and odd ones, 8 and 16 bit.  Bit for bit against the oracle's decoding and a
view made from unprepared sources."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bd", [8, 10, 16])
@pytest.mark.parametrize("w,h", [(2, 2), (4, 2), (6, 4), (254, 6), (256, 8), (258, 10), (514, 2), (7, 5), (255, 9)])
def test_decode(torch_cuda, w, h, bd):
    torch = torch_cuda
    print("case decode %dx%d %d bit" % (w, h, bd), flush=True)
    rng = np.random.default_rng(w * h + bd)
    dt = np.uint8 if bd <= 8 else np.uint16
    y, u, v = (rng.integers(0, 1 << bd, s).astype(dt) for s in ((h, w), (h // 2, w // 2), (h // 2, w // 2)))
    raw = rng.integers(0, 1 << bd, (h, w)).astype(dt)
    dev = [torch.from_numpy(p.view(np.int16) if dt == np.uint16 else p).cuda() for p in (y, u, v, raw)]
    col = torch.empty((h, w, 3), dtype=torch.float32, device="cuda")
    dep = torch.empty((h, w), dtype=torch.float32, device="cuda")
    R.decode_yuv420(*dev[:3], bd, R.scale_of(bd), col)
    R.decode_depth(dev[3], bd, R.scale_of(bd), 0.5, 25.0, True, dep)
    assert np.array_equal(col.cpu().numpy(), ob.decode_color(y, u, v, bd))
    assert np.array_equal(dep.cpu().numpy(), ob.decode_depth(raw, bd, 0.5, 25.0), equal_nan=True)


@pytest.mark.parametrize("bd", [8, 10, 16])
@pytest.mark.parametrize("w,h", [(66, 34), (68, 36), (70, 38), (67, 35)])
def test_prepared_sources(torch_cuda, w, h, bd):
    torch = torch_cuda
    print("case prepared %dx%d %d bit" % (w, h, bd), flush=True)
    rng = np.random.default_rng(bd)
    dt = np.uint8 if bd <= 8 else np.uint16
    planes = [rng.integers(0, 1 << bd, s).astype(dt) for s in ((h, w), (h // 2, w // 2), (h // 2, w // 2))]
    planes.append(rng.integers(20000, 60000, (h, w)).astype(np.uint16))
    c = R.cam(0, w, h, f=(60.0, 60.0), p=(w / 2.0, h / 2.0))
    t = R.make_target(R.cam(0, 64, 32, f=(50.0, 50.0), p=(32.0, 16.0)), [0.0, 0.02, 0.01], [3.0, 1.0, 0.0], 10, 1.0,
                      R.scale_of(bd), R.scale_of(16))
    outs = []
    for prep in (False, True):
        s = R.DeviceSource(c, [0.0] * 3, [0.0] * 3, bd, 16, 0.5, 25.0, planes)
        if prep:
            s.prepare(R.scale_of(16))
        out = R.Synthesizer([s], t).run()
        outs.append({k: out[k].cpu().numpy() for k in ("y", "u", "v", "color", "depth", "quality")})
    for k in outs[0]:
        assert np.array_equal(outs[0][k], outs[1][k], equal_nan=outs[0][k].dtype.kind == "f"), k
