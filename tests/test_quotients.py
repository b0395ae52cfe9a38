"""GPU: the quotients that share a divisor, through the reprojection stage,
against IEEE division: every mantissa of the divisor (the depth of an unrotated
camera at the source's own place), numerators of many sizes, divisors at and
beyond the ends of the range that takes the reciprocal."""
import numpy as np
import pytest

import rvs_amd as R

pytestmark = pytest.mark.gpu

W, H = 4096, 2048   # 2^23 pixels, a mantissa each


# exponent of the depth; focal lengths of the target and of the source
@pytest.mark.parametrize("e,ft,fs", [(-31, 700.0, 321.5), (-30, 1.0, 1.0), (-30, 3.7e5, 0.37), (0, 1200.0, 1199.0),
                                     (1, 0.013, 777.7), (7, 640.0, 0.001), (39, 1.0, 3.3), (39, 1e-6, 5e4),
                                     (40, 250.0, 250.0)])
def test_every_divisor_mantissa(torch_cuda, e, ft, fs):
    torch = torch_cuda
    print("case quotients exponent %d focal %g / %g" % (e, ft, fs), flush=True)
    f32 = np.float32
    rng = np.random.default_rng(e + 100)
    bits = (np.uint32((e + 127) << 23) | rng.permutation(1 << 23).astype(np.uint32)).reshape(H, W)
    d = bits.view(f32)
    p = rng.uniform(0, 2000, 2).astype(f32)
    src = R.cam(0, W, H, f=(fs, fs * 1.7), p=(float(p[0]), float(p[1])))
    dst = R.cam(0, W, H, f=(ft, ft * 0.3), p=(0.0, 0.0))
    uv = torch.empty((H, W, 2), dtype=torch.float32, device="cuda")
    vd = torch.empty((H, W), dtype=torch.float32, device="cuda")
    R.reproject(src, dst, np.eye(3), np.zeros(3), torch.from_numpy(d).cuda(), None, 1.0, uv, vd)
    uv, vd = uv.cpu().numpy(), vd.cpu().numpy()
    at = [np.arange(W, dtype=f32)[None, :] + f32(0.5), np.arange(H, dtype=f32)[:, None] + f32(0.5)]
    assert np.array_equal(vd.view(np.uint32), bits)
    for k in range(2):
        y = -(d / f32(src.f[k])) * (at[k] - p[k])
        n = -f32(dst.f[k]) * y
        with np.errstate(over="ignore"):
            want = n / d + f32(0)
        bad = np.flatnonzero((uv[..., k].view(np.uint32) != want.view(np.uint32)).ravel())
        assert bad.size == 0, (k, bad.size, d.ravel()[bad[:4]], n.ravel()[bad[:4]])
