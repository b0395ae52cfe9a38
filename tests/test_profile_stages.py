"""GPU: the binning stage's time includes the culling tables a call builds for
sources without resident ones."""
import numpy as np
import pytest

import rvs_amd as R

pytestmark = pytest.mark.gpu


def test_binning_includes_the_tables_built_per_call(torch_cuda):
    torch = torch_cuda
    print("case profile stages", flush=True)
    n, w, h = 6, 4096, 2048
    raw = np.full((h, w), 20000, np.uint16)
    planes = [np.full(s, 128, np.uint8) for s in ((h, w), (h // 2, w // 2), (h // 2, w // 2))]
    srcs = [R.DeviceSource(R.cam(1, w, h), [0.0] * 3, [0.0] * 3, 8, 16, 1.0, 10.0, planes + [raw]) for _ in range(n)]
    # a few degrees of view: hardly an item survives the culling
    t = R.make_target(R.cam(0, 64, 48, f=(900.0, 900.0), p=(32.0, 24.0)), [0.0] * 3, [0.0] * 3, 8, 1.0, R.scale_of(8),
                      R.scale_of(16))
    best = []
    for prepared in (False, True):
        if prepared:
            for s in srcs:
                s.prepare(R.scale_of(16))
        syn = R.Synthesizer(srcs, t)
        syn.run()
        R.profile_enable(True)
        try:
            ms = []
            for _ in range(20):
                syn.run()
                ms.append(R.profile_read()["bin"])
        finally:
            R.profile_enable(False)
        best.append(min(ms))
    # every table reads its 16-bit depth plane: not faster than 8 TB/s
    tables = n * w * h * 2 / 8e12 * 1e3
    print("  bin ms without / with tables at hand", best, "tables at least", tables, flush=True)
    assert best[0] - best[1] > tables
