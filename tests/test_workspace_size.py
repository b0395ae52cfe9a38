"""Workspace planning (host code) for batches of uneven views, and on the GPU
the inpainting whose per-tile arrays it packs view by view."""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R
import workloads as W


def _cam(w, h):
    return R.cam(0, w, h, f=(w / 2.0, w / 2.0), p=(w / 2.0, h / 2.0))


def _plan(sizes, ns=2):
    srcs = (R.RvsSource * ns)()
    for s in srcs:
        s.cam = _cam(640, 480)
    z = [0.0] * 3
    tgts = (R.RvsTarget * len(sizes))(*[R.make_target(_cam(w, h), z, z, 8, 1.0, R.scale_of(8), R.scale_of(16))
                                        for w, h in sizes])
    n = R.hip().rvs_synth_batch_workspace_size(srcs, ns, tgts, len(sizes), 0)
    assert n > 0, R.hip().rvs_last_error()
    return n


def test_uneven_batches_pay_for_their_own_views():
    """A batch takes no more than its views apart: many small views beside a
    large one are not sized like it."""
    small, large = _plan([(64, 64)]), _plan([(4096, 2048)])
    for n in (1, 63, 1000):
        assert _plan([(4096, 2048)] + [(64, 64)] * n) <= large + n * small, n
    assert _plan([(64, 2048)] * 8 + [(4096, 64)] * 8) <= 8 * (_plan([(64, 2048)]) + _plan([(4096, 64)]))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [16, 32])
def test_uneven_batch_inpainted(torch_cuda, tile):
    """Views with holes, one to many inpainting tiles wide and high, the widest
    and the highest of them between smaller ones; bit for bit against the oracle."""
    print("case uneven inpainting, tile %d" % tile, flush=True)
    rg = W.rig("persp11_2048", scale=16)
    planes = W.render_sources(rg)
    sizes = ((34, 30), (310, 66), (32, 32), (66, 250), (30, 34), (128, 96))
    tgts = W.batch_targets(rg, len(sizes), seed=5, sizes=sizes)
    outs = R.BatchSynthesizer(W.device_sources(rg, planes), tgts, tile=tile).run()
    holes = 0
    for k, (t, out) in enumerate(zip(tgts, outs)):
        ref = ob.synthesize(W.oracle_sources(rg, planes, ob), W.oracle_cam(t.cam, ob), list(t.pos), list(t.rot),
                            t.bitdepth, t.blending_exp)
        holes += int((ref["quality"] <= 0).sum())
        assert np.array_equal(out["color"].cpu().numpy().view(np.uint32), ref["color"].view(np.uint32)), k
        for p in ("y", "u", "v"):
            assert np.array_equal(out[p].cpu().numpy().view(ref[p].dtype), ref[p]), (k, p)
    assert holes > 1000


def test_one_source_keeps_no_replay_results(monkeypatch):
    """The replay's per-source results exist for launch sets of several
    sources only: a stage raster and a one-source view ask for none."""
    tile = 16 * 16 * 5 * 4
    for w, h in ((640, 480), (1366, 766)):
        def sizes():
            return _plan([(w, h)], 1), R.hip().rvs_raster_workspace_size(w, h, w, h, 0), _plan([(w, h)], 2)

        monkeypatch.delenv("RVS_REPLAY_TILES", raising=False)
        planned = sizes()
        monkeypatch.setenv("RVS_REPLAY_TILES", "0")   # none at all
        none = sizes()
        assert none[:2] == planned[:2]
        assert planned[2] - none[2] >= 16 * 2 * tile   # two sources: at least sixteen tiles
