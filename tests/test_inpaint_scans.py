"""The inpainting's two sweeps as quadrant minima.

On the CPU: the closed form (smallest key over the upper-left quadrant, then
over the lower-right one) restated in numpy equals the oracle's sweeps, map for
map.  On the GPU: image sizes around the 32-pixel tiles and the 64-tile scan
chunks, with holes from a few pixels to nearly everything; every map entry and
colour equals the oracle's.
"""
import numpy as np
import pytest

import oracle_bind as ob
import rvs_amd as R

NONE = np.int64(1) << 62


def closed_form(known):
    h, w = known.shape
    X, Y = np.meshgrid(np.arange(w, dtype=np.int64), np.arange(h, dtype=np.int64))
    down, right = np.zeros_like(known), np.zeros_like(known)
    down[:-1], right[:, :-1] = known[1:], known[:, 1:]
    pos = 2 * (X * h + Y) + np.where(known | down, 0, 1)
    key = np.where(known | down | right, (np.where(known, 0, 1) + w + h - X - Y << 32) | pos, NONE)
    P = np.minimum.accumulate(np.minimum.accumulate(key, 1), 0)
    has = P < NONE
    F = np.where(known, 0, np.where(has, (P >> 32) - (w + h) + X + Y, w + h))
    q = P & 0xffffffff
    qx, qy = (q >> 1) // h, (q >> 1) % h
    next_to = (P >> 32) + qx + qy != w + h
    src = (qy + (next_to & (q % 2 == 0))) * w + qx + (next_to & (q % 2 == 1))
    src = np.where(known | ~has, Y * w + X, src)

    def suffix(a, ax):
        return np.flip(np.minimum.accumulate(np.flip(a, ax), ax), ax)

    H = F + X + Y
    own = suffix(np.where(known | has, (H << 32) | Y, NONE), 0)
    row = np.full_like(H, NONE)
    row[:, :-1] = suffix(np.where(known | has, (H << 32) | ((h - 1 - Y) * w + X), NONE), 1)[:, 1:]
    cols = suffix(row, 0)
    use = (own >> 32) <= (cols >> 32)
    best = np.where(use, own, cols)
    found = best < NONE
    lo = best & 0xffffffff
    qy = np.where(found, np.where(use, lo, h - 1 - lo // w), Y)
    qx = np.where(found, np.where(use, X, lo % w), X)
    s = src[qy, qx]
    return np.stack([s % w, s // w, np.where(found, (best >> 32) - X - Y, w + h)], -1)


def masks(h, w, seed):
    rng = np.random.default_rng(seed)
    for frac in (0.003, 0.05, 0.5, 0.98):
        yield rng.random((h, w)) < frac
    k = np.ones((h, w), bool)
    k[h // 8: h - h // 7, w // 9: w - w // 10] = False
    yield k
    k = rng.random((h, w)) < 0.9
    k[:, w - (w + 2) // 3:] = False      # an uncovered right border
    yield k
    yield np.add.outer(np.arange(h), 2 * np.arange(w)) % 5 == 0


@pytest.mark.parametrize("h,w", [(1, 1), (1, 17), (13, 1), (9, 14), (33, 40), (24, 7)])
def test_closed_form_equals_the_sweeps(h, w):
    for k, known in enumerate(masks(h, w, 10 * h + w)):
        _, m, _ = ob.inpaint(np.zeros((h, w, 3), np.float32), known.astype(np.float32), want_map=True)
        assert np.array_equal(m, closed_form(known)), (h, w, k)


@pytest.mark.gpu
@pytest.mark.parametrize("h,w", [(1, 1), (1, 70), (31, 33), (32, 32), (33, 31), (64, 65), (97, 130),
                                 (40, 2049), (2080, 35), (70, 4130)])
def test_tile_and_chunk_edges(torch_cuda, h, w):
    torch = torch_cuda
    col = np.random.default_rng(3).random((h, w, 3)).astype(np.float32)
    for k, known in enumerate(masks(h, w, h + w)):
        print("case inpaint scans %dx%d mask %d" % (w, h, k), flush=True)
        q = known.astype(np.float32)
        rcol, rmap, _ = ob.inpaint(col, q, want_map=True)
        gcol = torch.from_numpy(col).cuda()
        gmap = torch.empty((h, w, 3), dtype=torch.int32, device="cuda")
        R.inpaint(gcol, torch.from_numpy(q).cuda(), map_out=gmap)
        assert np.array_equal(gmap.cpu().numpy(), rmap), (h, w, k)
        assert np.array_equal(gcol.cpu().numpy(), rcol), (h, w, k)
