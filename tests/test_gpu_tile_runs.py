"""The tile sort by runs: every integer output and the image, bit for bit, on both
sides of the grid sizes that it takes (256 columns, 255 rows), at the edges of a
chunk (1,024 runs of a row) and of the pairs staged at a time, and with several
chunks to a group.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import compare_forward, gpu_forward, uniforms_for

pytestmark = pytest.mark.gpu


def _line(n, w, h, log_scale, seed):
    """n splats spread over a w x h image, depths in no order."""
    from brush_amd.camera import Camera

    rng = np.random.default_rng(seed)
    focal = 40.0
    tr = np.zeros((n, 10), np.float32)
    tr[:, 0] = rng.uniform(-0.5, 0.5, n) * w / focal * 3.0
    tr[:, 1] = rng.uniform(-0.5, 0.5, n) * h / focal * 3.0
    tr[:, 2] = rng.uniform(-0.2, 0.2, n)
    tr[:, 3] = 1.0
    tr[:, 7:10] = rng.uniform(log_scale - 0.3, log_scale + 0.3, (n, 3))
    sh = rng.normal(0.0, 0.5, (n, 1, 3)).astype(np.float32)
    opac = rng.normal(-2.0, 0.5, n).astype(np.float32)
    return tr, sh, opac, Camera.from_focal((0.0, 0.0, -3.0), (0.0, 0.0, 0.0, 1.0), focal, w, h)


def _check(tr, sh, opac, cam, w, h, flags):
    n = tr.shape[0]
    print(f"[case] {w}x{h} n={n} flags={flags}", flush=True)
    u = uniforms_for(cam, w, h, n, 0)
    o = O.render_forward(u, tr, sh, opac, flags)
    for _ in range(2):  # sized from the counts or an earlier plan, then from this scene's
        compare_forward(gpu_forward(u, tr, sh, opac, flags), o)
    return o


# 4,096 pixels are 256 columns of tiles (4,097: 257), 4,080 are 255 rows of 16
# and 2,040 of 8
@pytest.mark.parametrize("w,h,fine", [(4096, 40, False), (4097, 40, False), (40, 4080, False), (40, 4081, False),
                                      (40, 2040, True), (40, 2041, True), (4096, 24, True), (16, 16, False)])
@pytest.mark.parametrize("log_scale", [-1.0, 1.5])
def test_grids(gpu, w, h, fine, log_scale):
    _check(*_line(1500, w, h, log_scale, w + h), w, h, O.FLAG_BWD_INFO | (O.FLAG_TILE_16X8 if fine else 0))


# one row of tiles: a splat of 4, 18 or 108 tiles is a run (or more, where a step
# of 64 items ends inside it), so a chunk's pairs fit the 6,912 staged at a
# time or take several rounds
@pytest.mark.parametrize("n", [1, 63, 64, 1023, 1024, 1025, 2049, 5000])
@pytest.mark.parametrize("log_scale", [-3.0, -1.0, 1.6])
def test_chunks(gpu, n, log_scale):
    _check(*_line(n, 2000, 16, log_scale, n), 2000, 16, O.FLAG_BWD_INFO)


# every splat over every tile: the pairs of tile t are all splats in depth order;
# above 16,777,216 pairs a group holds more than one chunk
@pytest.mark.parametrize("n,w,h", [(300, 4096, 32), (5000, 960, 960)])
def test_full_cover(gpu, n, w, h):
    tr, sh, opac, cam = _line(n, w, h, 1.0, n)
    tr[:, 0:2] = 0.0
    tr[:, 7:10] = 9.0
    opac[:] = 2.0
    print(f"[case] {w}x{h} n={n}", flush=True)
    g = gpu_forward(uniforms_for(cam, w, h, n, 0), tr, sh, opac, 0)
    tiles = -(-w // 16) * -(-h // 16)
    assert g["num_intersections"] == n * tiles
    ids = g["compact_gid_from_isect"][:n * tiles].reshape(tiles, n)
    assert np.array_equal(ids, np.broadcast_to(np.arange(n, dtype=ids.dtype), ids.shape))
    assert np.array_equal(g["tile_id_from_isect"][:n * tiles].reshape(tiles, n)[:, [0, -1]],
                          np.arange(tiles)[:, None].repeat(2, 1))
    first = np.arange(tiles, dtype=np.int64) * n
    assert np.array_equal(np.asarray(g["tile_offsets_pre"], np.int64).reshape(tiles, 2), np.stack([first, first + n], 1))
