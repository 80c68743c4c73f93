"""The blend and the rasterize backward of small frames (four waves per 8x8
block) and the one-wave kernels of larger ones, on both sides of the block
counts where the choice changes, at ragged sizes and at batch edges: images bit
for bit, gradient lanes to rtol 1e-3 plus each entry's own rounding noise.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import (OracleGrads, check_fused_backward, compare_forward, compare_lanes, gpu_forward, keep_lanes,
                           random_scene, uniforms_for)

pytestmark = pytest.mark.gpu


def _both_backwards(name, tr, sh, opac, cam, w, h, smooth, depth, fine=False):
    import torch
    from brush_amd import render as R

    print(f"[case] {name} {w}x{h} n={tr.shape[0]} smooth={smooth} depth={depth} fine={fine}", flush=True)
    n, deg = tr.shape[0], int(round(sh.shape[1] ** 0.5)) - 1
    dev = torch.device("cuda", 0)
    leaves = [torch.from_numpy(x).to(dev).requires_grad_(True) for x in (tr, sh, opac)]
    chans = 5 if depth else 4
    v = np.random.default_rng(w + h).standard_normal((h, w, chans)).astype(np.float32)
    vt = torch.from_numpy(v).to(dev)
    tiles = R.Rasterizer.Candidate if fine else R.Rasterizer.Legacy
    with keep_lanes():
        res = R.render_splats_diff(R.Splats(*leaves), cam, (w, h), raster_pass=R.RasterPass.BackwardSmoothCutoff
                                   if smooth else R.RasterPass.Backward, raster_mode=R.RasterizationMode.RgbaAndDepth
                                   if depth else R.RasterizationMode.Rgba, rasterizer=tiles)
        grads = torch.autograd.grad(res.img, leaves, vt)
    u = uniforms_for(cam, w, h, n, deg)
    flags = O.FLAG_BWD_INFO | (O.FLAG_SMOOTH_CUTOFF if smooth else 0) | (O.FLAG_RENDER_DEPTH if depth else 0) | \
        (O.FLAG_TILE_16X8 if fine else 0)
    o = O.render_forward(u, tr, sh, opac, flags)
    g = gpu_forward(u, tr, sh, opac, flags)
    compare_forward(g, o)
    want = OracleGrads(o, tr, sh, opac, v, (flags & ~O.FLAG_BWD_INFO) | O.FLAG_REFINE_WEIGHT)
    got = dict(zip(("v_transforms", "v_coeffs", "v_raw_opac"), (x.cpu().numpy() for x in grads)))
    check_fused_backward(name, res._cfg.state, tr, sh, opac, got, want)
    out = g["out"]
    lanes = R.rasterize_bwd(out.out_img, out.projected_splats, out.compact_gid_from_isect, out.aux.tile_offsets,
                            (0.0, 0.0, 0.0), (w, h), vt, smooth, depth, True, tiles)
    compare_lanes(f"{name} replay", lanes.cpu().numpy(), want)


# 6,144 blocks (768x512) and 8,192 (1024x512) are the last the four-wave blend
# and backward take; one pixel more is a further column of tiles
@pytest.mark.parametrize("w,h,fine", [(768, 512, False), (769, 512, False), (1024, 512, False), (1025, 512, False),
                                      (512, 768, True), (3, 2, False), (9, 17, False), (41, 23, True)])
def test_sizes(gpu, w, h, fine):
    from brush_amd.camera import Camera

    n = 3000 if w > 100 else 700
    tr, sh, opac = random_scene(w * 7 + h, n, 1, log_scale=(-3.0, 0.6))
    cam = Camera.from_focal((0.0, 0.1, -3.0), (0.0, 0.0, 0.0, 1.0), 0.6 * max(w, 8), w, h)
    _both_backwards("sizes", tr, sh, opac, cam, w, h, smooth=(h % 2 == 1), depth=(w % 2 == 1), fine=fine)


# a stack over every pixel of one tile: lengths at the edges of the batches
# (128 and 256 candidates) and of a step (4), faint (no pixel saturates) and
# opaque (every pixel does, in different steps)
@pytest.mark.parametrize("n", [1, 3, 4, 5, 127, 128, 129, 255, 256, 257, 600])
@pytest.mark.parametrize("logit", [-4.5, 0.0])
def test_stacks(gpu, n, logit):
    from brush_amd.camera import Camera

    rng = np.random.default_rng(n)
    tr = np.zeros((n, 10), np.float32)
    tr[:, 0:2] = rng.uniform(-0.02, 0.02, (n, 2))
    tr[:, 2] = np.linspace(0.0, 1.0, n)
    tr[:, 3] = 1.0
    tr[:, 7:10] = rng.uniform(-2.5, -1.0, (n, 3))
    sh = rng.normal(0.0, 0.5, (n, 1, 3)).astype(np.float32)
    opac = (logit + rng.normal(0.0, 0.3, n)).astype(np.float32)
    cam = Camera.from_focal((0.0, 0.0, -3.0), (0.0, 0.0, 0.0, 1.0), 40.0, 16, 16)
    _both_backwards(f"stack {n}", tr, sh, opac, cam, 16, 16, smooth=False, depth=True)
