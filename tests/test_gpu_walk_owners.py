"""The tile walk where its owner search has corners: waves with no, one or many
splats to a step of 64 tiles, culled splats between visible ones, splats of a few
tiles and of the whole frame; both tile heights, and a grid of 263 columns, whose
map writes pairs instead of runs.  Every integer output and the image against the
restatement."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import compare_forward, gpu_forward, uniforms_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 300])
@pytest.mark.parametrize("log_scale", [-5.0, -2.0, 0.5])
@pytest.mark.parametrize("w,h,fine", [(300, 215, False), (300, 215, True), (4200, 40, False)])
def test_owners(gpu, n, log_scale, w, h, fine):
    from brush_amd.camera import Camera

    print(f"[case] walk owners n={n} log_scale={log_scale} {w}x{h} fine={fine}", flush=True)
    rng = np.random.default_rng(n + int(10 * log_scale) + 100)
    tr = np.zeros((n, 10), np.float32)
    tr[:, :3] = rng.uniform(-1.0, 1.0, (n, 3))
    tr[:, 0] *= w / h
    tr[rng.random(n) < 0.4, 2] = -50.0  # behind the camera
    tr[0, 2] = 0.0
    tr[:, 3:7] = rng.standard_normal((n, 4))
    tr[:, 7:] = log_scale + 0.5 * rng.standard_normal((n, 3))
    sh = rng.standard_normal((n, 1, 3)).astype(np.float32)
    opac = rng.standard_normal(n).astype(np.float32)
    cam = Camera.from_focal((0.0, 0.0, -4.0), (0.0, 0.0, 0.0, 1.0), float(h), w, h)
    u = uniforms_for(cam, w, h, n, 0)
    flags = O.FLAG_BWD_INFO | (O.FLAG_TILE_16X8 if fine else 0)
    compare_forward(gpu_forward(u, tr, sh, opac, flags), O.render_forward(u, tr, sh, opac, flags))
