"""The SSIM loss's strips: widths and heights around the strip's 64 columns and
its row counts, both directions bit for bit against the restatement, and the
VJP of a captured stream (which takes the kernel without a workspace)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bits_equal

pytestmark = pytest.mark.gpu


def _inputs(h, w, stride, ch, seed):
    rng = np.random.default_rng(seed)
    pred = rng.random((h, w, stride), dtype=np.float32)
    b = rng.integers(0, 256, (h, w, 4), dtype=np.uint8).astype(np.uint32)
    gt = (b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16) | (b[..., 3] << 24)).astype(np.uint32)
    return pred, gt, rng.standard_normal((h, w, ch)).astype(np.float32)


@pytest.mark.parametrize("h,w,stride,ch,cfg", [
    (1, 64, 3, 3, (0.8, -0.2, None, False)), (2, 65, 4, 3, (0.8, -0.2, None, True)),
    (11, 63, 4, 4, (0.5, 0.5, (0.1, 0.2, 0.3), False)), (33, 129, 7, 4, (0.8, -0.2, None, True)),
    (300, 5, 5, 3, (0.8, -0.2, None, False)), (257, 1300, 4, 3, (0.8, -0.2, None, False)),
    (3, 2, 6, 4, (1.0, 0.0, (0.1, 0.2, 0.3), True)), (1100, 70, 3, 3, (0.0, 1.0, None, False)),
])
def test_strips_match_checker(gpu, h, w, stride, ch, cfg):
    import torch
    from brush_amd import loss as L

    print(f"[case] loss strips {h}x{w} stride={stride} ch={ch} cfg={cfg}", flush=True)
    pred, gt, chain = _inputs(h, w, stride, ch, h * 31 + w)
    view = torch.from_numpy(pred).to(gpu)[..., :ch]
    tg = torch.from_numpy(gt.view(np.int32)).to(gpu)
    c, oc = L.ImageLossConfig(*cfg), O.loss_config(*cfg)
    assert_bits_equal("map", L.image_loss_forward_raw(view, tg, c).cpu().numpy(), O.image_loss_forward(pred, ch, gt, oc))
    g = L.image_loss_backward_raw(view, tg, c, torch.from_numpy(chain).to(gpu)).cpu().numpy()
    assert_bits_equal("vjp", g, O.image_loss_backward(pred, ch, gt, oc, chain))


def test_non_finite_pixels_spread_as_in_the_checker(gpu):
    """An infinity or NaN in the prediction reaches every pixel within ten of it,
    also across the image's edge, and no other."""
    import torch
    from brush_amd import loss as L

    pred, gt, chain = _inputs(40, 90, 3, 3, 3)
    pred[2, 3, 0], pred[20, 70, 1], pred[39, 89, 2] = np.inf, np.nan, -np.inf
    c, oc = L.ImageLossConfig(0.8, -0.2), O.loss_config(0.8, -0.2, None, False)
    tp, tg = torch.from_numpy(pred).to(gpu), torch.from_numpy(gt.view(np.int32)).to(gpu)
    m, wm = L.image_loss_forward_raw(tp, tg, c).cpu().numpy(), O.image_loss_forward(pred, 3, gt, oc)
    g = L.image_loss_backward_raw(tp, tg, c, torch.from_numpy(chain).to(gpu)).cpu().numpy()
    wg = O.image_loss_backward(pred, 3, gt, oc, chain)
    for name, got, want in (("map", m, wm), ("vjp", g, wg)):
        assert np.array_equal(np.isnan(got), np.isnan(want)), name
        ok = ~np.isnan(want)
        assert_bits_equal(name, got[ok], want[ok])


def test_captured_vjp(gpu):
    import torch
    from brush_amd import loss as L

    pred, gt, chain = _inputs(50, 70, 4, 3, 9)
    c, oc = L.ImageLossConfig(0.8, -0.2), O.loss_config(0.8, -0.2, None, False)
    tp, tg = torch.from_numpy(pred).to(gpu), torch.from_numpy(gt.view(np.int32)).to(gpu)
    tc = torch.from_numpy(chain).to(gpu)
    out = torch.empty_like(tp)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        L.image_loss_backward_raw(tp[..., :3], tg, c, tc, out)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            L.image_loss_backward_raw(tp[..., :3], tg, c, tc, out)
        for k in range(3):
            scaled = pred * np.float32(0.5 + 0.2 * k)
            tp.copy_(torch.from_numpy(scaled))
            out.zero_()
            graph.replay()
            stream.synchronize()
            assert_bits_equal(f"replay {k}", out.cpu().numpy(), O.image_loss_backward(scaled, 3, gt, oc, chain))
            # eager work between the replays reuses the pool's blocks
            L.image_loss_backward_raw(tp[..., :3], tg, c, tc)
            stream.synchronize()
    torch.cuda.synchronize()
