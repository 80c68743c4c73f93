"""The SSIM partials that a forward leaves to its VJP: map and VJP bit for bit
against the restatement at the strips' edges, in every option, with infinities
and NaN, through autograd and under capture."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_bits_equal
from tests.test_gpu_loss_strips import _inputs

pytestmark = pytest.mark.gpu


def _same(name, got, want):
    assert np.array_equal(np.isnan(got), np.isnan(want)), name
    ok = ~np.isnan(want)
    assert_bits_equal(name, got[ok], want[ok])


@pytest.mark.parametrize("h,w,stride,ch,cfg", [
    (1, 1, 3, 3, (0.8, -0.2, None, False)), (1, 64, 4, 3, (0.8, -0.2, None, True)),
    (11, 65, 4, 4, (0.5, 0.5, (0.1, 0.2, 0.3), True)), (33, 129, 7, 4, (0.8, -0.2, None, False)),
    (300, 5, 5, 3, (0.8, -0.2, None, True)), (257, 1300, 4, 3, (0.8, -0.2, None, False)),
    (3, 2, 6, 4, (1.0, 0.0, (0.1, 0.2, 0.3), True)), (1100, 70, 3, 3, (0.0, 1.0, None, False)),
])
@pytest.mark.parametrize("finite", [True, False])
def test_partials_match_checker(gpu, h, w, stride, ch, cfg, finite):
    import torch
    from brush_amd import loss as L

    print(f"[case] loss partials {h}x{w} stride={stride} ch={ch} cfg={cfg} finite={finite}", flush=True)
    pred, gt, chain = _inputs(h, w, stride, ch, h * 37 + w)
    if not finite:
        pred[h // 2, w // 2, 0], pred[0, 0, 1], chain[h - 1, w - 1, 2] = np.nan, np.inf, -np.inf
    view = torch.from_numpy(pred).to(gpu)[..., :ch]
    tg = torch.from_numpy(gt.view(np.int32)).to(gpu)
    c, oc = L.ImageLossConfig(*cfg), O.loss_config(*cfg)
    partials = L.ssim_partials(view, c)
    assert (partials is None) == (cfg[1] == 0.0)
    if partials is not None:
        partials.fill_(float("nan"))  # every one that is read was written
    _same("map", L.image_loss_forward_raw(view, tg, c, partials).cpu().numpy(), O.image_loss_forward(pred, ch, gt, oc))
    g = L.image_loss_backward_raw(view, tg, c, torch.from_numpy(chain).to(gpu), partials=partials).cpu().numpy()
    _same("vjp", g, O.image_loss_backward(pred, ch, gt, oc, chain))


def test_autograd_keeps_partials(gpu):
    """Two backwards of one forward, two forwards before their backwards, and
    none kept for a prediction without a gradient."""
    import torch
    from brush_amd import loss as L

    c, oc = L.ImageLossConfig(0.8, -0.2), O.loss_config(0.8, -0.2, None, False)
    runs = []
    for seed in (1, 2):
        pred, gt, chain = _inputs(37, 70, 4, 3, seed)
        tp = torch.from_numpy(pred).to(gpu).requires_grad_()
        runs.append((pred, gt, chain, tp, L.image_loss(tp[..., :3], torch.from_numpy(gt.view(np.int32)).to(gpu), c)))
    for pred, gt, chain, tp, m in runs:
        for scale in (1.0, -2.0):
            ch = chain * np.float32(scale)
            (g,) = torch.autograd.grad(m, (tp,), torch.from_numpy(ch).to(gpu), retain_graph=True)
            assert_bits_equal("vjp", g.cpu().numpy(), O.image_loss_backward(pred, 3, gt, oc, ch))
    m = L.image_loss(torch.from_numpy(pred).to(gpu)[..., :3], torch.from_numpy(gt.view(np.int32)).to(gpu), c)
    assert m.grad_fn is None
    assert_bits_equal("map", m.cpu().numpy(), O.image_loss_forward(pred, 3, gt, oc))


def test_captured_forward_and_vjp(gpu):
    import torch
    from brush_amd import loss as L

    pred, gt, chain = _inputs(50, 70, 4, 3, 9)
    c, oc = L.ImageLossConfig(0.8, -0.2), O.loss_config(0.8, -0.2, None, False)
    tp, tg = torch.from_numpy(pred).to(gpu), torch.from_numpy(gt.view(np.int32)).to(gpu)
    tc = torch.from_numpy(chain).to(gpu)
    out = torch.empty_like(tp)

    def step():
        partials = L.ssim_partials(tp[..., :3], c)
        m = L.image_loss_forward_raw(tp[..., :3], tg, c, partials)
        L.image_loss_backward_raw(tp[..., :3], tg, c, tc, out, partials)
        return m

    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        step()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            m = step()
        for k in range(3):
            scaled = pred * np.float32(0.5 + 0.2 * k)
            tp.copy_(torch.from_numpy(scaled))
            out.zero_()
            graph.replay()
            stream.synchronize()
            assert_bits_equal(f"map {k}", m.cpu().numpy(), O.image_loss_forward(scaled, 3, gt, oc))
            assert_bits_equal(f"vjp {k}", out.cpu().numpy(), O.image_loss_backward(scaled, 3, gt, oc, chain))
            step()  # eager work between the replays
            stream.synchronize()
    torch.cuda.synchronize()
