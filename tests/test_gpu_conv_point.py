"""Layers with filters of 1 x 1, whose passes are products of matrices without transforms (conv_point.hip),
against fp64 products; which calls those are, and what the others still give."""
import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import POINT, conv_route, dev, rel

pytestmark = pytest.mark.gpu


def bar(terms):
    # chains of at most 32 roundings (eight instructions of four terms) of 2^-24, then one per chain and, of a weight
    # gradient, per range: sums grow like the square root of their terms
    return np.sqrt(32 + terms / 32 + 8) * 2.0 ** -24


def products(x, w, g):
    """out, gradInput and gradWeight in 64 bits"""
    xd, wd, gd = x.double().flatten(2), w.double()[:, :, 0, 0], g.double().flatten(2)
    out = torch.stack([wd @ i for i in xd]).view(g.shape)
    gin = torch.stack([wd.T.contiguous() @ i for i in gd]).view(x.shape)
    gw = sum(j @ i.T.contiguous() for i, j in zip(xd, gd))
    return out, gin, gw[:, :, None, None]


def run(x, w, g, N, accumulate=False, scale=1.0, before=None, point=(True, True, True)):
    (B, cin, H, W), cout = x.shape, w.shape[0]
    d = dev()
    for p in (0, 1, 2):
        if point[p] is not None:
            assert (conv_route(p, N, B, cin, cout, H, W, 1)[0] == POINT) == point[p]
    size = max(F.conv_workspace_image(p, B, cin, cout, H, W, 1, 1, N) for p in (0, 1, 2))
    ws = torch.full((size + 256,), 77, dtype=torch.uint8, device=d)
    large = [torch.full((t.shape[0], t.shape[1] + 2) + tuple(t.shape[2:]), 7.0, device=d) for t in (g, x)]
    out, gin = (t[:, 1:-1] for t in large)
    gw = torch.full((cout, cin + 1, 1, 1), 7.0, device=d)
    if before is not None:
        gw[:, :cin] = before
    assert F.conv_fprop(x, w, out, N, ws[:size]) == F.Success
    assert F.conv_bprop(g, w, gin, N, ws[:size]) == F.Success
    assert F.conv_accgrad(x, g, gw[:, :cin], N, ws[:size], scale=scale, accumulate=accumulate) == F.Success
    torch.cuda.synchronize()
    assert bool((ws[size:] == 77).all()) and bool((gw[:, cin] == 7.0).all())
    assert all(bool((t[:, 0] == 7.0).all()) and bool((t[:, -1] == 7.0).all()) for t in large)
    return out, gin, gw[:, :cin]


def operands(B, cin, cout, H, W, extra=0):
    d = dev()
    x = synth.normal((B, cin + extra, H, W), seed=60).to(d)[:, extra:]
    w = synth.normal((cout, cin, 1, 1), seed=61).to(d)
    g = synth.normal((B, cout + extra, H, W), seed=62).to(d)[:, extra:]
    return x, w, g


def compare(x, w, g, got, scale=1.0, before=0.0):
    B, cin, H, W = x.shape
    for a, b, terms in zip(got, products(x, w, g), (cin, w.shape[0], B * H * W)):
        if terms == B * H * W:
            b = scale * b + before
        assert rel(a.cpu().numpy(), b.cpu().numpy()) < bar(terms)


# pixels that are no multiple of four, as few as four, images that end inside a wave; planes of either side at the ends of
# 16 and 32 rows, of 64, of the 4 planes of a step and the 128 that wait in LDS
@pytest.mark.parametrize("B,cin,cout,H,W", [
    (40, 33, 65, 23, 23), (300, 16, 17, 2, 2), (77, 130, 64, 5, 3), (9, 300, 129, 31, 30), (16, 3, 200, 57, 61),
    (3, 128, 250, 64, 63), (5, 127, 96, 100, 31), (1, 257, 300, 41, 45), (20, 65, 33, 37, 29), (260, 40, 140, 7, 1),
    (64, 5, 31, 90, 91), (130, 32, 32, 64, 64), (128, 20, 48, 66, 65),
    # 64 pixels of a weight gradient's turn out of many images, the last turn partly filled; one to three turns in a range
    (1, 40, 50, 2, 2), (17, 33, 40, 3, 3), (3, 47, 46, 7, 7), (40, 20, 50, 7, 7), (138, 47, 46, 7, 7), (33, 110, 346, 8, 8),
    (500, 9, 70, 5, 1), (129, 65, 20, 3, 5), (64, 31, 33, 6, 11)])
def test_products_vs_fp64(B, cin, cout, H, W):
    x, w, g = operands(B, cin, cout, H, W, extra=1)
    # (small passes are summed in one launch by conv_small.hip)
    compare(x, w, g, run(x, w, g, 0, point=(None, None, True)))


def test_which_calls():
    B, cin, cout, H, W = 16, 60, 100, 60, 61
    x, w, g = operands(B, cin, cout, H, W)
    compare(x, w, g, run(x, w, g, 0))
    compare(x, w, g, run(x, w, g, 64))
    compare(x, w, g, run(x, w, g, 32, point=(False,) * 3))
    compare(x, w, g, run(x, w, g, 16, point=(False,) * 3))
    assert conv_route(2, 0, 4, 5, 6, 1, 3, 1)[0] != POINT and conv_route(2, 0, 4, 5, 6, 1, 4, 1)[0] == POINT


def test_filters_in_another_order_scale_and_accumulate():
    B, cin, cout, H, W = 30, 70, 90, 29, 31
    d = dev()
    x, _, g = operands(B, cin, cout, H, W)
    w = synth.normal((1, cin, 1, cout), seed=63).to(d).permute(3, 1, 0, 2)
    before = synth.normal((cout, cin, 1, 1), seed=64).to(d)
    got = run(x, w, g, 0, accumulate=True, scale=0.5, before=before)
    compare(x, w, g, got, 0.5, before.double())
    again = run(x, w, g, 0, accumulate=True, scale=0.5, before=before)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_planes_with_gaps_and_results_in_place():
    """What does not lie in whole planes, or overlaps what it is made from, keeps the transforms."""
    B, c, H, W = 12, 64, 40, 40
    x, w, g = operands(B, c, c, H, 2 * W)
    x, g = x[..., ::2], g[..., 1::2]
    compare(x, w, g, run(x, w, g, 0))
    y = x.contiguous()
    ws = torch.empty(F.conv_workspace_image(0, B, c, c, H, W, 1, 1, 0), dtype=torch.uint8, device=dev())
    want = products(x, w, g)[0]
    assert F.conv_fprop(y, w, y, 0, ws) == F.Success
    torch.cuda.synchronize()
    assert rel(y.cpu().numpy(), want.cpu().numpy()) < 1e-6


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_not_finite_values_stay_with_their_pixel_and_filter(value):
    B, cin, cout, H, W = 24, 61, 90, 40, 39
    x, w, g = operands(B, cin, cout, H, W)
    clean = [t.clone() for t in run(x, w, g, 0)]
    x[5, cin - 1, 39, 38] = value
    out, _, gw = run(x, w, g, 0)
    meets = torch.zeros((B, 1, H, W), dtype=torch.bool, device=dev())
    meets[5, 0, 39, 38] = True
    assert not bool(torch.isfinite(out[5, :, 39, 38]).any())
    assert torch.equal(out.masked_fill(meets, 0), clean[0].masked_fill(meets, 0))
    assert not bool(torch.isfinite(gw[:, cin - 1]).any()) and torch.equal(gw[:, :-1], clean[2][:, :-1])
    x[5, cin - 1, 39, 38] = 1.0
    w[7, 3] = value
    out, gin, _ = run(x, w, g, 0)
    others = torch.arange(cout, device=dev()) != 7
    assert not bool(torch.isfinite(out[:, 7]).any()) and not bool(torch.isfinite(gin[:, 3]).any())
    assert bool(torch.isfinite(out[:, others]).all())


def test_replays_of_a_captured_training_step():
    B, cin, cout, H, W = 16, 60, 100, 60, 61
    x, w, g = operands(B, cin, cout, H, W)
    d = dev()
    size = max(F.conv_workspace_image(p, B, cin, cout, H, W, 1, 1, 0) for p in (0, 1, 2))
    ws = torch.empty(size, dtype=torch.uint8, device=d)
    out, gin, gw = torch.empty_like(g), torch.empty_like(x), torch.empty_like(w)

    def step():
        assert F.conv_fprop(x, w, out, 0, ws) == F.Success
        assert F.conv_bprop(g, w, gin, 0, ws) == F.Success
        assert F.conv_accgrad(x, g, gw, 0, ws) == F.Success
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for i in range(3):
        x.normal_()
        step()
        want = [t.clone() for t in (out, gin, gw)]
        for t in (out, gin, gw):
            t.zero_()
        ws.fill_(i)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip((out, gin, gw), want))
