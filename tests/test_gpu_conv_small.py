"""Small layers that would run on the library's own choice of transform size, whose forward pass
and input gradient sum over the taps in one launch (conv_small.hip), against the fp64 direct
convolution; and which layers those are."""
import ctypes

import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import SMALL, conv_route, dev, pass_size, rel

pytestmark = pytest.mark.gpu


def runs_small(pass_, B, cin, cout, H, W, k):
    fn = F.lib()._ZN9fbfft_amd9runsSmallEiiiiiiiii
    fn.argtypes, fn.restype = [ctypes.c_int] * 9, ctypes.c_bool
    N = F.conv_choose_fft_size(pass_, B, cin, cout, H, W, k, k)
    return fn(pass_, N, B, cin, cout, H, W, k, k)


def bar(taps):
    # a wave's chain of taps / 8 multiply-adds and the eight waves' sum: at most sqrt(taps / 8 + 8)
    # roundings of 2^-24 of a sum that grows like the square root of its terms
    return np.sqrt(taps / 8 + 8) * 2.0 ** -24


def workspace(B, cin, cout, H, W, k):
    return torch.empty(max(F.conv_workspace_image(p, B, cin, cout, H, W, k, k, 0) for p in (0, 1)),
                       dtype=torch.uint8, device=dev())


# forward, every filter width, and the input gradient of those of them that it is summed for, too; pixels and planes that do not fill the last workgroup, several images to a
# workgroup, fewer filter rows than waves, one plane on either side
@pytest.mark.parametrize("B,cin,cout,H,W,k", [
    (3, 7, 9, 8, 9, 1), (5, 10, 8, 7, 8, 2), (9, 5, 9, 8, 7, 3), (2, 4, 17, 11, 23, 4),
    (2, 3, 5, 9, 9, 5), (1, 3, 16, 30, 9, 6), (2, 5, 8, 12, 12, 7), (2, 3, 7, 21, 20, 8),
    (1, 3, 9, 20, 20, 9), (2, 3, 10, 32, 30, 10), (1, 3, 8, 33, 31, 11),
    (65, 1, 1, 3, 2, 1), (1, 1, 9, 64, 64, 3), (2, 6, 3, 50, 64, 2), (1, 250, 8, 4, 4, 1)])
def test_both_passes_vs_fp64(oracle, B, cin, cout, H, W, k):
    d = dev()
    x = synth.normal((B, cin, H, W), seed=30)
    w = synth.normal((cout, cin, k, k), seed=31)
    g = synth.normal((B, cout, H - k + 1, W - k + 1), seed=32)
    ws = workspace(B, cin, cout, H, W, k)
    assert runs_small(0, B, cin, cout, H, W, k)
    out = torch.full(tuple(g.shape), float("nan"), device=d)
    assert F.conv_fprop(x.to(d), w.to(d), out, 0, ws) == F.Success
    torch.cuda.synchronize()
    assert rel(out.cpu().numpy(), oracle.corr2d_valid(x.numpy(), w.numpy())) < bar(cin * k * k)
    if runs_small(1, B, cin, cout, H, W, k):
        gi = torch.full(tuple(x.shape), float("nan"), device=d)
        assert F.conv_bprop(g.to(d), w.to(d), gi, 0, ws) == F.Success
        torch.cuda.synchronize()
        assert rel(gi.cpu().numpy(), oracle.corr2d_grad_input(g.numpy(), w.numpy(), H, W)) < bar(cout * k * k)


# input gradients of the filter widths that are left, sides that differ, and as many filter values as LDS holds
@pytest.mark.parametrize("B,cin,cout,H,W,kH,kW", [
    (11, 4, 2, 7, 7, 6, 6), (1, 61, 3, 28, 28, 9, 9), (4, 42, 3, 23, 23, 10, 10), (14, 3, 4, 33, 33, 11, 11),
    (3, 7, 9, 14, 13, 1, 5), (2, 9, 17, 20, 16, 7, 2), (3, 7, 9, 14, 13, 3, 11), (2, 9, 17, 20, 16, 11, 1),
    (2, 9, 17, 20, 16, 2, 9), (3, 7, 9, 14, 13, 5, 4), (1, 8, 2048, 6, 6, 1, 1)])
def test_input_gradient_and_sides_that_differ_vs_fp64(oracle, B, cin, cout, H, W, kH, kW):
    d = dev()
    x, w = synth.normal((B, cin, H, W), seed=30), synth.normal((cout, cin, kH, kW), seed=31)
    g = synth.normal((B, cout, H - kH + 1, W - kW + 1), seed=32)
    ws = torch.empty(max(F.conv_workspace_image(p, B, cin, cout, H, W, kH, kW, 0) for p in (0, 1)),
                     dtype=torch.uint8, device=d)
    # (61 and 42 input planes: the forward pass has too many taps)
    assert [conv_route(p, 0, B, cin, cout, H, W, kH, kW)[0] == SMALL for p in (0, 1)] == [cin < 42, True]
    gi, out = torch.full(tuple(x.shape), float("nan"), device=d), torch.full(tuple(g.shape), float("nan"), device=d)
    assert F.conv_bprop(g.to(d), w.to(d), gi, 0, ws) == F.Success
    assert F.conv_fprop(x.to(d), w.to(d), out, 0, ws) == F.Success
    torch.cuda.synchronize()
    assert rel(gi.cpu().numpy(), oracle.corr2d_grad_input(g.numpy(), w.numpy(), H, W)) < bar(cout * kH * kW)
    assert rel(out.cpu().numpy(), oracle.corr2d_valid(x.numpy(), w.numpy())) < bar(cin * kH * kW)


def test_infinite_filter_value_in_an_input_gradient(oracle):
    """What the padding around a gradient meets counts as zero times the filter, so an infinite filter
    value makes every element of its input plane infinite or not a number, and nothing else."""
    B, cin, cout, H, k = 3, 7, 5, 9, 3
    d = dev()
    w, g = synth.normal((cout, cin, k, k), seed=31).to(d), synth.normal((B, cout, H - 2, H - 2), seed=32).to(d)
    ws = workspace(B, cin, cout, H, H, k)
    assert runs_small(1, B, cin, cout, H, H, k)
    results = []
    for value in (0.5, float("inf")):
        w[1, 4, 0, 2] = value
        gi = torch.empty((B, cin, H, H), device=d)
        assert F.conv_bprop(g, w, gi, 0, ws) == F.Success
        results.append(gi)
    torch.cuda.synchronize()
    others = torch.arange(cin, device=d) != 4
    assert torch.equal(results[0][:, others], results[1][:, others])
    assert not bool(torch.isfinite(results[1][:, 4]).any())


def test_strided_views(oracle):
    """Planes, rows and columns apart, filters in another order, a result inside a larger tensor
    whose other elements stay."""
    B, cin, cout, H, W, k = 3, 5, 9, 12, 13, 3
    d = dev()
    x = synth.normal((B, cin, 2 * H + 1, 2 * W + 3), seed=30).to(d)[:, :, 1:2 * H + 1:2, 2:2 * W + 2:2]
    w = synth.normal((k, k, cin, cout), seed=31).to(d).permute(3, 2, 1, 0)
    big = torch.full((cout, B, H + 2, 2 * W), 7.0, device=d)
    out = big.transpose(0, 1)[:, :, 1:H - k + 2, 1:2 * (W - k + 1):2]
    ws = workspace(B, cin, cout, H, W, k)
    assert runs_small(0, B, cin, cout, H, W, k) and runs_small(1, B, cin, cout, H, W, k)
    assert F.conv_fprop(x, w, out, 0, ws) == F.Success
    torch.cuda.synchronize()
    xh, wh = x.cpu().contiguous().numpy(), w.cpu().contiguous().numpy()
    assert rel(out.cpu().numpy(), oracle.corr2d_valid(xh, wh)) < bar(cin * k * k)
    assert int((big == 7.0).sum()) == big.numel() - out.numel()
    gi = torch.full((B, cin, H, W), float("nan"), device=d)
    assert F.conv_bprop(out, w, gi, 0, ws) == F.Success
    torch.cuda.synchronize()
    want = oracle.corr2d_grad_input(out.cpu().contiguous().numpy(), wh, H, W)
    assert rel(gi.cpu().numpy(), want) < bar(cout * k * k)


def test_result_in_place_of_an_operand(oracle):
    """A result that overlaps what it is made from takes the way that has read it all before."""
    B, c, H = 4, 8, 9
    d = dev()
    x, w = synth.normal((B, c, H, H), seed=30), synth.normal((c, c, 1, 1), seed=31)
    ws = workspace(B, c, c, H, H, 1)
    assert runs_small(0, B, c, c, H, H, 1)
    xd = x.to(d)
    assert F.conv_fprop(xd, w.to(d), xd, 0, ws) == F.Success
    torch.cuda.synchronize()
    assert rel(xd.cpu().numpy(), oracle.corr2d_valid(x.numpy(), w.numpy())) < 1e-6


def test_other_layers_keep_the_transforms():
    assert not runs_small(2, 9, 5, 9, 8, 7, 3)             # weight gradients
    assert not runs_small(0, 128, 64, 192, 27, 27, 5)     # a large layer
    assert not runs_small(0, 1, 8, 8, 14, 14, 12)         # filters wider than 11
    assert not runs_small(0, 1, 2049, 8, 4, 4, 1)          # more filter values than LDS holds


def test_named_sizes():
    """The chosen size by its name is the same call; another size is a transform of that size."""
    d = dev()
    x, w = synth.normal((9, 5, 8, 7), seed=30).to(d), synth.normal((9, 5, 3, 3), seed=31).to(d)
    ws = torch.empty(F.conv_workspace(0, 9, 5, 9, 16), dtype=torch.uint8, device=d)
    chosen = F.conv_choose_fft_size(0, 9, 5, 9, 8, 7, 3, 3)
    assert chosen == 8 and pass_size(0, 16, 9, 5, 9, 8, 7, 3)[0] == 8 and runs_small(0, 9, 5, 9, 8, 7, 3)
    out = {n: torch.empty((9, 9, 6, 5), device=d) for n in (0, 8, 16)}
    for n, o in out.items():
        assert F.conv_fprop(x, w, o, n, ws) == F.Success
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[8]) and torch.equal(out[0], out[16])
    y, v = synth.normal((1, 2, 30, 30), seed=32).to(d), synth.normal((3, 2, 3, 3), seed=33).to(d)
    chosen = F.conv_choose_fft_size(0, 1, 2, 3, 30, 30, 3, 3)
    other = next(n for n in (8, 16, 32) if pass_size(0, n, 1, 2, 3, 30, 30, 3)[0] == n != chosen)
    ws = torch.empty(F.conv_workspace_image(0, 1, 2, 3, 30, 30, 3, 3, other), dtype=torch.uint8, device=d)
    a, b = (torch.empty((1, 3, 28, 28), device=d) for _ in range(2))
    assert F.conv_fprop(y, v, a, other, ws) == F.Success
    wide = torch.empty(F.conv_workspace_image(0, 1, 2, 3, 30, 30, 3, 3, 0), dtype=torch.uint8, device=d)
    assert F.conv_fprop(y, v, b, 0, wide) == F.Success
    torch.cuda.synchronize()
    assert not torch.equal(a, b) and rel(a.cpu().numpy(), b.cpu().numpy()) < 1e-6
