"""Every kernel that a layer's contraction runs on, in every pass, with the reduction whole and cut
into ranges: each case asserts the kernel before it is compared with the fp64 direct convolution, so
that a changed rule of dispatch cannot leave one untested.  And what the ways that a pass may run make
of values that are not finite."""
import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import (DIRECT64, DIRECT128, PLANE_MAJOR, REGS_NARROW, REGS_SPLIT_K, REGS_WIDE, SMALL, SPLIT, check,
                      conv_route, dev)

pytestmark = pytest.mark.gpu

# (kernel, ranges, pass, points, B, cin, cout, H, W, kH, kW): ends of tiles on both sides and of k-slices,
# images that fit the transform and images cut into windows
CASES = [
    (REGS_SPLIT_K, 1, 0, 16, 4, 1, 1, 19, 18, 6, 3), (REGS_SPLIT_K, 2, 0, 8, 1, 60, 1, 4, 5, 3, 5),
    (REGS_SPLIT_K, 1, 1, 32, 1, 5, 1, 21, 20, 4, 6), (REGS_SPLIT_K, 2, 1, 8, 1, 2, 67, 9, 8, 4, 6),
    (REGS_SPLIT_K, 1, 2, 32, 1, 2, 1, 33, 35, 6, 6), (REGS_SPLIT_K, 3, 2, 16, 421, 1, 1, 9, 8, 5, 6),
    # ... with several 32 x 32 tiles per bin, either side the longer one
    (REGS_SPLIT_K, 1, 0, 8, 33, 80, 34, 8, 8, 6, 6), (REGS_SPLIT_K, 1, 0, 8, 3, 200, 65, 14, 14, 5, 5),
    (REGS_SPLIT_K, 1, 1, 8, 33, 34, 80, 8, 8, 3, 3), (REGS_SPLIT_K, 1, 2, 8, 80, 33, 65, 8, 8, 3, 3),
    (REGS_WIDE, 1, 0, 16, 18, 3, 199, 8, 10, 1, 2), (REGS_WIDE, 7, 0, 8, 21, 218, 20, 9, 12, 5, 3),
    (REGS_WIDE, 1, 1, 32, 20, 33, 5, 18, 18, 2, 6), (REGS_WIDE, 2, 1, 16, 129, 17, 62, 8, 10, 4, 4),
    (REGS_WIDE, 1, 2, 16, 2, 17, 197, 14, 14, 5, 6), (REGS_WIDE, 15, 2, 8, 30, 18, 26, 17, 17, 6, 5),
    (REGS_NARROW, 1, 0, 32, 1, 1, 34, 26, 25, 3, 2), (REGS_NARROW, 4, 0, 16, 44, 129, 3, 9, 9, 3, 4),
    (REGS_NARROW, 1, 1, 16, 1, 41, 1, 10, 9, 3, 1), (REGS_NARROW, 2, 1, 8, 20, 2, 62, 12, 14, 6, 6),
    (REGS_NARROW, 1, 2, 32, 1, 1, 33, 30, 28, 6, 6), (REGS_NARROW, 5, 2, 16, 39, 1, 36, 17, 17, 6, 3),
    (DIRECT64, 1, 0, 16, 39, 27, 52, 10, 11, 5, 3), (DIRECT64, 2, 0, 8, 17, 255, 41, 17, 15, 6, 6),
    (DIRECT64, 1, 1, 32, 40, 36, 5, 21, 19, 6, 5), (DIRECT64, 2, 1, 16, 10, 38, 286, 19, 17, 5, 5),
    (DIRECT64, 1, 2, 32, 7, 39, 33, 30, 32, 6, 1), (DIRECT64, 9, 2, 8, 106, 33, 33, 16, 14, 6, 6),
    (DIRECT128, 1, 0, 32, 86, 2, 227, 18, 18, 3, 6), (DIRECT128, 1, 0, 8, 303, 3, 90, 17, 15, 6, 6),
    (DIRECT128, 1, 1, 16, 119, 200, 12, 17, 16, 6, 5), (DIRECT128, 1, 2, 32, 20, 201, 84, 28, 29, 6, 5),
    (SPLIT, 1, 0, 8, 237, 51, 230, 4, 7, 3, 4), (SPLIT, 2, 0, 16, 17, 266, 91, 24, 22, 4, 3),
    (SPLIT, 1, 1, 8, 476, 82, 61, 4, 5, 2, 5), (SPLIT, 2, 1, 16, 178, 45, 252, 9, 7, 4, 5),
    (SPLIT, 1, 1, 32, 210, 65, 114, 20, 18, 4, 6), (SPLIT, 1, 2, 16, 190, 107, 79, 9, 9, 3, 6),
    (SPLIT, 4, 2, 8, 562, 73, 67, 4, 5, 2, 3), (SPLIT, 3, 2, 8, 32, 68, 150, 16, 17, 2, 6),
    (SPLIT, 1, 2, 32, 137, 135, 86, 19, 17, 1, 5),
    (PLANE_MAJOR, 1, 0, 64, 3, 5, 4, 60, 57, 5, 5), (PLANE_MAJOR, 1, 1, 64, 6, 5, 7, 61, 64, 20, 20),
    (PLANE_MAJOR, 1, 2, 128, 2, 3, 2, 100, 128, 7, 7)]


def some(n, count):
    """The first, the last and evenly spaced ones between."""
    return np.unique(np.linspace(0, n - 1, min(n, count)).astype(int))


def take(t, first, second):
    return t.cpu().numpy()[first][:, second].copy()


@pytest.mark.parametrize("kind,ranges,pass_,N,B,cin,cout,H,W,kH,kW", CASES)
def test_every_contraction_kernel_vs_fp64(oracle, kind, ranges, pass_, N, B, cin, cout, H, W, kH, kW):
    assert conv_route(pass_, N, B, cin, cout, H, W, kH, kW) == (kind, N, ranges)
    d = dev()
    # the operands as slices of larger tensors, which stay as they are around the result
    x = synth.normal((B, cin + 1, H, W), seed=40).to(d)[:, 1:]
    w = synth.normal((cout, cin, kH, kW + 2), seed=41).to(d)[..., 1:1 + kW]
    g = synth.normal((B, cout + 2, H - kH + 1, W - kW + 1), seed=42).to(d)[:, 1:-1]
    size = F.conv_workspace_image(pass_, B, cin, cout, H, W, kH, kW, N)
    space = torch.full((size + 256,), 77, dtype=torch.uint8, device=d)
    like = (g, x, w)[pass_]
    large = torch.full((like.shape[0], like.shape[1] + 2) + tuple(like.shape[2:]), 7.0, device=d)
    out = large[:, 1:-1]
    if pass_ == 0:
        rc = F.conv_fprop(x, w, out, N, space[:size])
    elif pass_ == 1:
        rc = F.conv_bprop(g, w, out, N, space[:size])
    else:
        rc = F.conv_accgrad(x, g, out, N, space[:size])
    torch.cuda.synchronize()
    assert rc == F.Success
    assert bool((space[size:] == 77).all()) and bool((large[:, 0] == 7.0).all()) and bool((large[:, -1] == 7.0).all())
    n, c, f = some(B, 4), some(cin, 5), some(cout, 5)
    every = slice(None)
    if pass_ == 0:
        K, got = cin, take(out, n, f)
        want = oracle.corr2d_valid(take(x, n, every), take(w, f, every))
    elif pass_ == 1:
        K, got = cout, take(out, n, c)
        want = oracle.corr2d_grad_input(take(g, n, every), take(w, every, c), H, W)
    else:
        windows = -(-(H - kH + 1) // (N - kH + 1)) * -(-(W - kW + 1) // (N - kW + 1)) if max(H, W) > N else 1
        K, got = B * windows, take(out, f, c)
        want = oracle.corr2d_grad_weight(take(x, every, c), take(g, every, f), kH, kW)
    # three transforms of at most 1.3e-7 (rel-L2, tests of the transforms), and of the contraction a rounding
    # of at most 2^-24 per two k of three sums of up to twice the result, which grow like the
    # square root of k: sqrt(K / 2 / 2) 2 2^-24
    check("kernel %d, pass %d, %d points, K = %d" % (kind, pass_, N, K), got, want, 3 * 1.3e-7 + np.sqrt(K) * 2.0 ** -24)


# layers of every way a forward pass may run, sizes as they name it
WAYS = [(SMALL, 0, 9, 5, 9, 8, 7, 3, 3), (REGS_SPLIT_K, 8, 33, 80, 34, 8, 8, 6, 6),
        (REGS_NARROW, 32, 9, 3, 34, 26, 25, 3, 3), (REGS_WIDE, 16, 18, 3, 199, 8, 10, 1, 2),
        (DIRECT64, 16, 39, 27, 52, 10, 11, 5, 3), (DIRECT128, 32, 90, 2, 230, 25, 25, 3, 3),
        (SPLIT, 8, 237, 51, 230, 6, 7, 3, 3), (PLANE_MAJOR, 64, 3, 5, 4, 60, 57, 5, 5)]


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("kind,N,B,cin,cout,H,W,kH,kW", WAYS)
def test_not_finite_values_stay_with_their_image_and_filter(kind, N, B, cin, cout, H, W, kH, kW, value):
    """One value of one image, then of one filter, that is not finite: every output whose taps meet it
    is not finite either, and no bit of another image's or filter's outputs changes."""
    assert conv_route(0, N, B, cin, cout, H, W, kH, kW)[0] == kind
    d = dev()
    x, w = synth.normal((B, cin, H, W), seed=50).to(d), synth.normal((cout, cin, kH, kW), seed=51).to(d)
    ws = torch.empty(F.conv_workspace_image(0, B, cin, cout, H, W, kH, kW, N), dtype=torch.uint8, device=d)

    def run():
        out = torch.empty((B, cout, H - kH + 1, W - kW + 1), device=d)
        assert F.conv_fprop(x, w, out, N, ws) == F.Success
        torch.cuda.synchronize()
        return out
    clean = run()
    image, filter_ = B // 2, cout // 3
    x[image, cin - 1, 1, 2] = value
    got = run()
    others = torch.arange(B, device=d) != image
    assert torch.equal(got[others], clean[others])
    assert not bool(torch.isfinite(got[image, :, max(0, 2 - kH):2, max(0, 3 - kW):3]).any())
    x[image, cin - 1, 1, 2] = 1.0
    clean = run()
    w[filter_, 0, kH - 1, 0] = value
    got = run()
    others = torch.arange(cout, device=d) != filter_
    assert torch.equal(got[:, others], clean[:, others])
    assert not bool(torch.isfinite(got[:, filter_]).any())
