"""Layers whose contraction splits its fp32 operands into bf16 pieces (binGemmSplit: 48 k or
more, at least 38 products per spectrum value, two 64 x 64 tiles per CU), against the fp64 direct convolution.
(Input gradients, weight gradients and reductions in ranges: test_gpu_conv_routes.py.)"""
import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import SPLIT, check, conv_route, dev

pytestmark = pytest.mark.gpu

# The three transforms of a convolution leave at most 1.3e-7 each (rel-L2, tests of the
# transforms); a sum over K complex values in 16-k steps of six piece products, re and im parts:
# 12 K / 16 roundings of at most 2^-24 of a partial sum that grows like the square root of the
# steps, so at most sqrt(12 K / 16 / 2) 2^-24.
def bar(K):
    return 3 * 1.3e-7 + np.sqrt(12 * K / 32) * 2.0 ** -24


def layer(N, B, cin, cout, H, k, scale=1.0):
    d = dev()
    assert conv_route(0, N, B, cin, cout, H, H, k)[0] == SPLIT
    x = synth.normal((B, cin, H, H), seed=30).to(d) * scale
    w = synth.normal((cout, cin, k, k), seed=31, std=0.05).to(d)
    ws = torch.empty(F.conv_workspace(0, B, cin, cout, N), dtype=torch.uint8, device=d)
    out = torch.full((B, cout, H - k + 1, H - k + 1), float("nan"), device=d)
    assert F.conv_fprop(x, w, out, N, ws) == F.Success
    torch.cuda.synchronize()
    return x, w, out


# 128 and 512 bins; one k-slice more and less than whole, ends of the 64 x 64 tiles and of their
# 32 x 32 parts, either operand on the rows
@pytest.mark.parametrize("N,B,cin,cout,H,k", [
    (16, 272, 64, 160, 15, 2), (16, 320, 65, 129, 16, 3), (16, 161, 87, 127, 14, 3),
    (16, 97, 120, 160, 16, 1), (16, 320, 97, 97, 13, 3), (16, 113, 161, 113, 16, 4),
    (32, 129, 136, 97, 31, 5)])
def test_pieces_vs_fp64(oracle, N, B, cin, cout, H, k):
    x, w, out = layer(N, B, cin, cout, H, k)
    rng = np.random.default_rng(B)
    oh = H - k + 1
    n = 4000
    at = np.stack([rng.integers(0, B, n), rng.integers(0, cout, n), rng.integers(0, oh, n),
                   rng.integers(0, oh, n)], axis=1).astype(np.int32)
    at[:4] = [[0, 0, 0, 0], [B - 1, cout - 1, oh - 1, oh - 1], [B - 1, 0, 0, oh - 1], [0, cout - 1, oh - 1, 0]]
    assert bool(torch.isfinite(out).all())
    want = oracle.corr2d_valid_at(x.cpu().numpy(), w.cpu().numpy(), at)
    got = out.cpu().numpy()[at[:, 0], at[:, 1], at[:, 2], at[:, 3]]
    check("%d points, %d x %d x %d" % (N, B, cout, cin), got, want, bar(cin))


@pytest.mark.parametrize("exponent", [-84, 60])
def test_pieces_scale_exactly(exponent):
    """Operands times a power of two: the pieces and the sums are the same, times that power."""
    a = layer(16, 128, 128, 128, 15, 2)[2]
    b = layer(16, 128, 128, 128, 15, 2, 2.0 ** exponent)[2]
    assert torch.equal(a * 2.0 ** exponent, b)


@pytest.mark.parametrize("exponent", [-100, -108, -116])
def test_pieces_of_small_values(oracle, exponent):
    """A piece that falls below the smallest normal number may be cut to zero: a spectrum value is off by
    at most 2^-126 then, nothing against 2^-100, a 2^-14 of a spectrum of 15 x 15 values of 2^-116."""
    N, B, cin, cout, H, k = 16, 272, 64, 160, 15, 2
    x, w, out = layer(N, B, cin, cout, H, k, 2.0 ** exponent)
    n = [0, 100, B - 1]
    want = oracle.corr2d_valid((x[n].double() * 2.0 ** -exponent).float().cpu().numpy(), w.cpu().numpy())
    got = out[n].double().cpu().numpy() * 2.0 ** -exponent
    check("values of 2^%d" % exponent, got, want, bar(cin) + 2.0 ** -126 / (15 * 2.0 ** exponent))
