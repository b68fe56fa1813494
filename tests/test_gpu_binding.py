"""The native calls (csrc/binding.cpp) against the general way through ctypes: the same bits on
strided, offset and padded operands and on another stream, and NotImplemented for what is not a
plain call, so that results and errors stay those of the general way."""
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import dev

pytestmark = pytest.mark.gpu


def both(fn, *results):
    """fn(stream=None) and fn(stream=<the current one>), which takes the general way: equal
    codes and results."""
    codes, kept = [], []
    for stream in (None, torch.cuda.current_stream()):
        for r in results:
            r.fill_(-3.0)
        codes.append(fn(stream))
        torch.cuda.synchronize()
        kept.append([r.clone() for r in results])
    assert codes[0] == codes[1]
    assert all(torch.equal(a, b) for a, b in zip(*kept))
    return codes[0]


@pytest.mark.parametrize("side", [False, True])
def test_same_as_the_general_way(side):
    d = dev()
    with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.current_stream()):
        wide = synth.normal((6, 70), seed=1).to(d)
        rows, spec, back = wide[::2, 3:67], torch.empty((3, 33, 2), device=d), torch.empty((3, 64), device=d)
        assert both(lambda s: F.fbfft1D(rows, spec, 0, s), spec) == F.Success
        assert both(lambda s: F.fbifft1D(back, spec, 0, s), back) == F.Success
        planes = synth.normal((5, 30, 40), seed=2).to(d)[:, 1:14, 2:15]
        sp, bk = torch.empty((5, 9, 16, 2), device=d), torch.empty((5, 13, 13), device=d)
        assert both(lambda s: F.fbfft2D(planes, sp, 2, 1, stream=s), sp) == F.Success
        assert both(lambda s: F.fbifft2D(sp, bk, 2, 1, stream=s), bk) == F.Success
        A, B = synth.normal((3, 4, 9, 16, 2), seed=3).to(d), synth.normal((5, 4, 9, 16, 2), seed=4).to(d)
        C = torch.empty((3, 5, 9, 16, 2), device=d)
        assert both(lambda s: F.transposeMM(A, B, C, 0.5, conjugateTransposeB=True, stream=s), C) == F.Success
        x, w = synth.normal((2, 3, 12, 13), seed=5).to(d), synth.normal((4, 3, 3, 3), seed=6).to(d)
        g = synth.normal((2, 4, 10, 11), seed=7).to(d)
        out, gi, gw = torch.empty_like(g), torch.empty_like(x), torch.empty_like(w)
        ws = torch.empty(max(F.conv_workspace_image(p, 2, 3, 4, 12, 13, 3, 3, 0) for p in range(3)),
                         dtype=torch.uint8, device=d)
        assert both(lambda s: F.conv_fprop(x, w, out, 0, ws, s), out) == F.Success
        assert both(lambda s: F.conv_bprop(g, w, gi, 0, ws, s), gi) == F.Success
        assert both(lambda s: F.conv_accgrad(x, g, gw, 0, ws, 0.5, True, s), gw) == F.Success
        # what the library refuses is refused with the same code
        assert both(lambda s: F.fbfft1D(rows, sp, 0, s)) != F.Success
        assert both(lambda s: F.conv_fprop(x, w, out, 0, ws[:64], s)) != F.Success


def test_plain_calls_are_native_and_others_are_not():
    d = dev()
    native = F._load_native()
    x, y = torch.zeros((4, 32), device=d), torch.zeros((4, 17, 2), device=d)
    assert native.r2c_1d(x, y, 0) == F.Success
    assert native.r2c_1d(torch.nn.Parameter(x), y, 0) == F.Success
    torch.cuda.synchronize()
    for args in [(x.cpu(), y, 0), (x.double(), y, 0), (x, y, 0.0), (x, y, 1 << 40), (None, y, 0), (x, y),
                 (x.to_sparse(), y, 0), (torch.zeros((1,) * 6, device=d), y, 0)]:
        assert native.r2c_1d(*args) is NotImplemented
    with pytest.raises(TypeError):
        F.fbfft1D(x.double(), y)
    with pytest.raises(ValueError):
        F.fbfft1D(x.cpu(), y)
    with pytest.raises(ValueError):
        F.fbfft1D(torch.zeros((1,) * 6, device=d), y)
