"""CPU-only checks of the boundary: the shared library loads and exports every
symbol include/fbfft_amd.h declares, the structs have the reference's layout,
and the host-side mirror behaves like the reference's parameter class."""
import ctypes
import os
import re
import subprocess
import sys
import warnings

import numpy as np
import pytest

import fbcuda_amd as F
from gpu_util import (DIRECT, LANES, POINT, REGISTERS, REGS_NARROW, REGS_SPLIT_K, REGS_WIDE, conv_route, pass_size,
                      product_route)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    src = open(os.path.join(ROOT, "include", "fbfft_amd.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(fbfft_[a-z0-9_]+)\s*\(", src)))


def test_header_and_python_agree():
    assert declared_symbols() == sorted(F.EXPORTS)


def test_library_exports_every_declared_symbol():
    if not os.path.exists(F.LIB_PATH):
        import __graft_entry__
        __graft_entry__.build()
    L = ctypes.CDLL(F.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(L, name), name


def test_struct_layouts():
    # fbfft_tensor: pointer, 5 strides, 5 sizes, rank
    assert F.Tensor.data.offset == 0 and F.Tensor.stride.offset == 8
    assert F.Tensor.size.offset == 28 and F.Tensor.dim.offset == 48
    # TiledDeviceTensor<float,4>: {int padL; int padU; {float* data; int stride[4]; int size[4];}}
    assert ctypes.sizeof(F.Tile) == 48
    assert (F.Tile.padL.offset, F.Tile.padU.offset, F.Tile.data.offset) == (0, 4, 8)
    assert (F.Tile.stride.offset, F.Tile.size.offset) == (16, 32)


def test_error_strings_and_twiddles():
    assert F.error_string(0) == "Success"
    assert F.error_string(1) == "UnsupportedSize"
    assert F.error_string(2) == "UnsupportedDimension"
    assert F.error_string(3) == "HipError"
    out = (ctypes.c_float * 256)()
    F.lib().fbfft_twiddle_table(out)
    tw = np.frombuffer(out, dtype=np.float32).reshape(128, 2)
    k = np.arange(128)
    assert np.array_equal(tw[:, 1], np.sin(np.pi * k / 128).astype(np.float32))
    assert tw[64, 0] == 0.0 and tw[0, 0] == 1.0


def test_parameters_mirror():
    p = F.FBFFTParameters()
    assert p.forwardFFT() and not p.inverseFFT() and not p.normalizeFFT()
    assert p.padLeft() == 0 and p.padUp() == 0
    q = p.inverse().normalize(True).withPadLeft(3).withPadUp(4)
    assert q is p and p.inverseFFT() and p.normalizeFFT() and (p.padLeft(), p.padUp()) == (3, 4)
    assert p.forward().forwardFFT()
    assert (p.Success, p.UnsupportedSize, p.UnsupportedDimension, p.CudaError) == (0, 1, 2, 3)
    assert [F.numHermitian(n) for n in (2, 8, 32, 256)] == [2, 5, 17, 129]


def test_cpu_tensors_are_rejected():
    import torch
    with pytest.raises(ValueError):
        F.fbfft2D(torch.zeros(1, 8, 8), torch.zeros(1, 5, 8, 2))


def test_synth_is_deterministic():
    from fbcuda_amd import synth
    a = synth.normal((4, 8), seed=3)
    b = synth.normal((4, 8), seed=3)
    assert a.dtype.is_floating_point and bool((a == b).all())
    assert not bool((a == synth.normal((4, 8), seed=4)).all())
    u = synth.uniform((1000,), seed=0)
    assert float(u.min()) >= -1.0 and float(u.max()) < 1.0


def test_cpp_facade_compiles_against_reference_include_paths():
    """Host code that includes cuda/fbfft/FBFFT.cuh, cuda/MM.cuh and
    cuda/fbfft/FFTIteratedConvolution.cuh and uses the reference's names builds and links."""
    import subprocess
    if not os.path.exists(F.LIB_PATH):
        import __graft_entry__
        __graft_entry__.build()
    subprocess.check_call(["make", "-C", os.path.join(ROOT, "tests", "cpp"), "-B"],
                          stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    assert os.path.exists(os.path.join(ROOT, "tests", "cpp", "facade_check"))


def test_cpp_device_tensor_and_complex_host_arithmetic():
    """tests/cpp/tensor_check.cpp: sizes / strides of downcast, upcast, transpose, permute,
    view and cast, and Complex's operators, against hand-written expectations (host only)."""
    import subprocess
    subprocess.check_call(["make", "-C", os.path.join(ROOT, "tests", "cpp"), "-B", "tensor_check"],
                          stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([os.path.join(ROOT, "tests", "cpp", "tensor_check")], capture_output=True,
                         text=True)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout


def test_cpp_in_register_transforms_on_the_host():
    """tests/cpp/regs_check.cpp: the butterfly and real-fix-up templates the kernels
    instantiate (fbcuda_amd/csrc/fft_regs.h), compiled for the host and compared with a
    naive fp64 DFT for 2 ... 128 complex points, both directions, and 4 ... 128 real points."""
    import subprocess
    subprocess.check_call(["make", "-C", os.path.join(ROOT, "tests", "cpp"), "-B", "regs_check"],
                          stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([os.path.join(ROOT, "tests", "cpp", "regs_check")], capture_output=True,
                         text=True)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout


def _fake_tensor(shape, base=0x10000000):
    """fbfft_tensor over memory that is never touched: the tile builder only does
    address arithmetic."""
    t = F.Tensor()
    t.data = base
    t.dim = len(shape)
    stride = 1
    for i in reversed(range(len(shape))):
        t.size[i] = shape[i]
        t.stride[i] = stride
        stride *= shape[i]
    return t


@pytest.mark.parametrize("H,W,kH,kW,N", [
    (256, 256, 9, 9, 32),    # configs[4]: 11 x 11 tiles, the last 16 wide in, 8 wide out
    (32, 32, 5, 5, 32), (40, 56, 9, 3, 32), (14, 17, 3, 3, 8), (30, 25, 5, 1, 16), (9, 9, 1, 1, 8)])
def test_make_tiles_grid(H, W, kH, kW, N):
    Bn, Cin, Cout = 3, 2, 5
    oH, oW = H - kH + 1, W - kW + 1
    ti, to = _fake_tensor((Bn, Cin, H, W)), _fake_tensor((Bn, Cout, oH, oW), 0x20000000)
    L = F.lib()
    n = L.fbfft_make_tiles(ti, to, kH, kW, N, None, None, 0)
    sy, sx = N - kH + 1, N - kW + 1
    ys, xs = list(range(0, oH, sy)), list(range(0, oW, sx))
    assert n == len(ys) * len(xs)
    a, b = (F.Tile * n)(), (F.Tile * n)()
    assert L.fbfft_make_tiles(ti, to, kH, kW, N, ctypes.cast(a, ctypes.c_void_p),
                              ctypes.cast(b, ctypes.c_void_p), n) == n
    covered = np.zeros((oH, oW), np.int32)
    for t, (y0, x0) in enumerate((y, x) for y in ys for x in xs):
        assert (a[t].padL, a[t].padU, b[t].padL, b[t].padU) == (0, 0, 0, 0)
        assert a[t].data == 0x10000000 + 4 * (y0 * W + x0)
        assert b[t].data == 0x20000000 + 4 * (y0 * oW + x0)
        assert list(a[t].stride) == [Cin * H * W, H * W, W, 1]
        assert list(b[t].stride) == [Cout * oH * oW, oH * oW, oW, 1]
        assert list(a[t].size) == [Bn, Cin, min(N, H - y0), min(N, W - x0)]
        assert list(b[t].size) == [Bn, Cout, min(sy, oH - y0), min(sx, oW - x0)]
        # the input window holds every sample the output window needs
        assert a[t].size[2] >= b[t].size[2] + kH - 1 and a[t].size[3] >= b[t].size[3] + kW - 1
        covered[y0:y0 + b[t].size[2], x0:x0 + b[t].size[3]] += 1
    assert (covered == 1).all()   # output windows partition the output plane
    if (H, N) == (256, 32):
        assert n == 121 and a[n - 1].size[2] == 16 and b[n - 1].size[2] == 8


def test_make_tiles_capacity_and_rejects():
    ti, to = _fake_tensor((1, 1, 40, 40)), _fake_tensor((1, 1, 36, 36))
    L = F.lib()
    a, b = (F.Tile * 2)(), (F.Tile * 2)()
    pa, pb = ctypes.cast(a, ctypes.c_void_p), ctypes.cast(b, ctypes.c_void_p)
    assert L.fbfft_make_tiles(ti, to, 5, 5, 16, pa, pb, 2) == 9    # 3 x 3 grid, two written
    assert a[1].data == 0x10000000 + 4 * 12
    assert L.fbfft_make_tiles(ti, to, 5, 5, 64, None, None, 0) == 0    # FFT size
    assert L.fbfft_make_tiles(ti, to, 3, 3, 16, None, None, 0) == 0    # output shape mismatch
    assert L.fbfft_make_tiles(ti, to, 5, 17, 16, None, None, 0) == 0   # kernel wider than the FFT
    assert F.lib().fbfft_conv_workspace(0, 128, 64, 192, 32) == \
        F.lib().fbfft_conv_fprop_workspace(128, 64, 192, 32) > 0
    for p in (0, 1, 2):
        assert F.lib().fbfft_conv_workspace(p, 4, 5, 6, 16) % 8 == 0
    # 64 / 128: plane-major half spectra of both operands and the result
    assert F.lib().fbfft_conv_workspace(0, 4, 5, 6, 64) == (20 + 30 + 24) * 33 * 64 * 8
    assert F.lib().fbfft_conv_workspace(2, 4, 5, 6, 128) == (20 + 30 + 24) * 65 * 128 * 8 + 30 * 128 * 128 * 4
    assert F.lib().fbfft_conv_workspace(0, 4, 5, 6, 256) == 0


def _descriptor_views(tiles, base_ptr, strides):
    """(y0, x0, h, w, padL, padU) of each descriptor, recovered from its address."""
    out = []
    for t in tiles:
        off = (t.data - base_ptr) // 4
        assert (t.data - base_ptr) % 4 == 0 and off >= 0
        y0, x0 = off // strides[2], off % strides[2]
        out.append((y0, x0, t.size[2], t.size[3], t.padL, t.padU))
    return out


@pytest.mark.parametrize("N,kH,kW,H,W", [(8, 3, 3, 14, 17), (16, 5, 3, 30, 41), (32, 9, 9, 70, 56),
                                         (8, 1, 1, 9, 9), (16, 16, 16, 16, 16), (8, 3, 2, 8, 6)])
def test_grad_input_tile_grid_partitions_and_reproduces_gradient(oracle, N, kH, kW, H, W):
    """fbfft_make_tiles_for_pass(FFT_UpdateGradInput) is host code: its gradInput windows
    tile the tensor exactly once, and the CPU transcription of the tiled pass run over its
    descriptors gives the fp64 input gradient (multi-tile, seams included)."""
    import torch
    from fbcuda_amd import synth
    Nb, Cin, Cout = 2, 3, 2
    gin = np.full((Nb, Cin, H, W), 7.0, np.float32)
    g = synth.normal((Nb, Cout, H - kH + 1, W - kW + 1), seed=60).numpy()
    w = synth.normal((Cout, Cin, kH, kW), seed=61, std=0.05).numpy()
    vi, vo = F.view(torch.from_numpy(gin)), F.view(torch.from_numpy(g))
    n = F.lib().fbfft_make_tiles_for_pass(1, vi, vo, kH, kW, N, None, None, 0)
    stepY, stepX = N - kH + 1, N - kW + 1
    assert n == -(-H // stepY) * -(-W // stepX)
    a, b = (F.Tile * n)(), (F.Tile * n)()
    assert F.lib().fbfft_make_tiles_for_pass(1, vi, vo, kH, kW, N, ctypes.cast(a, ctypes.c_void_p),
                                             ctypes.cast(b, ctypes.c_void_p), n) == n
    iv = _descriptor_views(a, gin.ctypes.data, [s // 4 for s in gin.strides])
    ov = _descriptor_views(b, g.ctypes.data, [s // 4 for s in g.strides])
    cover = np.zeros((H, W), np.int32)
    for (y0, x0, h, wd, padL, padU), (gy, gx, gh, gw, gpl, gpu) in zip(iv, ov):
        cover[y0:y0 + h, x0:x0 + wd] += 1
        assert (padU, padL) == (kH - 1, kW - 1) and h >= 1 and wd >= 1
        assert gh >= 1 and gw >= 1 and gpu + gh <= N and gpl + gw <= N
        assert gy - gpu == y0 - (kH - 1) and gx - gpl == x0 - (kW - 1)
    assert (cover == 1).all()
    assert oracle.iterated_conv(N, gin, iv, g.copy(), ov, w, 1) == 1
    from oracle import rel_l2
    assert rel_l2(gin, oracle.corr2d_grad_input(g, w, H, W)) < 1e-4
    # passes 0 and 2 share the grid of fbfft_make_tiles
    assert F.lib().fbfft_make_tiles_for_pass(2, vi, vo, kH, kW, N, None, None, 0) == \
        F.lib().fbfft_make_tiles(vi, vo, kH, kW, N, None, None, 0)
    assert F.lib().fbfft_make_tiles_for_pass(3, vi, vo, kH, kW, N, None, None, 0) == 0


def test_view_rejects_strides_beyond_32_bits():
    import torch
    t = torch.empty(4).as_strided((1, 2), (2 ** 31, 1))
    with pytest.raises(ValueError):
        F.view(t)
    assert F.view(torch.empty(4).as_strided((1, 2), (2 ** 31 - 1, 1))).stride[0] == 2 ** 31 - 1


@pytest.mark.parametrize("shape", [(), (3,), (5, 0), (7, 17, 2), (2, 3, 9, 5), (2, 3, 17, 32, 2)])
def test_packed_descriptor_is_the_view(shape):
    """The byte string that a call passes is the fbfft_tensor that view fills in, for every rank,
    contiguous and strided, and operands that view refuses raise the same error."""
    import torch
    t = torch.zeros(shape)
    for u in (t, t.transpose(0, -1) if t.dim() else t, t[1:] if t.dim() else t):
        assert F._desc(u) == bytes(F.view(u))
    for bad in (t.double(), torch.zeros((1,) * 6), torch.empty(4).as_strided((1, 2), (2 ** 31, 1)),
                torch.empty(1).expand(2 ** 31)):
        with pytest.raises((TypeError, ValueError)) as want:
            F.view(bad)
        with pytest.raises(want.type, match="^" + re.escape(str(want.value)) + "$"):
            F._desc(bad)


def test_iterated_conv_refuses_filters_larger_than_the_transform():
    """Validated on the host before anything is launched: returns 0 (not launched)."""
    import torch
    w = torch.zeros((1, 1, 9, 3))
    ins, outs = (F.Tile * 1)(), (F.Tile * 1)()
    rc = F.lib().fbfft_iterated_conv(8, ctypes.cast(ins, ctypes.c_void_p),
                                     ctypes.cast(outs, ctypes.c_void_p), F.view(w), 0,
                                     ctypes.c_float(1.0), 1, 1, None)
    assert rc == 0


def test_iterated_conv_refuses_more_pairs_than_32_bits_count():
    """A weight gradient over 2^31 (tile, image) pairs is not launched (it came out as zeros):
    decided on the host, descriptors are not read."""
    import torch
    w = torch.zeros((1, 1, 1, 1))
    ins, outs = (F.Tile * 1)(), (F.Tile * 1)()
    for batch, tiles in ((1 << 16, 1 << 15), (2 ** 31 - 1, 1), (1, 1 << 31), (3, (1 << 64) // 3 + 1)):
        assert F.lib().fbfft_iterated_conv(8, ctypes.cast(ins, ctypes.c_void_p),
                                           ctypes.cast(outs, ctypes.c_void_p), F.view(w), 2,
                                           ctypes.c_float(1.0), batch, tiles, None) == 0


@pytest.mark.parametrize("pass_,N,B,cin,cout,H,W,k,want", [
    # ranges: the largest number that the named workspace has room for (16: as many as planned)
    (2, 128, 153, 3, 33, 73, 70, 2, (16, 15)),
    (2, 64, 95, 13, 34, 43, 43, 2, (16, 7)),
    (2, 128, 8, 5, 52, 125, 125, 3, (16, 3)),
    (2, 64, 85, 32, 66, 33, 61, 7, (64, 16)),      # 3 ranges of 6: plane-major 124 us, windows 173
    (2, 64, 36, 18, 107, 56, 62, 8, (64, 16)),     # 1 range of 2: 85, 92
    # windows that fit with all ranges and are slower all the same
    (2, 64, 173, 80, 362, 63, 64, 3, (64, 16)),    # 1375, 1992
    (2, 64, 162, 299, 115, 60, 60, 6, (64, 16)),   # 1346, 1796
    (2, 128, 93, 193, 41, 122, 119, 8, (128, 16)),  # 1360, 1772
    (0, 64, 57, 247, 190, 63, 64, 8, (64, 16)),    # 799, 954
    # and faster ones
    (0, 64, 32, 32, 64, 60, 60, 5, (32, 16)),
    (1, 64, 32, 32, 64, 60, 60, 5, (16, 1)),       # 1 range of 2
    (2, 64, 32, 32, 64, 60, 60, 5, (32, 16)),
    (2, 128, 16, 32, 64, 100, 100, 8, (32, 16)),
    # 32 points: three fifths of the named workspace
    (0, 32, 32, 64, 192, 27, 27, 5, (16, 16)),     # 42 %
    (2, 32, 32, 64, 192, 27, 27, 5, (16, 16)),     # 55 %
    (0, 32, 128, 64, 192, 27, 27, 5, (32, 16)),    # 80 %
    # 16 points: the same, and no smaller product left to less of the chip
    (0, 16, 9, 20, 40, 8, 8, 1, (8, 16)),
    (1, 16, 64, 96, 128, 14, 14, 3, (16, 16)),     # 137 %
    (0, 16, 28, 45, 15, 8, 9, 3, (16, 16)),        # 50 %, 14.8 us, on 8 points 16.6
    (1, 16, 2, 4, 50, 12, 12, 1, (16, 16)),        # 51 %, 14.8, 16.4
    (2, 16, 4, 310, 175, 25, 25, 6, (16, 16)),     # 60 %, 38.9, 49.3
    (2, 16, 2, 64, 300, 10, 10, 3, (8, 16)),
])
def test_transform_size_of_a_named_layer(pass_, N, B, cin, cout, H, W, k, want):
    """The size and the ranges that a layer pass runs on, decided on the host from the layer
    alone, on both sides of each line of the rule."""
    assert pass_size(pass_, N, B, cin, cout, H, W, k) == want


def test_conv_choose_fft_size():
    """fftSize = 0 of the layer entry points: the choices recorded next to the measurements
    they came from (forward pass / input gradient / weight gradient, us per pass at
    fftSize 8, 16, 32 on one MI355X), and the properties every choice has."""
    L = F.lib()
    measured = [
        # batch, cin, cout, H, k: chosen size per pass
        ((128, 64, 192, 27, 5), (16, 32, 16)),    # configs[3]: 196/92/102, 236/184/99, 226/104/104
        ((16, 32, 32, 256, 9), (32, 32, 32)),     # configs[4]: -/499/285, -/506/283, -/549/310
        ((32, 32, 64, 60, 5), (32, 16, 32)),      # 68/45/36, 81/55/76, 123/76/55
        ((128, 96, 256, 13, 3), (8, 16, 16)),     # 46/50/168, 94/56/181, 58/53/186
        ((128, 256, 256, 13, 3), (8, 16, 16)),    # 87/92/351, 161/92/356, 97/91/365
        ((32, 64, 64, 56, 3), (16, 16, 32)),      # 51/43/50, 60/43/50, 82/60/56
    ]
    for (B, cin, cout, H, k), want in measured:
        got = tuple(L.fbfft_conv_choose_fft_size(p, B, cin, cout, H, H, k, k) for p in range(3))
        assert got == want, ((B, cin, cout, H, k), got)
    for (H, W, kH, kW) in [(27, 27, 5, 5), (8, 8, 3, 3), (12, 40, 3, 5), (16, 16, 1, 1),
                           (100, 7, 7, 7), (33, 33, 17, 2), (9, 9, 9, 9), (500, 300, 32, 32)]:
        for p in range(3):
            N = L.fbfft_conv_choose_fft_size(p, 4, 3, 5, H, W, kH, kW)
            assert N in (8, 16, 32) and N >= max(kH, kW), (p, H, W, kH, kW, N)
            # the workspace of size 0 is the workspace of the chosen size
            assert L.fbfft_conv_workspace_image(p, 4, 3, 5, H, W, kH, kW, 0) == \
                L.fbfft_conv_workspace_image(p, 4, 3, 5, H, W, kH, kW, N) > 0
    # an image that fits one 32-point window is one window for the input gradient too (its
    # 30..32 rows are more than the 28 a window advances by, but there is nothing to advance to)
    for H in (29, 30, 31, 32):
        assert L.fbfft_conv_choose_fft_size(1, 128, 64, 192, H, H, 5, 5) == 32, H
    # no size holds the filter, the filter is larger than the image, bad pass or counts
    assert L.fbfft_conv_choose_fft_size(0, 4, 3, 5, 64, 64, 33, 3) == 0
    assert L.fbfft_conv_choose_fft_size(0, 4, 3, 5, 4, 4, 5, 5) == 0
    assert L.fbfft_conv_choose_fft_size(3, 4, 3, 5, 27, 27, 5, 5) == 0
    assert L.fbfft_conv_choose_fft_size(0, 0, 3, 5, 27, 27, 5, 5) == 0
    assert L.fbfft_conv_workspace_image(0, 4, 3, 5, 64, 64, 33, 3, 0) == 0


# timed on both kernels (N points; matrix kernel / lanes): 11.5 / 17.1, 13.9 / 26.8, 19.9 / 26.1, 6.8 / 7.9, 16.9
# / 27.9 us; 77.9 / 9.4, 13.3 / 11.6, 8.3 / 3.6, 17.3 / 12.2 us
@pytest.mark.parametrize("I,J,K,N,kind", [
    (253, 100, 2, 16, DIRECT), (369, 460, 1, 8, DIRECT), (198, 265, 1, 16, DIRECT), (80, 32, 3, 32, DIRECT),
    (81, 28, 55, 32, DIRECT),
    (1, 30, 323, 16, LANES), (27, 54, 24, 32, LANES), (9, 16, 5, 32, LANES), (18, 100, 17, 32, LANES)])
def test_mm_route_is_the_faster_kernel(I, J, K, N, kind):
    import torch
    space = torch.empty(2 * (N // 2 + 1) * N * (I * K + K * J + I * J))
    A, B, C = (t.view(d0, d1, N // 2 + 1, N, 2) for t, d0, d1 in zip(
        space.split([2 * (N // 2 + 1) * N * n for n in (I * K, K * J, I * J)]), (I, K, I), (K, J, J)))
    assert product_route(A, B, C, False, False)[0] == kind


@pytest.mark.parametrize("I,J,K", [(16, 8, 8), (8, 16, 16), (32, 32, 32), (5, 3, 3), (150, 8, 8)])
def test_mm_small_products_in_place_keep_the_kernels_that_read_first(I, J, K):
    """A small product goes to the kernel whose tiles are separate workgroups only where C lies
    apart from A and B: in place of one of them, or with one element in common, it keeps the matrix
    kernels, and just beside them it does not."""
    import torch
    xy = 544
    space = torch.empty((3, 160, 160 * xy * 2 + 2))  # no element is read or written

    def operand(n, d0, d1, shift=0):
        return space[n].view(-1).as_strided((d0, d1, xy, 2), (d1 * xy * 2, xy * 2, 2, 1),
                                            space[n].storage_offset() + shift)
    A, B, C = operand(0, I, K), operand(1, K, J), operand(2, I, J)
    assert product_route(A, B, C, False, False)[0] == LANES
    for other, into in ((A, 0), (B, 1)):
        assert product_route(A, B, operand(into, I, J), False, False)[0] == DIRECT
        last = other.numel()
        assert product_route(A, B, operand(into, I, J, last - 4), False, False)[0] == DIRECT
        assert product_route(A, B, operand(into, I, J, last - 2), False, False)[0] == REGISTERS  # 8-byte aligned
        assert product_route(A, B, operand(into, I, J, last), False, False)[0] == LANES


# timed both ways, transforms / sums: 10.8 / 18.6, 14.4 / 23.8, 13.5 / 18.9, 28.7 / 41.5 us; 11.1
# / 3.9, 19.2 / 6.1, 26.2 / 6.4 us
@pytest.mark.parametrize("pass_,B,cin,cout,H,W,kH,kW,small", [
    (0, 81, 12, 22, 6, 6, 6, 6, False), (0, 25, 59, 75, 5, 5, 4, 4, False), (0, 71, 32, 15, 5, 5, 4, 4, False),
    (1, 15, 6, 2, 112, 112, 2, 9, False),
    (0, 9, 5, 9, 8, 7, 3, 3, True), (0, 7, 4, 10, 55, 55, 2, 2, True), (1, 47, 11, 143, 10, 11, 1, 1, True)])
def test_small_layers_run_the_faster_way(pass_, B, cin, cout, H, W, kH, kW, small):
    fn = F.lib()._ZN9fbfft_amd9runsSmallEiiiiiiiii
    fn.argtypes, fn.restype = [ctypes.c_int] * 9, ctypes.c_bool
    n = F.conv_choose_fft_size(pass_, B, cin, cout, H, W, kH, kW)
    assert fn(pass_, n, B, cin, cout, H, W, kH, kW) == small


# contractions with a short side that would leave most of the chip idle: 32 x 32 tiles, but not for up to 16
# rows and few slices of k (11.7 us on 32 rows, 12.5 on the tiles, 11.0 on 16 rows: the first of these)
@pytest.mark.parametrize("pass_,N,B,cin,cout,H,W,k,kind", [
    (2, 16, 1, 171, 2, 12, 9, 8, REGS_NARROW), (2, 0, 2, 362, 3, 14, 14, 2, REGS_NARROW),
    (2, 16, 48, 171, 2, 12, 9, 8, REGS_SPLIT_K), (2, 16, 8, 171, 20, 12, 9, 8, REGS_SPLIT_K),
    (2, 32, 8, 171, 20, 30, 30, 8, REGS_WIDE)])
def test_contraction_of_a_short_side(pass_, N, B, cin, cout, H, W, k, kind):
    assert conv_route(pass_, N, B, cin, cout, H, W, k)[0] == kind


def test_the_library_builds_without_python():
    """The C ABI's own target needs hipcc only; the Python package's module is a target apart."""
    csrc = os.path.join(ROOT, "fbcuda_amd", "csrc")
    plan = subprocess.run(["make", "-C", csrc, "-n", "-B", "PYTHON=/nonexistent"], capture_output=True, text=True)
    assert plan.returncode == 0 and "libfbfft_amd.so" in plan.stdout and "/nonexistent" not in plan.stderr
    assert "binding" not in plan.stdout
    assert "binding.cpp" in subprocess.run(["make", "-C", csrc, "-n", "-B", "binding"], capture_output=True,
                                           text=True).stdout


@pytest.mark.parametrize("built", [False, True])
def test_calls_without_the_native_module_go_the_general_way(monkeypatch, tmp_path, built):
    """Not built: the general way's results and errors, without a word; built and not loading: the
    same, with a warning."""
    import torch
    monkeypatch.setattr(F, "_native", None)
    monkeypatch.setattr(F, "_HERE", str(tmp_path))
    monkeypatch.delattr(F, "_binding", raising=False)
    monkeypatch.setitem(sys.modules, "fbcuda_amd._binding", None)
    if built:
        (tmp_path / "_binding.so").write_bytes(b"")
    calls = []
    monkeypatch.setattr(F, "_on_gpu", lambda *ts: calls.append("on_gpu"))
    monkeypatch.setattr(F, "_stream", lambda stream: 0)
    x, y = torch.zeros((2, 300)), torch.zeros((2, 151, 2))  # refused on the host, nothing is launched
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        assert F.fbfft1D(x, y) == F.UnsupportedSize
        assert F.fbfft1D(x, y) == F.UnsupportedSize
    assert calls == ["on_gpu"] * 2
    assert [w.category for w in seen] == ([RuntimeWarning] if built else [])


# filters of 1 x 1 whose results are too few for a workgroup per CU: a long chain over the contracted planes keeps the
# transforms, which cut it into ranges (us, transforms / product: 52 / 192, 73 / 236, 69 / 83, 28 / 47, 45 / 108); not where the
# transforms take longer (295 / 237, 446 / 197, 55 / 51), nor where results are many
@pytest.mark.parametrize("pass_,N,B,cin,cout,H,W,product", [
    (0, 0, 1, 4000, 64, 4, 4, False), (0, 64, 64, 4100, 64, 8, 8, False), (0, 0, 64, 1400, 256, 8, 8, False),
    (1, 0, 64, 64, 1000, 8, 8, False), (1, 0, 1, 64, 2000, 56, 56, False),
    (0, 0, 1, 4100, 400, 28, 28, True), (0, 64, 1, 4096, 1000, 2, 2, True),
    (0, 0, 64, 4100, 256, 14, 14, True), (1, 0, 64, 600, 4100, 14, 14, True), (2, 0, 1, 4000, 64, 4, 4, True)])
def test_long_chains_of_1x1_filters_keep_the_transforms(pass_, N, B, cin, cout, H, W, product):
    assert (conv_route(pass_, N, B, cin, cout, H, W, 1)[0] == POINT) == product
