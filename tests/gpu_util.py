"""Shared helpers of the GPU parity tests: they call the product through its C ABI
(fbcuda_amd -> libfbfft_amd.so) and check it against the CPU oracle."""
import ctypes

import numpy as np
import torch

import fbcuda_amd as F

TOL_FFT = 1e-5    # rel-L2 per transform (vs the fp32 transcription and vs the fp64 DFT)
TOL_CONV = 1e-4   # rel-L2 per full convolution


class PassSize(ctypes.Structure):
    _fields_ = [("N", ctypes.c_int), ("maxSplits", ctypes.c_int)]


def pass_size(pass_, N, B, cin, cout, H, W, k):
    """(points, ranges at most) that a layer pass named N points runs on: the library's own
    host function, which is no part of the C ABI (common.h)."""
    fn = F.lib()._ZN9fbfft_amd8passSizeEiiiiiiiii
    fn.argtypes, fn.restype = [ctypes.c_int] * 9, PassSize
    r = fn(pass_, N, B, cin, cout, H, W, k, k)
    return r.N, r.maxSplits


class ProductRoute(ctypes.Structure):
    _fields_ = [(f, ctypes.c_int) for f in ("kind", "rows", "cols", "waves")]


REGISTERS, DIRECT, LANES = range(3)


def product_route(A, B, C, conjA, conjB):
    """The kernel (REGISTERS, DIRECT or LANES), rows and columns of its tile and waves that
    transposeMM runs on A, B, C [d0][d1]...[2]: the library's own host function (common.h), which
    looks at addresses, strides and sizes only."""
    fn = F.lib()._ZN9fbfft_amd12productRouteEPKfllS1_llS1_lliiiibb
    l, i, b = ctypes.c_long, ctypes.c_int, ctypes.c_bool
    fn.argtypes, fn.restype = [ctypes.c_void_p, l, l] * 3 + [i] * 4 + [b] * 2, ProductRoute
    I, K = (A.shape[1], A.shape[0]) if conjA else A.shape[:2]
    xy = int(np.prod(C.shape[2:-1]))
    r = fn(*(v for t in (A, B, C) for v in (t.data_ptr(), t.stride(0), t.stride(1))), I, C.shape[1], K, xy,
           conjA, conjB)
    return r.kind, r.rows, r.cols, r.waves


class ConvRoute(ctypes.Structure):
    _fields_ = [("kind", ctypes.c_int), ("N", ctypes.c_int), ("splits", ctypes.c_int)]


# what a layer pass runs on: convSmall, plane-major spectra, windows with binGemm<name>, or the products of filters of 1 x 1
SMALL, PLANE_MAJOR, REGS_SPLIT_K, REGS_WIDE, REGS_NARROW, DIRECT64, DIRECT128, SPLIT, POINT = range(9)


def conv_route(pass_, N, B, cin, cout, H, W, kH, kW=None):
    """(kind, points, ranges of the reduction) of a layer pass named N points (0: the library's
    choice), from the library's own host function (common.h)."""
    fn = F.lib()._ZN9fbfft_amd9convRouteEiiiiiiiii
    fn.argtypes, fn.restype = [ctypes.c_int] * 9, ConvRoute
    kW = kH if kW is None else kW
    r = fn(pass_, N, B, cin, cout, H, W, kH, kW)
    return r.kind, r.N, r.splits


def dev():
    return torch.device("cuda:0")


def c(a):
    a = np.asarray(a)
    return a[..., 0] + 1j * a[..., 1]


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    wide = np.complex128 if (np.iscomplexobj(a) or np.iscomplexobj(b)) else np.float64
    a, b = a.astype(wide).ravel(), b.astype(wide).ravel()
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def check(label, got, want, tol):
    """Asserts rel-L2(got, want) < tol and prints the observed figure (`pytest -s` shows it:
    the parity numbers quoted in the documents come from these lines)."""
    e = rel(got, want)
    print("parity %-58s rel-L2 %.2e (bar %.0e)" % (label, e, tol))
    assert e < tol, "%s: rel-L2 %.3e >= %.0e" % (label, e, tol)
    return e


def fft2d(x, N, padL=0, padU=0):
    """numpy real [B][h][w] -> numpy [B][N/2+1][N][2] through the C ABI."""
    xd = torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev())
    out = torch.full((x.shape[0], N // 2 + 1, N, 2), float("nan"), device=dev())
    rc = F.fbfft2D(xd, out, padL, padU)
    torch.cuda.synchronize()
    return rc, out.cpu().numpy()


def ifft2d(spec, h, w, padL=0, padU=0, fill=float("nan")):
    sd = torch.from_numpy(np.ascontiguousarray(spec, dtype=np.float32)).to(dev())
    out = torch.full((spec.shape[0], h, w), fill, device=dev())
    rc = F.fbifft2D(sd, out, padL, padU)
    torch.cuda.synchronize()
    return rc, out.cpu().numpy()
