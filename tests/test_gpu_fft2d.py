"""GPU parity of fbfft2D / fbifft2D (C ABI fbfft_r2c_2d / fbfft_c2r_2d) against
the CPU oracle: fp32 transcription, fp64 DFT, golden fixtures, edge cases and
size-independent properties at the benchmark's full size."""
import os

import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import TOL_FFT, c, check, dev, fft2d, ifft2d, rel

pytestmark = pytest.mark.gpu
GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "fft_vectors.npz"))
SIZES = [8, 16, 32, 64, 128]


@pytest.mark.parametrize("key", [k[4:] for k in GOLD.files if k.startswith("x2d_")])
def test_golden(key):
    N, h, w, padL, padU = map(int, key.split("_"))
    rc, out = fft2d(GOLD["x2d_" + key], N, padL, padU)
    assert rc == F.Success
    assert rel(c(out), GOLD["f2d_" + key]) < TOL_FFT


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("case", ["full", "ragged", "padded", "tiny"])
@pytest.mark.parametrize("B", [1, 5, 67])
def test_forward_inverse_vs_oracle(oracle, N, case, B):
    h, w, padL, padU = {"full": (N, N, 0, 0), "ragged": (N - 5, N - 3, 0, 0),
                        "padded": (N - 5, N - 4, 2, 3), "tiny": (5, 5, 0, 0)}[case]
    x = synth.normal((B, h, w), seed=N + B).numpy()
    rc, got = fft2d(x, N, padL, padU)
    assert rc == F.Success
    _, want32 = oracle.fbfft2d(x, N, padL, padU)
    want64 = oracle.dft2d_r2c(x, N, padL, padU)
    assert rel(got, want32) < TOL_FFT
    assert rel(got, want64) < TOL_FFT
    # inverse of the oracle's spectrum, cropped on store; cells outside stay untouched
    rc, back = ifft2d(want32, h, w, padL, padU)
    assert rc == F.Success
    _, back32 = oracle.fbifft2d(want32, h, w, padL, padU)
    assert rel(back, back32) < TOL_FFT
    assert rel(back, N * N * x.astype(np.float64)) < TOL_FFT


@pytest.mark.parametrize("N", SIZES)
def test_inverse_writes_only_the_window(oracle, N):
    """crop-on-store: a real tensor smaller than N x N receives exactly its window."""
    x = synth.normal((3, N, N), seed=77).numpy()
    _, spec = oracle.fbfft2d(x, N)
    h, w, padL, padU = N - 9 if N > 9 else 3, N - 5, 1, 2
    rc, got = ifft2d(spec, h, w, padL, padU)
    assert rc == F.Success
    want = N * N * x[:, padU:padU + h, padL:padL + w].astype(np.float64)
    assert rel(got, want) < TOL_FFT


@pytest.mark.parametrize("N", [8, 16, 32])
def test_inverse_lane0_quirk(oracle, N):
    """Imaginary parts of F[0][0] and F[N/2][0] are ignored (fbfft/FFT2D32.cuh:313-315)."""
    x = synth.normal((2, N, N), seed=5).numpy()
    _, spec = oracle.fbfft2d(x, N)
    spec[:, 0, 0, 1] = 3.0
    spec[:, N // 2, 0, 1] = -4.0
    _, got = ifft2d(spec, N, N)
    _, want = oracle.fbifft2d(spec, N, N)
    assert rel(got, want) < TOL_FFT
    assert rel(got, N * N * x.astype(np.float64)) < TOL_FFT


@pytest.mark.parametrize("N", SIZES)
def test_strided_operands(oracle, N):
    """Non-contiguous views: padded batch / row strides on both operands."""
    B = 6
    x = synth.normal((B, N, N), seed=9).numpy()
    big = torch.zeros((B, N + 3, N + 4), device=dev())
    real = big[:, 1:N + 1, 2:N + 2]
    real.copy_(torch.from_numpy(x))
    wide = torch.full((B, N // 2 + 2, N + 2, 2), float("nan"), device=dev())
    spec = wide[:, :N // 2 + 1, 1:N + 1, :]
    assert F.fbfft2D(real, spec) == F.Success
    torch.cuda.synchronize()
    _, want = oracle.fbfft2d(x, N)
    assert rel(spec.cpu().numpy(), want) < TOL_FFT
    back = torch.zeros_like(big)
    assert F.fbifft2D(spec, back[:, 1:N + 1, 2:N + 2]) == F.Success
    torch.cuda.synchronize()
    assert rel(back[:, 1:N + 1, 2:N + 2].cpu().numpy(), N * N * x.astype(np.float64)) < TOL_FFT
    assert float(back[:, 0].abs().max()) == 0.0  # nothing outside the view was written


def test_error_codes():
    d = dev()
    real = torch.zeros((4, 32, 32), device=d)
    assert F.fbfft2D(real, torch.zeros((4, 17, 32, 2), device=d)) == F.Success
    assert F.fbfft2D(real, torch.zeros((4, 129, 256, 2), device=d)) == F.UnsupportedSize
    assert F.fbfft2D(real, torch.zeros((4, 7, 12, 2), device=d)) == F.UnsupportedSize
    assert F.fbfft2D(real, torch.zeros((4, 15, 32, 2), device=d)) == F.UnsupportedSize
    assert F.fbfft2D(real, torch.zeros((4, 16, 32, 2), device=d)) == F.Success  # packed rows
    assert F.fbfft2D(torch.zeros((4, 64, 64), device=d),
                     torch.zeros((4, 32, 64, 2), device=d)) == F.UnsupportedSize  # N <= 32 only
    assert F.fbfft2D(real, torch.zeros((3, 17, 32, 2), device=d)) == F.UnsupportedDimension
    assert F.fbfft2D(real, torch.zeros((4, 17, 32), device=d)) == F.UnsupportedDimension
    assert F.fbfft2D(torch.zeros((4, 40, 32), device=d),
                     torch.zeros((4, 17, 32, 2), device=d)) == F.UnsupportedSize
    assert F.fbifft2D(torch.zeros((4, 129, 256, 2), device=d), real) == F.UnsupportedSize
    # empty batch is a successful no-op
    assert F.fbfft2D(torch.zeros((0, 32, 32), device=d), torch.zeros((0, 17, 32, 2), device=d)) == F.Success
    torch.cuda.synchronize()


def per_plane_rel(got, want):
    """Largest rel-L2 of any single plane (a whole-tensor norm could hide one bad plane)."""
    B = got.shape[0]
    a = np.asarray(got, np.float64).reshape(B, -1)
    b = np.asarray(want, np.float64).reshape(B, -1)
    return float((np.linalg.norm(a - b, axis=1) / np.maximum(np.linalg.norm(b, axis=1), 1e-300)).max())


@pytest.mark.parametrize("N,B", [(32, 16384), (8, 1 << 20), (16, 1 << 18), (64, 16384), (128, 4096)])
def test_full_size_properties(oracle, N, B):
    """Benchmark sizes: round trip ifft(fft(x)) = N^2 x on the whole tensor, linearity, and
    parity with the CPU transcription plane by plane - on every one of configs[1]'s 16384
    planes, on 256 seeded planes (first and last included) of each configs[2] size - for
    the forward transform and, on the transcription's own spectra, for the inverse."""
    d = dev()
    seed = {32: 1, 8: 5, 16: 6, 64: 8, 128: 9}[N]
    x = synth.normal((B, N, N), seed=seed, device=d)
    spec = torch.empty((B, N // 2 + 1, N, 2), device=d)
    assert F.fbfft2D(x, spec) == F.Success
    back = torch.empty_like(x)
    assert F.fbifft2D(spec, back) == F.Success
    torch.cuda.synchronize()
    err = (back / (N * N) - x).double().norm() / x.double().norm()
    print("parity round trip %dx%d over all %d planes: %.2e" % (N, N, B, float(err)))
    assert float(err) < TOL_FFT
    if N == 32:
        pick = np.arange(B)
    else:
        pick = np.unique(np.concatenate([[0, 1, B - 2, B - 1],
                                         np.random.default_rng(seed).choice(B, 252, replace=False)]))
    xp = x.cpu().numpy()[pick]
    rc, want = oracle.fbfft2d(xp, N)
    assert rc == 0
    got = spec.cpu().numpy()[pick]
    tag = "%dx%d, %d of %d planes" % (N, N, len(pick), B)
    check("fbfft2D vs transcription (%s)" % tag, got, want, TOL_FFT)
    check("fbfft2D vs fp64 DFT (first 64 of them)", got[:64], oracle.dft2d_r2c(xp[:64], N), TOL_FFT)
    worst = per_plane_rel(got, want)
    print("parity fbfft2D worst single plane (%s): %.2e" % (tag, worst))
    assert worst < TOL_FFT
    # inverse: the same spectra (the transcription's) into both implementations
    rc, want_back = oracle.fbifft2d(want, N, N)
    assert rc == 0
    sd = torch.from_numpy(want).to(d)
    bd = torch.full((len(pick), N, N), float("nan"), device=d)
    assert F.fbifft2D(sd, bd) == F.Success
    torch.cuda.synchronize()
    check("fbifft2D vs transcription, same spectra (%s)" % tag, bd.cpu().numpy(), want_back, TOL_FFT)
    assert per_plane_rel(bd.cpu().numpy(), want_back) < TOL_FFT
    del sd, bd
    # linearity on a slice: F(2x + y) = 2F(x) + F(y)
    n = min(B // 2, 4096)
    z = (2 * x[:n] + x[n:2 * n]).contiguous()
    sz = torch.empty((n, N // 2 + 1, N, 2), device=d)
    assert F.fbfft2D(z, sz) == F.Success
    torch.cuda.synchronize()
    lin = (sz - (2 * spec[:n] + spec[n:2 * n])).double().norm() / sz.double().norm()
    assert float(lin) < TOL_FFT


@pytest.mark.parametrize("N,B", [(32, 9001), (16, 33333), (8, 110001)])
def test_two_groups_per_wave_tail(oracle, N, B):
    """Batch sizes in the one-to-two-round regime, where a wave transforms two groups
    of planes and prefetches the second: odd group counts and a ragged last group."""
    d = dev()
    x = synth.normal((B, N, N), seed=12, device=d)
    spec = torch.full((B, N // 2 + 1, N, 2), float("nan"), device=d)
    back = torch.full((B, N, N), float("nan"), device=d)
    assert F.fbfft2D(x, spec) == F.Success
    assert F.fbifft2D(spec, back) == F.Success
    torch.cuda.synchronize()
    assert bool(torch.isfinite(spec).all()) and bool(torch.isfinite(back).all())
    err = (back / (N * N) - x).double().norm() / x.double().norm()
    assert float(err) < TOL_FFT
    pick = [0, 1, B // 2, B - 130, B - 5, B - 4, B - 3, B - 2, B - 1]
    _, want = oracle.fbfft2d(x[pick].cpu().numpy(), N)
    assert rel(spec[pick].cpu().numpy(), want) < TOL_FFT


@pytest.mark.parametrize("N", [2, 4])
@pytest.mark.parametrize("B", [1, 2, 5, 1000])
def test_warp_kernel_sizes(oracle, N, B):
    """N = 2 and 4 (the reference's plane-pairing warp kernel, fbfft/FBFFT2D-inl.cuh:611-612):
    transposed [kx half][ky] layout, odd batches, windows and padding."""
    for h, w, padL, padU in [(N, N, 0, 0), (N - 1, N, 0, 0), (N - 1, N - 1, 1, 1)]:
        x = synth.normal((B, h, w), seed=100 + N + B).numpy()
        rc, got = fft2d(x, N, padL, padU)
        assert rc == F.Success
        _, want32 = oracle.fbfft2d(x, N, padL, padU)
        assert rel(got, want32) < TOL_FFT
        assert rel(got, oracle.dft2d_r2c(x, N, padL, padU)) < TOL_FFT
        rc, back = ifft2d(want32, h, w, padL, padU)
        assert rc == F.Success
        _, back32 = oracle.fbifft2d(want32, h, w, padL, padU)
        assert rel(back, back32) < TOL_FFT
        assert rel(back, N * N * x.astype(np.float64)) < TOL_FFT
    # strided views on both sides
    x = synth.normal((B, N, N), seed=7).numpy()
    big = torch.zeros((B, N + 1, N + 3), device=dev())
    real = big[:, 1:, 2:N + 2]
    real.copy_(torch.from_numpy(x))
    wide = torch.full((B, N // 2 + 2, N + 1, 2), float("nan"), device=dev())
    spec = wide[:, 1:, :N, :]
    assert F.fbfft2D(real, spec) == F.Success
    torch.cuda.synchronize()
    assert rel(spec.cpu().numpy(), oracle.dft2d_r2c(x, N)) < TOL_FFT
    assert bool(torch.isnan(wide[:, 0]).all()) and bool(torch.isnan(wide[:, :, N]).all())


@pytest.mark.parametrize("seed", range(40))
def test_random_windows_and_views(oracle, seed):
    """Seeded random draw over size, batch, window, padding (also windows that
    hang over the right / bottom edge, which MemoryAccess.cuh:19-25 clips), and
    views that are transposed or padded in memory."""
    rng = np.random.default_rng(1000 + seed)
    N = int(rng.choice([2, 4, 8, 16, 32, 64, 128]))
    B = int(rng.integers(1, 20))
    h, w = int(rng.integers(1, N + 1)), int(rng.integers(1, N + 1))
    padL, padU = (int(rng.integers(0, N // 2 + 1)), int(rng.integers(0, N // 2 + 1))) \
        if rng.random() < 0.6 else (0, 0)
    x = synth.normal((B, h, w), seed=seed).numpy()
    d = dev()
    kind = int(rng.integers(0, 3))
    if kind == 0:                                   # contiguous
        real = torch.from_numpy(x).to(d)
    elif kind == 1:                                 # padded rows and batch stride
        big = torch.zeros((B, h + 2, w + 3), device=d)
        real = big[:, 1:h + 1, 2:w + 2]
        real.copy_(torch.from_numpy(x))
    else:                                           # x and y swapped in memory
        real = torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1))).to(d).transpose(1, 2)
    if rng.random() < 0.5:
        spec = torch.full((B, N // 2 + 1, N, 2), float("nan"), device=d)
    else:
        wide = torch.full((B + 1, N // 2 + 2, N + 1, 2), float("nan"), device=d)
        spec = wide[1:, 1:, :N, :]
    assert F.fbfft2D(real, spec, padL, padU) == F.Success
    torch.cuda.synchronize()
    _, want32 = oracle.fbfft2d(x, N, padL, padU)
    got = spec.cpu().numpy()
    assert rel(got, want32) < TOL_FFT, (N, B, h, w, padL, padU, kind)
    assert rel(got, oracle.dft2d_r2c(x, N, padL, padU)) < TOL_FFT
    # and back into a view of the same geometry
    # (cells of the window that hang over the edge keep what they held)
    back = torch.full_like(real, 7.0)
    assert F.fbifft2D(spec, back, padL, padU) == F.Success
    torch.cuda.synchronize()
    _, back32 = oracle.fbifft2d(want32, h, w, padL, padU, out=np.full((B, h, w), 7.0, np.float32))
    assert rel(back.cpu().numpy(), back32) < TOL_FFT, (N, B, h, w, padL, padU, kind)


@pytest.mark.parametrize("N,h,w,padL,padU", [
    (64, 60, 60, 0, 0), (64, 60, 60, 4, 3), (64, 17, 8, 8, 40), (64, 64, 64, 4, 1),
    (128, 124, 124, 0, 0), (128, 124, 120, 4, 2), (128, 31, 64, 60, 100), (128, 5, 4, 124, 0)])
def test_windows_that_move_as_16_byte_words(oracle, N, h, w, padL, padU):
    """Windows whose rows start on 16-byte boundaries with width and left edge
    multiples of 4 take the float4 loader of the 64 / 128 kernels (also hanging
    over the right edge)."""
    B = 5
    x = synth.normal((B, h, w), seed=N + h).numpy()
    rc, got = fft2d(x, N, padL, padU)
    assert rc == F.Success
    _, want32 = oracle.fbfft2d(x, N, padL, padU)
    assert rel(got, want32) < TOL_FFT
    assert rel(got, oracle.dft2d_r2c(x, N, padL, padU)) < TOL_FFT


@pytest.mark.parametrize("N", [8, 16, 32])
def test_odd_plane_stride_mixes_the_window_load_paths(oracle, N):
    """Even window, even row stride, odd plane stride: every other plane starts on an
    8-byte boundary, so the planes of one wave take different load paths."""
    B, h, w = 11, N // 2, N // 2 - 2
    x = synth.normal((B, h, w), seed=5 * N).numpy()
    flat = torch.zeros(B * (h * w + 1) + 8, device=dev())
    real = flat.as_strided((B, h, w), (h * w + 1, w, 1))
    real.copy_(torch.from_numpy(x))
    spec = torch.full((B, N // 2 + 1, N, 2), float("nan"), device=dev())
    assert F.fbfft2D(real, spec, 2, 1) == F.Success
    torch.cuda.synchronize()
    _, want = oracle.fbfft2d(x, N, 2, 1)
    assert rel(spec.cpu().numpy(), want) < TOL_FFT
    back = torch.zeros_like(flat).as_strided((B, h, w), (h * w + 1, w, 1))
    assert F.fbifft2D(spec, back, 2, 1) == F.Success
    torch.cuda.synchronize()
    assert rel(back.cpu().numpy(), N * N * x.astype(np.float64)) < TOL_FFT


@pytest.mark.parametrize("N", [4, 8, 32, 64])
@pytest.mark.parametrize("h,w", [(0, 3), (3, 0)])
def test_empty_window_gives_zero_spectra(N, h, w):
    """B > 0 planes whose real window is empty are all padding: zeros, not stale data."""
    x = torch.zeros((3, h, w), device=dev())
    out = torch.full((3, N // 2 + 1, N, 2), float("nan"), device=dev())
    assert F.fbfft2D(x, out) == F.Success
    torch.cuda.synchronize()
    assert float(out.abs().max()) == 0.0


@pytest.mark.parametrize("N,B", [(32, 8195), (32, 12289), (32, 14336), (32, 14339), (16, 30727),
                                 (16, 53760), (16, 53767), (8, 98317), (8, 172032), (8, 172049)])
def test_batches_either_side_of_the_two_groups_per_wave_switch(oracle, N, B):
    """Batches just above one round of resident waves, at 1.75 rounds (the last that pair)
    and just beyond (one group per wave again), odd tails included: every plane of the
    forward transform against the transcription, and the inverse on its spectra."""
    d = dev()
    x = synth.normal((B, N, N), seed=70 + N, device=d)
    spec = torch.full((B, N // 2 + 1, N, 2), float("nan"), device=d)
    assert F.fbfft2D(x, spec) == F.Success
    back = torch.full_like(x, float("nan"))
    assert F.fbifft2D(spec, back) == F.Success
    torch.cuda.synchronize()
    rc, want = oracle.fbfft2d(x.cpu().numpy(), N)
    assert rc == 0
    got = spec.cpu().numpy()
    assert np.isfinite(got).all()
    assert per_plane_rel(got, want) < TOL_FFT
    err = (back / (N * N) - x).double().norm() / x.double().norm()
    assert bool(torch.isfinite(back).all()) and float(err) < TOL_FFT


# windows in planes of 64 and 128 points that begin and end beside the rows of a wave (16 and 8 at a time, 32 and
# 64 rows apart), whose samples move as words, as pairs and one by one, and spectra that do not move as words
@pytest.mark.parametrize("N,h,w,padL,padU", [
    (64, 1, 4, 0, 63), (64, 15, 60, 4, 1), (64, 16, 7, 1, 16), (64, 17, 64, 0, 15), (64, 33, 62, 2, 31),
    (64, 64, 1, 63, 0), (64, 48, 33, 8, 16), (128, 1, 128, 0, 127), (128, 7, 6, 122, 1), (128, 8, 126, 2, 8),
    (128, 9, 5, 1, 7), (128, 65, 127, 0, 63), (128, 128, 1, 127, 0), (128, 120, 100, 28, 8)])
def test_windows_beside_the_rows_of_a_wave(oracle, N, h, w, padL, padU):
    B = 3
    x = synth.normal((B, h, w), seed=h + w).numpy()
    rc, got = fft2d(x, N, padL, padU)
    want = oracle.dft2d_r2c(x, N, padL, padU)
    # fourteen (twelve) steps of butterflies, three roots and a fix-up, each a rounding of at most 2^-24 in both
    # parts of a value that grows like the square root of its terms
    bar = np.sqrt(2 * (np.log2(N) * 2 + 4)) * 2.0 ** -24
    assert rc == F.Success and rel(got, want) < bar
    d = dev()
    wide = torch.full((B, N // 2 + 1, N, 4), 7.0, device=d)
    view = wide[..., :2]
    assert F.fbfft2D(torch.from_numpy(x).to(d), view, padL, padU) == F.Success
    torch.cuda.synchronize()
    assert np.array_equal(view.cpu().numpy(), got) and bool((wide[..., 2:] == 7.0).all())
    back = torch.full((B, h + 2, w + 2), 7.0, device=d)
    assert F.fbifft2D(view, back[:, 1:-1, 1:-1], padL, padU) == F.Success
    torch.cuda.synchronize()
    inner = back[:, 1:-1, 1:-1].cpu().numpy()
    assert rel(inner, N * N * x.astype(np.float64)) < 2 * bar * np.sqrt(N * N / (h * w))
    back[:, 1:-1, 1:-1] = 7.0
    assert bool((back == 7.0).all())


# windows one after the other in memory that move as streams of 16-byte words, either side of the batches that
# do (1024 groups of 128 / N planes; forward up to 16 points only), whole and partly filled last groups, whose
# floats end between two words, and windows beside them in memory that do not move that way
@pytest.mark.parametrize("N,B,h,w,padL,padU", [
    (32, 4096, 27, 27, 0, 0), (32, 4093, 27, 27, 0, 0), (32, 4097, 27, 27, 0, 0), (32, 4095, 5, 31, 1, 2), (32, 4094, 1, 1, 31, 31),
    (32, 9001, 28, 28, 2, 1), (16, 8185, 13, 13, 1, 2), (16, 8191, 16, 15, 0, 0), (16, 8186, 1, 3, 13, 15),
    (16, 31003, 13, 13, 0, 0), (8, 16369, 7, 7, 0, 1), (8, 16371, 3, 5, 3, 4), (8, 100003, 7, 5, 1, 1), (8, 100001, 1, 1, 7, 0),
    # inverse windows either side of four ninths of a plane, at 8 points a quarter
    (32, 4101, 15, 31, 0, 0), (32, 4101, 14, 32, 0, 1), (16, 8203, 9, 13, 2, 0), (16, 8203, 8, 14, 0, 0),
    (8, 16389, 4, 4, 1, 2), (8, 16389, 3, 5, 0, 0),
    # forward either side of half a plane and, below it, of one and a half rounds of waves; pairs of 8 points
    (16, 9001, 9, 15, 1, 0), (16, 9002, 8, 15, 0, 2), (16, 46003, 8, 15, 0, 0), (8, 160001, 6, 8, 0, 1), (8, 160003, 5, 8, 0, 0)])
def test_windows_that_move_as_streams(oracle, N, B, h, w, padL, padU):
    d = dev()
    x = synth.normal((B, h, w), seed=B).to(d)
    spec = torch.full((B + 1, N // 2 + 1, N, 2), 7.0, device=d)
    assert F.fbfft2D(x, spec[:B], padL, padU) == F.Success
    flat = torch.full((B * h * w + 8,), 7.0, device=d)
    back = flat[:B * h * w].view(B, h, w)
    assert F.fbifft2D(spec[:B], back, padL, padU) == F.Success
    other = torch.full((B, h + 1, w + 1), 7.0, device=d)  # the same windows, not one after the other
    wide = torch.zeros((B, h, w + 1), device=d)
    wide[:, :, :w] = x
    spec2 = torch.empty_like(spec[:B])
    assert F.fbfft2D(wide[:, :, :w], spec2, padL, padU) == F.Success
    assert F.fbifft2D(spec[:B], other[:, :h, :w], padL, padU) == F.Success
    torch.cuda.synchronize()
    assert bool((spec[B] == 7.0).all()) and bool((flat[B * h * w:] == 7.0).all())
    # (the compiler need not contract the same products to multiply-adds in both: roundings of 2^-24 apart)
    assert rel(spec[:B].cpu().numpy(), spec2.cpu().numpy()) < 3e-7
    assert rel(other[:, :h, :w].cpu().numpy(), back.cpu().numpy()) < 3e-7 * np.sqrt(N * N / (h * w))
    at = np.unique(np.r_[0:16, B // 2:B // 2 + 16, B - 40:B])
    assert rel(spec[:B].cpu().numpy()[at], oracle.dft2d_r2c(x.cpu().numpy()[at], N, padL, padU)) < TOL_FFT
    assert rel(back.cpu().numpy(), N * N * x.cpu().numpy().astype(np.float64)) < TOL_FFT * np.sqrt(N * N / (h * w))


# windows one after the other in memory, in batches that move as streams, that reach past the transform's right edge,
# its bottom edge or both, or are larger than it: what it does not cover keeps what it held
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("N", [8, 16, 32])
@pytest.mark.parametrize("dh,dw,padL,padU", [(0, 0, 1, 0), (0, 0, 0, 1), (-1, -2, 5, 3), (0, 3, 0, 0), (2, 0, 0, 0),
                                             (5, 7, 2, 3), (0, 0, 1 << 30, 0), (-3, 0, 0, 2147483647)])
def test_inverse_windows_past_the_transform(oracle, N, packed, dh, dw, padL, padU):
    B, h, w = 4096 * 32 // N + 3, N + dh, N + dw
    d = dev()
    x = synth.normal((B, N, N), seed=N).to(d)
    spec = torch.empty((B, N // 2 + (not packed), N, 2), device=d)
    assert F.fbfft2D(x, spec) == F.Success
    flat = torch.full((B * h * w + 8,), 7.0, device=d)
    back = flat[:B * h * w].view(B, h, w)
    assert F.fbifft2D(spec, back, padL, padU) == F.Success
    torch.cuda.synchronize()
    ch, cw = max(0, min(h, N - padU)), max(0, min(w, N - padL))
    assert bool((flat[B * h * w:] == 7.0).all())
    assert bool((back[:, ch:] == 7.0).all()) and bool((back[:, :, cw:] == 7.0).all())
    if ch and cw:
        want = N * N * x[:, padU:padU + ch, padL:padL + cw].double()
        got = back[:, :ch, :cw].double()
        assert float((got - want).norm() / want.norm()) < TOL_FFT * np.sqrt(N * N / (ch * cw))
        at = np.r_[0:8, B - 8:B]
        rc, ref = oracle.fbifft2d(oracle.fbfft2d(x.cpu().numpy()[at], N)[1], N, N)
        assert rc == 0 and rel(got.cpu().numpy()[at], ref[:, padU:padU + ch, padL:padL + cw]) < TOL_FFT


# how the 64-point forward transform reads: four samples at a time from any float on, windows whose ends cut such words
# on either side at each place, windows narrower than one, samples that lie 2 and 7 apart, turned planes, and batches whose
# planes lie between each other
@pytest.mark.parametrize("h,w,padL,padU", [(64, 64, 0, 0), (61, 61, 2, 1), (50, 62, 1, 9), (33, 59, 4, 31), (7, 4, 59, 50),
                                           (64, 5, 3, 0), (20, 6, 58, 44), (40, 7, 30, 10), (9, 3, 61, 3), (12, 1, 17, 0),
                                           (64, 63, 7, 5), (30, 64, 62, 40)])
@pytest.mark.parametrize("layout", ["off1", "off3", "gap", "apart2", "apart7", "turned", "between"])
def test_forward_64_reads_any_layout(oracle, layout, h, w, padL, padU):
    B, d = 37, dev()
    x = synth.normal((B, h, w), seed=h + w)
    at = {"off1": lambda: torch.empty(B * h * w + 1, device=d)[1:].view(B, h, w),
          "off3": lambda: torch.empty(B * h * w + 3, device=d)[3:].view(B, h, w),
          "gap": lambda: torch.full((B, h + 1, 64 + 4), float("nan"), device=d)[:, 1:, 2:2 + w],
          "apart2": lambda: torch.full((B, h, w, 2), float("nan"), device=d)[..., 1],
          "apart7": lambda: torch.full((B, h, w, 7), float("nan"), device=d)[..., 3],
          "turned": lambda: torch.empty((B, w, h), device=d).transpose(1, 2),
          "between": lambda: torch.empty((h, w, B), device=d).permute(2, 0, 1)}[layout]()
    at.copy_(x)
    spec = torch.full((B + 1, 33, 64, 2), 7.0, device=d)
    assert F.fbfft2D(at, spec[:B], padL, padU) == F.Success
    torch.cuda.synchronize()
    assert bool((spec[B] == 7.0).all())
    plane = np.zeros((B, 64, 64), np.float32)
    ch, cw = min(h, 64 - padU), min(w, 64 - padL)
    plane[:, padU:padU + ch, padL:padL + cw] = x.numpy()[:, :ch, :cw]
    rc, want = oracle.fbfft2d(plane, 64)
    assert rc == 0 and per_plane_rel(spec[:B].cpu().numpy(), want) < TOL_FFT


# how the 64-point inverse writes: four samples at a time to any float, row ends within a word at each place, windows that hang over
# the transform's right edge or its bottom (what is not covered keeps what it held), narrower ones, and other layouts
@pytest.mark.parametrize("h,w,padL,padU", [(64, 64, 0, 0), (61, 61, 2, 1), (50, 62, 1, 9), (33, 59, 4, 31), (7, 9, 59, 50),
                                           (64, 5, 3, 0), (20, 6, 58, 44), (40, 7, 30, 10), (9, 3, 61, 3), (12, 1, 17, 0),
                                           (64, 63, 7, 5), (30, 64, 62, 40), (70, 81, 0, 3), (8, 8, 64, 0)])
@pytest.mark.parametrize("layout", ["off1", "off3", "gap", "apart2", "turned", "between"])
def test_inverse_64_writes_any_layout(oracle, layout, h, w, padL, padU):
    B, d = 37, dev()
    spec = oracle.fbfft2d(synth.normal((B, 64, 64), seed=h + w).numpy(), 64)[1]
    n = B * h * w
    flat = torch.full((2 * n + 100 * B * (h + 1) + 8,), 7.0, device=d)
    view = {"off1": flat[1:1 + n].view(B, h, w), "off3": flat[3:3 + n].view(B, h, w),
            "gap": flat[:B * (h + 1) * 100].view(B, h + 1, 100)[:, 1:, 2:2 + w],
            "apart2": flat[:2 * n].view(B, h, w, 2)[..., 1], "turned": flat[:n].view(B, w, h).transpose(1, 2),
            "between": flat[:n].view(h, w, B).permute(2, 0, 1)}[layout]
    assert F.fbifft2D(torch.from_numpy(spec).to(d), view, padL, padU) == F.Success
    torch.cuda.synchronize()
    got = view.cpu().numpy().copy()
    view.fill_(7.0)
    assert bool((flat == 7.0).all())
    ch, cw = max(0, min(h, 64 - padU)), max(0, min(w, 64 - padL))
    assert (got[:, ch:] == 7.0).all() and (got[:, :, cw:] == 7.0).all()
    if ch and cw:
        rc, full = oracle.fbifft2d(spec, 64, 64)
        want = full[:, padU:padU + ch, padL:padL + cw]
        # (of a few samples the largest may be small beside the others' roundings: the bar is on the plane's scale)
        err = np.abs(got[:, :ch, :cw].astype(np.float64) - want).max() / np.sqrt((full.astype(np.float64) ** 2).mean())
        assert rc == 0 and err < TOL_FFT


# spectra that lie in memory the other way round, [ky][kx], and so with gaps between rows and values
@pytest.mark.parametrize("N,B,h,w,padL,padU", [(64, 1, 64, 64, 0, 0), (64, 9, 40, 51, 3, 20), (128, 1, 128, 128, 0, 0),
                                               (128, 7, 128, 128, 0, 0), (128, 5, 77, 101, 9, 30), (128, 300, 31, 128, 0, 97)])
@pytest.mark.parametrize("gaps", [False, True])
def test_turned_spectra(oracle, N, B, h, w, padL, padU, gaps):
    d = dev()
    x = synth.normal((B, h, w), seed=N + B)
    hold = torch.full((B + 1, N + gaps, N // 2 + 1 + 2 * gaps, 2), 7.0, device=d)
    view = hold[:B, gaps:, gaps:gaps + N // 2 + 1].transpose(1, 2)
    assert F.fbfft2D(x.to(d), view, padL, padU) == F.Success
    back = torch.full((B, h, w), float("nan"), device=d)
    assert F.fbifft2D(view, back, padL, padU) == F.Success
    torch.cuda.synchronize()
    rc, want = oracle.fbfft2d(x.numpy(), N, padL, padU)
    assert rc == 0 and per_plane_rel(view.cpu().numpy(), want) < TOL_FFT
    assert per_plane_rel(back.cpu().numpy(), N * N * x.numpy().astype(np.float64)) < TOL_FFT * np.sqrt(N * N / (h * w))
    view.fill_(7.0)
    assert bool((hold == 7.0).all())


# batches whose planes lie between each other: consecutive planes share an XCD, and the grid ends on a multiple of eight
@pytest.mark.parametrize("N,h,w", [(64, 64, 64), (64, 37, 50), (128, 128, 128), (128, 75, 110)])
@pytest.mark.parametrize("B", [1, 2, 7, 8, 9, 45])
def test_planes_between_each_other(oracle, N, h, w, B):
    d = dev()
    x = synth.normal((B, h, w), seed=N + B + h)
    hold = torch.full((h, w, B + 2), 7.0, device=d)
    view = hold[..., 1:1 + B].permute(2, 0, 1)
    view.copy_(x)
    spec = torch.full((B + 1, N // 2 + 1, N, 2), 7.0, device=d)
    assert F.fbfft2D(view, spec[:B], N - w, 0) == F.Success
    view.fill_(float("nan"))
    assert F.fbifft2D(spec[:B], view, N - w, 0) == F.Success
    torch.cuda.synchronize()
    rc, want = oracle.fbfft2d(x.numpy(), N, N - w, 0)
    assert rc == 0 and per_plane_rel(spec[:B].cpu().numpy(), want) < TOL_FFT
    assert per_plane_rel(view.cpu().numpy(), N * N * x.numpy().astype(np.float64)) < TOL_FFT * np.sqrt(N * N / (h * w))
    assert bool((spec[B] == 7.0).all()) and bool((hold[..., 0] == 7.0).all()) and bool((hold[..., B + 1] == 7.0).all())


# and the same of spectra: one value of every plane, then the next (real planes whole, cut, and between each other as well)
@pytest.mark.parametrize("N,h,w", [(64, 64, 64), (64, 37, 50), (128, 128, 128), (128, 75, 110)])
@pytest.mark.parametrize("B,both", [(2, False), (7, True), (9, False), (45, True)])
def test_spectra_between_each_other(oracle, N, h, w, B, both):
    d = dev()
    x = synth.normal((B, h, w), seed=N + B + w).to(d)
    real = torch.empty((h, w, B), device=d).permute(2, 0, 1) if both else torch.empty((B, h, w), device=d)
    real.copy_(x)
    hold = torch.full((N // 2 + 1, N, B + 2, 2), 7.0, device=d)
    view = hold[:, :, 1:1 + B].permute(2, 0, 1, 3)
    assert F.fbfft2D(real, view, 0, N - h) == F.Success
    real.fill_(float("nan"))
    assert F.fbifft2D(view, real, 0, N - h) == F.Success
    torch.cuda.synchronize()
    rc, want = oracle.fbfft2d(x.cpu().numpy(), N, 0, N - h)
    assert rc == 0 and per_plane_rel(view.cpu().numpy(), want) < TOL_FFT
    assert per_plane_rel(real.cpu().numpy(), N * N * x.cpu().numpy().astype(np.float64)) < TOL_FFT * np.sqrt(N * N / (h * w))
    view.fill_(7.0)
    assert bool((hold == 7.0).all())


# samples four floats apart: planes and windows of 128 points either side of 104 columns, which are read row by row from there on
@pytest.mark.parametrize("h,w,padL,padU", [(128, 128, 0, 0), (128, 104, 3, 0), (77, 103, 9, 30), (5, 111, 17, 60), (61, 128, 0, 67),
                                           (128, 127, 5, 9), (1, 120, 8, 127)])
@pytest.mark.parametrize("B", [1, 9])
@pytest.mark.parametrize("turned", [False, True])
def test_forward_128_of_samples_four_apart(oracle, h, w, padL, padU, B, turned):
    d = dev()
    x = synth.normal((B, h, w), seed=h + w + B)
    hold = torch.full((B, h, w, 4), float("nan"), device=d)
    hold[..., 2] = x.to(d)
    spec = torch.full((B + 1, 128, 65, 2) if turned else (B + 1, 65, 128, 2), 7.0, device=d)
    view = spec[:B].transpose(1, 2) if turned else spec[:B]
    assert F.fbfft2D(hold[..., 2], view, padL, padU) == F.Success
    torch.cuda.synchronize()
    assert bool((spec[B] == 7.0).all())
    plane = np.zeros((B, 128, 128), np.float32)
    ch, cw = min(h, 128 - padU), min(w, 128 - padL)
    plane[:, padU:padU + ch, padL:padL + cw] = x.numpy()[:, :ch, :cw]
    rc, want = oracle.fbfft2d(plane, 128)
    assert rc == 0 and per_plane_rel(view.cpu().numpy(), want) < TOL_FFT


@pytest.mark.parametrize("N", [64, 128])  # (up to 32 points pairs of columns travel together instead)
def test_inverse_rows_whose_even_samples_overflow_keep_the_odd_ones(N):
    """Of the two ends of a spectrum's rows even samples are the sums, odd ones the differences."""
    d = dev()
    spec = torch.zeros(3, N // 2 + 1, N, 2)
    spec[0, 0, 0, 0], spec[0, N // 2, 0, 0] = 2e38, 1.5e38
    spec[1, 0, 0, 0], spec[1, N // 2, 0, 0] = -2e38, 1.5e38
    back = torch.full((3, N, N), 7.0, device=d)
    wide = torch.full((3, N, N + 1), 7.0, device=d)
    for to in (back, wide[:, :, :N]):
        assert F.fbifft2D(spec.to(d), to) == F.Success
        torch.cuda.synchronize()
        got = to.cpu()
        assert bool((got[0, :, ::2] == float("inf")).all()) and bool((got[1, :, 1::2] == float("-inf")).all())
        assert float((got[0, :, 1::2].double() / 0.5e38 - 1).abs().max()) < 1e-6
        assert float((got[1, :, ::2].double() / -0.5e38 - 1).abs().max()) < 1e-6
        assert bool((got[2] == 0.0).all())
