"""GPU parity of fbfft1D / fbifft1D (C ABI fbfft_r2c_1d / fbfft_c2r_1d)."""
import os

import numpy as np
import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import check, TOL_FFT, c, dev, rel

pytestmark = pytest.mark.gpu
GOLD = np.load(os.path.join(os.path.dirname(__file__), "golden", "fft_vectors.npz"))
SIZES = [2, 4, 8, 16, 32, 64, 128, 256]


def fft1d(x, padL=0):
    xd = torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev())
    B, N = x.shape
    out = torch.full((B, N // 2 + 1, 2), float("nan"), device=dev())
    rc = F.fbfft1D(xd, out, padL)
    torch.cuda.synchronize()
    return rc, out.cpu().numpy()


def ifft1d(spec, padL=0, fill=float("nan")):
    sd = torch.from_numpy(np.ascontiguousarray(spec, dtype=np.float32)).to(dev())
    B, nc, _ = spec.shape
    out = torch.full((B, 2 * (nc - 1)), fill, device=dev())
    rc = F.fbifft1D(out, sd, padL)
    torch.cuda.synchronize()
    return rc, out.cpu().numpy()


@pytest.mark.parametrize("N", [8, 32, 256])
def test_golden(N):
    rc, out = fft1d(GOLD["x1d_%d" % N])
    assert rc == F.Success
    assert rel(c(out), GOLD["f1d_%d" % N]) < TOL_FFT


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("B", [1, 2, 7, 300, 1025])
def test_vs_oracle(oracle, N, B):
    x = synth.uniform((B, N), seed=N + B).numpy()
    rc, got = fft1d(x)
    assert rc == F.Success
    _, want32 = oracle.fbfft1d(x)
    assert rel(got, want32) < TOL_FFT
    assert rel(got, oracle.dft1d_r2c(x)) < TOL_FFT
    rc, back = ifft1d(want32)
    assert rc == F.Success
    _, back32 = oracle.fbifft1d(want32)
    assert rel(back, back32) < TOL_FFT
    assert rel(back, N * x.astype(np.float64)) < TOL_FFT


def test_config0_full(oracle):
    """4096 rows of 32 points, U[-1,1], seed 0, whole tensor."""
    x = synth.uniform((4096, 32), seed=0).numpy()
    rc, got = fft1d(x)
    assert rc == F.Success and got.shape == (4096, 17, 2)
    _, want = oracle.fbfft1d(x)
    check("configs[0] fbfft1D vs transcription (4096 rows)", got, want, TOL_FFT)
    check("configs[0] fbfft1D vs fp64 DFT", got, oracle.dft1d_r2c(x), TOL_FFT)
    rc, back = ifft1d(got)
    check("configs[0] round trip", back, 32 * x.astype(np.float64), TOL_FFT)


@pytest.mark.parametrize("N", [4, 16, 32, 128])
def test_padl_quirk(oracle, N):
    """padL shifts right and drops the tail on load; the inverse writes the first
    row of each pair un-shifted and the second shifted (fbfft/FBFFTCommon.cuh:325, :425-427)."""
    padL, B = 3 if N > 4 else 1, 5
    x = synth.uniform((B, N), seed=11).numpy()
    rc, got = fft1d(x, padL)
    _, want = oracle.fbfft1d(x, padL)
    assert rc == F.Success and rel(got, want) < TOL_FFT
    rc, back = ifft1d(want, padL, fill=777.0)
    _, back32 = oracle.fbifft1d(want, padL, out=np.full((B, N), 777.0, np.float32))
    assert rc == F.Success
    assert np.array_equal(back == 777.0, back32 == 777.0)
    assert rel(back, back32) < TOL_FFT


def test_strided_and_errors(oracle):
    d = dev()
    N, B = 64, 9
    x = synth.uniform((B, N), seed=3).numpy()
    big = torch.zeros((B, 2 * N + 2), device=d)
    real = big[:, 1:2 * N + 1:2]                       # x stride 2, odd offset
    real.copy_(torch.from_numpy(x))
    wide = torch.full((B, N, 2), float("nan"), device=d)
    spec = wide[:, :N // 2 + 1, :]                     # padded batch stride
    assert F.fbfft1D(real, spec) == F.Success
    torch.cuda.synchronize()
    _, want = oracle.fbfft1d(x)
    assert rel(spec.cpu().numpy(), want) < TOL_FFT
    assert F.fbifft1D(real, spec) == F.Success
    torch.cuda.synchronize()
    assert rel(real.cpu().numpy(), N * x.astype(np.float64)) < TOL_FFT
    assert float(big[:, 0::2].abs().max()) == 0.0
    # unsupported sizes and shapes
    for n in (3, 6, 512):
        assert F.fbfft1D(torch.zeros((2, n), device=d), torch.zeros((2, n // 2 + 1, 2), device=d)) == F.UnsupportedSize
    assert F.fbfft1D(torch.zeros((2, 32), device=d), torch.zeros((2, 16, 2), device=d)) == F.UnsupportedDimension
    assert F.fbfft1D(torch.zeros((2, 32), device=d), torch.zeros((3, 17, 2), device=d)) == F.UnsupportedDimension
    assert F.fbfft1D(torch.zeros((0, 32), device=d), torch.zeros((0, 17, 2), device=d)) == F.Success
    torch.cuda.synchronize()


@pytest.mark.parametrize("N,B", [(32, 1 << 21), (64, (1 << 20) + 77), (128, (1 << 19) + 5), (256, 1 << 18)])
def test_large_batch_roundtrip(N, B):
    d = dev()
    x = synth.uniform((B, N), seed=2, device=d)
    spec = torch.empty((B, N // 2 + 1, 2), device=d)
    back = torch.empty_like(x)
    assert F.fbfft1D(x, spec) == F.Success
    assert F.fbifft1D(back, spec) == F.Success
    torch.cuda.synchronize()
    assert float((back / N - x).double().norm() / x.double().norm()) < TOL_FFT


@pytest.mark.parametrize("seed", range(30))
def test_random_batches_pads_and_views(oracle, seed):
    """Seeded random draw over size, batch (odd tails), padL and memory layout of
    both operands; forward against the transcription and the fp64 DFT of the
    shifted row, inverse against the transcription (sentinel where it writes nothing)."""
    rng = np.random.default_rng(2000 + seed)
    N = int(rng.choice(SIZES))
    B = int(rng.integers(1, 600))
    padL = int(rng.integers(0, N // 2 + 1)) if rng.random() < 0.4 else 0
    x = synth.uniform((B, N), seed=seed).numpy()
    d = dev()
    kind = int(rng.integers(0, 3))
    if kind == 0:
        real = torch.from_numpy(x).to(d)
    elif kind == 1:                                    # padded batch stride
        big = torch.zeros((B, N + 6), device=d)
        real = big[:, 4:N + 4]
        real.copy_(torch.from_numpy(x))
    else:                                              # rows along the slow axis
        real = torch.from_numpy(np.ascontiguousarray(x.T)).to(d).t()
    if rng.random() < 0.5:
        spec = torch.full((B, N // 2 + 1, 2), float("nan"), device=d)
    else:
        wide = torch.full((B, N // 2 + 3, 2), float("nan"), device=d)
        spec = wide[:, 1:N // 2 + 2, :]
    assert F.fbfft1D(real, spec, padL) == F.Success
    torch.cuda.synchronize()
    _, want = oracle.fbfft1d(x, padL)
    got = spec.cpu().numpy()
    assert rel(got, want) < TOL_FFT, (N, B, padL, kind)
    shifted = np.zeros_like(x)
    shifted[:, padL:] = x[:, :N - padL]
    assert rel(got, oracle.dft1d_r2c(shifted)) < TOL_FFT
    back = torch.full_like(real, 777.0)
    assert F.fbifft1D(back, spec, padL) == F.Success
    torch.cuda.synchronize()
    _, back32 = oracle.fbifft1d(want, padL, out=np.full((B, N), 777.0, np.float32))
    bh = back.cpu().numpy()
    assert np.array_equal(bh == 777.0, back32 == 777.0), (N, B, padL, kind)
    assert rel(bh, back32) < TOL_FFT, (N, B, padL, kind)


# rows of 256 points: whole and partly filled waves (8 rows) and workgroups (32), odd counts, whose last
# spectrum ends between two 16-byte words
@pytest.mark.parametrize("B", [1, 7, 8, 9, 24, 31, 32, 33, 4099])
def test_rows_of_256(oracle, B):
    x = synth.normal((B, 256), seed=B).numpy()
    d = dev()
    spec = torch.full((B + 1, 129, 2), 7.0, device=d)
    back = torch.full((B + 1, 256), 7.0, device=d)
    assert F.fbfft1D(torch.from_numpy(x).to(d), spec[:B]) == F.Success
    assert F.fbifft1D(back[:B], spec[:B]) == F.Success
    torch.cuda.synchronize()
    assert bool((spec[B] == 7.0).all()) and bool((back[B] == 7.0).all())
    # 128 = 16 x 8 points, a root and the fix-up: ten roundings of at most 2^-24 of a value that grows with
    # the square root of its terms, each the 2-norm of two parts
    bar = np.sqrt(2 * 10) * 2.0 ** -24
    assert rel(spec[:B].cpu().numpy(), oracle.dft1d_r2c(x)) < bar
    assert rel(back[:B].cpu().numpy(), 256 * x.astype(np.float64)) < 2 * bar


def test_inverse_of_256_ignores_imaginary_ends(oracle):
    """The imaginary parts of the first and last bin reach no real result, whatever they hold."""
    spec = oracle.dft1d_r2c(synth.normal((5, 256), seed=3).numpy()).astype(np.float32)
    rc, clean = ifft1d(spec)
    spec[:, [0, 128], 1] = np.nan
    rc2, got = ifft1d(spec)
    assert rc == rc2 == F.Success and np.array_equal(got, clean)


# ends of the workgroups of 64 rows (up to 64 points; 256 forward between one and 1.8 rounds of waves) and of 64 and 128
# (128 points, either side of the switch)
@pytest.mark.parametrize("N,B", [(8, 63), (8, 65), (16, 64), (16, 129), (32, 127), (32, 4097), (64, 1), (64, 191),
                                 (128, 63), (128, 65), (128, 32768), (128, 32769), (128, 32897),
                                 (64, 147456), (64, 147457), (64, 200003), (64, 265408), (64, 265409)])
def test_ends_of_workgroups(oracle, N, B):
    x = synth.normal((B, N), seed=N + B)
    d = dev()
    spec = torch.full((B + 1, N // 2 + 1, 2), 7.0, device=d)
    back = torch.full((B + 1, N), 7.0, device=d)
    xd = x.to(d)
    assert F.fbfft1D(xd, spec[:B]) == F.Success
    assert F.fbifft1D(back[:B], spec[:B]) == F.Success
    torch.cuda.synchronize()
    assert bool((spec[B] == 7.0).all()) and bool((back[B] == 7.0).all())
    at = np.unique(np.r_[0:min(B, 70), max(0, B - 200):B])
    # log2(N) + 2 roundings of at most 2^-24 in both parts of values that grow like the root of their terms
    bar = np.sqrt(2 * (np.log2(N) + 2)) * 2.0 ** -24
    assert rel(spec[:B].cpu().numpy()[at], oracle.dft1d_r2c(x.numpy()[at])) < bar
    assert rel(back[:B].cpu().numpy(), N * x.numpy().astype(np.float64)) < 2 * bar


@pytest.mark.parametrize("N", [8, 32, 64, 128, 256])
def test_ends_of_spectra_near_and_beyond_the_largest_float(N):
    """F[0] and F[N/2] are real and overflow only where their own sum does; and backwards a finite pair of them
    gives finite samples, an infinite one infinities of its signs."""
    inf, nan = float("inf"), float("nan")
    d = dev()
    x = torch.zeros(5, N)
    x[0, 0], x[0, 1] = 2e38, -1e38
    x[1, 3], x[2, 4], x[3, 2] = inf, -inf, nan
    x[4, N // 2], x[4, N // 2 + 1] = -3e38, 3e38
    spec = torch.full((5, N // 2 + 1, 2), 7.0, device=d)
    assert F.fbfft1D(x.to(d), spec) == F.Success
    back = torch.zeros(5, N // 2 + 1, 2)
    back[0, 0, 0], back[0, -1, 0] = inf, 1.0
    back[1, 0, 0], back[1, -1, 0] = 1.0, inf
    back[2, 0, 0], back[2, -1, 0] = 1.5e38, 1e38
    back[3, 0, 0], back[3, -1, 0] = -2e38, -1e38
    back[4, 0, 0], back[4, -1, 0] = 2.0, -inf
    y = torch.full((5, N), 7.0, device=d)
    assert F.fbifft1D(y, back.to(d)) == F.Success
    torch.cuda.synchronize()
    ends = spec[:, [0, N // 2]].cpu()
    assert bool((ends[..., 1] == 0.0).all())
    want = torch.tensor([x[0, :2].tolist(), x[4, N // 2:N // 2 + 2].tolist()])
    assert torch.equal(ends[[0, 4], 0, 0], want.sum(1)) and bool(torch.isinf(ends[4, 1, 0]))
    assert torch.equal(ends[0, 1, 0], want[0, 0] - want[0, 1])
    even = 1.0 - 2.0 * (torch.arange(N) % 2)
    assert torch.equal(y.cpu(), torch.stack([torch.full((N,), inf), inf * even, 1.5e38 + 1e38 * even, -2e38 - 1e38 * even,
                                             -inf * even]))
