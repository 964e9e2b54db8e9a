"""The library's own transform passes at sizes that reach every radix (2 .. 8), stage
count, odd half length and ragged column tile, against numpy in double precision, and a
size with a large prime factor (hipFFT). The bound is the normwise one of an FFT of n
points with correctly rounded roots, 5 u log2 n, u = 2^-53, doubled for the two passes of
the real transform and numpy's own error."""
import math

import numpy as np
import pytest
import torch

from test_gpu_parity import dev, host

pytestmark = pytest.mark.gpu

SIZES = [4, 6, 8, 10, 14, 18, 28, 30, 42, 48, 50, 54, 64, 98, 100, 126, 160]


def bound(N):
    return 2 * 5 * 2.0 ** -53 * math.log2(N ** 3)


@pytest.mark.parametrize("N", SIZES + [22])
def test_transforms_match_numpy(cfl, N):
    print(f"case fft N={N}", flush=True)
    rng = np.random.default_rng(N)
    f = rng.standard_normal((N, N, N))
    plan = cfl.SpectrumPlan(N)
    fd = dev(f.reshape(-1))
    k = plan.d2z(fd)
    assert torch.equal(fd, dev(f.reshape(-1))), "the transform changed its input"
    got = host(k).view(np.complex128).reshape(N, N, N // 2 + 1)
    want = np.fft.rfftn(f)
    assert np.linalg.norm(got - want) <= bound(N) * np.linalg.norm(want)
    g = want + 1j * rng.standard_normal(want.shape) * 1e-3  # not the transform of a real field: rows still are
    back = host(plan.z2d(dev(np.ascontiguousarray(want).view(np.float64).reshape(-1))))
    assert np.linalg.norm(back.reshape(N, N, N) - f * N ** 3) <= bound(N) * np.linalg.norm(f) * N ** 3
    one = host(plan.z2d(dev(np.ascontiguousarray(g).view(np.float64).reshape(-1)))).reshape(N, N, N)
    ref = np.fft.irfft(np.fft.ifft2(g, axes=(0, 1), norm="forward"), n=N, axis=2, norm="forward")
    assert np.linalg.norm(one - ref) <= bound(N) * np.linalg.norm(ref)


def s_index(N):
    i = np.minimum(np.arange(N), N - np.arange(N)) ** 2
    return i[:, None, None] + i[None, :, None] + i[None, None, : N // 2 + 1]


@pytest.mark.parametrize("N", SIZES + [22])
def test_spectra_and_scaled_modes(cfl, N):
    """Folded-power spectra against the full definition per bin, and the scaled inverse."""
    print(f"case spectra N={N}", flush=True)
    rng = np.random.default_rng(100 + N)
    x = rng.standard_normal(2 * N ** 3)
    plan = cfl.SpectrumPlan(N)
    xd = dev(x)
    L, m, a = 1.5 * N, 1.1, 1.7
    fk = [np.abs(np.fft.rfftn(x[q * N ** 3:(q + 1) * N ** 3].reshape(N, N, N))) ** 2 for q in range(2)]
    w = np.full(N // 2 + 1, 2.0)
    w[0] = w[-1] = 1.0
    s = s_index(N)
    nb = cfl.nbins(N)
    power = np.bincount(s.reshape(-1), (fk[0] * w).reshape(-1), nb)
    om = m * m + (2 * np.pi / L) ** 2 * s / (a * a)
    mode = np.bincount(s.reshape(-1), ((fk[0] + fk[1] / om) * w).reshape(-1), nb)
    for got, want in ((host(plan.power_spectrum(xd[: N ** 3])), power),
                      (host(plan.mode_power_spectrum(xd, L, m, a)), mode)):
        assert np.all(np.abs(got - want) <= 1e-10 * want + 1e-18 * want.max())
        assert np.all(got[want == 0] == 0)
    assert torch.equal(xd, dev(x))
    kern = rng.uniform(0.5, 1.5, nb)
    out = host(plan.scaled_fourier_modes(xd[: N ** 3], dev(kern))).reshape(N, N, N)
    ref = np.fft.irfftn(np.fft.rfftn(x[: N ** 3].reshape(N, N, N)) * kern[s], s=(N, N, N), axes=(0, 1, 2))
    assert np.linalg.norm(out - ref) <= 2 * bound(N) * np.linalg.norm(ref)


def test_odd_alignment(cfl):
    """Fields and spectra that start on an odd double (the passes move 16 bytes a lane)."""
    N = 18
    x = np.random.default_rng(5).standard_normal(N ** 3)
    plan = cfl.SpectrumPlan(N)
    base = torch.zeros(N ** 3 + 1, dtype=torch.float64, device="cuda")
    base[1:] = dev(x)
    kbuf = torch.zeros(2 * N * N * (N // 2 + 1) + 1, dtype=torch.float64, device="cuda")
    back = torch.zeros(N ** 3 + 1, dtype=torch.float64, device="cuda")
    plan.d2z(base[1:], out=kbuf[1:])
    assert torch.equal(kbuf[1:], plan.d2z(dev(x)))
    ref = plan.z2d(kbuf[1:].clone())
    plan.z2d(kbuf[1:], out=back[1:])
    assert torch.equal(back[1:], ref)
