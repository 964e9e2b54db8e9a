"""The library's transform passes at sizes whose plans have four, five and six stages, or
whose lines take more than 64 KB of LDS (N > 448), against torch's transforms in double
precision: forward, inverse, scaled inverse, spectra, and the pair of fields behind Psi.
Bounds as in tests/test_gpu_fft_sizes.py."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
# stages of the passes along a and b (length N) and along c (N / 2)
SIZES = {108: (4, 3), 162: (4, 4), 250: (4, 3), 324: (5, 4), 486: (5, 5), 972: (6, 5), 1024: (4, 3)}


def stages(n):
    """Radices 7, 5, 3 and 8, 4, 2, a two and a three merged where twos are left over."""
    e = {f: 0 for f in (2, 3, 5, 7)}
    for f in e:
        while n % f == 0:
            n //= f
            e[f] += 1
    assert n == 1
    merged = e[2] % 3 == 1 and e[3] > 0
    twos = e[2] - merged
    return e[7] + e[5] + e[3] + -(-twos // 3)


def test_sizes_have_the_stages_they_stand_for():
    assert {n: (stages(n), stages(n // 2)) for n in SIZES} == SIZES


def bound(N):
    return 2 * 5 * U * math.log2(N ** 3)


def gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def s_index(N):
    i = torch.arange(N, device="cuda")
    i = torch.minimum(i, N - i) ** 2
    return i[:, None, None] + i[None, :, None] + i[None, None, : N // 2 + 1]


@pytest.mark.parametrize("N", SIZES)
def test_transforms_and_spectra(cfl, N):
    print(f"case fft stages N={N}", flush=True)
    f = torch.randn((N, N, N), dtype=torch.float64, device="cuda", generator=gen(N))
    plan = cfl.SpectrumPlan(N)
    want = torch.fft.rfftn(f)
    got = torch.view_as_complex(plan.d2z(f.reshape(-1)).view(N, N, N // 2 + 1, 2))
    assert torch.linalg.vector_norm(got - want) <= bound(N) * torch.linalg.vector_norm(want)
    # every line takes part: no plane of the spectrum is worse than the rest
    worst = torch.linalg.vector_norm(got - want, dim=(1, 2)) / torch.linalg.vector_norm(want, dim=(1, 2))
    assert worst.max() <= 2 * bound(N)
    del got
    s = s_index(N)
    w = torch.full((N // 2 + 1,), 2.0, dtype=torch.float64, device="cuda")
    w[0] = w[-1] = 1.0
    power = torch.bincount(s.reshape(-1), (torch.view_as_real(want).square().sum(-1) * w).reshape(-1), cfl.nbins(N))
    bins = plan.power_spectrum(f.reshape(-1))
    assert torch.all((bins - power).abs() <= 1e-10 * power + 1e-18 * power.max())
    back = plan.z2d(torch.view_as_real(want).contiguous().reshape(-1)).view(N, N, N)
    assert torch.linalg.vector_norm(back / N ** 3 - f) <= bound(N) * torch.linalg.vector_norm(f)
    del back
    kern = torch.rand(cfl.nbins(N), dtype=torch.float64, device="cuda", generator=gen(N + 1)) + 0.5
    out = plan.scaled_fourier_modes(f.reshape(-1), kern).view(N, N, N)
    want *= kern[s]
    del s
    ref = torch.fft.irfftn(want, s=(N, N, N))
    assert torch.linalg.vector_norm(out - ref) <= 2 * bound(N) * torch.linalg.vector_norm(ref)
    plan.close()


@pytest.mark.parametrize("N", [4, 6, 14, 64, 126, 128, 140])
def test_small_inverse(cfl, N):
    """Inverses whose passes along b and c share a kernel (N <= 128), from the smallest plane to
    the first lattice past the line; the imaginary parts that a real transform has no use
    for (columns 0 and N/2) are not read."""
    print(f"case fft plane N={N}", flush=True)
    f = torch.randn((N, N, N), dtype=torch.float64, device="cuda", generator=gen(N))
    plan = cfl.SpectrumPlan(N)
    k = torch.fft.fftn(f)[:, :, : N // 2 + 1].contiguous()
    back = plan.z2d(torch.view_as_real(k).clone().reshape(-1)).view(N, N, N)
    assert torch.linalg.vector_norm(back / N ** 3 - f) <= bound(N) * torch.linalg.vector_norm(f)
    # rows that are no half of a real field's spectrum: complex along a and b, then each row
    k = torch.view_as_complex(torch.randn((N, N, N // 2 + 1, 2), dtype=torch.float64, device="cuda", generator=gen(1)))
    rows = torch.fft.ifft2(k, dim=(0, 1), norm="forward")
    rows[:, :, 0].imag.zero_()
    rows[:, :, -1].imag.zero_()
    want = torch.fft.irfft(rows, n=N, dim=2, norm="forward")
    out = plan.z2d(torch.view_as_real(k).clone().reshape(-1)).view(N, N, N)
    assert torch.linalg.vector_norm(out - want) <= bound(N) * torch.linalg.vector_norm(want)
    plan.close()


@pytest.mark.parametrize("N", [4, 14, 64, 108, 126, 128, 140, 162, 324, 486])
def test_psi_pair(cfl, N):
    """Psi and dPsi/dt of the comoving curvature. The factors' own error: a few roundings of
    |k| eta / sqrt(3) = w and of the sines and cosines, 8 u of every term's size."""
    print(f"case psi stages N={N}", flush=True)
    L, t, cosmo = 0.05 * N, 1.3, cfl.radiation(a1=1.0, H1=0.5, t1=1.0)
    field = torch.randn((N, N, N), dtype=torch.float64, device="cuda", generator=gen(N))
    R = torch.fft.rfftn(field)
    v = cfl.Variant(cfl.kg_params(N, L, 1.0, 0.0, cosmo), cfl.CF_VAR_COMOVING_CURVATURE,
                    torch.view_as_real(R).contiguous().reshape(-1))
    H = cfl.cosmo_H(cosmo, t)
    w = s_index(N).double().sqrt() * (2 * math.pi / L * cfl.cosmo_eta(cosmo, t) / math.sqrt(3.0))
    w[0, 0, 0] = 1.0
    sv, cv, c = torch.sin(w), torch.cos(w), 2 / w ** 3
    factors = ((sv - w * cv) * c, H * (3 * w * cv + (w * w - 3) * sv) * c)
    slack = (8 * U * c * (1 + w + w * w), 8 * U * H * c * (3 + 3 * w + w * w + w ** 3))
    for got, tr, d in zip(v.psi(t), factors, slack):
        tr[0, 0, 0] = d[0, 0, 0] = 0.0
        want = torch.fft.irfftn(R * tr, s=(N, N, N))
        tol = 2 * bound(N) * torch.linalg.vector_norm(want) + \
            math.sqrt(2.0) * torch.linalg.vector_norm(R.abs() * d) / N ** 1.5
        assert torch.linalg.vector_norm(got.view(N, N, N) - want) <= tol
    v.close()
