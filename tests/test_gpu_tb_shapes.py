"""The blocked step over every region shape its launch rule can pick: lattices smaller
than a tile, one column or row past a tile edge, chunks of one plane and ragged last
chunks, in the three storage forms, bit for bit against the oracle; and the ensemble's
28 x 36 regions against single-lattice runs."""
import numpy as np
import pytest
import torch

from test_gpu_parity import assert_bitwise, dev, host, rand_state

pytestmark = pytest.mark.gpu

FRW = dict(a1=1.0, H1=0.5, t1=1.0)

# (N, chunk): below the smallest tile; 8 x 16 and 10 x 32 tiles with a remainder; chunks of
# 1, 3 and 5 planes; sizes at which 24 x 32, 26 x 64 / 18 x 64 and 11 x 128 tiles are picked
CASES = [(10, 1), (18, 0), (34, 3), (66, 5), (98, 0), (130, 0), (200, 67), (260, 0), (384, 0)]


@pytest.mark.parametrize("mode", ["f64", "f32c", "f32s"])
@pytest.mark.parametrize("N,chunk", CASES)
def test_step_bitwise_oracle(cfl, O, N, chunk, mode):
    print(f"case tb shapes {mode} N={N} chunk={chunk}", flush=True)
    lam, L, t = (0.1 if N % 4 else 0.0), 1.25 * N, 1.15
    eq = O.Equation(N, L, 1.0, lam, O.Cosmo.radiation(**FRW))
    p = cfl.kg_params(N, L, 1.0, lam, cfl.radiation(**FRW))
    x = rand_state(N, 31, amp=0.5)
    if mode == "f64":
        out = torch.full((2 * N ** 3,), float("nan"), dtype=torch.float64, device="cuda")
        cfl.rk4_step_tb_f64(p, dev(x), out, t, 0.05, chunk=chunk)
        eq.rk4_step(x, t, 0.05)
        assert_bitwise(host(out), x, "state")
        return
    hi = x.astype(np.float32)
    lo = (x - hi.astype(np.float64)).astype(np.float32)
    ho = torch.full((2 * N ** 3,), float("nan"), dtype=torch.float32, device="cuda")
    lw = torch.full_like(ho, float("nan"))
    step = cfl.rk4_step_tb_f32c if mode == "f32c" else cfl.rk4_step_tb_f32s
    step(p, dev(hi.copy()), dev(lo.copy()), ho, lw, t, 0.05, chunk=chunk)
    (eq.rk4_step_f32c if mode == "f32c" else eq.rk4_step_f32s)(hi, lo, t, 0.05)
    assert_bitwise(host(ho), hi, "hi")
    assert_bitwise(host(lw), lo, "lo")


@pytest.mark.parametrize("prec,grid", [(0, 0), (0, -1), (1, -1), (2, 0), (2, -1)])
def test_ensemble_28x36_keeps_bits(cfl, prec, grid):
    print(f"case ensemble 28x36 prec={prec} grid={grid}", flush=True)
    Ns = [16, 34, 48, 34]
    ens = cfl.Ensemble(Ns, [float(n) for n in Ns], 1.0, 0.1, cfl.radiation(**FRW), prec)
    ens.init_grf([1, 2, 3, 4], cfl.CF_SPEC_GAUSS, (0.25,), 1.0)
    start = [ens.state(r) for r in range(len(Ns))]
    for n in (16, 34, 48):
        ens.set_region(n, cfl.CF_ENS_REGION_28X36)
        assert ens.get_region(n) == cfl.CF_ENS_REGION_28X36
    ens.set_plan(34, 13, 5 if grid == 0 else grid)
    ens.run(1.0, 0, 3, 0.05)
    for r, n in enumerate(Ns):
        p = cfl.kg_params(n, float(n), 1.0, 0.1, cfl.radiation(**FRW))
        if prec == 0:
            x = start[r].clone()
            cfl.rk4_run_tb_f64(p, x, 1.0, 0, 3, 0.05, cfl.alloc_tb_work(n))
        else:
            hi, lo = cfl.split_f64(start[r])
            run = cfl.rk4_run_tb_f32c if prec == 1 else cfl.rk4_run_tb_f32s
            run(p, hi, lo, 1.0, 0, 3, 0.05, cfl.alloc_tb_work(n, prec))
            x = cfl.join_f64(hi, lo)
        torch.cuda.synchronize()
        assert torch.equal(ens.state(r), x), f"realisation {r}"


@pytest.mark.parametrize("N", [18, 98])
def test_odd_alignment(cfl, N):
    """States that start on an odd double / float (the step moves two columns a lane)."""
    print(f"case tb odd alignment N={N}", flush=True)
    n = 2 * N ** 3
    p = cfl.kg_params(N, float(N), 1.0, 0.1, cfl.radiation(**FRW))
    x = dev(rand_state(N, 33, amp=0.5))
    a = torch.empty(n + 1, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    a[1:] = x
    ref = torch.empty_like(x)
    cfl.rk4_step_tb_f64(p, x, ref, 1.0, 0.05)
    cfl.rk4_step_tb_f64(p, a[1:], b[1:], 1.0, 0.05)
    assert torch.equal(b[1:], ref)
    hi, lo = cfl.split_f64(x)
    h2, l2 = torch.empty_like(hi), torch.empty_like(lo)
    bufs = [torch.empty(n + 1, dtype=torch.float32, device="cuda") for _ in range(4)]
    bufs[0][1:], bufs[1][1:] = hi, lo
    for step in (cfl.rk4_step_tb_f32s, cfl.rk4_step_tb_f32c):
        step(p, hi, lo, h2, l2, 1.0, 0.05)
        step(p, *[t[1:] for t in bufs], 1.0, 0.05)
        assert torch.equal(bufs[2][1:], h2) and torch.equal(bufs[3][1:], l2)


@pytest.mark.parametrize("kind,N,chunk", [(1, 66, 3), (1, 130, 0), (1, 260, 0), (2, 130, 0), (2, 302, 0), (3, 98, 0)])
def test_variant_step_equals_stage_kernels(cfl, O, kind, N, chunk):
    """The variants' region shapes (10 x 32, 24 x 32, 18 x 64 tiles with remainders): two
    blocked steps give the bits of the stage kernels, from a state on an odd double too."""
    print(f"case tb shapes variant {kind} N={N} chunk={chunk}", flush=True)
    p = cfl.kg_params(N, float(N), 1.0, 0.0, cfl.radiation(**FRW))
    if kind == 3:
        g = torch.Generator(device="cuda").manual_seed(5)
        field = 1e-2 * torch.randn(2 * N * N * (N // 2 + 1), dtype=torch.float64, device="cuda", generator=g)
    else:
        field = dev(0.02 * rand_state(N, 34)[: N ** 3]) if kind == 1 else None
    v = cfl.Variant(p, kind, field, f_a=1.3)
    x = dev(rand_state(N, 35, amp=0.3))
    ref = x.clone()
    v.rk4_run(ref, 1.0, 0, 2, 0.05)
    odd = torch.empty(2 * N ** 3 + 1, dtype=torch.float64, device="cuda")
    odd[1:] = x
    y, z = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    v.rk4_step_tb(odd[1:], y, 1.0, 0.05, chunk=chunk)
    v.rk4_step_tb(y, z, 1.05, 0.05, chunk=chunk)
    assert torch.equal(z, ref)
    v.close()


@pytest.mark.parametrize("prec,grid", [(0, -1), (1, -1), (2, 5), (2, -1)])
def test_ensemble_15x68_keeps_bits(cfl, prec, grid):
    """11 x 64 tiles: a lattice inside one tile, one of 64 columns, one just past a tile."""
    print(f"case ensemble 15x68 prec={prec} grid={grid}", flush=True)
    Ns = [10, 64, 66]
    ens = cfl.Ensemble(Ns, [float(n) for n in Ns], 1.0, 0.1, cfl.radiation(**FRW), prec)
    ens.init_grf([1, 2, 3], cfl.CF_SPEC_GAUSS, (0.25,), 1.0)
    start = [ens.state(r) for r in range(len(Ns))]
    for n in Ns:
        ens.set_region(n, cfl.CF_ENS_REGION_15X68)
        assert ens.get_region(n) == cfl.CF_ENS_REGION_15X68
    ens.set_plan(66, 13, grid)
    ens.run(1.0, 0, 3, 0.05)
    for r, n in enumerate(Ns):
        p = cfl.kg_params(n, float(n), 1.0, 0.1, cfl.radiation(**FRW))
        if prec == 0:
            x = start[r].clone()
            cfl.rk4_run_tb_f64(p, x, 1.0, 0, 3, 0.05, cfl.alloc_tb_work(n))
        else:
            hi, lo = cfl.split_f64(start[r])
            run = cfl.rk4_run_tb_f32c if prec == 1 else cfl.rk4_run_tb_f32s
            run(p, hi, lo, 1.0, 0, 3, 0.05, cfl.alloc_tb_work(n, prec))
            x = cfl.join_f64(hi, lo)
        torch.cuda.synchronize()
        assert torch.equal(ens.state(r), x), f"realisation {r}"
