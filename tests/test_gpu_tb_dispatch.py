"""The blocked step where its launch rule leaves the ordinary: large regions with the quartic
term and a ragged last tile, paced launches of the widest region. Bit for bit against the
oracle; tests/test_tb_geometry.py checks which region shapes these sizes reach."""
import numpy as np
import pytest
import torch

from test_gpu_parity import assert_bitwise, dev, host, rand_state

pytestmark = pytest.mark.gpu

FRW = dict(a1=1.0, H1=0.5, t1=1.0)


def check_step(cfl, O, N, chunk, mode, lam):
    """One step into poisoned buffers against the oracle's."""
    L, t = 1.25 * N, 1.15
    eq = O.Equation(N, L, 1.0, lam, O.Cosmo.radiation(**FRW))
    p = cfl.kg_params(N, L, 1.0, lam, cfl.radiation(**FRW))
    x = rand_state(N, 41, amp=0.5)
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


@pytest.mark.parametrize("mode", ["f64", "f32c", "f32s"])
@pytest.mark.parametrize("N,chunk", [(126, 0), (250, 0), (250, 21), (254, 0)])
def test_ragged_large_regions_with_lambda(cfl, O, N, chunk, mode):
    print(f"case tb dispatch {mode} N={N} chunk={chunk}", flush=True)
    check_step(cfl, O, N, chunk, mode, 0.1)


@pytest.mark.parametrize("lam", [0.0, 0.1])
def test_paced_widest_region(cfl, O, lam):
    """15 x 132 regions with a ragged last tile, held to 3 us a plane."""
    N = 126
    print(f"case tb dispatch paced lam={lam}", flush=True)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or \
        cfl.rk4_tb_geometry(N, cfl.CF_PREC_F32S)[:2] == (15, 132)
    cfl.rk4_tb_set_pace(N, 300)
    try:
        check_step(cfl, O, N, 0, "f32s", lam)
    finally:
        cfl.rk4_tb_set_pace(N, 0)


@pytest.mark.parametrize("mode", ["f64", "f32s"])
@pytest.mark.parametrize("lam", [0.0, 0.1])
def test_shorter_tiles(cfl, O, mode, lam):
    """Tiles of fewer rows than the region holds (a given chunk that would leave units idle)."""
    N, chunk = 202, 101
    print(f"case tb dispatch shorter tiles {mode} lam={lam}", flush=True)
    rb, _, tb, *_ = cfl.rk4_tb_geometry(N, cfl.CF_PREC_F64 if mode == "f64" else cfl.CF_PREC_F32S, chunk)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or tb < rb - 4
    check_step(cfl, O, N, chunk, mode, lam)
