"""What the blocked step's launches run over (cf_rk4_tb_geometry): the query's contract, and
that the sizes which the GPU tests compare with the oracle reach every region shape in every
storage form. Without a GPU the library plans for 256 compute units."""
import ctypes as C

import pytest
import torch

import cfl_amd as cfl
from cfl_amd import _lib as lib

SHAPES = {cfl.CF_PREC_F64: {(12, 20), (14, 36), (28, 36), (30, 68)},
          cfl.CF_PREC_F32C: {(14, 36), (28, 36), (22, 68)},
          cfl.CF_PREC_F32S: {(12, 20), (14, 36), (28, 36), (30, 68), (15, 132)}}


def plans_for_256():
    return not torch.cuda.is_available() or torch.cuda.get_device_properties(0).multi_processor_count == 256


def test_query_arguments():
    g = (C.c_int * 6)()
    assert lib.load().cf_rk4_tb_geometry(15, 0, 0, g) == lib.CF_E_INVALID
    assert lib.load().cf_rk4_tb_geometry(16, 3, 0, g) == lib.CF_E_INVALID
    assert lib.load().cf_rk4_tb_geometry(16, 0, 0, None) == lib.CF_E_INVALID


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("N,chunk", [(4, 0), (16, 0), (32, 0), (100, 7), (128, 0), (250, 0), (256, 128), (512, 0),
                                     (1024, 0), (2048, 0)])
def test_geometry_covers_the_lattice(prec, N, chunk):
    rb, rc, tb, tc, A, blocks = cfl.rk4_tb_geometry(N, prec, chunk)
    assert (rb, rc) in SHAPES[prec]
    assert 1 <= tb <= min(N, rb - 4) and tc == min(N, rc - 4) and 1 <= A <= N
    assert chunk == 0 or A == chunk
    assert blocks == -(-N // tb) * -(-N // tc) * -(-N // A)
    threads = {(12, 20): 128, (14, 36): 512 if prec == 1 else 256, (28, 36): 1024 if prec == 1 else 512,
               (30, 68): 1024, (15, 132): 1024, (22, 68): 768}[rb, rc]
    assert blocks * threads < 2 ** 32  # what a launch can hold


# the (N, chunk) that tests/test_gpu_tb_shapes.py and tests/test_gpu_tb_dispatch.py run
BITWISE = [(10, 1), (18, 0), (34, 3), (66, 5), (98, 0), (130, 0), (200, 67), (260, 0), (384, 0)]
RAGGED = [(126, 0), (250, 0), (250, 21), (254, 0)]


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_bitwise_sizes_reach_every_shape(prec):
    if not plans_for_256():
        pytest.skip("the sizes are chosen for 256 compute units")
    lam = {k: set() for k in (False, True)}
    for N, chunk in BITWISE + RAGGED:
        lam[N % 4 != 0].add(cfl.rk4_tb_geometry(N, prec, chunk)[:2])
    assert lam[False] | lam[True] == SHAPES[prec]
    assert lam[True] == SHAPES[prec]  # with the quartic term as well


@pytest.mark.parametrize("prec,least", [(cfl.CF_PREC_F64, 0.7), (cfl.CF_PREC_F32S, 0.9)])
@pytest.mark.parametrize("N,chunk", [(202, 101), (224, 112), (256, 128), (300, 300), (320, 320)])
def test_given_chunk_leaves_few_units_idle(prec, least, N, chunk):
    """A long chunk in a lattice beyond the cache: shorter tiles, not a fraction of the chip."""
    if not plans_for_256():
        pytest.skip("the sizes are chosen for 256 compute units")
    assert least * 256 <= cfl.rk4_tb_geometry(N, prec, chunk)[5] <= 256
