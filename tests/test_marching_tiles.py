"""The marching tile kernels word for word where their tiles and level chunks end: planes a tile
wide, one more and one less, the fewest levels, single-level chunks and chunks with a remainder."""

from __future__ import annotations

import pytest
import test_advection5 as scalar_tests
import test_momentum5 as momentum_tests

DIMS = [(64, 8, 8), (65, 9, 9), (63, 8, 83), (129, 17, 8), (140, 100, 37)]
SIDES = [(2, 2, 2, 2), (1, 1, 1, 1), (2, 4, 1, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("nrk", [1, 3])
@pytest.mark.parametrize("sides", SIDES + [None])
@pytest.mark.parametrize("dims", DIMS)
def test_gpu_scalar_tiles(device, nrk, sides, dims):
    print("scalar tiles", dims, sides, nrk, flush=True)
    scalar_tests.test_gpu_scalar_advection_bit_exact(device, nrk, sides, dims)


@pytest.mark.gpu
@pytest.mark.parametrize("sides", SIDES)
@pytest.mark.parametrize("dims", DIMS)
def test_gpu_momentum_tiles(device, sides, dims):
    print("momentum tiles", dims, sides, flush=True)
    momentum_tests.test_gpu_momentum_advection_bit_exact(device, sides, dims)
