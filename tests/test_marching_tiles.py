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


@pytest.mark.gpu
@pytest.mark.parametrize("weps", [1.0e-17, 1.0e-20, 1.0e-30])
@pytest.mark.parametrize("field", ["steps", "decades", "signed zeros", "huge"])
def test_gpu_weno_words_over_the_whole_range(device, field, weps):
    """The short evaluation and the statement it stands for: smooth and broken stencils, words over twenty
    decades, exact cancellation, zeros of either sign, smoothness above and weps below the short form's range."""
    import numpy as np
    import torch

    from gm1_amd.advection5 import launch_cuda_scalar_advection5
    from helpers import F, assert_bits_equal, shapes, to_dev, to_host
    from oracle import advection5 as oa

    print("weno words", field, weps, flush=True)
    ni, nj, nk = 70, 21, 16
    rng = np.random.default_rng(len(field))
    a, m, _ = scalar_tests._random_case(rng, ni, nj, nk)
    sh = shapes(ni, nj, nk)
    for k in ("rru", "rrv", "rrw"):
        a[k] = rng.standard_normal(a[k].shape).astype(F)
    x = rng.standard_normal(sh["s"])
    if field == "steps":
        s = 300.0 + np.round(2.0 * x) + 1e-6 * x
    elif field == "decades":
        s = x * 10.0 ** rng.uniform(-18.0, 4.0, x.shape)
    elif field == "signed zeros":
        s = np.where(rng.random(x.shape) < 0.8, np.copysign(0.0, x), 1e-3 * x)
    else:
        s = x * 10.0 ** rng.uniform(2.0, 12.0, x.shape)
    s = s.astype(F)
    divx = (rng.standard_normal((nk, nj, ni)) * 1e-3).astype(F)
    want = np.zeros((nk, nj, ni), F)
    fl = {"x": np.zeros(sh["u"], F), "y": np.zeros(sh["v"], F), "z": np.zeros(sh["w"], F)}
    dfl = to_dev(fl, device)
    kw = dict(ni=ni, nj=nj, nk=nk, nrk=3, dx=250.0, dy=200.0, dz=150.0, weps=weps, lateral_sides=(1, 1, 1, 1))
    oa.cpu_scalar_advection5_inplace(s, a, m, divx, want, fl, **kw)
    got = torch.zeros((nk, nj, ni), dtype=torch.float32, device=device)
    launch_cuda_scalar_advection5(to_dev(s, device), to_dev(a, device), to_dev(m, device), to_dev(divx, device), got,
                                  dfl, **kw)
    torch.cuda.synchronize()
    # the top and bottom faces' limiter takes max(0, x) of zeros of either sign, whose sign IEEE 754 leaves open:
    # with signed zeros the words compared are those of the faces that WENO alone forms
    zeros = field == "signed zeros"
    faces = {"x": slice(None), "y": slice(None), "z": slice(4, nk - 1) if zeros else slice(None)}
    for d in "xyz":
        assert_bits_equal(to_host(dfl[d])[faces[d]], fl[d][faces[d]], f"flux {d}")
    if not zeros:
        assert_bits_equal(to_host(got), want, "tendency")


@pytest.mark.gpu
@pytest.mark.parametrize("field,weps", [("infinities", 1.0e-17), ("infinities", 1.0e-6), ("steps", 1.0e30),
                                        ("steps", 1.0e31), ("steps", 1.0e51), ("steps", 1.0e60), ("steps", 1.0e300)])
def test_gpu_weno_words_at_infinities_and_huge_weps(device, field, weps):
    """An infinite word beside one above 2^126 has a NaN smoothness, which the statement's min() drops: the word is
    then infinite, not NaN.  A weps whose sixth power is no binary64 number leaves the linear weights."""
    import numpy as np
    import torch

    from gm1_amd.advection5 import launch_cuda_scalar_advection5
    from helpers import F, assert_bits_equal, shapes, to_dev, to_host
    from oracle import advection5 as oa

    print("weno words", field, weps, flush=True)
    ni, nj, nk = 70, 21, 16
    rng = np.random.default_rng(5)
    a, m, _ = scalar_tests._random_case(rng, ni, nj, nk)
    sh = shapes(ni, nj, nk)
    for k in ("rru", "rrv", "rrw"):
        a[k] = rng.standard_normal(a[k].shape).astype(F)
    if field == "steps":
        x = rng.standard_normal(sh["s"])
        s = (300.0 + np.round(2.0 * x) + 1e-6 * x).astype(F)
    else:
        s = rng.choice(np.array([0.0, 1.0, -1.0, 2.0, 1.2e38, -1.2e38, 3e38, -3e38, np.inf, -np.inf], F), sh["s"])
    divx = (rng.standard_normal((nk, nj, ni)) * 1e-3).astype(F)
    want = np.zeros((nk, nj, ni), F)
    fl = {"x": np.zeros(sh["u"], F), "y": np.zeros(sh["v"], F), "z": np.zeros(sh["w"], F)}
    dfl = to_dev(fl, device)
    kw = dict(ni=ni, nj=nj, nk=nk, nrk=3, dx=250.0, dy=200.0, dz=150.0, weps=weps, lateral_sides=(1, 1, 1, 1))
    with np.errstate(all="ignore"):
        oa.cpu_scalar_advection5_inplace(s, a, m, divx, want, fl, **kw)
    got = torch.zeros((nk, nj, ni), dtype=torch.float32, device=device)
    launch_cuda_scalar_advection5(to_dev(s, device), to_dev(a, device), to_dev(m, device), to_dev(divx, device), got,
                                  dfl, **kw)
    torch.cuda.synchronize()
    # (a NaN's payload is the machine's; the z faces compared are those that WENO alone forms, as above)
    one_nan = lambda v: np.where(np.isnan(v), F(np.nan), v)  # noqa: E731
    faces = {"x": slice(None), "y": slice(None), "z": slice(4, nk - 1) if field == "infinities" else slice(None)}
    for d in "xyz":
        assert_bits_equal(one_nan(to_host(dfl[d])[faces[d]]), one_nan(fl[d][faces[d]]), f"flux {d}")
    if field == "steps":
        assert np.isfinite(want).all()
        assert_bits_equal(to_host(got), want, "tendency")
    else:
        assert np.isinf(fl["x"]).sum() > 100
