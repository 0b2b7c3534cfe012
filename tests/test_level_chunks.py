"""The marching tile kernels over chunks of many levels, word for word against the oracle.

A chunk carries words from level to level (seven-level windows, two LDS buffers in turn, planes requested a
level ahead, the pdef repair's five candidates), and the small grids of the other tests march one level a
chunk.  These grids march 8 to 11 levels a chunk and a ragged chunk at the top.
"""

from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import test_advection5 as scalar_tests
import test_large_step as terrain_tests
import test_momentum5 as momentum_tests
import test_stretched as flat_tests
from helpers import F, NG, assert_bits_equal, seeded_metrics, shapes, to_dev, to_host
from oracle import boundary as obc
from oracle import large_step as ol
from oracle import momentum5 as omom
from oracle import pdef as op
from oracle import sound as osound
from oracle import stage as ost
from oracle.advection5 import cpu_scalar_advection5_inplace, cpu_terrain_mass_flux5_inplace

NARROW, WIDE = (9, 1241, 31), (70, 621, 31)  # one tile column, and two of which one is ragged
TX, TY = 64, 8


@pytest.mark.parametrize("dims", [NARROW, WIDE])
def test_these_grids_march_many_levels_a_chunk(dims):
    """Every kernel's chunk (two or three workgroups a CU; w marches nk - 1 levels) has at least eight levels, and
    the top one is ragged."""
    from gm1_amd import _native, advection5  # noqa: F401

    ni, nj, nk = dims
    tiles = -(-ni // TX) * -(-nj // TY)
    for levels, per_cu in ((nk, 2), (nk, 3), (nk - 1, 3)):
        chunk = _native.query("gm1hip_tile_chunk_levels", tiles, levels, per_cu)
        assert chunk >= 8 and levels % chunk, (levels, per_cu, chunk)


def _storm(host, seed):
    """Cloud and rain in places, with holes, so that the positive-definite repair acts."""
    rng = np.random.default_rng(seed)
    q = host["arrays"]["q3d"]
    for sp, size in ((1, 1e-3), (2, 2e-3)):
        q[sp] = np.where(rng.random(q[sp].shape) < 0.4, size * rng.random(q[sp].shape), 0.0).astype(F)
    host["arrays"]["qa"][...] = q


@pytest.mark.gpu
@pytest.mark.parametrize("sides", [(2, 2, 2, 2), (1, 1, 1, 1)])
@pytest.mark.parametrize("family", ["flat", "terrain"])
def test_gpu_moist_large_step(device, family, sides):
    """A whole moist step: momentum with its held tendencies and the flat buoyancy, the paired compose, WENO theta'
    and the pdef chain of three species, all from unpadded carriers."""
    import torch

    from gm1_amd.fields import large_stretched_c3
    from gm1_amd.large_step import create_gm1_large_step_state, host_initial_state, launch_cuda_gm1_large_step

    ni, nj, nk = NARROW
    print(f"level chunks: {family} step {ni}x{nj}x{nk} sides {sides}", flush=True)
    if family == "flat":
        cfg = replace(large_stretched_c3(ni, nj, nk), lateral_sides=sides,
                      stretched=(nk * 100.0, 0.0, nk * 100.0, 60.0, 140.0))
    else:
        cfg = terrain_tests.moist_case(ni, nj, nk, sides)
    host = host_initial_state(cfg)
    _storm(host, 3)
    st = create_gm1_large_step_state(host, device)
    a = {k: v.copy() for k, v in host["arrays"].items()}
    launch_cuda_gm1_large_step(st)
    torch.cuda.synchronize()
    corr = float(st.dry_mass.correction.cpu().numpy()[0])
    if family == "flat":
        lv = host["levels"]
        ol.large_step(a, host["metrics"], host["base"], host["prof"], flat_tests.cfg_dict(cfg), zt=F(lv.ztop),
                      mass_correction=corr, flat=lv)
    else:
        ol.large_step(a, host["metrics"], host["base"], osound.terrain_coordinate_profiles(nk, cfg.dz),
                      flat_tests.cfg_dict(cfg), zt=F(nk * cfg.dz), mass_correction=corr)
    for name in terrain_tests.MOIST_FIELDS:
        assert_bits_equal(to_host(st.a[name]), a[name], name)


@pytest.mark.gpu
@pytest.mark.parametrize("nrk", [1, 3])
@pytest.mark.parametrize("sides", [(2, 2, 2, 2), (2, 4, 1, 1), None])
def test_gpu_terrain_scalar_tendency(device, nrk, sides):
    print("level chunks: scalar", WIDE, sides, nrk, flush=True)
    scalar_tests.test_gpu_scalar_advection_bit_exact(device, nrk, sides, WIDE)


@pytest.mark.gpu
@pytest.mark.parametrize("sides", [(2, 2, 2, 2), (1, 1, 2, 3)])
def test_gpu_terrain_momentum(device, sides):
    print("level chunks: momentum", WIDE, sides, flush=True)
    momentum_tests.test_gpu_momentum_advection_bit_exact(device, sides, WIDE)


def _levels(nk):
    from gm1_amd.grid import build_vertical_levels

    return build_vertical_levels(stretch_z=1, nk=nk, dz=100.0, ztop=nk * 100.0, str_bot=0.0, str_top=nk * 100.0,
                                 dz_bot=60.0, dz_top=140.0)


def _column_metrics(rng, ni, nj, nk):
    """Flat metrics, one word a level."""
    m = seeded_metrics(rng, ni, nj, nk, terrain=False)
    return {n: np.ascontiguousarray(np.broadcast_to(v[..., :1, :1], v.shape)) if v.ndim == 3 else v
            for n, v in m.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("sides", [(2, 2, 2, 2), (1, 1, 2, 3)])
def test_gpu_flat_momentum(device, sides):
    import torch

    from gm1_amd.stretched import flat_stretched_column, launch_cuda_gm1_child_stretched_momentum5

    ni, nj, nk = WIDE
    print("level chunks: flat momentum", WIDE, sides, flush=True)
    rng = np.random.default_rng(11)
    a, _ = momentum_tests._case(rng, ni, nj, nk)
    m, lv = _column_metrics(rng, ni, nj, nk), _levels(nk)
    d, dm = to_dev(a, device), to_dev(m, device)
    divx = np.zeros((nk, nj, ni), F)
    ddivx = to_dev(divx, device)
    launch_cuda_gm1_child_stretched_momentum5(d, dm, flat_stretched_column(lv, device), ni=ni, nj=nj, nk=nk, nrk=2,
                                              dx=250.0, dy=200.0, divx=ddivx, lateral_sides=sides)
    torch.cuda.synchronize()
    omom.cpu_terrain_open_momentum_advection5_inplace(a, m, divx, ni=ni, nj=nj, nk=nk, nrk=2, dx=250.0, dy=200.0,
                                                      dz=100.0, lateral_sides=sides, flat=lv)
    for n in ("rru", "rrv", "rrw", "uten", "vten", "wten"):
        assert_bits_equal(to_host(d[n]), a[n], n)
    assert_bits_equal(to_host(ddivx), divx, "divx")


@pytest.mark.gpu
@pytest.mark.parametrize("row", ["theta-nrk1", "theta-nrk3", "qv-pdef", "qc-pdef"])
@pytest.mark.parametrize("family,sides", [("terrain", (3, 4, 2, 2)), ("flat", (2, 2, 1, 1))])
def test_gpu_scalar_stage_from_padded_and_unpadded_carriers(device, family, sides, row):
    """One scalar's stage (compose, or pdef chain and repair) from a padded carrier, from an unpadded one, and as the
    batch's only and first scalar, against the oracle's pack, fill, advection and compose."""
    import torch

    from gm1_amd import scalar_moist_rk as sm
    from gm1_amd import stretched

    ni, nj, nk = WIDE
    print("level chunks: scalar stage", family, WIDE, sides, row, flush=True)
    rng = np.random.default_rng(40 + len(row))
    sh, cell = shapes(ni, nj, nk), (nk, nj, ni)
    flat = _levels(nk) if family == "flat" else None
    m = _column_metrics(rng, ni, nj, nk) if flat else seeded_metrics(rng, ni, nj, nk)
    a = {"u3d": (4 * rng.standard_normal(sh["u"])).astype(F), "v3d": (4 * rng.standard_normal(sh["v"])).astype(F),
         "w3d": (2 * rng.standard_normal(sh["w"])).astype(F), "rru": np.zeros(sh["u"], F),
         "rrv": np.zeros(sh["v"], F), "rrw": np.zeros(sh["w"], F)}
    divx = np.zeros(cell, F)
    dt, dx, dy, dz = 1.5, 250.0, 300.0, 200.0
    if flat:
        omom.mass_flux_and_divergence(a, m, divx, ni=ni, nj=nj, nk=nk, dx=dx, dy=dy, dz=dz, flat=flat)
    else:
        cpu_terrain_mass_flux5_inplace(a, m, divx, ni=ni, nj=nj, nk=nk, dx=dx, dy=dy, dz=dz)
    d = lambda x: to_dev(x, device)  # noqa: E731
    zeros = lambda: torch.zeros(cell, dtype=torch.float32, device=device)  # noqa: E731
    mass, dm, ddivx = {k: d(a[k]) for k in ("rru", "rrv", "rrw")}, d(m), d(divx)
    grid = dict(ni=ni, nj=nj, nk=nk, dt=dt, dx=dx, dy=dy, lateral_sides=sides)
    vertical = stretched.flat_stretched_column(flat, device) if flat else None
    column = vertical.column if flat else None
    rdz = float(flat.rdz) if flat else float(F(1.0) / F(dz))
    s = np.zeros(sh["s"], F)
    got = {}
    if row.startswith("theta"):
        nrk = int(row[-1])
        th0 = (F(300.0) + np.linspace(0.0, 40.0, nk)).astype(F)
        x, a0 = (rng.normal(0.0, 2.0, cell).astype(F) for _ in range(2))
        held, divterm = (rng.normal(0.0, 1e-3, cell).astype(F) for _ in range(2))
        ost.pack_theta(th0, x, s, ni=ni, nj=nj, nk=nk)
        obc.fill(s, obc.KIND_SCALAR, sides, ni=ni, nj=nj, nk=nk)
        adv = np.zeros(cell, F)
        fl = {"x": np.zeros(sh["u"], F), "y": np.zeros(sh["v"], F), "z": np.zeros(sh["w"], F)}
        weps = float(F(F(10.0) * F(1e-18)))
        cpu_scalar_advection5_inplace(s, a, m, divx, adv, fl, ni=ni, nj=nj, nk=nk, nrk=nrk, dx=dx, dy=dy, dz=dz,
                                      weps=weps, lateral_sides=sides, flat=flat)
        want = ost.compose_theta(a0, held, divterm, adv, F(F(dt) / F(4 - nrk)))
        dx_, dth0, da0, dheld, ddiv = d(x), d(th0), d(a0), d(held), d(divterm)
        out = zeros()
        if flat:
            stretched.launch_flat_scalar_rk_compose(d(s), mass, dm, vertical, ddivx, da0, dheld, ddiv, out, nrk=nrk,
                                                    weps=weps, **grid)
        else:
            sm.launch_scalar_rk_compose(d(s), mass, dm, ddivx, da0, dheld, ddiv, out, nrk=nrk, weps=weps, dz=dz, **grid)
        got["padded"] = out
        got["unpadded"] = zeros()
        sm.launch_scalar_stage_from_carrier(dx_, dth0, mass, dm, ddivx, da0, dheld, ddiv, got["unpadded"], nrk=nrk,
                                            rdz=rdz, weps=weps, flat_column=column, copy_back=False, **grid)
        if nrk == 1:
            for ns in (1, 2):
                outs = [zeros() for _ in range(ns)]
                sm.launch_scalar_stages_from_carriers([dx_] * ns, [dth0] * ns, mass, dm, ddivx, [da0] * ns,
                                                      [dheld] * ns, [ddiv] * ns, outs, nrk=nrk, rdz=rdz,
                                                      flat_column=column, **grid)
                got.update({f"batch {q} of {ns}": o for q, o in enumerate(outs)})
    else:
        species = 0 if row.startswith("qv") else 1
        q = np.abs(rng.normal(0.0, 1e-3, cell)).astype(F)
        q[rng.random(cell) < 0.3] = F(0.0)
        a0 = np.abs(q + rng.normal(0.0, 2e-4, cell)).astype(F)
        a0[rng.random(cell) < 0.3] = F(0.0)
        held = rng.normal(0.0, 1e-7, cell).astype(F)
        s[1 : nk + 1, NG : NG + nj, NG : NG + ni] = q
        obc.fill(s, obc.KIND_SCALAR, sides, ni=ni, nj=nj, nk=nk)
        adv = op.pdef_advection(a0, s, a, m, divx, ni=ni, nj=nj, nk=nk, dt=F(dt), dx=dx, dy=dy, dz=dz,
                                weps=float(F(F(1e-2) * F(1e-18))), pdefweno=species != 0, sides=sides, flat=flat)
        want = ost.compose_moisture(a0, held, adv, F(dt))
        da0, dheld, out, ps = d(a0), d(held), zeros(), {n: zeros() for n in ("advx", "advy", "advz")}
        if flat:
            stretched.launch_cuda_gm1_child_stretched_pdef_moisture(d(s), mass, dm, vertical, ddivx, da0, dheld, out, ps,
                                                                    species=species, **grid)
        else:
            sm.launch_pdef_moisture(d(s), mass, dm, ddivx, da0, dheld, out, ps, species=species, dz=dz, **grid)
        got["padded"] = out
        got["unpadded"] = zeros()
        sm.launch_scalar_stage_from_carrier(d(q), None, mass, dm, ddivx, da0, dheld, None, got["unpadded"], nrk=3,
                                            rdz=rdz, flat_column=column, pdef_species=species, pdef_scratch=ps,
                                            copy_back=False, **grid)
    torch.cuda.synchronize()
    for name, out in got.items():
        assert_bits_equal(to_host(out), want, f"{row} {name}")
