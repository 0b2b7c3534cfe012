"""The acoustic stage's column passes against its general one, word for word, where their rules branch."""

from __future__ import annotations

import numpy as np
import pytest
from helpers import assert_bits_equal, to_host

OUT = ("u3d", "v3d", "w3d", "pp3d", "ppd", "ppx", "rru", "rrv", "rrw", "radbcw", "radbce", "radbcs", "radbcn")


@pytest.mark.gpu
@pytest.mark.parametrize("nloop", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("sides,ni,nj,nk", [((2, 2, 2, 2), 33, 9, 18), ((1, 1, 2, 2), 32, 11, 16), ((2, 4, 1, 1), 31, 8, 33),
                                            ((4, 2, 2, 4), 64, 9, 66), ((1, 1, 1, 1), 9, 33, 17)])
def test_gpu_flat_resident_stage_equals_the_staged_one(device, monkeypatch, nloop, sides, ni, nj, nk):
    """Odd and even counts of small steps (time averages are added two steps at a time), mixed lateral families
    (ppd's halo words are taken from the cells the fill copies), tiles with and without a ragged edge."""
    from dataclasses import replace

    import torch

    from gm1_amd import stretched
    from gm1_amd.fields import large_stretched_c3
    from gm1_amd.large_step import create_gm1_large_step_state, host_initial_state, launch_cuda_gm1_large_step

    cfg = replace(large_stretched_c3(ni, nj, nk), lateral_sides=sides,
                  stretched=(nk * 100.0, 0.0, nk * 100.0, 60.0, 140.0))
    print(f"resident stage {ni}x{nj}x{nk} sides {sides} nloop {nloop}", flush=True)
    st = create_gm1_large_step_state(host_initial_state(cfg), device)
    launch_cuda_gm1_large_step(st)
    torch.cuda.synchronize()
    g = torch.Generator(device=device).manual_seed(nloop)
    for n in ("ppi", "ppx", "uten", "vten", "wten", "ua", "va", "wa", "u3d", "v3d", "w3d"):
        scale = 1e-4 if n in ("ppi", "ppx") else 1e-3 if n.endswith("ten") else 1.0
        st.a[n] += scale * torch.randn(st.a[n].shape, device=device, generator=g)
    schedule = stretched.sound3_stage_schedule_f32
    monkeypatch.setattr(stretched, "sound3_stage_schedule_f32", lambda dt, ns, nrk: (nloop, schedule(dt, ns, nrk)[1]))
    runs = {}
    for column_pass in ("staged", "resident", "resident16"):
        a = {k: v.clone() for k, v in st.a.items()}
        out = []
        for nrk in (1, 3):
            stretched.launch_cuda_gm1_flat_acoustic_stage(a, st.metrics, ni=ni, nj=nj, nk=nk, nrk=nrk, dt=cfg.dt,
                                                          nsound=cfg.nsound, dx=cfg.dx, dy=cfg.dy, vertical=st.flat,
                                                          lateral_sides=sides, column_pass=column_pass)
            torch.cuda.synchronize()
            out.append({n: to_host(a[n]) for n in OUT})
        runs[column_pass] = out
    for column_pass in ("resident", "resident16"):
        for got, want, nrk in zip(runs[column_pass], runs["staged"], (1, 3)):
            for n in OUT:
                assert_bits_equal(got[n], want[n], f"{column_pass} stage {nrk} {n}")
    assert np.isfinite(runs["staged"][1]["w3d"]).all() and np.abs(runs["staged"][1]["w3d"]).max() > 0.0


@pytest.mark.gpu
@pytest.mark.parametrize("nloop", [1, 2, 3])
def test_gpu_flat_resident_stage_with_w_held_in_place(device, monkeypatch, nloop):
    """A caller whose w3d is its wa: rrw starts from the words before the first small step on every pass."""
    from dataclasses import replace

    import torch

    from gm1_amd import stretched
    from gm1_amd.fields import large_stretched_c3
    from gm1_amd.large_step import create_gm1_large_step_state, host_initial_state, launch_cuda_gm1_large_step

    cfg = replace(large_stretched_c3(33, 9, 18), stretched=(1800.0, 0.0, 1800.0, 60.0, 140.0))
    print(f"w in place, nloop {nloop}", flush=True)
    st = create_gm1_large_step_state(host_initial_state(cfg), device)
    launch_cuda_gm1_large_step(st)
    torch.cuda.synchronize()
    schedule = stretched.sound3_stage_schedule_f32
    monkeypatch.setattr(stretched, "sound3_stage_schedule_f32", lambda dt, ns, nrk: (nloop, schedule(dt, ns, nrk)[1]))
    runs = {}
    for column_pass in ("staged", "resident"):
        for nrk in (1, 3):
            a = {k: v.clone() for k, v in st.a.items()}
            a["wa"] = a["w3d"]
            stretched.launch_cuda_gm1_flat_acoustic_stage(a, st.metrics, ni=33, nj=9, nk=18, nrk=nrk, dt=cfg.dt,
                                                          nsound=cfg.nsound, dx=cfg.dx, dy=cfg.dy, vertical=st.flat,
                                                          lateral_sides=cfg.lateral_sides, column_pass=column_pass)
            torch.cuda.synchronize()
            runs[column_pass, nrk] = {n: to_host(a[n]) for n in OUT}
    for nrk in (1, 3):
        for n in OUT:
            assert_bits_equal(runs["resident", nrk][n], runs["staged", nrk][n], f"stage {nrk} {n}")
    assert np.abs(runs["staged", 1]["rrw"]).max() > 0.0


@pytest.mark.gpu
@pytest.mark.parametrize("sides,ni,nj", [((2, 2, 1, 1), 1, 9), ((1, 1, 2, 2), 9, 1), ((2, 2, 2, 2), 2, 2)])
def test_gpu_flat_resident_stage_on_a_grid_one_cell_wide(device, monkeypatch, sides, ni, nj):
    """Both faces of a cell open: the second face steps beside the first one's new word, as in the staged stage."""
    import torch
    from helpers import to_dev
    from test_sound import _acoustic_case
    from test_stretched import uniform_flat

    from gm1_amd import stretched

    nk = 18
    print(f"resident stage {ni}x{nj}x{nk} sides {sides}", flush=True)
    a0, m0 = _acoustic_case(np.random.default_rng(ni + 2 * nj), ni, nj, nk, terrain=False)
    m = to_dev(m0, device)
    column = stretched.flat_stretched_column(uniform_flat(nk, 100.0), device)
    monkeypatch.setattr(stretched, "sound3_stage_schedule_f32", lambda dt, ns, nrk: (3, float(np.float32(dt / ns))))
    runs = {}
    for column_pass in ("staged", "resident"):
        a = to_dev(a0, device)
        stretched.launch_cuda_gm1_flat_acoustic_stage(a, m, ni=ni, nj=nj, nk=nk, nrk=1, dt=0.5, nsound=8, dx=250.0,
                                                      dy=200.0, vertical=column, lateral_sides=sides,
                                                      column_pass=column_pass)
        torch.cuda.synchronize()
        runs[column_pass] = {n: to_host(a[n]) for n in OUT}
    for n in OUT:
        assert_bits_equal(runs["resident"][n], runs["staged"][n], n)
    assert np.isfinite(runs["staged"]["u3d"]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("nloop", [1, 2, 3, 6])
@pytest.mark.parametrize("sides,ni,nj,nk,slopes", [((2, 2, 2, 2), 33, 9, 18, True), ((1, 1, 2, 2), 32, 11, 49, False),
                                                   ((2, 4, 1, 1), 31, 8, 65, True), ((4, 2, 2, 4), 64, 9, 81, False),
                                                   ((1, 1, 1, 1), 9, 33, 128, True), ((2, 2, 1, 1), 40, 8, 130, True)])
def test_gpu_terrain_pipelined_stage_equals_the_staged_one(device, monkeypatch, nloop, sides, ni, nj, nk, slopes):
    """The resident terrain pass (up to 128 levels; beyond, the seven-plane one) and the pressure gradient's levels,
    averages and mapped halo words, with and without slopes, on every chunk of levels a thread may own."""
    import torch
    from helpers import to_dev
    from test_sound import _acoustic_case

    from gm1_amd import psolver3

    print(f"terrain stage {ni}x{nj}x{nk} sides {sides} nloop {nloop}", flush=True)
    a0, m0 = _acoustic_case(np.random.default_rng(nk + nloop), ni, nj, nk, terrain=slopes)
    m = to_dev(m0, device)
    monkeypatch.setattr(psolver3, "sound3_stage_schedule_f32", lambda dt, ns, nrk: (nloop, float(np.float32(dt / ns))))
    runs = {}
    for column_pass in ("staged", "pipelined", "pipelined16"):
        a = to_dev(a0, device)
        out = []
        for nrk in (1, 3):
            psolver3.launch_cuda_psolver3_terrain_open_stage(a, m, ni=ni, nj=nj, nk=nk, nrk=nrk, dt=0.5, nsound=8,
                                                             dx=250.0, dy=200.0, dz=150.0, lateral_sides=sides,
                                                             column_pass=column_pass, terrain_slopes_zero=not slopes)
            torch.cuda.synchronize()
            out.append({n: to_host(a[n]) for n in OUT + ("qk", "pk1", "pk2", "mm")})
        runs[column_pass] = out
    for column_pass in ("pipelined", "pipelined16"):
        for got, want, nrk in zip(runs[column_pass], runs["staged"], (1, 3)):
            for n in got:
                assert_bits_equal(got[n], want[n], f"{column_pass} stage {nrk} {n}")
    assert np.isfinite(runs["staged"][1]["w3d"]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nk,nsound", [(17, 5, 3, 4), (16, 4, 32, 6), (15, 3, 33, 4), (33, 6, 65, 8), (48, 3, 97, 4),
                                             (9, 4, 128, 6), (8, 3, 130, 4)])
def test_gpu_periodic_column_passes_equal_the_oracle(ni, nj, nk, nsound):
    """Every chunk of levels a slot may own (1 to 4 levels of 32 slots), ragged tiles, both parities of the averages'
    pairs, and a column too tall for the staged pass: every compared output, after each stage, word for word."""
    from test_sound3_periodic import _to_device, differing, seeded_case

    from gm1_amd.sound3_periodic import launch_cuda_sound3_periodic_stage
    from oracle import sound3_periodic as osp

    a = seeded_case(ni, nj, nk, nk)
    for n in ("tri_aa", "tri_bb", "tri_cc", "tri_dd", "tri_pivot", "tri_residual", "divh", "hadvp", "elim_c", "elim_d"):
        a[n][...] = np.float32(7.0)  # words that a stage zeroes or writes
    d = _to_device(a, "cuda")
    params = dict(dt=2.0, nsound=nsound, rdx=1e-3, rdy=1e-3, rdz=1 / 500)
    print(f"periodic stage {ni}x{nj}x{nk} nsound {nsound}", flush=True)
    for nrk in (1, 2, 3):
        launch_cuda_sound3_periodic_stage(d, ni=ni, nj=nj, nk=nk, nrk=nrk, **params)
        osp.stage(a, ni=ni, nj=nj, nk=nk, nrk=nrk, **params)
        assert differing({n: d[n].cpu().numpy() for n in osp.COMPARE_OUTPUT_NAMES}, a) == {}, f"stage {nrk}"
