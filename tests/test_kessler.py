"""Kessler warm rain: the oracle against the reference's CPU functions, closed forms, GPU parity.

The oracle (``oracle/kessler.py``) must reproduce ``cpu_gm1_kessler_driver_inplace``,
``cpu_gm1_kessler_large_step_inplace`` and ``cpu_apmasscon_inplace`` word for
word (same NumPy transcendentals), including the binary64 budgets.
"""

from __future__ import annotations

import numpy as np
import pytest

from helpers import F, assert_bits_equal, golden, to_host
from oracle import kessler as ok

FIELDS = ("rho", "rr", "pp3d", "th3d", "prs", "qv", "qc", "qr", "fall_velocity", "rain", "prate")


def _inputs(g, prefix):
    return {k[len(prefix):]: g[k].copy() for k in g.files if k.startswith(prefix)}


@pytest.mark.parametrize("case", [0, 1, 2])
def test_driver_matches_reference(case):
    g = golden("kessler")
    a = _inputs(g, f"d{case}_in_")
    dt, dz, eqt = (float(v) for v in g[f"d{case}_params"])
    res = ok.kessler_driver(a, dx=250.0, dy=250.0, dz=dz, dt=dt, equation_set=int(eqt))
    for name in FIELDS:
        assert_bits_equal(a[name], g[f"d{case}_out_{name}"], f"case {case} {name}")
    np.testing.assert_array_equal(res["iterations"], g[f"d{case}_iterations"])
    assert res["max_fall_substeps"] == int(g[f"d{case}_nfall"])
    np.testing.assert_array_equal(a["asq"], g[f"d{case}_out_asq"])
    np.testing.assert_array_equal(a["qbudget"], g[f"d{case}_out_qbudget"])


def test_driver_cases_exercise_the_branches():
    g = golden("kessler")
    assert int(g["d1_nfall"]) > 1 and int(g["d0_nfall"]) == 1
    it = g["d0_iterations"]
    assert (it > 1).any() and (it == 0).any()
    assert (g["d0_in_qc"] < 0).any() and (g["d0_in_qr"] < 0).any()


def test_large_step_transition_matches_reference():
    g = golden("kessler")
    a = _inputs(g, "t_in_")
    held = {k: a.pop(k) for k in ("qpten", "qtten", "qvten", "qcten")}
    ok.large_step_transition(a, held, dx=250.0, dy=250.0, dz=250.0, dt=1.5, equation_set=2)
    for name in FIELDS:
        assert_bits_equal(a[name], g[f"t_out_{name}"], name)
    for name in held:
        assert_bits_equal(held[name], g[f"t_out_{name}"], name)


def test_apmasscon_matches_reference():
    g = golden("kessler")
    a = _inputs(g, "m_in_")
    r = ok.apmasscon(a, float(g["m_mass1"]))
    mass2, psum, corr, after = g["m_result"]
    assert r["mass2"] == mass2 and r["pressure_sum"] == psum and r["correction"] == corr
    for name in ("pp3d", "prs", "rho"):
        assert_bits_equal(a[name], g[f"m_out_{name}"], name)
    # the ledger after the correction is the reference's, and the gap to mass1 shrank tenfold
    m1 = float(g["m_mass1"])
    assert ok.dry_mass(a["rho"], a["ruh"], a["rvh"], a["rmh"]) == after
    assert abs(after / m1 - 1.0) < 0.2 * abs(mass2 / m1 - 1.0)


def test_water_changes_only_by_surface_rain():
    """Closed form: column-integrated rho*(qv+qc+qr) before minus after equals the rain that left."""
    g = golden("kessler")
    a = _inputs(g, "d0_in_")
    # start from a state pdefq leaves alone so its rescaling does not enter
    for q in ("qc", "qr"):
        a[q] = np.where(a[q] < F(1e-14), F(0.0), a[q]).astype(F)
    a["qv"] = np.maximum(a["qv"], F(0.0))
    rho0 = a["rho"].astype(np.float64).copy()
    w0 = (rho0 * (a["qv"] + a["qc"] + a["qr"]).astype(np.float64)).sum(axis=0)
    ok.kessler_driver(a, dx=250.0, dy=250.0, dz=250.0, dt=1.5, equation_set=2, budgets=False)
    # fallout moves rho*qr*dz through the floor; the local and satadj steps conserve q totals per cell
    w1 = (rho0 * (a["qv"] + a["qc"] + a["qr"]).astype(np.float64)).sum(axis=0)
    fell = a["rain"][0].astype(np.float64) / 0.1 / 250.0
    # binary32 rounding of ~0.01 kg/kg values over 12 levels is a few 1e-9; the rain signal is ~1e-4
    assert fell.max() > 1e-5
    np.testing.assert_allclose(w0 - w1, fell, rtol=0, atol=3e-8)


# ---------------------------------------------------------------- branch decisions
# The north star asks for identical saturation / autoconversion branch decisions.  The
# decision word (oracle.kessler.decision_words, and the device driver's per-cell output)
# records every branch of the local conversion (cuda_gm1_kessler_local.py:290-416), whether
# the saturation adjustment ran, and its iteration count (cuda_gm1_kessler_driver.py:337-428).
BRANCH_MASK = 0xFF  # local-conversion branches and "satadj ran"
ITER_SHIFT = ok.DECISION_ITER_SHIFT


def c2_like_kessler_fields(ni=64, nj=64, nk=80, seed=7):
    """Kessler mass arrays on the 320x320x80 case's column (250 m layers, moist WK sounding) with cloud and rain.

    qv is drawn at 0.75..1.06 of saturation, qc and qr are log-normal in 40 % of the cells: the
    autoconversion, accretion, evaporation and update branches and the saturation adjustment are
    exercised across the column.  Evaporation capped at saturation and the ar + cr > qc limiter
    are out of reach at dt = 1.5 s (the capped rate needs er > qvs - qv, about 100 times the
    evaporation a step allows); both words still have to agree there.
    """
    from gm1_amd.fields import moist_c2
    from gm1_amd.large_step import host_initial_state
    from oracle import large_step as ol

    cfg = moist_c2(ni, nj, nk)
    host = host_initial_state(cfg)
    a = {k: v.copy() for k, v in host["arrays"].items()}
    a["pp_mass"][...] = a["pp3d"][1 : nk + 1, 1 : nj + 1, 1 : ni + 1]
    k = {n: (v.copy() if isinstance(v, np.ndarray) else v) for n, v in ol.kessler_arrays(a).items()}
    ok.eos(k)
    k["rr"][...] = k["rho"]
    rng = np.random.default_rng(seed)
    t = (k["th0"] + k["th3d"]) * (k["pi0"] + k["pp3d"])
    qvs = ok.saturation_qv(t, k["prs"], k["prs"])
    k["qv"][...] = (qvs * rng.uniform(0.75, 1.06, qvs.shape)).astype(F)
    k["qc"][...] = np.where(rng.random(qvs.shape) < 0.4, rng.lognormal(np.log(8e-4), 1.0, qvs.shape), 0).astype(F)
    k["qr"][...] = np.where(rng.random(qvs.shape) < 0.4, rng.lognormal(np.log(4e-4), 1.2, qvs.shape), 0).astype(F)
    return cfg, k


def _decisions(a, mode, *, dz, dt, eqt, dx=250.0):
    b = {n: (v.copy() if isinstance(v, np.ndarray) else v) for n, v in a.items()}
    with ok.transcendentals(mode):
        res = ok.kessler_driver(b, dx=dx, dy=dx, dz=dz, dt=dt, equation_set=eqt, budgets=False)
    return res["decisions"], res["iterations"]


@pytest.mark.parametrize("case", [0, 1, 2])
def test_branch_decisions_of_both_transcendental_forms_match_the_reference_on_its_vectors(case):
    """On the golden cells the reference's float32 transcendentals and the device's rounded ones take every branch
    alike, and both give the reference's own satadj iteration counts."""
    g = golden("kessler")
    a = _inputs(g, f"d{case}_in_")
    dt, dz, eqt = (float(v) for v in g[f"d{case}_params"])
    dn, itn = _decisions(a, "numpy", dz=dz, dt=dt, eqt=int(eqt))
    dr, itr = _decisions(a, "rounded", dz=dz, dt=dt, eqt=int(eqt))
    np.testing.assert_array_equal(itn, g[f"d{case}_iterations"])
    np.testing.assert_array_equal(dn, dr)
    np.testing.assert_array_equal((dn >> ITER_SHIFT) & 0xFF, g[f"d{case}_iterations"])


def test_branch_decisions_on_c2_like_fields():
    """327 680 cells of cloud and rain on the 320x320x80 column: the local-conversion branches and the saturation
    adjustment's on/off decision are identical for the reference's transcendentals and the device's; the
    adjustment's iteration count (its |dT| <= 2e-4 test) moves by one in a few cells in 10^4, where the two exp
    results straddle the threshold."""
    cfg, k = c2_like_kessler_fields()
    dn, _ = _decisions(k, "numpy", dz=cfg.dz, dt=cfg.dt, eqt=2)
    dr, _ = _decisions(k, "rounded", dz=cfg.dz, dt=cfg.dt, eqt=2)
    for bit in range(8):
        assert ((dn >> bit) & 1).sum() > 1000 or bit in (4, 5), f"bit {bit} not exercised"
    np.testing.assert_array_equal(dn & BRANCH_MASK, dr & BRANCH_MASK)
    it_n = ((dn >> ITER_SHIFT) & 0xFF).astype(np.int64)
    it_r = ((dr >> ITER_SHIFT) & 0xFF).astype(np.int64)
    moved = it_n != it_r
    assert moved.mean() < 5e-4 and np.abs(it_n - it_r).max() <= 1


# ---------------------------------------------------------------- GPU parity
def _device_arrays(a, device):
    import torch

    out = {}
    for k, v in a.items():
        out[k] = torch.from_numpy(np.ascontiguousarray(v)).to(device)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("case", [0, 1, 2])
def test_gpu_driver_bit_exact_against_rounded_oracle(device, case):
    """Fields bit for bit against the oracle with binary64-rounded transcendentals; budgets to 1e-12."""
    import torch

    from gm1_amd.kessler import Gm1KesslerDriverSelection, launch_cuda_gm1_kessler_driver

    g = golden("kessler")
    ni, nj, nk = (int(v) for v in g["dims"])
    a = _inputs(g, f"d{case}_in_")
    dt, dz, eqt = (float(v) for v in g[f"d{case}_params"])
    da = _device_arrays(a, device)
    ws = launch_cuda_gm1_kessler_driver(da, ni=ni, nj=nj, nk=nk, dx=250.0, dy=250.0, dz=dz, dt=dt,
                                        selection=Gm1KesslerDriverSelection(equation_set=int(eqt)))
    torch.cuda.synchronize()
    with ok.transcendentals("rounded"):
        res = ok.kessler_driver(a, dx=250.0, dy=250.0, dz=dz, dt=dt, equation_set=int(eqt))
    for name in FIELDS:
        assert_bits_equal(da[name].cpu().numpy(), a[name], f"case {case} {name}")
    np.testing.assert_allclose(da["asq"].cpu().numpy(), a["asq"], rtol=1e-12, atol=1e-30)
    np.testing.assert_allclose(da["qbudget"].cpu().numpy(), a["qbudget"], rtol=1e-12, atol=1e-30)
    status = ws.status.cpu().numpy()
    assert status[0] == int(res["iterations"].max()) and status[1] == 0
    # and the reference's own words to the stated 1e-5 relative max-norm (its NumPy float32
    # transcendentals differ from correctly rounded ones by an ulp); pi' and theta' are measured
    # as the total Exner function and potential temperature they perturb
    totals = {"pp3d": g[f"d{case}_in_pi0"], "th3d": g[f"d{case}_in_th0"]}
    for name in FIELDS:
        off = totals.get(name, 0.0)
        want = g[f"d{case}_out_{name}"].astype(np.float64) + off
        got = da[name].cpu().numpy().astype(np.float64) + off
        scale = max(np.abs(want).max(), 1e-30)
        assert np.abs(got - want).max() / scale < 1e-5, name


@pytest.mark.gpu
@pytest.mark.parametrize("hook", [False, True])
def test_gpu_transition_matches_oracle(device, hook):
    import torch

    from gm1_amd.kessler import (Gm1KesslerDriverSelection, create_cuda_gm1_kessler_driver_workspace,
                                 create_dry_mass_workspace, launch_cuda_gm1_kessler_transition)

    g = golden("kessler")
    ni, nj, nk = (int(v) for v in g["dims"])
    a = _inputs(g, "t_in_")
    held = {k: a.pop(k) for k in ("qpten", "qtten", "qvten", "qcten")}
    mass1 = ok.dry_mass(a["rho"], a["ruh"], a["rvh"], a["rmh"]) * (1.0 + 3e-6)
    da, dh = _device_arrays(a, device), _device_arrays(held, device)
    ws = create_cuda_gm1_kessler_driver_workspace(ni, nj, nk, device)
    dm = create_dry_mass_workspace(ni, nj, nk, device)
    launch_cuda_gm1_kessler_transition(da, dh, ni=ni, nj=nj, nk=nk, dx=250.0, dy=250.0, dz=250.0, dt=1.5,
                                       selection=Gm1KesslerDriverSelection(equation_set=2), workspace=ws,
                                       mass1=mass1 if hook else None, dry_mass=dm)
    torch.cuda.synchronize()
    hookfn = None
    if hook:
        corr = float(dm.correction.cpu().numpy()[0])
        ledger = dm.ledger.cpu().numpy()

        def hookfn(arr):
            r = ok.apmasscon({k: v.copy() for k, v in arr.items()}, mass1)
            # the device's ledger is the same sum in another order
            assert abs(ledger[0] / r["mass2"] - 1.0) < 1e-13 and abs(ledger[1] / r["pressure_sum"] - 1.0) < 1e-13
            assert abs(corr - r["correction"]) <= 1e-6 * abs(r["correction"])
            ok.apply_mass_correction(arr, F(corr))
    with ok.transcendentals("rounded"):
        ok.large_step_transition(a, held, dx=250.0, dy=250.0, dz=250.0, dt=1.5, equation_set=2, hook=hookfn)
    for name in FIELDS:
        assert_bits_equal(da[name].cpu().numpy(), a[name], name)
    for name in held:
        assert_bits_equal(dh[name].cpu().numpy(), held[name], name)


@pytest.mark.gpu
def test_gpu_fused_transition_and_dry_mass_equal_the_two_calls(device):
    """gm1hip_kessler_transition_pre_apmasscon writes the words of gm1hip_kessler_transition_pre (copy_rr = 0)
    then gm1hip_apmasscon: every field, the held rates, the binary64 ledger and the correction, bit for bit."""
    import torch

    from gm1_amd import _native
    from gm1_amd._device import ptr
    from gm1_amd.kessler import create_dry_mass_workspace, launch_cuda_apmasscon

    g = golden("kessler")
    ni, nj, nk = (int(v) for v in g["dims"])
    a = _inputs(g, "t_in_")
    held = {k: a.pop(k) for k in ("qpten", "qtten", "qvten", "qcten")}
    mass1 = ok.dry_mass(a["rho"], a["ruh"], a["rvh"], a["rmh"]) * (1.0 + 3e-6)
    runs = []
    for fused in (False, True):
        da, dh = _device_arrays(a, device), _device_arrays(held, device)
        dm = create_dry_mass_workspace(ni, nj, nk, device)
        pre = (None, ptr(da["pp3d"]), ptr(da["th3d"]), ptr(da["qv"]), ptr(da["qc"]), ptr(dh["qpten"]),
               ptr(dh["qtten"]), ptr(dh["qvten"]), ptr(dh["qcten"]), ptr(da["pi0"]), ptr(da["th0"]), ptr(da["prs"]),
               ptr(da["rho"]), ptr(da["rr"]))
        if fused:
            _native.call("gm1hip_kessler_transition_pre_apmasscon", *pre, ptr(da["ruh"]), ptr(da["rvh"]),
                         ptr(da["rmh"]), ptr(dm.ledger), ptr(dm.correction), float(mass1), ptr(dm.scratch),
                         dm.scratch.numel(), ni, nj, nk, 1.5, 2, 0)
        else:
            _native.call("gm1hip_kessler_transition_pre", *pre, ni, nj, nk, 1.5, 2, 0, 0)
            launch_cuda_apmasscon(da, ni=ni, nj=nj, nk=nk, mass1=float(mass1), workspace=dm)
        torch.cuda.synchronize()
        runs.append(({**{n: to_host(t) for n, t in da.items()}, **{n: to_host(t) for n, t in dh.items()}},
                     to_host(dm.ledger)[:2].copy(), to_host(dm.correction)[:1].copy()))
    (f0, l0, c0), (f1, l1, c1) = runs
    for n in f0:
        assert_bits_equal(f1[n], f0[n], n)
    assert l1.tobytes() == l0.tobytes() and c1.tobytes() == c0.tobytes()


def _device_decisions(a, device, *, dz, dt, eqt, ni, nj, nk, dx=250.0):
    import torch

    from gm1_amd.kessler import Gm1KesslerDriverSelection, launch_cuda_gm1_kessler_driver

    da = _device_arrays({n: v for n, v in a.items() if isinstance(v, np.ndarray)}, device)
    out = torch.zeros((nk, nj, ni), dtype=torch.int32, device=device)
    launch_cuda_gm1_kessler_driver(da, ni=ni, nj=nj, nk=nk, dx=dx, dy=dx, dz=dz, dt=dt,
                                   selection=Gm1KesslerDriverSelection(equation_set=eqt), decisions=out)
    torch.cuda.synchronize()
    return out.cpu().numpy().view(np.uint32), da


@pytest.mark.gpu
@pytest.mark.parametrize("case", [0, 1, 2])
def test_gpu_branch_decisions_match_the_reference_on_its_vectors(device, case):
    """Every cell's branch word from the device equals the oracle's in both transcendental forms and carries the
    reference's satadj iteration counts."""
    g = golden("kessler")
    ni, nj, nk = (int(v) for v in g["dims"])
    a = _inputs(g, f"d{case}_in_")
    dt, dz, eqt = (float(v) for v in g[f"d{case}_params"])
    got, _ = _device_decisions(a, device, dz=dz, dt=dt, eqt=int(eqt), ni=ni, nj=nj, nk=nk)
    dr, _ = _decisions(a, "rounded", dz=dz, dt=dt, eqt=int(eqt))
    dn, _ = _decisions(a, "numpy", dz=dz, dt=dt, eqt=int(eqt))
    np.testing.assert_array_equal(got, dr)
    np.testing.assert_array_equal(got, dn)
    np.testing.assert_array_equal((got >> ITER_SHIFT) & 0xFF, g[f"d{case}_iterations"])


@pytest.mark.gpu
def test_gpu_branch_decisions_on_c2_like_fields(device):
    """327 680 cloudy and rainy cells: the device's words equal the rounded oracle's bit for bit (fields too), and
    the reference-transcendental oracle's in every branch bit."""
    cfg, k = c2_like_kessler_fields()
    print(f"kessler decisions {cfg.ni}x{cfg.nj}x{cfg.nk}", flush=True)
    got, da = _device_decisions(k, device, dz=cfg.dz, dt=cfg.dt, eqt=2, ni=cfg.ni, nj=cfg.nj, nk=cfg.nk)
    b = {n: (v.copy() if isinstance(v, np.ndarray) else v) for n, v in k.items()}
    with ok.transcendentals("rounded"):
        res = ok.kessler_driver(b, dx=250.0, dy=250.0, dz=cfg.dz, dt=cfg.dt, equation_set=2, budgets=False)
    np.testing.assert_array_equal(got, res["decisions"])
    for name in FIELDS:
        assert_bits_equal(da[name].cpu().numpy(), b[name], name)
    dn, _ = _decisions(k, "numpy", dz=cfg.dz, dt=cfg.dt, eqt=2)
    np.testing.assert_array_equal(got & BRANCH_MASK, dn & BRANCH_MASK)
    assert (((got >> ITER_SHIFT) & 0xFF) != ((dn >> ITER_SHIFT) & 0xFF)).mean() < 5e-4


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nk", [(70, 512, 8), (70, 512, 13), (70, 513, 9), (70, 513, 14), (9, 8, 17)])
def test_gpu_column_pass_of_either_batch(device, ni, nj, nk):
    """1024 waves of columns (eight levels a batch) and 1026 (four), with whole and ragged batches, word for word."""
    import torch

    from gm1_amd.kessler import Gm1KesslerDriverSelection, launch_cuda_gm1_kessler_driver

    print(f"kessler columns {ni}x{nj}x{nk}", flush=True)
    _, a = c2_like_kessler_fields(ni, nj, nk, seed=nk)
    da = _device_arrays(a, device)
    launch_cuda_gm1_kessler_driver(da, ni=ni, nj=nj, nk=nk, dx=250.0, dy=250.0, dz=250.0, dt=6.0,
                                   selection=Gm1KesslerDriverSelection(equation_set=2))
    torch.cuda.synchronize()
    with ok.transcendentals("rounded"):
        ok.kessler_driver(a, dx=250.0, dy=250.0, dz=250.0, dt=6.0, equation_set=2)
    for name in FIELDS:
        assert_bits_equal(da[name].cpu().numpy(), a[name], name)
    np.testing.assert_allclose(da["qbudget"].cpu().numpy(), a["qbudget"], rtol=1e-12, atol=1e-30)
