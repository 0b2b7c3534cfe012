"""The terrain stage's column passes word for word where their level slots and chunks end."""

from __future__ import annotations

import numpy as np
import pytest
from helpers import assert_bits_equal, to_dev, to_host
from test_large_step import F, _stage_inputs, ost


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nk", [(64, 3, 8), (65, 2, 9), (3, 4, 17), (7, 5, 33), (5, 3, 127), (9, 2, 128), (6, 3, 129)])
def test_gpu_post_acoustic_and_buoyancy_columns(device, ni, nj, nk):
    """Whole and ragged slots and chunks, one column past a wavefront, the tallest slotted column and one above it."""
    import torch

    from gm1_amd import _native
    from gm1_amd._device import ptr, stream_handle

    print(f"stage columns {ni}x{nj}x{nk}", flush=True)
    rng = np.random.default_rng(ni + 7 * nk)
    a, m, _, _, _ = _stage_inputs(rng, ni, nj, nk)
    a["thterm"] = rng.standard_normal((nk, nj, ni)).astype(F)
    a["dum8"] = rng.standard_normal(a["dum8"].shape).astype(F)
    ha = {k: v.copy() for k, v in a.items()}
    div, tdiv, divx = (np.zeros((nk, nj, ni), F) for _ in range(3))
    ost.buoyancy(ha, m, ni=ni, nj=nj, nk=nk)
    ost.getdiv(ha, m, div, tdiv, ha["thterm"], ni=ni, nj=nj, nk=nk, dx=250.0, dy=300.0, dz=200.0)
    ost.getdivx(ha, m, divx, ni=ni, nj=nj, nk=nk, dx=250.0, dy=300.0, dz=200.0)
    da, dm = to_dev(a, device), to_dev(m, device)
    dd = {n: torch.zeros((nk, nj, ni), dtype=torch.float32, device=device) for n in ("div", "tdiv", "divx")}
    h = stream_handle(None)
    _native.call("gm1hip_buoyancy", ptr(da["dum8"]), ptr(dm["c1"]), ptr(dm["c2"]), ptr(dm["gxu"]), ptr(dm["gyv"]),
                 ptr(da["uten"]), ptr(da["vten"]), ptr(da["wten"]), ni, nj, nk, h)
    _native.call("gm1hip_post_acoustic", ptr(da["rru"]), ptr(da["rrv"]), ptr(da["rrw"]), ptr(dm["rho0_3d"]),
                 ptr(dm["rf0"]), ptr(dm["rgzu"]), ptr(dm["rgzv"]), ptr(dm["dzdx"]), ptr(dm["dzdy"]), ptr(dm["gz"]),
                 ptr(da["thterm"]), ptr(dd["div"]), ptr(dd["tdiv"]), ptr(dd["divx"]), ni, nj, nk, 250.0, 300.0,
                 200.0, h)
    torch.cuda.synchronize()
    for name, want in (("div", div), ("tdiv", tdiv), ("divx", divx)):
        assert_bits_equal(to_host(dd[name]), want, name)
    got = to_host(da)
    for name in ("rru", "rrv", "rrw", "uten", "vten", "wten"):
        assert_bits_equal(got[name], ha[name], name)
