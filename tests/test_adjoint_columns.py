"""The halo-free step's staged column passes at the level counts where their chunks branch."""

from __future__ import annotations

import numpy as np
import pytest
from test_adjoint_step import FIELDS, _oracle64_trajectory, _rel, state32, unpad_np


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nk", [(33, 6, 6), (32, 7, 16), (8, 9, 33), (35, 6, 65), (6, 6, 128), (9, 7, 130)])
def test_gpu_staged_columns_forward_words_and_adjoint(device, ni, nj, nk):
    """Chunks of 1, 1, 3, 5 and 8 levels (four- and eight-level instances), ragged tiles, and a column that takes the
    passes of one thread a cell: the forward step equals the binary32 restatement word for word and its adjoint the
    binary64 adjoint within 1e-4, the bound the stage's own test uses.  theta' is bounded in the 2-norm by 1e-3:
    its differentiated WENO weights are ratios of binary32 smoothness indicators of this noisy state (floor
    1e-17), whose rounding single cells amplify; the passes of one thread a cell give the same 3.2e-4 (2-norm)
    and 3.2e-3 (largest cell) at 128 levels."""
    import torch

    from gm1_amd.adjoint_step import DryPeriodicStep
    from oracle import large_step as ol

    print(f"adjoint columns {ni}x{nj}x{nk}", flush=True)
    cfg, host, a, prof, c = state32(seed=nk, ni=ni, nj=nj, nk=nk)
    S32 = unpad_np(a, ni, nj, nk)
    a1 = {k: v.copy() for k, v in a.items()}
    ol.large_step(a1, host["metrics"], host["base"], prof, c, zt=np.float32(nk * cfg.dz))
    ref = unpad_np(a1, ni, nj, nk)
    step = DryPeriodicStep(cfg, host["metrics"], host["base"], device)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(device)  # noqa: E731
    out = step.forward({n: dev(v) for n, v in S32.items()})
    torch.cuda.synchronize()
    for n in FIELDS:
        assert np.array_equal(out[n].cpu().numpy(), ref[n]), n
    _, als, p = _oracle64_trajectory(a, host, cfg, prof, c)
    S = {n: v.astype(np.float64) for n, v in S32.items()}
    end, T = als.Step(p).forward(S)
    rng = np.random.default_rng(nk)
    Sb = {n: rng.standard_normal(end[n].shape) for n in FIELDS}
    want = als.Step(p).adjoint(T, Sb)
    got = step.adjoint({n: dev(v) for n, v in S32.items()}, {n: dev(v) for n, v in Sb.items()})
    torch.cuda.synchronize()
    for n in FIELDS:
        g = got[n].cpu().numpy()
        if n == "th":
            assert np.linalg.norm(g - want[n]) <= 1e-3 * np.linalg.norm(want[n])
        else:
            assert _rel(g, want[n]) <= 1e-4, n


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nk", [(33, 6, 6), (32, 7, 16), (8, 9, 33), (9, 8, 64), (35, 6, 65), (6, 6, 128), (9, 7, 130)])
def test_gpu_staged_columns_adjoint_at_every_cell(device, ni, nj, nk):
    """With the WENO weights held at their forward values nothing amplifies a rounding, and every field, theta' too
    (where the column's coefficient adjoints of thv and ppterm end), meets the stage test's 1e-4 at each cell: a
    level taken wrong where two slots meet would not."""
    import torch

    from gm1_amd.adjoint_step import DryPeriodicStep

    print(f"adjoint columns, weights held {ni}x{nj}x{nk}", flush=True)
    cfg, host, a, prof, c = state32(seed=nk, ni=ni, nj=nj, nk=nk)
    S32 = unpad_np(a, ni, nj, nk)
    step = DryPeriodicStep(cfg, host["metrics"], host["base"], device, weno="frozen")
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(device)  # noqa: E731
    _, als, p = _oracle64_trajectory(a, host, cfg, prof, c)
    end, T = als.Step(p).forward({n: v.astype(np.float64) for n, v in S32.items()}, als.Tape(exact=False))
    rng = np.random.default_rng(nk)
    Sb = {n: rng.standard_normal(end[n].shape) for n in FIELDS}
    want = als.Step(p).adjoint(T, Sb)
    got = step.adjoint({n: dev(v) for n, v in S32.items()}, {n: dev(v) for n, v in Sb.items()})
    torch.cuda.synchronize()
    errs = {n: _rel(got[n].cpu().numpy(), want[n]) for n in FIELDS}
    print({n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    for n, e in errs.items():
        assert e <= 1e-4, (n, e)
