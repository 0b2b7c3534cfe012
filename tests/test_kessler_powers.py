"""The Kessler passes' binary64-rounded powers, word for word, over the whole binary32 range."""

from __future__ import annotations

import numpy as np
import pytest

F = np.float32


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [1, 2])
def test_gpu_equation_of_state_power_is_the_rounded_binary64_power(device, seed):
    """prs = (pi0 + pp)^(cp/rd) * p00 of the transition: random words of every exponent, words at the ends of the
    short form's range (powers of two and sqrt(2) and their neighbours), zeros, infinities, NaN, denormals and
    negatives, and 250 000 words of the range a column has."""
    import torch

    from gm1_amd import _native
    from gm1_amd._device import ptr, stream_handle

    rng = np.random.default_rng(seed)
    words = rng.integers(0, 1 << 32, 250_000, dtype=np.uint64).astype(np.uint32)
    edges = np.array([(e << 23) | m for e in range(0, 256) for m in (0, 1, 0x3504F2, 0x3504F3, 0x3504F4, 0x7FFFFF)], np.uint32)
    column = rng.uniform(0.2, 1.1, 250_000).astype(F).view(np.uint32)
    x = np.concatenate([words, edges, edges | np.uint32(1 << 31), column])
    n = (x.size + 63) // 64 * 64
    x = np.concatenate([x, np.full(n - x.size, 0x3F800000, np.uint32)]).view(F)
    ni, nj, nk = 64, n // 64, 1
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v, F)).to(device)  # noqa: E731
    pi0, zero, one = t(x), t(np.zeros(n)), t(np.ones(n))
    a = {k: zero.clone() for k in ("pp", "th", "qv", "qc", "prs", "rho", "rr", "h1", "h2", "h3", "h4")}
    print(f"powers of {n} words", flush=True)
    _native.call("gm1hip_kessler_transition_pre", None, *(ptr(a[k]) for k in ("pp", "th", "qv", "qc", "h1", "h2", "h3", "h4")),
                 ptr(pi0), ptr(one), ptr(a["prs"]), ptr(a["rho"]), ptr(a["rr"]), ni, nj, nk, 1.0, 1, 1,
                 stream_handle(None))
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        e = np.float64(F(1005.7) / F(287.04))
        want = np.power(x.astype(np.float64), e).astype(F) * F(1.0e5)
    got = a["prs"].cpu().numpy()
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), (x[~same][:5], got[~same][:5], want[~same][:5], int((~same).sum()))
