"""The Kessler passes' binary64-rounded powers and exponentials, word for word.

On the device: the equation of state's power over the whole binary32 range.  On the CPU: the source's own short forms
built for the host, for the exponential and every exponent the passes use, against the C library's binary64 functions
rounded once (and against its 80-bit ones for the stated error).
"""

from __future__ import annotations

import subprocess
from pathlib import Path

import numpy as np
import pytest

F = np.float32
SOURCE = Path(__file__).resolve().parents[1] / "gm1_amd" / "csrc" / "kessler.hip"

# the short forms as the source states them; the hardware's reciprocal (within one unit in the last place) is
# played by the rounded one moved by -1, 0 or 1 units
HOST = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
static unsigned __float_as_uint(float f) { unsigned u; memcpy(&u, &f, 4); return u; }
static float __uint_as_float(unsigned u) { float f; memcpy(&f, &u, 4); return f; }
static long long __double_as_longlong(double d) { long long u; memcpy(&u, &d, 8); return u; }
static int nudge = 0;
static float __builtin_amdgcn_rcpf(float x) { return __uint_as_float(__float_as_uint(1.0f / x) + nudge); }
#define GM1_DEV static inline
%s
static std::mt19937_64 r(%d);
static double uniform() { return (double)(r() >> 11) * 0x1p-53; }
static float word() { return __uint_as_float((unsigned)r()); }
static long wrong = 0, checked = 0, decided = 0;
static double worst = 0.0;
static void check(double y, bool ok, float want, long double exact, float a, float e) {
  ++checked;
  if (!ok) return;
  ++decided;
  const double err = std::fabs((double)(((long double)y - exact) / exact));
  if (err > worst) worst = err;
  if (__float_as_uint((float)y) != __float_as_uint(want) && ++wrong <= 5)
    printf("word of %%a (exponent %%a): %%a, want %%a\n", a, e, (float)y, want);
}
static void power(float b, float e) {
  nudge = (int)(r() %% 3) - 1;
  const Near l = log_near(b);
  const double t = std::fma(l.ex, (double)e, l.log_m * ((double)e * LOG2E));
  const double y = exp2_near(std::fmin(std::fmax(t, -200.0), 200.0));
  const float want = (float)std::pow((double)b, (double)e);
  check(y, l.ok && rounds_safely(y), want, powl((long double)b, (long double)e), b, e);
}
static void exponential(float x) {
  const double y = exp2_near((double)std::fmin(std::fmax(x, -200.0f), 200.0f) * LOG2E);
  const float want = (float)std::exp((double)x);
  check(y, rounds_safely(y), want, expl((long double)x), x, 0.0f);
}
int main() {
  const float RD = 287.04f, CP = 1005.7f;
  const float es[] = {0.1346f, 0.2046f, 0.525f, 0.875f, RD / CP, RD / (CP - RD), CP / RD};
  for (float e : es) {
    for (long n = 0; n < 300000; ++n) {
      power(word(), e);                                               // every exponent, either sign, NaN, denormals
      power((float)std::pow(10.0, -14.0 + 20.0 * uniform()), e);      // rain and pressures
      power((float)(0.2 + 0.9 * uniform()), e);                       // Exner functions
      // a base whose power lies beside the midpoint of two binary32 words
      const double mid = (double)__uint_as_float((unsigned)(0x30000000u + r() %% 0x20000000u)) * (1.0 + 0x1p-24);
      power((float)std::pow(mid, 1.0 / (double)e), e);
    }
    for (unsigned x = 0; x < 256; ++x)
      for (unsigned m : {0u, 1u, 0x3504f2u, 0x3504f3u, 0x3504f4u, 0x7fffffu}) {
        power(__uint_as_float(x << 23 | m), e);
        power(__uint_as_float(1u << 31 | x << 23 | m), e);
      }
  }
  for (long n = 0; n < 2000000; ++n) {
    exponential(word());
    exponential((float)(-110.0 + 210.0 * uniform()));  // past both ends of the binary32 results
    const float t = (float)(180.0 + 150.0 * uniform());
    exponential((17.67f * (t - 273.15f)) / (t - 29.65f));  // saturation
    exponential((float)std::log((double)__uint_as_float((unsigned)(0x00800000u + r() %% 0x7e000000u)) * (1.0 + 0x1p-24)));
  }
  for (float x : {0.0f, -0.0f, 1e-45f, -1e-45f, INFINITY, -INFINITY, NAN, 200.0f, -200.0f, 88.722839f, 88.72284f, -87.33655f})
    exponential(x);
  printf("checked %%ld decided %%ld wrong %%ld worst 2^%%.2f\n", checked, decided, wrong, std::log2(worst));
  return wrong || worst > 0x1p-44 || decided < checked / 2;
}
"""


@pytest.mark.parametrize("seed", [1, 2])
def test_short_forms_give_the_rounded_binary64_words(tmp_path, seed):
    """Wherever the short form decides a word it is the library's, and its error is below the stated 2^-44."""
    text = SOURCE.read_text()
    log_form = text[text.index("struct Near {"):text.index("// binary64 rounded once: the words that decide")]
    log_form += text[text.index("GM1_DEV Near log_near"):text.index("GM1_DEV float exp_r")]
    source = tmp_path / "powers.cpp"
    source.write_text(HOST % (log_form, seed))
    program = tmp_path / "powers"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(program), str(source)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


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
