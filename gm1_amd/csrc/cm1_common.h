// Shared device helpers for the CM1 large-step kernels (gfx950).
//
// Arithmetic contract: every float operation is one IEEE binary32 operation
// rounded to nearest, in the association order the CM1 transcription spells.
// The translation units are compiled with -ffp-contract=off and without fast
// math, so `a*b + c` is a rounded product followed by a rounded sum and never
// a fused multiply-add; division and sqrt are the correctly rounded forms.
// Denormals are preserved (no flush to zero).
#pragma once
#pragma clang fp contract(off)

#include <algorithm>
#include <hip/hip_runtime.h>
#include <stdint.h>

#define GM1_DEV __device__ __forceinline__

// Field layout (z, y, x), C order, i fastest.  Winds and scalars carry a
// three-cell lateral halo (ng = 3); the pressure family carries one cell.
namespace gm1 {

constexpr int NG = 3;

struct Dims {
  int ni, nj, nk;
};

// Index of (k, j, i) in an array with row length nx and nz*ny*nx words.
GM1_DEV int64_t ix3(int k, int j, int i, int ny, int nx) {
  return ((int64_t)k * ny + j) * (int64_t)nx + i;
}

// Padded-array extents for the four staggerings.
GM1_DEV int sx(int ni) { return ni + 2 * NG; }      // scalar / w row length
GM1_DEV int sy(int nj) { return nj + 2 * NG; }      // scalar / w / u rows
GM1_DEV int ux(int ni) { return ni + 1 + 2 * NG; }  // u row length
GM1_DEV int vy(int nj) { return nj + 1 + 2 * NG; }  // v rows

// Tile index for linear workgroup id `linear` of `n`, chosen so that each of
// the eight XCDs -- which receive workgroups round-robin in dispatch order --
// works on one contiguous range of tiles, keeping neighbouring rows in the
// same L2.
GM1_DEV int xcd_tile(int linear, int n) {
  constexpr int X = 8;
  const int per = n / X, rem = n % X;
  const int x = linear % X, r = linear / X;
  return (x < rem) ? x * (per + 1) + r : rem * (per + 1) + (x - rem) * per + r;
}

// Level chunks of a kernel of `tiles` 512-lane tiles marching nk levels, per_cu
// workgroups resident on each of the 256 CUs: the count whose estimated time is
// least (of counts within a hundredth, the largest).  A chunk takes a level more than
// it has (its window and first plane), full rounds of resident workgroups take a
// chunk's time each, and a last round takes 0.5 + 0.5 f of it where its fullest CU
// holds a fraction f of per_cu (fewer waves on a CU each run faster).  The rule lands
// within 2 % of the measured minima (its own count first): 200 tiles of 80 levels at two
// per CU, 5 chunks 154 us, 10 160, 16 173, 4 179; 200 of 80 at three, 10 142, 5 140,
// 3 152, 4 167; 48 of 64 at three, 16 36 us, 10 40, 5 44; 960 of 80 at three, 4 604 us,
// 5 612, 10 640, 2 625.
inline int tile_chunks(int tiles, int nk, int per_cu, int* kchunk) {
  auto cost = [&](int kc) {
    const int64_t groups = (int64_t)tiles * ((nk + kc - 1) / kc), slots = 256 * per_cu;
    const int64_t last = (groups % slots + 255) / 256;  // workgroups on the last round's fullest CU
    return (kc + 1) * ((double)(groups / slots) + (last ? 0.5 + 0.5 * (double)last / per_cu : 0.0));
  };
  double least = cost(nk);
  for (int kc = 1; kc < nk; ++kc) least = std::min(least, cost(kc));
  *kchunk = 1;
  while (cost(*kchunk) > 1.01 * least) ++*kchunk;
  return (nk + *kchunk - 1) / *kchunk;
}

// The word at a 32-bit byte offset from a base the whole workgroup shares:
// the load takes the base in scalar registers and the offset in one vector
// register (the hardware adds them), so a thread's level-k address costs no
// 64-bit vector arithmetic.  The offset must stay below 4 GiB.
GM1_DEV float ldo(const float* base, uint32_t byte_offset) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + byte_offset);
}
GM1_DEV void sto(float* base, uint32_t byte_offset, float v) {
  *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + byte_offset) = v;
}

// Pressure family (nk+2, nj+2, ni+2).
GM1_DEV int64_t pix(int k, int j, int i, int ni, int nj) {
  return ((int64_t)k * (nj + 2) + j) * (int64_t)(ni + 2) + i;
}

// Constant weights: each is the binary64 quotient rounded once to binary32,
// which is how the CM1 transcription forms them.
constexpr float C2_60 = (float)(2.0 / 60.0);
constexpr float CM13_60 = (float)(-13.0 / 60.0);
constexpr float C47_60 = (float)(47.0 / 60.0);
constexpr float C27_60 = (float)(27.0 / 60.0);
constexpr float CM3_60 = (float)(-3.0 / 60.0);
constexpr float CM1_6 = (float)(-1.0 / 6.0);
constexpr float C1_6 = (float)(1.0 / 6.0);
constexpr float C2_6 = (float)(2.0 / 6.0);
constexpr float C5_6 = (float)(5.0 / 6.0);
constexpr float CM7_6 = (float)(-7.0 / 6.0);
constexpr float C11_6 = (float)(11.0 / 6.0);
constexpr float C13_12 = (float)(13.0 / 12.0);

// Third-order upwind face value (adv_routines.F flx3).
GM1_DEV float flx3(float s1, float s2, float s3) {
  float r = CM1_6 * s1;
  r = r + C5_6 * s2;
  return r + C2_6 * s3;
}

// Fifth-order upwind-biased face value (adv_routines.F flx5).
GM1_DEV float flx5(float s1, float s2, float s3, float s4, float s5) {
  float r = C2_60 * s1;
  r = r + CM13_60 * s2;
  r = r + C47_60 * s3;
  r = r + C27_60 * s4;
  return r + CM3_60 * s5;
}

// WENO-Z (siform 2) face value: binary32 smoothness indicators and
// candidate stencils, binary64 nonlinear weights (adv_routines.F weno5).
//
// The kernels that form it are bound by its four binary64 divisions, so the word is
// decided by a shorter evaluation first (Ziv 1991, as the Kessler powers): over the
// common denominator (a1 a2 a3)^2, a_i = b_i + weps, the weights are
// g_i (a_i^2 + tau^2) a_j^2 a_k^2 and one reciprocal remains.  With u = 2^-53 and P the
// largest |p_i|: the statement below is within 16 u P of the exact value of its a_i and
// tau (5 u a weight, 8 u the sums, a quotient), the short form within 25 u P (7 u a
// weight, 9 u each sum, the reciprocal of two Newton steps and a product), together
// under 2^-47 P; where v - 2^-45 P and v + 2^-45 P round to one binary32 word it is the
// statement's.  Elsewhere (about one lane in 2^20, zeros of either sign) and outside
// b_i <= 1e9, 1e-21 <= weps <= 1e30, the statement itself: there a smoothness may be
// NaN or infinite (the statement's min() drops it, so its word can be finite), min(1e30, .)
// could act, or a product could leave the binary64 range (inside, every a_i lies in
// 1e-21 .. 1.1e30, a weight over the common denominator in 1e-127 .. 1e181).  WENO compose
// 677 -> 617 us and pdef tendencies 600 -> 515 at 640x768x80, 154 -> 134 and 141 -> 121
// at 320x320x80 (terrain).
GM1_DEV float weno5(float s1, float s2, float s3, float s4, float s5,
                    double weps) {
  float d1 = (s1 - 2.0f * s2) + s3;
  float e1 = (s1 - 4.0f * s2) + 3.0f * s3;
  float b1r = C13_12 * (d1 * d1) + 0.25f * (e1 * e1);
  float d2 = (s2 - 2.0f * s3) + s4;
  float e2 = s2 - s4;
  float b2r = C13_12 * (d2 * d2) + 0.25f * (e2 * e2);
  float d3 = (s3 - 2.0f * s4) + s5;
  float e3 = (3.0f * s3 - 4.0f * s4) + s5;
  float b3r = C13_12 * (d3 * d3) + 0.25f * (e3 * e3);
  float p1 = (C2_6 * s1 + CM7_6 * s2) + C11_6 * s3;
  float p2 = (CM1_6 * s2 + C5_6 * s3) + C2_6 * s4;
  float p3 = (C2_6 * s3 + C5_6 * s4) + CM1_6 * s5;
  double b1 = (double)b1r, b2 = (double)b2r, b3 = (double)b3r;
  const double g1 = (double)0.1f, g2 = (double)0.6f, g3 = (double)0.3f;
  const double a1 = b1 + weps, a2 = b2 + weps, a3 = b3 + weps;
  {
    const double t = b1 - b3, t1 = a1 * a1, t2 = a2 * a2, t3 = a3 * a3;
    const double v1 = (g1 * __builtin_fma(t, t, t1)) * (t2 * t3);
    const double v2 = (g2 * __builtin_fma(t, t, t2)) * (t1 * t3);
    const double v3 = (g3 * __builtin_fma(t, t, t3)) * (t1 * t2);
    const double den = (v1 + v2) + v3;
    const double num = __builtin_fma(v3, (double)p3, __builtin_fma(v2, (double)p2, v1 * (double)p1));
    double r = __builtin_amdgcn_rcp(den);
    r = __builtin_fma(__builtin_fma(-den, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-den, r, 1.0), r, r);
    const double v = num * r;
    const double e = 0x1p-45 * (double)fmaxf(fmaxf(fabsf(p1), fabsf(p2)), fabsf(p3));
    const float lo = (float)(v - e), hi = (float)(v + e);
    // (as integers, which order the smoothnesses as floats do, with infinity and NaN above all)
    const uint32_t above = (weps >= 1.0e-21 && weps <= 1.0e30) ? 0x4e6e6b29u /* the float after 1e9 */ : 0u;
    const uint32_t smooth = max(max(__float_as_uint(b1r), __float_as_uint(b2r)), __float_as_uint(b3r));
    if (__float_as_uint(lo) == __float_as_uint(hi) && smooth < above) return lo;
  }
  double tau = fabs(b1 - b3);
  double q1 = fmin(1.0e30, tau / a1);
  double q2 = fmin(1.0e30, tau / a2);
  double q3 = fmin(1.0e30, tau / a3);
  double w1 = g1 * (1.0 + q1 * q1);
  double w2 = g2 * (1.0 + q2 * q2);
  double w3 = g3 * (1.0 + q3 * q3);
  double num = (w1 * (double)p1 + w2 * (double)p2) + w3 * (double)p3;
  return (float)(num / ((w1 + w2) + w3));
}

// Positive-definite third-order limiter used at the WENO lower closures
// (adv_routines.F upstrpd).
GM1_DEV float upstrpd(float s1, float s2, float s3, float weps) {
  float dd = s2 - s1;
  float se = copysignf(fabsf(weps), dd);
  float rr = (s3 - s2) / (se + dd);
  float cand = C1_6 + C2_6 * rr;
  float phi = fmaxf(0.0f, fminf(rr, fminf(cand, 1.0f)));
  return s2 + phi * (s2 - s1);
}

GM1_DEV float recon5(float s1, float s2, float s3, float s4, float s5,
                     bool use_weno, double weps) {
  return use_weno ? weno5(s1, s2, s3, s4, s5, weps)
                  : flx5(s1, s2, s3, s4, s5);
}

// CM1's lateral family word: wbc | ebc<<4 | sbc<<8 | nbc<<12 with each side
// 1 periodic, 2 open-radiative, 3/4 rigid.  Zero is a tile-local launch.
__host__ __device__ inline unsigned side_of(unsigned obc, unsigned side) {
  return (obc >> (4u * side)) & 15u;
}

}  // namespace gm1

// Status handling shared by every C entry point.
#define GM1_LAUNCH_CHECK()                          \
  do {                                              \
    hipError_t e_ = hipGetLastError();              \
    if (e_ != hipSuccess) return (int)e_;           \
  } while (0)

inline int gm1_blocks(int64_t n, int threads) {
  int64_t b = (n + threads - 1) / threads;
  return (int)(b < 1 ? 1 : b);
}
