// Fifth-order flux-form momentum advection for gfx950.
//
// Replaces the kernel family of cuda_momentum_advection5.py: terrain mass
// fluxes, divx, and the advu/advv/advw increments added to uten/vten/wten,
// for any CM1 lateral family (periodic sides read across the seam at the
// wrapped index; open sides take the inflow edits).
//   * k_mom_mass_{terrain,flat}: rru on faces 0..ni, rrv on faces 0..nj, rrw at
//                      every w level and divx in one pass.
//   * k_mom_adv{u,v,w}_tile: an LDS-staged tile marching a chunk of levels,
//                      one lane per flux point.
#include "cm1_common.h"
#include "timing.h"

using namespace gm1;

namespace {

struct MomArgs {
  const float* u;
  const float* v;
  const float* w;
  const float* rru;
  const float* rrv;
  const float* rrw;
  const float* divx;
  const float* rho0;
  const float* c2;
  const float* gzu;
  const float* gzv;
  const float* rrf0;
  const float* gz;
  const float* uh;
  const float* vh;
  float* uten;
  float* vten;
  float* wten;
  int ni, nj, nk;
  float rdx, rdy, rdz;
  unsigned obc;
  // Flat stretched column (terrain_flag=.false.): mh (nk+2) then mf (nk+3),
  // CM1-indexed; null on the terrain-coordinate family.  rr0 is the base
  // state's reciprocal density, read at the first column.
  const float* flat;
  const float* rr0;
  // Held tendencies seeding the update (uten = uten1 + advection), or null:
  // the update then adds to uten as it stands -- unless zero_held, where the
  // held tendencies are +0 everywhere (no solve1 contribution) and the update
  // forms 0 + advection without reading them.
  const float* u1 = nullptr;
  const float* v1 = nullptr;
  const float* w1 = nullptr;
  int zero_held = 0;
  // The flat column's buoyancy added to the w update in the same statement
  // order, wten = (wten1 + advw) + (c1*dum8(k-1) + c2*dum8(k)), or null.
  const float* dum8 = nullptr;
  const float* c1 = nullptr;
};

GM1_DEV bool per(unsigned obc, unsigned s) { return side_of(obc, s) == 1u; }
GM1_DEV bool opn(unsigned obc, unsigned s) { return side_of(obc, s) == 2u; }
// periodic wrap of a cell index (0..n-1) and of a face index (0..n)
GM1_DEV int wc(int i, int n, bool lo, bool hi) { return (lo && i < 0) ? i + n : ((hi && i >= n) ? i - n : i); }
GM1_DEV int wf(int i, int n, bool lo, bool hi) { return (lo && i < 0) ? i + n : ((hi && i > n) ? i - n : i); }
GM1_DEV int clampi(int a, int n) { return a < 0 ? 0 : (a >= n ? n - 1 : a); }

// ------------------------------------------------------------- mass fluxes
// Levels per thread of the mass-flux kernels (loads of MKB levels in flight).
constexpr int MKB = 8;

// The terrain mass fluxes in one pass: rru on faces 0..ni, rrv on faces 0..nj, rrw at
// w levels 1..nk+1 (0 at both ends) and divx of the cell below.  A cell forms its east
// and north faces' products itself (the same products its neighbours write) and a
// chunk its lower level's again, so no thread reads a word another writes.  Words are
// requested a level ahead by loads no lane skips.  Against the horizontal and the
// vertical part as two passes, which read rru and rrv back: 58 + 74 -> 95 us at 320x320x80.
__global__ __launch_bounds__(64) void k_mom_mass_terrain(
    const float* __restrict__ u, const float* __restrict__ v, const float* __restrict__ w,
    const float* __restrict__ rho0, const float* __restrict__ rf0, const float* __restrict__ rgzu,
    const float* __restrict__ rgzv, const float* __restrict__ dzdx, const float* __restrict__ dzdy,
    const float* __restrict__ gz, float* __restrict__ rru, float* __restrict__ rrv, float* __restrict__ rrw,
    float* __restrict__ divx, int ni, int nj, int nk, float dz, float rdx, float rdy) {
  const int i = blockIdx.x * 64 + threadIdx.x;  // 0..ni (face or cell)
  const int j = blockIdx.y;                     // 0..nj
  if (i > ni) return;
  const int nxu = ux(ni), nyu = sy(nj), nxs = sx(ni), nyv = vy(nj);
  const int64_t ust = (int64_t)nyu * nxu, vst = (int64_t)nyv * nxs, wst = (int64_t)nyu * nxs, mst = (int64_t)nj * ni;
  const bool uface = j < nj, vface = i < ni, cell = uface && vface;
  const int ic = min(i, ni - 1), jc = min(j, nj - 1), ie = min(i + 1, ni), jn = min(j + 1, nj);
  const uint32_t oc = (uint32_t)(jc * ni + ic) * 4u, ol = (uint32_t)(jc * ni + max(i - 1, 0)) * 4u,
                 oe = (uint32_t)(jc * ni + min(i + 1, ni - 1)) * 4u, os = (uint32_t)(max(j - 1, 0) * ni + ic) * 4u,
                 on = (uint32_t)(min(j + 1, nj - 1) * ni + ic) * 4u;
  const uint32_t ow = (uint32_t)((jc + NG) * nxu + i + NG) * 4u, oue = (uint32_t)((jc + NG) * nxu + ie + NG) * 4u;
  const uint32_t ov = (uint32_t)((j + NG) * nxs + ic + NG) * 4u, ovn = (uint32_t)((jn + NG) * nxs + ic + NG) * 4u;
  const uint32_t owc = (uint32_t)((jc + NG) * nxs + ic + NG) * 4u;
  const float gw = rgzu[(int64_t)jc * (ni + 1) + i], ge = rgzu[(int64_t)jc * (ni + 1) + ie];
  const float gs = rgzv[(int64_t)j * ni + ic], gn = rgzv[(int64_t)jn * ni + ic];
  const float ddx = ldo(dzdx, oc), ddy = ldo(dzdy, oc), g = ldo(gz, oc);
  const float half = 0.5f;
  const float zt = (float)nk * dz, rzt = 1.0f / zt, rdz = 1.0f / dz;
  struct In {
    float uw, ue, vs, vn, rc, rl, re, rs, rn, w, rf;
  };
  auto load = [&](int k) {
    const float *U = u + (int64_t)k * ust, *V = v + (int64_t)k * vst, *R = rho0 + (int64_t)(k - 1) * mst;
    return In{ldo(U, ow), ldo(U, oue), ldo(V, ov), ldo(V, ovn), ldo(R, oc), ldo(R, ol), ldo(R, oe), ldo(R, os),
              ldo(R, on), ldo(w + (int64_t)k * wst, owc), ldo(rf0 + (int64_t)(k - 1) * mst, oc)};
  };
  struct Faces {
    float w, e, s, n;
  };
  auto faces = [&](const In& x) {
    return Faces{(half * (x.rl + x.rc)) * (x.uw * gw), (half * (x.rc + x.re)) * (x.ue * ge),
                 (half * (x.rs + x.rc)) * (x.vs * gs), (half * (x.rc + x.rn)) * (x.vn * gn)};
  };
  // rrw at w level kf (0 at kf = 1 and nk + 1) from level kf's words and the faces of levels kf and kf - 1
  auto rrw_at = [&](int kf, const In& x, const Faces& hi, const Faces& lo) {
    if (kf <= 1 || kf > nk) return 0.0f;
    const float sf = (float)(kf - 1) * dz, sm = (float)((double)kf - 1.5) * dz;
    float r2 = (sf - sm) * rdz;
    const float r1 = half * (1.0f - r2);
    r2 = half * r2;
    const float uxv = r2 * (hi.w + hi.e) + r1 * (lo.w + lo.e);
    const float vyv = r2 * (hi.s + hi.n) + r1 * (lo.s + lo.n);
    float t = uxv * ddx + vyv * ddy;
    t = t * (sf - zt);
    t = t * g;
    t = t * rzt;
    return x.rf * x.w + t;
  };
  const int kb = 1 + (int)blockIdx.z * MKB;
  const In x0 = load(max(kb - 1, 1)), x1 = load(kb);
  In nx = load(min(kb + 1, nk));
  Faces lo = faces(x1);
  float below = rrw_at(kb, x1, lo, faces(x0));
  if (cell && kb == 1) sto(rrw + wst, owc, 0.0f);
#pragma unroll
  for (int q = 0; q < MKB; ++q) {
    const int k = kb + q;
    if (k > nk) break;
    const In cu = nx;  // level k + 1 (the top level again above it, where rrw is 0)
    nx = load(min(k + 2, nk));
    const Faces hi = faces(cu);
    const float val = rrw_at(k + 1, cu, hi, lo);
    if (uface) sto(rru + (int64_t)k * ust, ow, lo.w);
    if (vface) sto(rrv + (int64_t)k * vst, ov, lo.s);
    if (cell) {
      sto(rrw + (int64_t)(k + 1) * wst, owc, val);
      float d = (lo.e - lo.w) * rdx + (lo.n - lo.s) * rdy;
      d = d + (val - below) * rdz;
      sto(divx + (int64_t)(k - 1) * mst, oc, (fabsf(d) < 1.0e-20f) ? 0.0f : d);
    }
    below = val;
    lo = hi;
  }
}

// Flat stretched column (solve2.F:493-520, 605-617 with terrain_flag=.false.):
// rru = rho0(1,1,k)*u, rrv = rho0(1,1,k)*v, rrw = rf0(1,1,k)*w (zero at both
// lids), divx's vertical term ((d*rdz)*mh(k)) and smeps 1e-30.
// The flat column's mass fluxes in one pass: rru = rho0(k)*u on faces
// 0..ni, rrv = rho0(k)*v on faces 0..nj, rrw = rf0(kf)*w on w levels 2..nk
// (0 at 1 and nk+1), and divx from them.  A cell forms its east and north
// faces' products itself (the same product its neighbour writes), so no
// thread reads a word another writes.
__global__ __launch_bounds__(256) void k_mom_mass_flat(
    const float* __restrict__ u, const float* __restrict__ v, const float* __restrict__ w,
    const float* __restrict__ rho0, const float* __restrict__ rf0, const float* __restrict__ mh,
    float* __restrict__ rru, float* __restrict__ rrv, float* __restrict__ rrw, float* __restrict__ divx, int ni,
    int nj, int nk, float rdx, float rdy, float rdz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // 0..ni
  const int j = blockIdx.y;                             // 0..nj
  if (i > ni) return;
  const int nxu = ux(ni), nyu = sy(nj), nxs = sx(ni), nyv = vy(nj);
  const int x = i + NG, y = j + NG;
  const int64_t plane = (int64_t)nj * ni;
  const int64_t ust = (int64_t)nyu * nxu, vst = (int64_t)nyv * nxs, wst = (int64_t)nyu * nxs;
  const int64_t uc = (int64_t)y * nxu + x, vc = (int64_t)y * nxs + x, wc = vc;
  const bool uface = j < nj, vface = i < ni, cell = i < ni && j < nj;
  auto rrw_at = [&](int kf) {
    return (kf <= 1 || kf > nk) ? 0.0f : rf0[(int64_t)(kf - 1) * plane] * w[(int64_t)kf * wst + wc];
  };
  const int kb = 1 + (int)blockIdx.z * MKB;
  // every word of the chunk requested first (levels past the top clamped to it), then formed
  float u0[MKB], u1[MKB], v0[MKB], v1[MKB], wk[MKB], rc[MKB], rf[MKB];
#pragma unroll
  for (int q = 0; q < MKB; ++q) {
    const int k = min(kb + q, nk), kf = min(k + 1, nk);
    rc[q] = rho0[(int64_t)(k - 1) * plane];
    rf[q] = rf0[(int64_t)(kf - 1) * plane];
    const float* uk = u + (int64_t)k * ust;
    const float* vk = v + (int64_t)k * vst;
    u0[q] = uface ? uk[uc] : 0.0f;
    v0[q] = vface ? vk[vc] : 0.0f;
    u1[q] = cell ? uk[uc + 1] : 0.0f;
    v1[q] = cell ? vk[vc + nxs] : 0.0f;
    wk[q] = cell ? w[(int64_t)kf * wst + wc] : 0.0f;
  }
  if (cell && kb == 1) rrw[wst + wc] = 0.0f;
  float below = cell ? rrw_at(kb) : 0.0f;
#pragma unroll
  for (int q = 0; q < MKB; ++q) {
    const int k = kb + q;
    if (k > nk) break;
    const float ru0 = rc[q] * u0[q], rv0 = rc[q] * v0[q];
    if (uface) rru[(int64_t)k * ust + uc] = ru0;
    if (vface) rrv[(int64_t)k * vst + vc] = rv0;
    if (cell) {
      const float ru1 = rc[q] * u1[q], rv1 = rc[q] * v1[q];
      const int kf = k + 1;
      const float val = (kf > nk) ? 0.0f : rf[q] * wk[q];
      rrw[(int64_t)kf * wst + wc] = val;
      float d = (ru1 - ru0) * rdx + (rv1 - rv0) * rdy;
      d = d + ((val - below) * rdz) * mh[k];
      divx[(int64_t)(k - 1) * plane + (int64_t)j * ni + i] = (fabsf(d) < 1.0e-30f) ? 0.0f : d;
      below = val;
    }
  }
}

// the words a column's vertical flux of u (stag 0) or v (stag 1) at w level kf
// takes beside its own: the pair of rrw and, where the face has a centred closure
// (kf = 2 and nk), the pair of c2
struct UvzWords { float r0, r1, c0, c1; };

template <int STAG>
GM1_DEV void uvz_c2(const MomArgs& a, int kf, int j, int i, UvzWords& w) {
  const int ni = a.ni, nj = a.nj;
  const float* c2k = a.c2 + (int64_t)(kf - 1) * nj * ni;
  const int jl = STAG == 0 ? clampi(j, nj) : clampi(j - 1, nj), jh = clampi(j, nj);
  const int il = STAG == 0 ? clampi(i - 1, ni) : clampi(i, ni), ih = clampi(i, ni);
  w.c0 = ldo(c2k, (uint32_t)(jl * ni + il) * 4u);
  w.c1 = ldo(c2k, (uint32_t)(jh * ni + ih) * 4u);
}

template <int STAG>
GM1_DEV UvzWords uvz_words(const MomArgs& a, int kf, int j, int i) {
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const int nxs = sx(ni), nys = sy(nj);
  UvzWords w;
  // the level's planes, each word at a 32-bit byte offset
  const float* R = a.rrw + (int64_t)kf * nys * nxs;
  if (STAG == 0) {
    const bool pw = per(a.obc, 0), pe = per(a.obc, 1);
    const int rb = (j + NG) * nxs + NG;
    w.r0 = ldo(R, (uint32_t)(rb + wc(i, ni, pw, pe)) * 4u);
    w.r1 = ldo(R, (uint32_t)(rb + wc(i - 1, ni, pw, pe)) * 4u);
  } else {
    const bool ps = per(a.obc, 2), pn = per(a.obc, 3);
    w.r0 = ldo(R, (uint32_t)((wc(j, nj, ps, pn) + NG) * nxs + i + NG) * 4u);
    w.r1 = ldo(R, (uint32_t)((wc(j - 1, nj, ps, pn) + NG) * nxs + i + NG) * 4u);
  }
  w.c0 = w.c1 = 0.0f;
  if (kf == 2 || kf == nk) uvz_c2<STAG>(a, kf, j, i, w);
  return w;
}

// the flux from those words and the column's (Q(level))
template <class Get>
GM1_DEV float uvz_g(const UvzWords& w, int kf, int nk, Get Q) {
  const float m = 0.5f * (w.r0 + w.r1);
  const float c2h = 0.5f * (w.c0 + w.c1);
  const float c1h = 1.0f - c2h;
  float r;
  if (kf == 2) {
    r = (m >= 0.0f) ? c1h * Q(1) + c2h * Q(2) : flx3(Q(3), Q(2), Q(1));
  } else if (kf == nk) {
    r = (m >= 0.0f) ? flx3(Q(nk - 2), Q(nk - 1), Q(nk)) : c1h * Q(nk - 1) + c2h * Q(nk);
  } else if (kf == 3) {
    r = (m >= 0.0f) ? flx3(Q(1), Q(2), Q(3)) : flx5(Q(5), Q(4), Q(3), Q(2), Q(1));
  } else if (kf == nk - 1) {
    r = (m >= 0.0f) ? flx5(Q(kf - 3), Q(kf - 2), Q(kf - 1), Q(kf), Q(kf + 1))
                    : flx3(Q(kf + 1), Q(kf), Q(kf - 1));
  } else {  // one value of the upwind words, whichever way the lanes' fluxes point
    const bool up = m >= 0.0f;
    const float q0 = Q(kf - 3), q1 = Q(kf - 2), q2 = Q(kf - 1), q3 = Q(kf), q4 = Q(kf + 1), q5 = Q(kf + 2);
    r = flx5(up ? q0 : q5, up ? q1 : q4, up ? q2 : q3, up ? q3 : q2, up ? q4 : q1);
  }
  return m * r;
}

// ... with the column read from the wind array
template <int STAG>
GM1_DEV float uvz(const MomArgs& a, int kf, int j, int i) {
  const int ni = a.ni, nj = a.nj;
  const float* q = (STAG == 0) ? a.u : a.v;
  const int nxq = (STAG == 0) ? ux(ni) : sx(ni);
  const int nyq = (STAG == 0) ? sy(nj) : vy(nj);
  const int64_t st = (int64_t)nyq * nxq;
  const float* col = q + (int64_t)(j + NG) * nxq + (i + NG);
  return uvz_g(uvz_words<STAG>(a, kf, j, i), kf, a.nk, [&](int lev) { return col[(int64_t)lev * st]; });
}


// ------------------------------------------------------------- tiled advu / advv
// advu / advv (cuda_momentum_advection5.py:1059-1064; the transport of
// _cpu_momentum_transport5, :753-1012) as a MTX x MTY tile marching a chunk
// of levels: per level the tile's wind plane (3-cell halo) is staged in LDS,
// every x and y flux point of the tile is formed once from it into LDS (the
// open fallback rows included), and the vertical flux comes from a 7-level
// register window of the thread's own column, the lower face's flux carried
// from the level below.  One lane per flux point: each lane forms the x and
// y points west and south of its own face (wavefront MTY-1 also the tile's
// east points, wavefront MTY-2 its north points); the byte offsets of the
// plane slots and of each point's mass-flux pair (periodic seams wrapped) are
// formed once into LDS.  A lane whose point lies outside reads word 0 and its
// flux is never consumed.
constexpr int MTX = 64, MTY = 8, MNT = MTX * MTY, MPX = MTX + 6;
constexpr int MPS = ((MTY + 6) * MPX + MNT - 1) / MNT;  // plane slots a lane
static_assert(MTX == 64, "a wavefront is one tile row");

// fifth-order upwind value of the six words q0..q5 around a flux point (q2|q3
// straddle it), times the mass flux m
GM1_DEV float point_flux(float m, float q0, float q1, float q2, float q3, float q4, float q5) {
  const bool up = m >= 0.0f;
  return m * flx5(up ? q0 : q5, up ? q1 : q4, up ? q2 : q3, up ? q3 : q2, up ? q4 : q1);
}

// u-momentum: faces f0 .. f0+nf-1 (tile columns), rows 0..nj-1 (tile rows).
// What bounds the three tiles is the latency of a level's words behind its barriers,
// so no lane skips a load (a word it has no use for is read at a clipped place and
// dropped: a wait then leaves exactly the younger loads in flight), every word is
// requested a level ahead, and a level has one barrier.  Measured against guarded
// loads, the z fluxes' words loaded where they are used and three barriers a level:
// u 442 -> 333, v 401 -> 340, w 420 -> 410 us at 640x768x80 (flat), 124 -> 78, 120 -> 78
// and 111 -> 77 at 320x320x80 (terrain).  Six waves per SIMD (three workgroups a CU), where the flat u
// and w tiles spill four and two registers; on the terrain family, whose u tile needs more, four
// waves are faster (82 -> 78 us at 320x320x80; flat, 364 against 333 at 640x768x80).
constexpr int advu_waves(bool flat) { return flat ? 6 : 4; }
template <bool FLAT>
__global__ __launch_bounds__(MNT) __attribute__((amdgpu_waves_per_eu(advu_waves(FLAT)))) void k_mom_advu_tile(MomArgs a, int f0, int nf, int kchunk, int nchunks) {
  // (plane and fluxes each in two buffers, levels taking turns)
  __shared__ float lp2[2][MPS * MNT];  // u: row r = padded row ja + r, col c = padded x fa + c (pitch MPX)
  __shared__ float lfx2[2][MTY][MTX + 1];  // x flux at centre fa - 1 + t
  __shared__ float lfy2[2][MTY + 1][MTX];  // y flux at corner row ja + r of face fa + t
  __shared__ uint32_t lpo[MPS * MNT];  // plane slot offsets within a level (read back by their own lane)
  __shared__ uint32_t lmo[6][MNT];     // mass-flux pairs: own x centre, own y corner, extra point
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const int tx = threadIdx.x % MTX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / MTX);  // (a wavefront is one row)
  const int gx = (nf + MTX - 1) / MTX, gy = (nj + MTY - 1) / MTY;
  const int tile = xcd_tile((int)blockIdx.x, gx * gy * nchunks);
  const int fa = f0 + (tile % gx) * MTX, ja = ((tile / gx) % gy) * MTY;
  const int kb = 1 + (tile / (gx * gy)) * kchunk, ke = min(nk, kb + kchunk - 1);
  const int fend = f0 + nf;  // one past the last face
  const bool pw = per(a.obc, 0), pe = per(a.obc, 1);
  const int nxu = ux(ni), nyu = sy(nj), nxv = sx(ni), nyv = vy(nj);
  const int64_t ust = (int64_t)nyu * nxu, vst = (int64_t)nyv * nxv, mst = (int64_t)nj * ni;
  const int f = fa + tx, j = ja + ty;
  const bool live = f < fend && j < nj;
  const int y = j + NG, x = f + NG;
  const bool xe = (ty == MTY - 1), yn = (ty == MTY - 2);  // the wavefronts forming the extra points
  {
#pragma unroll
    for (int q = 0; q < MPS; ++q) {
      const int sl = threadIdx.x + q * MNT;
      const int r = sl / MPX, c = sl % MPX;
      const int yy = ja + r, xx = fa + c;
      lpo[sl] = (sl < (MTY + 6) * MPX && yy < nyu && xx < nxu) ? (uint32_t)(yy * nxu + xx) * 4u : 0u;
    }
    // x centre cc of row jj: the rru faces wf(cc), wf(cc+1)
    auto xpair = [&](int slot, int cc, int jj) {
      const bool ok = jj < nj && cc < fend;
      const int rb = (jj + NG) * nxu + NG;
      lmo[slot][threadIdx.x] = ok ? (uint32_t)(rb + wf(cc, ni, pw, pe)) * 4u : 0u;
      lmo[slot + 1][threadIdx.x] = ok ? (uint32_t)(rb + wf(cc + 1, ni, pw, pe)) * 4u : 0u;
    };
    // y corner p of face ff: the rrv faces wc(ff), wc(ff-1)
    auto ypair = [&](int slot, int p, int ff) {
      const bool ok = p <= nj && ff < fend;
      const int rb = (p + NG) * nxv + NG;
      lmo[slot][threadIdx.x] = ok ? (uint32_t)(rb + wc(ff, ni, pw, pe)) * 4u : 0u;
      lmo[slot + 1][threadIdx.x] = ok ? (uint32_t)(rb + wc(ff - 1, ni, pw, pe)) * 4u : 0u;
    };
    xpair(0, f - 1, j);
    ypair(2, j, f);
    if (xe) xpair(4, fa - 1 + MTX, ja + tx);  // lanes tx < MTY are read
    else if (yn) ypair(4, ja + MTY, f);
    else lmo[4][threadIdx.x] = lmo[5][threadIdx.x] = 0u;
  }
  // a level's words sit at 32-bit byte offsets from the level's base
  const uint32_t ocol = live ? (uint32_t)(y * nxu + x) * 4u : 0u;  // this face in the u family
  float win[7];  // u(k-3 .. k+3) of this face's column
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    const int lev = kb - 3 + q;
    win[q] = (live && lev >= 0 && lev <= nk + 1) ? ldo(a.u + (int64_t)lev * ust, ocol) : 0.0f;
  }
  auto zf = [&](int kf, const float* b, const UvzWords& z) {  // b[0] = u(kf - 3)
    return uvz_g(z, kf, nk, [&](int lev) { return b[lev - (kf - 3)]; });
  };
  auto zwords = [&](int kf, float r0, float r1) {
    UvzWords z{r0, r1, 0.0f, 0.0f};
    if (kf == 2 || kf == nk) uvz_c2<0>(a, kf, j, f, z);
    return z;
  };
  float zlo = (live && kb >= 2) ? zf(kb, win, uvz_words<0>(a, kb, j, f)) : 0.0f;
  // the top z face's pair of rrw words
  const uint32_t oz0 = live ? (uint32_t)((j + NG) * nxv + NG + wc(f, ni, pw, pe)) * 4u : 0u;
  const uint32_t oz1 = live ? (uint32_t)((j + NG) * nxv + NG + wc(f - 1, ni, pw, pe)) * 4u : 0u;
  // One barrier a level: a level's fluxes are formed from its u plane while the
  // plane above it, requested a level earlier, is stored to the other buffer; the
  // mass-flux pairs (the top z face's included) are requested a level ahead too.
  // the scalar cells west and east of the face
  const uint32_t olo = live ? (uint32_t)(j * ni + wc(f - 1, ni, pw, pe)) * 4u : 0u;
  const uint32_t ohi = live ? (uint32_t)(j * ni + wc(f, ni, pw, pe)) * 4u : 0u;
  const float gzl = (!FLAT && live) ? a.gzu[(int64_t)j * (ni + 1) + f] : 0.0f;
  struct Lv {
    float m[6];
    float unext;
    float z0, z1;
  };
  float pln[MPS];  // a plane in flight
  auto fetch_plane = [&](int k) {
    const float* plane = a.u + (int64_t)k * ust;
#pragma unroll
    for (int q = 0; q < MPS; ++q) pln[q] = ldo(plane, lpo[threadIdx.x + q * MNT]);
  };
  auto store_plane = [&](int k) {
#pragma unroll
    for (int q = 0; q < MPS; ++q) lp2[k & 1][threadIdx.x + q * MNT] = pln[q];
  };
  auto fetch = [&](int k) {
    Lv v;
    const int lnext = k + 4;
    v.unext = ldo(a.u + (int64_t)min(lnext, nk + 1) * ust, ocol);
    const float* Rw = a.rrw + (int64_t)min(k + 1, nk) * nyu * nxv;
    v.z0 = ldo(Rw, oz0);
    v.z1 = ldo(Rw, oz1);
    const float* Ru = a.rru + (int64_t)k * ust;
    const float* Rv = a.rrv + (int64_t)k * vst;
    v.m[0] = ldo(Ru, lmo[0][threadIdx.x]);
    v.m[1] = ldo(Ru, lmo[1][threadIdx.x]);
    v.m[2] = ldo(Rv, lmo[2][threadIdx.x]);
    v.m[3] = ldo(Rv, lmo[3][threadIdx.x]);
    const float* R = xe ? Ru : Rv;
    v.m[4] = ldo(R, lmo[4][threadIdx.x]);
    v.m[5] = ldo(R, lmo[5][threadIdx.x]);
    return v;
  };
  // x point (row r, centre fa-1+t): the mean of the two rru faces times u's
  // fifth-order upwind value
  auto xflux = [&](int k, int r, int t, float m0, float m1) {
    const float m = 0.5f * (m0 + m1);
    const float* L = lp2[k & 1] + (r + 3) * MPX + t;  // L[c] = u at padded x (cc + NG) - 2 + c
    lfx2[k & 1][r][t] = point_flux(m, L[0], L[1], L[2], L[3], L[4], L[5]);
  };
  // y point (corner row p = ja+r of face ff = fa+t); on an open south/north
  // side an inflowing edge corner takes the next row's flux
  auto yflux = [&](int k, int r, int t, float m0, float m1) {
    const int p = ja + r, ff = fa + t;
    const float mt = m0 + m1;
    int pb = p;
    if (p == 0 && opn(a.obc, 2) && mt >= 0.0f) pb = 1;
    else if (p == nj && opn(a.obc, 3) && mt <= 0.0f) pb = nj - 1;
    float m;
    if (pb == p) {
      m = 0.5f * mt;
    } else {  // (p is 0 or nj, so the point lies inside when its face does)
      const float* Rb = a.rrv + (int64_t)k * vst;
      const int rb = (pb + NG) * nxv + NG;
      m = (ff < fend) ? 0.5f * (ldo(Rb, (uint32_t)(rb + wc(ff, ni, pw, pe)) * 4u) +
                                ldo(Rb, (uint32_t)(rb + wc(ff - 1, ni, pw, pe)) * 4u))
                      : 0.0f;
    }
    const float* L = lp2[k & 1] + (pb - ja) * MPX + t + 3;  // u at padded row pb + NG - 3 + q
    lfy2[k & 1][r][t] = point_flux(m, L[0], L[MPX], L[2 * MPX], L[3 * MPX], L[4 * MPX], L[5 * MPX]);
  };
  fetch_plane(kb);
  Lv nx = fetch(kb);
  store_plane(kb);
  fetch_plane(min(kb + 1, ke));
  __syncthreads();
  for (int k = kb; k <= ke; ++k) {
    const auto& lfx = lfx2[k & 1];
    const auto& lfy = lfy2[k & 1];
    const Lv cu = nx;
    // this level's point words, requested before its fluxes are formed
    float e_dxe = 0.0f, e_dxw = 0.0f, e_sc0 = 0.0f, e_rw = 0.0f, e_re = 0.0f, e_ten = 0.0f;
    const int64_t lm = (int64_t)(k - 1) * mst;
    e_dxe = ldo(a.divx + lm, ohi);
    e_dxw = ldo(a.divx + lm, olo);
    if (FLAT) {
      e_sc0 = a.rr0[lm];
    } else {
      e_sc0 = gzl;
      e_rw = ldo(a.rho0 + lm, olo);
      e_re = ldo(a.rho0 + lm, ohi);
    }
    e_ten = ldo((a.zero_held ? a.u : a.u1 ? a.u1 : a.uten) + (int64_t)k * ust, ocol);  // (unread when the held tendencies are zero)
    nx = fetch(min(k + 1, ke));
    xflux(k, ty, tx, cu.m[0], cu.m[1]);
    yflux(k, ty, tx, cu.m[2], cu.m[3]);
    if (xe) {
      if (tx < MTY) xflux(k, tx, MTX, cu.m[4], cu.m[5]);
    } else if (yn) {
      yflux(k, MTY, tx, cu.m[4], cu.m[5]);
    }
    float zhi = 0.0f;
    if (live && k + 1 <= nk) zhi = zf(k + 1, win + 1, zwords(k + 1, cu.z0, cu.z1));
    if (k < ke) store_plane(k + 1);  // (the buffer was last read before the barrier below of the level below)
    fetch_plane(min(k + 2, ke));
    __syncthreads();
    if (live) {
      const int west = wc(f - 1, ni, pw, pe), east = wc(f, ni, pw, pe);
      float ax = (-(lfx[ty][tx + 1] - lfx[ty][tx])) * a.rdx;
      float ay = (-(lfy[ty + 1][tx] - lfy[ty][tx])) * a.rdy;
      const float uc = win[3];
      if (j == 0 && opn(a.obc, 2)) {
        const float* R0 = a.rrv + ix3(k, NG, 0, nyv, nxv);
        const float* R1 = a.rrv + ix3(k, NG + 1, 0, nyv, nxv);
        const float m = R0[east + NG] + R0[west + NG];
        if (m >= 0.0f) {
          const float c = (R1[west + NG] - R0[west + NG]) + (R1[east + NG] - R0[east + NG]);
          ay = FLAT ? ay - (((uc * 0.5f) * c) * a.rdy) * a.vh[y] : ay - (uc * 0.5f) * (c * (a.rdy * a.vh[y]));
        }
      } else if (j == nj - 1 && opn(a.obc, 3)) {
        const float* RN = a.rrv + ix3(k, NG + nj, 0, nyv, nxv);
        const float* R0 = a.rrv + ix3(k, y, 0, nyv, nxv);
        const float* R1 = a.rrv + ix3(k, y + 1, 0, nyv, nxv);
        const float m = RN[east + NG] + RN[west + NG];
        if (m <= 0.0f) {
          const float c = (R1[west + NG] - R0[west + NG]) + (R1[east + NG] - R0[east + NG]);
          ay = FLAT ? ay - (((uc * 0.5f) * c) * a.rdy) * a.vh[y] : ay - (uc * 0.5f) * (c * (a.rdy * a.vh[y]));
        }
      }
      float az;
      if (k == 1) az = (-zhi) * a.rdz;
      else if (k == nk) az = zlo * a.rdz;
      else az = (-(zhi - zlo)) * a.rdz;
      if constexpr (FLAT) az = az * a.flat[k];
      float tot = (ax + ay) + az;
      tot = tot + uc * (0.5f * (e_dxe + e_dxw));
      const float sc = FLAT ? e_sc0 : e_sc0 / (0.5f * (e_rw + e_re));
      sto(a.uten + (int64_t)k * ust, ocol, (a.zero_held ? 0.0f : e_ten) + tot * sc);
    }
    zlo = zhi;
#pragma unroll
    for (int q = 0; q < 6; ++q) win[q] = win[q + 1];
    win[6] = (k + 4 <= nk + 1) ? cu.unext : 0.0f;
  }
}

// v-momentum: faces g0 .. g0+nr-1 (tile rows), columns 0..ni-1 (tile columns)
template <bool FLAT>
__global__ __launch_bounds__(MNT) __attribute__((amdgpu_waves_per_eu(6))) void k_mom_advv_tile(MomArgs a, int g0, int nr, int kchunk, int nchunks) {
  // (plane and fluxes each in two buffers, levels taking turns)
  __shared__ float lp2[2][MPS * MNT];  // v: row r = padded row ga + r, col c = padded x ia + c (pitch MPX)
  __shared__ float lfx2[2][MTY][MTX + 1];  // x flux at corner column ia + t of face row ga + r
  __shared__ float lfy2[2][MTY + 1][MTX];  // y flux at centre ga - 1 + r of column ia + t
  __shared__ uint32_t lpo[MPS * MNT];  // plane slot offsets within a level (read back by their own lane)
  __shared__ uint32_t lmo[6][MNT];     // mass-flux pairs: own x corner, own y centre, extra point
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const int tx = threadIdx.x % MTX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / MTX);  // (a wavefront is one row)
  const int gx = (ni + MTX - 1) / MTX, gy = (nr + MTY - 1) / MTY;
  const int tile = xcd_tile((int)blockIdx.x, gx * gy * nchunks);
  const int ia = (tile % gx) * MTX, ga = g0 + ((tile / gx) % gy) * MTY;
  const int kb = 1 + (tile / (gx * gy)) * kchunk, ke = min(nk, kb + kchunk - 1);
  const int gend = g0 + nr;
  const bool ps = per(a.obc, 2), pn = per(a.obc, 3);
  const int nxu = ux(ni), nyu = sy(nj), nxv = sx(ni), nyv = vy(nj);
  const int64_t vst = (int64_t)nyv * nxv, ust = (int64_t)nyu * nxu, mst = (int64_t)nj * ni;
  const int i = ia + tx, g = ga + ty;
  const bool live = i < ni && g < gend;
  const int y = g + NG, x = i + NG;
  const bool xe = (ty == MTY - 1), yn = (ty == MTY - 2);  // the wavefronts forming the extra points
  {
#pragma unroll
    for (int q = 0; q < MPS; ++q) {
      const int sl = threadIdx.x + q * MNT;
      const int r = sl / MPX, c = sl % MPX;
      const int yy = ga + r, xx = ia + c;
      lpo[sl] = (sl < (MTY + 6) * MPX && yy < nyv && xx < nxv) ? (uint32_t)(yy * nxv + xx) * 4u : 0u;
    }
    // x corner p of face row gg: the rru faces of rows wc(gg), wc(gg-1)
    auto xpair = [&](int slot, int p, int gg) {
      const bool ok = gg < gend && p <= ni;
      const int rn = wc(gg, nj, ps, pn) + NG, rs = wc(gg - 1, nj, ps, pn) + NG;
      lmo[slot][threadIdx.x] = ok ? (uint32_t)(rn * nxu + p + NG) * 4u : 0u;
      lmo[slot + 1][threadIdx.x] = ok ? (uint32_t)(rs * nxu + p + NG) * 4u : 0u;
    };
    // y centre pc of column ii: the rrv faces of rows wf(pc), wf(pc+1)
    auto ypair = [&](int slot, int pc, int ii) {
      const bool ok = ii < ni && pc < gend;
      lmo[slot][threadIdx.x] = ok ? (uint32_t)((wf(pc, nj, ps, pn) + NG) * nxv + ii + NG) * 4u : 0u;
      lmo[slot + 1][threadIdx.x] = ok ? (uint32_t)((wf(pc + 1, nj, ps, pn) + NG) * nxv + ii + NG) * 4u : 0u;
    };
    xpair(0, i, g);
    ypair(2, g - 1, i);
    if (xe) xpair(4, ia + MTX, ga + tx);  // lanes tx < MTY are read
    else if (yn) ypair(4, ga - 1 + MTY, i);
    else lmo[4][threadIdx.x] = lmo[5][threadIdx.x] = 0u;
  }
  // a level's words sit at 32-bit byte offsets from the level's base
  const uint32_t ocol = live ? (uint32_t)(y * nxv + x) * 4u : 0u;  // this face in the v family
  float win[7];
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    const int lev = kb - 3 + q;
    win[q] = (live && lev >= 0 && lev <= nk + 1) ? ldo(a.v + (int64_t)lev * vst, ocol) : 0.0f;
  }
  auto zf = [&](int kf, const float* b, const UvzWords& z) {  // b[0] = v(kf - 3)
    return uvz_g(z, kf, nk, [&](int lev) { return b[lev - (kf - 3)]; });
  };
  auto zwords = [&](int kf, float r0, float r1) {
    UvzWords z{r0, r1, 0.0f, 0.0f};
    if (kf == 2 || kf == nk) uvz_c2<1>(a, kf, g, i, z);
    return z;
  };
  float zlo = (live && kb >= 2) ? zf(kb, win, uvz_words<1>(a, kb, g, i)) : 0.0f;
  // the top z face's pair of rrw words
  const uint32_t oz0 = live ? (uint32_t)((wc(g, nj, ps, pn) + NG) * nxv + i + NG) * 4u : 0u;
  const uint32_t oz1 = live ? (uint32_t)((wc(g - 1, nj, ps, pn) + NG) * nxv + i + NG) * 4u : 0u;
  // One barrier a level and the words requested a level ahead, as in the u tile.
  // the scalar cells south and north of the face
  const uint32_t olo = live ? (uint32_t)(wc(g - 1, nj, ps, pn) * ni + i) * 4u : 0u;
  const uint32_t ohi = live ? (uint32_t)(wc(g, nj, ps, pn) * ni + i) * 4u : 0u;
  const float gzl = (!FLAT && live) ? a.gzv[(int64_t)g * ni + i] : 0.0f;
  struct Lv {
    float m[6];
    float vnext;
    float z0, z1;
  };
  float pln[MPS];  // a plane in flight
  auto fetch_plane = [&](int k) {
    const float* plane = a.v + (int64_t)k * vst;
#pragma unroll
    for (int q = 0; q < MPS; ++q) pln[q] = ldo(plane, lpo[threadIdx.x + q * MNT]);
  };
  auto store_plane = [&](int k) {
#pragma unroll
    for (int q = 0; q < MPS; ++q) lp2[k & 1][threadIdx.x + q * MNT] = pln[q];
  };
  auto fetch = [&](int k) {
    Lv v;
    const int lnext = k + 4;
    v.vnext = ldo(a.v + (int64_t)min(lnext, nk + 1) * vst, ocol);
    const float* Rw = a.rrw + (int64_t)min(k + 1, nk) * nyu * nxv;
    v.z0 = ldo(Rw, oz0);
    v.z1 = ldo(Rw, oz1);
    const float* Ru = a.rru + (int64_t)k * ust;
    const float* Rv = a.rrv + (int64_t)k * vst;
    v.m[0] = ldo(Ru, lmo[0][threadIdx.x]);
    v.m[1] = ldo(Ru, lmo[1][threadIdx.x]);
    v.m[2] = ldo(Rv, lmo[2][threadIdx.x]);
    v.m[3] = ldo(Rv, lmo[3][threadIdx.x]);
    const float* R = xe ? Ru : Rv;
    v.m[4] = ldo(R, lmo[4][threadIdx.x]);
    v.m[5] = ldo(R, lmo[5][threadIdx.x]);
    return v;
  };
  // x point (face row gg = ga+r, corner column p = ia+t); on an open
  // west/east side an inflowing edge corner takes the next column's
  auto xflux = [&](int k, int r, int t, float m0, float m1) {
    const int p = ia + t, gg = ga + r;
    const float mt = m0 + m1;
    int pb = p;
    if (p == 0 && opn(a.obc, 0) && mt >= 0.0f) pb = 1;
    else if (p == ni && opn(a.obc, 1) && mt <= 0.0f) pb = ni - 1;
    float m;
    if (pb == p) {
      m = 0.5f * mt;
    } else {  // (p is 0 or ni, so the point lies inside when its row does)
      const float* R = a.rru + (int64_t)k * ust;
      const int rn = wc(gg, nj, ps, pn) + NG, rs = wc(gg - 1, nj, ps, pn) + NG;
      m = (gg < gend) ? 0.5f * (ldo(R, (uint32_t)(rn * nxu + pb + NG) * 4u) +
                                ldo(R, (uint32_t)(rs * nxu + pb + NG) * 4u))
                      : 0.0f;
    }
    const float* L = lp2[k & 1] + (r + 3) * MPX + (pb - ia);  // L[c] = v at padded x (pb + NG) - 3 + c
    lfx2[k & 1][r][t] = point_flux(m, L[0], L[1], L[2], L[3], L[4], L[5]);
  };
  // y point (centre pc = ga-1+r of column ia+t)
  auto yflux = [&](int k, int r, int t, float m0, float m1) {
    const float m = 0.5f * (m0 + m1);
    // LDS row of v at padded row (pc + NG) - 2 is pc + 1 - ga = r
    const float* L = lp2[k & 1] + r * MPX + t + 3;
    lfy2[k & 1][r][t] = point_flux(m, L[0], L[MPX], L[2 * MPX], L[3 * MPX], L[4 * MPX], L[5 * MPX]);
  };
  fetch_plane(kb);
  Lv nx = fetch(kb);
  store_plane(kb);
  fetch_plane(min(kb + 1, ke));
  __syncthreads();
  for (int k = kb; k <= ke; ++k) {
    const auto& lfx = lfx2[k & 1];
    const auto& lfy = lfy2[k & 1];
    const Lv cu = nx;
    // this level's point words, requested before its fluxes are formed
    float e_dxn = 0.0f, e_dxs = 0.0f, e_sc0 = 0.0f, e_rs = 0.0f, e_rn = 0.0f, e_ten = 0.0f;
    const int64_t lm = (int64_t)(k - 1) * mst;
    e_dxn = ldo(a.divx + lm, ohi);
    e_dxs = ldo(a.divx + lm, olo);
    if (FLAT) {
      e_sc0 = a.rr0[lm];
    } else {
      e_sc0 = gzl;
      e_rs = ldo(a.rho0 + lm, olo);
      e_rn = ldo(a.rho0 + lm, ohi);
    }
    e_ten = ldo((a.zero_held ? a.v : a.v1 ? a.v1 : a.vten) + (int64_t)k * vst, ocol);  // (unread when the held tendencies are zero)
    nx = fetch(min(k + 1, ke));
    xflux(k, ty, tx, cu.m[0], cu.m[1]);
    yflux(k, ty, tx, cu.m[2], cu.m[3]);
    if (xe) {
      if (tx < MTY) xflux(k, tx, MTX, cu.m[4], cu.m[5]);
    } else if (yn) {
      yflux(k, MTY, tx, cu.m[4], cu.m[5]);
    }
    float zhi = 0.0f;
    if (live && k + 1 <= nk) zhi = zf(k + 1, win + 1, zwords(k + 1, cu.z0, cu.z1));
    if (k < ke) store_plane(k + 1);  // (the buffer was last read before the barrier below of the level below)
    fetch_plane(min(k + 2, ke));
    __syncthreads();
    if (live) {
      const int south = wc(g - 1, nj, ps, pn), north = wc(g, nj, ps, pn);
      float ax = (-(lfx[ty][tx + 1] - lfx[ty][tx])) * a.rdx;
      float ay = (-(lfy[ty + 1][tx] - lfy[ty][tx])) * a.rdy;
      const float vc = win[3];
      const float* Rs = a.rru + ix3(k, south + NG, 0, nyu, nxu);
      const float* Rn = a.rru + ix3(k, north + NG, 0, nyu, nxu);
      if (i == 0 && opn(a.obc, 0)) {
        const float m = Rn[NG] + Rs[NG];
        if (m >= 0.0f) {
          const float c = (Rs[NG + 1] - Rs[NG]) + (Rn[NG + 1] - Rn[NG]);
          ax = FLAT ? ax - (((vc * 0.5f) * c) * a.rdx) * a.uh[NG] : ax - (vc * 0.5f) * (c * (a.rdx * a.uh[NG]));
        }
      } else if (i == ni - 1 && opn(a.obc, 1)) {
        const float m = Rn[NG + ni] + Rs[NG + ni];
        if (m <= 0.0f) {
          const float c = (Rs[x + 1] - Rs[x]) + (Rn[x + 1] - Rn[x]);
          ax = FLAT ? ax - (((vc * 0.5f) * c) * a.rdx) * a.uh[x] : ax - (vc * 0.5f) * (c * (a.rdx * a.uh[x]));
        }
      }
      float az;
      if (k == 1) az = (-zhi) * a.rdz;
      else if (k == nk) az = zlo * a.rdz;
      else az = (-(zhi - zlo)) * a.rdz;
      if constexpr (FLAT) az = az * a.flat[k];
      float tot = (ax + ay) + az;
      tot = tot + vc * (0.5f * (e_dxn + e_dxs));
      const float sc = FLAT ? e_sc0 : e_sc0 / (0.5f * (e_rs + e_rn));
      sto(a.vten + (int64_t)k * vst, ocol, (a.zero_held ? 0.0f : e_ten) + tot * sc);
    }
    zlo = zhi;
#pragma unroll
    for (int q = 0; q < 6; ++q) win[q] = win[q + 1];
    win[6] = (k + 4 <= nk + 1) ? cu.vnext : 0.0f;
  }
}

template <bool FLAT>
void launch_advu_tile(const MomArgs& a, int f0, int nf, hipStream_t s) {
  int kchunk = 1;
  const int tiles = ((nf + MTX - 1) / MTX) * ((a.nj + MTY - 1) / MTY);
  const int chunks = tile_chunks(tiles, a.nk, advu_waves(FLAT) / 2, &kchunk);
  GM1_TIMED(TK_MOM_ADVU, s, hipLaunchKernelGGL(k_mom_advu_tile<FLAT>, dim3(tiles * chunks), dim3(MNT), 0, s, a, f0,
                                               nf, kchunk, chunks));
}

template <bool FLAT>
void launch_advv_tile(const MomArgs& a, int g0, int nr, hipStream_t s) {
  int kchunk = 1;
  const int tiles = ((a.ni + MTX - 1) / MTX) * ((nr + MTY - 1) / MTY);
  const int chunks = tile_chunks(tiles, a.nk, 3, &kchunk);
  GM1_TIMED(TK_MOM_ADVV, s, hipLaunchKernelGGL(k_mom_advv_tile<FLAT>, dim3(tiles * chunks), dim3(MNT), 0, s, a, g0,
                                               nr, kchunk, chunks));
}

// ------------------------------------------------------------- advw
// vertical flux of w at scalar level k (wz) with the column read through Q
template <class Get>
GM1_DEV float wz_g(float m, int k, int nk, Get Q) {
  float r;
  if (k == 1) r = (m >= 0.0f) ? 0.5f * (Q(1) + Q(2)) : flx3(Q(3), Q(2), Q(1));
  else if (k == 2) r = (m >= 0.0f) ? flx3(Q(1), Q(2), Q(3)) : flx5(Q(5), Q(4), Q(3), Q(2), Q(1));
  else if (k == nk - 1) r = (m >= 0.0f) ? flx5(Q(k - 2), Q(k - 1), Q(k), Q(k + 1), Q(k + 2)) : flx3(Q(k + 2), Q(k + 1), Q(k));
  else if (k == nk) r = (m >= 0.0f) ? flx3(Q(k - 1), Q(k), Q(k + 1)) : 0.5f * (Q(k) + Q(k + 1));
  else {  // one value of the upwind words, whichever way the lanes' fluxes point
    const bool up = m >= 0.0f;
    const float q0 = Q(k - 2), q1 = Q(k - 1), q2 = Q(k), q3 = Q(k + 1), q4 = Q(k + 2), q5 = Q(k + 3);
    r = flx5(up ? q0 : q5, up ? q1 : q4, up ? q2 : q3, up ? q3 : q2, up ? q4 : q1);
  }
  return m * r;
}

// advw (cuda_momentum_advection5.py:1064, cm1_mom5_advw_v1; the transport of
// _cpu_momentum_transport5, :871-1012) as a MTX x MTY tile of cells marching a
// chunk of w levels 2..nk: per level the tile's w plane (3-cell halo) and its
// c2 plane (1-cell halo, clamped as the face weights clamp) are staged in LDS,
// every x and y face flux of the tile is formed once into LDS together with
// its mass flux (the open sides' fallback to the neighbouring face reads it),
// and the vertical flux comes from a 7-level window of the thread's own
// column, the lower flux, rru/rrv of the level below, divx and dum8 carried.
// One lane per face, as in the u and v tiles: each lane forms its cell's west
// x face and south y face (wavefront MTY-1 also the tile's east faces,
// wavefront MTY-2 its north faces); the plane slots' byte offsets are formed
// once into LDS.
constexpr int WLX = MTX + 6, WLY = MTY + 6, WCX = MTX + 2;
constexpr int WPS = (WLY * WLX + MNT - 1) / MNT, WCS = ((MTY + 2) * WCX + MNT - 1) / MNT;
template <bool FLAT>
__global__ __launch_bounds__(MNT) __attribute__((amdgpu_waves_per_eu(6)))
void k_mom_advw_tile(MomArgs a, int kchunk, int nchunks) {
  // (planes and fluxes each in two buffers, levels taking turns)
  __shared__ float lw2[2][WPS * MNT];       // w: row r = padded row ja + r, col c = padded x ia + c (pitch WLX)
  __shared__ float lc2[2][WCS * MNT];       // c2 of cells (clamp(ja-1+r), clamp(ia-1+c)) at level kf-1 (pitch WCX)
  __shared__ float lfx2[2][MTY][MTX + 1], lmx2[2][MTY][MTX + 1];  // x flux and mass flux at face ia + t
  __shared__ float lfy2[2][MTY + 1][MTX], lmy2[2][MTY + 1][MTX];  // y flux and mass flux at face ja + r
  __shared__ uint32_t lpo[WPS * MNT], lco[WCS * MNT];     // slot offsets (read back by their own lane)
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const int tx = threadIdx.x % MTX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / MTX);  // (a wavefront is one row)
  const int gx = (ni + MTX - 1) / MTX, gy = (nj + MTY - 1) / MTY;
  const int tile = xcd_tile((int)blockIdx.x, gx * gy * nchunks);
  const int ia = (tile % gx) * MTX, ja = ((tile / gx) % gy) * MTY;
  const int kb = 2 + (tile / (gx * gy)) * kchunk, ke = min(nk, kb + kchunk - 1);
  const int i = ia + tx, j = ja + ty;
  const bool live = i < ni && j < nj;
  const int nxu = ux(ni), nyu = sy(nj), nxs = sx(ni), nys = sy(nj), nyv = vy(nj);
  const int64_t wst = (int64_t)nys * nxs, plane = (int64_t)nj * ni;
  const int64_t ust = (int64_t)nyu * nxu, vst = (int64_t)nyv * nxs;
  const int y = j + NG, x = i + NG;
  const int64_t h = (int64_t)j * ni + i;
  const bool xe = (ty == MTY - 1), yn = (ty == MTY - 2);  // the wavefronts forming the extra faces
  // a level's words sit at 32-bit byte offsets from the level's base
  const uint32_t oh = live ? (uint32_t)(j * ni + i) * 4u : 0u, ow = live ? (uint32_t)(y * nxs + x) * 4u : 0u;
  // the lane's faces: west x face (i, j), south y face (i, j), and the extra face
  const uint32_t orx = (j < nj && i <= ni) ? (uint32_t)(y * nxu + x) * 4u : 0u;
  const uint32_t ory = (i < ni && j <= nj) ? (uint32_t)(y * nxs + x) * 4u : 0u;
  uint32_t ore = 0u;
  if (xe && tx < MTY && ja + tx < nj && ia + MTX <= ni) ore = (uint32_t)((ja + tx + NG) * nxu + ia + MTX + NG) * 4u;
  if (yn && ja + MTY <= nj && i < ni) ore = (uint32_t)((ja + MTY + NG) * nxs + x) * 4u;
#pragma unroll
  for (int q = 0; q < WPS; ++q) {
    const int sl = threadIdx.x + q * MNT;
    const int r = sl / WLX, c = sl % WLX;
    const int yy = ja + r, xx = ia + c;
    lpo[sl] = (sl < WLY * WLX && yy < nys && xx < nxs) ? (uint32_t)(yy * nxs + xx) * 4u : 0u;
  }
#pragma unroll
  for (int q = 0; q < WCS; ++q) {
    const int sl = threadIdx.x + q * MNT;
    const int r = sl / WCX, c = sl % WCX;
    lco[sl] = (sl < (MTY + 2) * WCX) ? (uint32_t)(clampi(ja - 1 + r, nj) * ni + clampi(ia - 1 + c, ni)) * 4u : 0u;
  }
  auto rface = [&](int k, uint32_t off, bool xface) {  // rru (x face) or rrv (y face) at level k
    return xface ? ldo(a.rru + (int64_t)k * ust, off) : ldo(a.rrv + (int64_t)k * vst, off);
  };
  float win[7];  // w(kf-3 .. kf+3) of this cell's column
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    const int lev = kb - 3 + q;
    win[q] = (live && lev >= 0 && lev <= nk + 2) ? ldo(a.w + (int64_t)lev * wst, ow) : 0.0f;
  }
  // the faces' mass fluxes of the level below
  float rxp = rface(kb - 1, orx, true), ryp = rface(kb - 1, ory, false);
  float rep = (xe || yn) ? rface(kb - 1, ore, xe) : 0.0f;
  float rrw_lo = 0.0f, rrw_hi = 0.0f, zlo = 0.0f, dxlo = 0.0f, d8lo = 0.0f;
  if (live) {
    rrw_lo = ldo(a.rrw + (int64_t)(kb - 1) * wst, ow);
    rrw_hi = ldo(a.rrw + (int64_t)kb * wst, ow);
    zlo = wz_g(0.5f * (rrw_lo + rrw_hi), kb - 1, nk, [&](int lev) { return win[lev - (kb - 3)]; });
    dxlo = ldo(a.divx + (int64_t)(kb - 2) * plane, oh);
    if (FLAT && a.dum8) d8lo = ldo(a.dum8 + (int64_t)(kb - 1) * wst, ow);
  }
  const float uhx = live ? a.uh[x] : 0.0f, vhy = live ? a.vh[y] : 0.0f;
  const float gzc = (!FLAT && live) ? a.gz[h] : 0.0f;
  struct Lv {
    float rx, ry, re;
    float wnext, rrwn, divx, base, d8, c1, rrf0;
  };
  // one barrier a level, as in the u and v tiles: the planes above are stored while
  // a level's fluxes are formed
  float pln[WPS], pc2[WCS];  // planes in flight
  auto fetch_plane = [&](int kf) {
    const float* wp = a.w + (int64_t)kf * wst;
#pragma unroll
    for (int q = 0; q < WPS; ++q) pln[q] = ldo(wp, lpo[threadIdx.x + q * MNT]);
    const float* c2k = a.c2 + (int64_t)(kf - 1) * plane;
#pragma unroll
    for (int q = 0; q < WCS; ++q) pc2[q] = ldo(c2k, lco[threadIdx.x + q * MNT]);
  };
  auto store_plane = [&](int kf) {
#pragma unroll
    for (int q = 0; q < WPS; ++q) lw2[kf & 1][threadIdx.x + q * MNT] = pln[q];
#pragma unroll
    for (int q = 0; q < WCS; ++q) lc2[kf & 1][threadIdx.x + q * MNT] = pc2[q];
  };
  auto fetch = [&](int kf) {
    Lv v;
    v.rx = rface(kf, orx, true);
    v.ry = rface(kf, ory, false);
    v.re = ldo(xe ? a.rru + (int64_t)kf * ust : a.rrv + (int64_t)kf * vst, ore);
    v.wnext = ldo(a.w + (int64_t)min(kf + 4, nk + 2) * wst, ow);
    v.rrwn = ldo(a.rrw + (int64_t)(kf + 1) * wst, ow);
    v.divx = ldo(a.divx + (int64_t)(kf - 1) * plane, oh);
    v.base = ldo((a.zero_held ? a.w : a.w1 ? a.w1 : a.wten) + (int64_t)kf * wst, ow);  // (unread when the held tendencies are zero)
    v.d8 = v.c1 = v.rrf0 = 0.0f;
    if (!FLAT) v.rrf0 = ldo(a.rrf0 + (int64_t)(kf - 1) * plane, oh);
    if (FLAT) {  // (dum8 and c1 unread without a dum8)
      v.d8 = ldo((a.dum8 ? a.dum8 : a.rrw) + (int64_t)kf * wst, ow);
      v.c1 = ldo((a.dum8 ? a.c1 : a.divx) + (int64_t)(kf - 1) * plane, oh);
    }
    return v;
  };
  // x face ia + t of row ja + r (wfx_base)
  auto xface = [&](int b, int r, int t, float mt, float mb) {
    const float c2h = 0.5f * (lc2[b][(r + 1) * WCX + t] + lc2[b][(r + 1) * WCX + t + 1]);
    const float c1h = 1.0f - c2h;
    const float m = c2h * mt + c1h * mb;
    const float* L = lw2[b] + (r + 3) * WLX + t;  // L[c] = w at padded x (ia + t + NG) - 3 + c
    lfx2[b][r][t] = point_flux(m, L[0], L[1], L[2], L[3], L[4], L[5]);
    lmx2[b][r][t] = m;
  };
  // y face ja + r of column ia + t (wfy_base)
  auto yface = [&](int b, int r, int t, float mt, float mb) {
    const float c2h = 0.5f * (lc2[b][r * WCX + t + 1] + lc2[b][(r + 1) * WCX + t + 1]);
    const float c1h = 1.0f - c2h;
    const float m = c2h * mt + c1h * mb;
    const float* L = lw2[b] + r * WLX + t + 3;
    lfy2[b][r][t] = point_flux(m, L[0], L[WLX], L[2 * WLX], L[3 * WLX], L[4 * WLX], L[5 * WLX]);
    lmy2[b][r][t] = m;
  };
  const bool pw = opn(a.obc, 0), pe = opn(a.obc, 1), ps = opn(a.obc, 2), pn = opn(a.obc, 3);
  fetch_plane(kb);
  Lv nx = fetch(kb);
  store_plane(kb);
  fetch_plane(min(kb + 1, ke));
  __syncthreads();
  for (int kf = kb; kf <= ke; ++kf) {
    const int b = kf & 1;
    const auto &lfx = lfx2[b], &lmx = lmx2[b];
    const auto &lfy = lfy2[b], &lmy = lmy2[b];
    const Lv cu = nx;
    nx = fetch(min(kf + 1, ke));
    xface(b, ty, tx, cu.rx, rxp);
    yface(b, ty, tx, cu.ry, ryp);
    if (xe) {
      if (tx < MTY) xface(b, tx, MTX, cu.re, rep);
    } else if (yn) {
      yface(b, MTY, tx, cu.re, rep);
    }
    const float c2 = lc2[b][(ty + 1) * WCX + tx + 1];
    float zhi = 0.0f;
    if (live) zhi = wz_g(0.5f * (rrw_hi + cu.rrwn), kf, nk, [&](int lev) { return win[lev - (kf - 3)]; });
    if (kf < ke) store_plane(kf + 1);
    fetch_plane(min(kf + 2, ke));
    __syncthreads();
    if (live) {
      // the open sides take the neighbouring face's flux where the mass flux points inward
      float fw = lfx[ty][tx], fe = lfx[ty][tx + 1];
      if (i == 0 && pw && lmx[ty][0] >= 0.0f) fw = lfx[ty][1];
      if (i == ni - 1 && pe && lmx[ty][tx + 1] <= 0.0f) fe = lfx[ty][tx];
      float fs = lfy[ty][tx], fn = lfy[ty + 1][tx];
      if (j == 0 && ps && lmy[0][tx] >= 0.0f) fs = lfy[1][tx];
      if (j == nj - 1 && pn && lmy[ty + 1][tx] <= 0.0f) fn = lfy[ty][tx];
      float ax, ay;
      if (FLAT) {
        ax = ((-(fe - fw)) * a.rdx) * uhx;
        ay = ((-(fn - fs)) * a.rdy) * vhy;
      } else {
        ax = (-(fe - fw)) * (a.rdx * uhx);
        ay = (-(fn - fs)) * (a.rdy * vhy);
      }
      const float c1 = 1.0f - c2;
      const float wc0 = win[3];
      if (i == 0 && pw) {
        const float* Rt = a.rru + ix3(kf, y, 0, nyu, nxu);
        const float* Rb = a.rru + ix3(kf - 1, y, 0, nyu, nxu);
        const float m = c2 * Rt[NG] + c1 * Rb[NG];
        if (m >= 0.0f) {
          const float c = c1 * (Rb[NG + 1] - Rb[NG]) + c2 * (Rt[NG + 1] - Rt[NG]);
          ax = FLAT ? ax - ((wc0 * c) * a.rdx) * uhx : ax - wc0 * (c * (a.rdx * uhx));
        }
      } else if (i == ni - 1 && pe) {
        const float* Rt = a.rru + ix3(kf, y, 0, nyu, nxu);
        const float* Rb = a.rru + ix3(kf - 1, y, 0, nyu, nxu);
        const float m = c2 * Rt[NG + ni] + c1 * Rb[NG + ni];
        if (m <= 0.0f) {
          const float c = c1 * (Rb[x + 1] - Rb[x]) + c2 * (Rt[x + 1] - Rt[x]);
          ax = FLAT ? ax - ((wc0 * c) * a.rdx) * uhx : ax - wc0 * (c * (a.rdx * uhx));
        }
      }
      if (j == 0 && ps) {
        const float m = c2 * a.rrv[ix3(kf, NG, x, nyv, nxs)] + c1 * a.rrv[ix3(kf - 1, NG, x, nyv, nxs)];
        if (m >= 0.0f) {
          const float c = c1 * (a.rrv[ix3(kf - 1, NG + 1, x, nyv, nxs)] - a.rrv[ix3(kf - 1, NG, x, nyv, nxs)]) +
                          c2 * (a.rrv[ix3(kf, NG + 1, x, nyv, nxs)] - a.rrv[ix3(kf, NG, x, nyv, nxs)]);
          ay = FLAT ? ay - ((wc0 * c) * a.rdy) * vhy : ay - wc0 * (c * (a.rdy * vhy));
        }
      } else if (j == nj - 1 && pn) {
        const float m = c2 * a.rrv[ix3(kf, NG + nj, x, nyv, nxs)] + c1 * a.rrv[ix3(kf - 1, NG + nj, x, nyv, nxs)];
        if (m <= 0.0f) {
          const float c = c1 * (a.rrv[ix3(kf - 1, y + 1, x, nyv, nxs)] - a.rrv[ix3(kf - 1, y, x, nyv, nxs)]) +
                          c2 * (a.rrv[ix3(kf, y + 1, x, nyv, nxs)] - a.rrv[ix3(kf, y, x, nyv, nxs)]);
          ay = FLAT ? ay - ((wc0 * c) * a.rdy) * vhy : ay - wc0 * (c * (a.rdy * vhy));
        }
      }
      float az = (-(zhi - zlo)) * a.rdz;
      if (FLAT) az = az * a.flat[(nk + 2) + kf];
      float tot = (ax + ay) + az;
      tot = tot + wc0 * (c2 * cu.divx + c1 * dxlo);
      const float sc = FLAT ? a.rrf0[(int64_t)(kf - 1) * plane]
                            : cu.rrf0 * gzc;
      float* wt_k = a.wten + (int64_t)kf * wst;
      const float wt = (a.zero_held ? 0.0f : cu.base) + tot * sc;
      if (FLAT && a.dum8) sto(wt_k, ow, wt + (cu.c1 * d8lo + c2 * cu.d8));
      else sto(wt_k, ow, wt);
      d8lo = cu.d8;
    }
    zlo = zhi;
    rrw_hi = cu.rrwn;
    dxlo = cu.divx;
    rxp = cu.rx;
    ryp = cu.ry;
    rep = cu.re;
#pragma unroll
    for (int q = 0; q < 6; ++q) win[q] = win[q + 1];
    win[6] = (kf + 4 <= nk + 2) ? cu.wnext : 0.0f;
  }
}

template <bool FLAT>
void launch_advw_tile(const MomArgs& a, hipStream_t s) {
  int kchunk = 1;
  const int tiles = ((a.ni + MTX - 1) / MTX) * ((a.nj + MTY - 1) / MTY);
  const int chunks = tile_chunks(tiles, a.nk - 1, 3, &kchunk);
  GM1_TIMED(TK_MOM_ADVW, s, hipLaunchKernelGGL(k_mom_advw_tile<FLAT>, dim3(tiles * chunks), dim3(MNT), 0, s, a,
                                               kchunk, chunks));
}

// The held tendencies' words that no advection statement writes: u on the
// row j = nj and on the faces i = 0, ni; v on the column i = ni and the
// faces j = 0, nj; w on the column i = ni and the row j = nj of levels
// 2..nk (level 1 by k_seed_w_surface) -- the rest of k_seed_held's region
// (faces 0..ni, rows 0..nj, levels 1..nk) is seeded by the advection updates
// themselves.  A face both seeds and an update write is seeded first and
// overwritten in stream order.  Null held tendencies seed +0 (the zeroed
// held fields of a step without a solve1 contribution).
__global__ __launch_bounds__(256) void k_seed_edges(const float* __restrict__ u1, const float* __restrict__ v1,
                                                    const float* __restrict__ w1, float* __restrict__ ut,
                                                    float* __restrict__ vt, float* __restrict__ wt, int ni, int nj,
                                                    int nk) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y + 1;
  if (e < ni + 1 + 2 * nj) {  // u
    int i, j;
    if (e <= ni) { i = e; j = nj; }
    else if (e < ni + 1 + nj) { i = 0; j = e - (ni + 1); }
    else { i = ni; j = e - (ni + 1 + nj); }
    const int64_t p = ix3(k, j + NG, i + NG, sy(nj), ux(ni));
    ut[p] = u1 ? u1[p] : 0.0f;
  }
  if (e < nj + 1 + 2 * ni) {  // v
    int i, j;
    if (e <= nj) { i = ni; j = e; }
    else if (e < nj + 1 + ni) { i = e - (nj + 1); j = 0; }
    else { i = e - (nj + 1 + ni); j = nj; }
    const int64_t p = ix3(k, j + NG, i + NG, vy(nj), sx(ni));
    vt[p] = v1 ? v1[p] : 0.0f;
  }
  if (k >= 2 && e < nj + 1 + ni) {  // w above the surface
    const int i = (e <= nj) ? ni : e - (nj + 1), j = (e <= nj) ? e : nj;
    const int64_t p = ix3(k, j + NG, i + NG, sy(nj), sx(ni));
    wt[p] = w1 ? w1[p] : 0.0f;
  }
}

__global__ __launch_bounds__(256) void k_seed_w_surface(const float* __restrict__ w1, float* __restrict__ wt, int ni,
                                                        int nj) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (ni + 1) * (nj + 1)) return;
  const int i = e % (ni + 1), j = e / (ni + 1);
  const int64_t p = ix3(1, j + NG, i + NG, sy(nj), sx(ni));
  wt[p] = w1 ? w1[p] : 0.0f;
}

void launch_seed_edges(const float* u1, const float* v1, const float* w1, float* ut, float* vt, float* wt, int ni,
                       int nj, int nk, hipStream_t s) {
  const int emax = max(ni + 1 + 2 * nj, nj + 1 + 2 * ni);
  hipLaunchKernelGGL(k_seed_edges, dim3((emax + 255) / 256, nk), dim3(256), 0, s, u1, v1, w1, ut, vt, wt, ni, nj,
                     nk);
  hipLaunchKernelGGL(k_seed_w_surface, dim3(((ni + 1) * (nj + 1) + 255) / 256), dim3(256), 0, s, w1, wt, ni, nj);
}

// The terrain-coordinate momentum advection; with held tendencies (u1, v1,
// w1) the k_seed_held copy is folded into the updates.
int momentum5_terrain(
    const float* u3d, const float* v3d, const float* w3d, const float* u1, const float* v1, const float* w1,
    float* uten, float* vten, float* wten, float* rru, float* rrv, float* rrw, const float* uh, const float* vh,
    const float* rho0_3d, const float* rf0, const float* rrf0, const float* c2, const float* gz, const float* gzu,
    const float* gzv, const float* rgzu, const float* rgzv, const float* dzdx, const float* dzdy,
    float* divx, int ni, int nj, int nk, float dx, float dy, float dz, unsigned obc,
    int stop_after_divergence, void* stream, bool zero_held = false) {
  hipStream_t s = (hipStream_t)stream;
  if (u1 || zero_held) {
    launch_seed_edges(u1, v1, w1, uten, vten, wten, ni, nj, nk, s);
    GM1_LAUNCH_CHECK();
  }
  const float rdx = 1.0f / dx, rdy = 1.0f / dy, rdz = 1.0f / dz;
  dim3 blk(64);
  hipLaunchKernelGGL(k_mom_mass_terrain, dim3((ni + 1 + 63) / 64, nj + 1, (nk + MKB - 1) / MKB), blk, 0, s, u3d,
                     v3d, w3d, rho0_3d, rf0, rgzu, rgzv, dzdx, dzdy, gz, rru, rrv, rrw, divx, ni, nj, nk, dz, rdx,
                     rdy);
  GM1_LAUNCH_CHECK();
  if (stop_after_divergence) return 0;
  MomArgs a;
  a.u = u3d; a.v = v3d; a.w = w3d; a.rru = rru; a.rrv = rrv; a.rrw = rrw; a.divx = divx;
  a.rho0 = rho0_3d; a.c2 = c2; a.gzu = gzu; a.gzv = gzv; a.rrf0 = rrf0; a.gz = gz; a.uh = uh; a.vh = vh;
  a.uten = uten; a.vten = vten; a.wten = wten; a.ni = ni; a.nj = nj; a.nk = nk;
  a.rdx = rdx; a.rdy = rdy; a.rdz = rdz; a.obc = obc;
  a.flat = nullptr; a.rr0 = nullptr;
  a.u1 = u1; a.v1 = v1; a.w1 = w1; a.zero_held = zero_held ? 1 : 0;
  const bool pw = side_of(obc, 0) == 1u, pe = side_of(obc, 1) == 1u;
  const bool ps = side_of(obc, 2) == 1u, pn = side_of(obc, 3) == 1u;
  const int f0 = pw ? 0 : 1, nf = ni - 1 + (pw ? 1 : 0) + (pe ? 1 : 0);
  const int g0 = ps ? 0 : 1, nr = nj - 1 + (ps ? 1 : 0) + (pn ? 1 : 0);
  launch_advu_tile<false>(a, f0, nf, s);
  GM1_LAUNCH_CHECK();
  launch_advv_tile<false>(a, g0, nr, s);
  GM1_LAUNCH_CHECK();
  launch_advw_tile<false>(a, s);
  GM1_LAUNCH_CHECK();
  return 0;
}

// The flat stretched column's momentum advection; with held tendencies the
// k_seed_held copy is folded into the updates, and with dum8 the flat
// buoyancy (k_buoyancy_flat) into the w update.
int momentum5_flat(
    const float* u3d, const float* v3d, const float* w3d, const float* u1, const float* v1, const float* w1,
    float* uten, float* vten, float* wten, float* rru, float* rrv, float* rrw, const float* uh, const float* vh,
    const float* rho0_3d, const float* rf0, const float* rr0, const float* rrf0, const float* c1, const float* c2,
    const float* dum8, const float* flat_column, float* divx, int ni, int nj, int nk, float dx, float dy, float rdz,
    unsigned obc, void* stream, bool zero_held = false) {
  if (!flat_column || (dum8 && !c1)) return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  if (u1 || zero_held) {
    launch_seed_edges(u1, v1, w1, uten, vten, wten, ni, nj, nk, s);
    GM1_LAUNCH_CHECK();
  }
  const float rdx = 1.0f / dx, rdy = 1.0f / dy;
  dim3 blk(64);
  hipLaunchKernelGGL(k_mom_mass_flat, dim3((ni + 1 + 63) / 64, nj + 1, (nk + MKB - 1) / MKB), blk, 0, s, u3d, v3d,
                     w3d, rho0_3d, rf0, flat_column, rru, rrv, rrw, divx, ni, nj, nk, rdx, rdy, rdz);
  GM1_LAUNCH_CHECK();
  MomArgs a;
  a.u = u3d; a.v = v3d; a.w = w3d; a.rru = rru; a.rrv = rrv; a.rrw = rrw; a.divx = divx;
  a.rho0 = rho0_3d; a.c2 = c2; a.gzu = nullptr; a.gzv = nullptr; a.rrf0 = rrf0; a.gz = nullptr; a.uh = uh;
  a.vh = vh; a.uten = uten; a.vten = vten; a.wten = wten; a.ni = ni; a.nj = nj; a.nk = nk;
  a.rdx = rdx; a.rdy = rdy; a.rdz = rdz; a.obc = obc; a.flat = flat_column; a.rr0 = rr0;
  a.u1 = u1; a.v1 = v1; a.w1 = w1; a.dum8 = dum8; a.c1 = c1; a.zero_held = zero_held ? 1 : 0;
  const bool pw = side_of(obc, 0) == 1u, pe = side_of(obc, 1) == 1u;
  const bool ps = side_of(obc, 2) == 1u, pn = side_of(obc, 3) == 1u;
  const int f0 = pw ? 0 : 1, nf = ni - 1 + (pw ? 1 : 0) + (pe ? 1 : 0);
  const int g0 = ps ? 0 : 1, nr = nj - 1 + (ps ? 1 : 0) + (pn ? 1 : 0);
  launch_advu_tile<true>(a, f0, nf, s);
  GM1_LAUNCH_CHECK();
  launch_advv_tile<true>(a, g0, nr, s);
  GM1_LAUNCH_CHECK();
  launch_advw_tile<true>(a, s);
  GM1_LAUNCH_CHECK();
  return 0;
}

}  // namespace

extern "C" {

int gm1hip_momentum_advection5(
    const float* u3d, const float* v3d, const float* w3d, float* uten, float* vten, float* wten,
    float* rru, float* rrv, float* rrw, const float* uh, const float* vh, const float* rho0_3d,
    const float* rf0, const float* rrf0, const float* c2, const float* gz, const float* gzu,
    const float* gzv, const float* rgzu, const float* rgzv, const float* dzdx, const float* dzdy,
    float* divx, int ni, int nj, int nk, float dx, float dy, float dz, unsigned obc,
    int stop_after_divergence, void* stream) {
  return momentum5_terrain(u3d, v3d, w3d, nullptr, nullptr, nullptr, uten, vten, wten, rru, rrv, rrw, uh, vh,
                           rho0_3d, rf0, rrf0, c2, gz, gzu, gzv, rgzu, rgzv, dzdx, dzdy, divx, ni, nj, nk, dx, dy,
                           dz, obc, stop_after_divergence, stream);
}

int gm1hip_momentum_stage(
    const float* u3d, const float* v3d, const float* w3d, const float* uten1, const float* vten1,
    const float* wten1, float* uten, float* vten, float* wten, float* rru, float* rrv, float* rrw,
    const float* uh, const float* vh, const float* rho0_3d, const float* rf0, const float* rrf0, const float* c2,
    const float* gz, const float* gzu, const float* gzv, const float* rgzu, const float* rgzv, const float* dzdx,
    const float* dzdy, float* divx, int ni, int nj, int nk, float dx, float dy, float dz, unsigned obc,
    void* stream) {
  // all three held tendencies null: they are +0 (no solve1 contribution) and are not read
  const bool zero_held = !uten1 && !vten1 && !wten1;
  if (!zero_held && (!uten1 || !vten1 || !wten1)) return (int)hipErrorInvalidValue;
  return momentum5_terrain(u3d, v3d, w3d, uten1, vten1, wten1, uten, vten, wten, rru, rrv, rrw, uh, vh, rho0_3d,
                           rf0, rrf0, c2, gz, gzu, gzv, rgzu, rgzv, dzdx, dzdy, divx, ni, nj, nk, dx, dy, dz, obc, 0,
                           stream, zero_held);
}

int gm1hip_momentum_transport5(
    const float* u3d, const float* v3d, const float* w3d, float* uten, float* vten, float* wten,
    const float* rru, const float* rrv, const float* rrw, const float* uh, const float* vh,
    const float* rho0_3d, const float* rrf0, const float* c2, const float* gz, const float* gzu,
    const float* gzv, const float* divx, int ni, int nj, int nk, float dx, float dy, float dz,
    unsigned obc, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  MomArgs a;
  a.u = u3d; a.v = v3d; a.w = w3d; a.rru = rru; a.rrv = rrv; a.rrw = rrw; a.divx = divx;
  a.rho0 = rho0_3d; a.c2 = c2; a.gzu = gzu; a.gzv = gzv; a.rrf0 = rrf0; a.gz = gz; a.uh = uh; a.vh = vh;
  a.uten = uten; a.vten = vten; a.wten = wten; a.ni = ni; a.nj = nj; a.nk = nk;
  a.rdx = 1.0f / dx; a.rdy = 1.0f / dy; a.rdz = 1.0f / dz; a.obc = obc;
  a.flat = nullptr; a.rr0 = nullptr;
  const bool pw = side_of(obc, 0) == 1u, pe = side_of(obc, 1) == 1u;
  const bool ps = side_of(obc, 2) == 1u, pn = side_of(obc, 3) == 1u;
  const int f0 = pw ? 0 : 1, nf = ni - 1 + (pw ? 1 : 0) + (pe ? 1 : 0);
  const int g0 = ps ? 0 : 1, nr = nj - 1 + (ps ? 1 : 0) + (pn ? 1 : 0);
  launch_advu_tile<false>(a, f0, nf, s);
  GM1_LAUNCH_CHECK();
  launch_advv_tile<false>(a, g0, nr, s);
  GM1_LAUNCH_CHECK();
  launch_advw_tile<false>(a, s);
  GM1_LAUNCH_CHECK();
  return 0;
}

// The flat stretched column's momentum advection (launch_cuda_gm1_child_stretched_momentum5
// with a flat column, cuda_gm1_child_stretched_momentum.py:655-757).
int gm1hip_momentum_advection5_flat(
    const float* u3d, const float* v3d, const float* w3d, float* uten, float* vten, float* wten,
    float* rru, float* rrv, float* rrw, const float* uh, const float* vh, const float* rho0_3d,
    const float* rf0, const float* rr0, const float* rrf0, const float* c2, const float* flat_column,
    float* divx, int ni, int nj, int nk, float dx, float dy, float rdz, unsigned obc, void* stream) {
  return momentum5_flat(u3d, v3d, w3d, nullptr, nullptr, nullptr, uten, vten, wten, rru, rrv, rrw, uh, vh, rho0_3d,
                        rf0, rr0, rrf0, nullptr, c2, nullptr, flat_column, divx, ni, nj, nk, dx, dy, rdz, obc, stream);
}

int gm1hip_momentum_stage_flat(
    const float* u3d, const float* v3d, const float* w3d, const float* uten1, const float* vten1,
    const float* wten1, float* uten, float* vten, float* wten, float* rru, float* rrv, float* rrw,
    const float* uh, const float* vh, const float* rho0_3d, const float* rf0, const float* rr0, const float* rrf0,
    const float* c1, const float* c2, const float* dum8, const float* flat_column, float* divx, int ni, int nj,
    int nk, float dx, float dy, float rdz, unsigned obc, void* stream) {
  // all three held tendencies null: they are +0 (no solve1 contribution) and are not read
  const bool zero_held = !uten1 && !vten1 && !wten1;
  if ((!zero_held && (!uten1 || !vten1 || !wten1)) || !dum8 || !c1) return (int)hipErrorInvalidValue;
  return momentum5_flat(u3d, v3d, w3d, uten1, vten1, wten1, uten, vten, wten, rru, rrv, rrw, uh, vh, rho0_3d, rf0,
                        rr0, rrf0, c1, c2, dum8, flat_column, divx, ni, nj, nk, dx, dy, rdz, obc, stream, zero_held);
}

}  // extern "C"
