// The flat, uniform, doubly periodic psolver=3 acoustic stage on gfx950.
//
// Layout (cuda_sound3_periodic.py:449-491): the scalar family (nk+2, nj+2,
// ni+2) with a one-cell periodic halo, u (nk+2, nj+2, ni+1), v (nk+2, nj+1,
// ni+2), w (nk+2, nj, ni) without lateral halo; 1-D metrics uf/uh (ni+2),
// vf/vh (nj+2), face weights dtu0 (nj+2, ni+1), dtv0 (nj+1, ni+2).  The
// statement order is cpu_sound3_periodic_stage_inplace's (:672-1064), which
// stores every elimination and tridiagonal diagnostic as an output.
//
// One stage is: prepare (coefficients, carriers, zeroed diagnostics), then per
// small step a face pass (pressure-gradient update of every live u and v face
// with the time average folded in), a column pass (divergence, pressure advection, fpk,
// Thomas solve, residual, pressure update and filter) and, between steps, the
// periodic ppd fill; the stage ends with the u/v and (nrk < 3) pp3d fills.  The
// fill runs once, after the last step but one: between steps the face pass reads
// the interior words the fill would copy.
#include <algorithm>

#include "cm1_common.h"

namespace {

using gm1::Dims;

// Pointer-table slots, in the order of cuda_sound3_periodic.ALL_ARRAY_NAMES.
enum Slot {
  MH, RR0, RF0, C1, C2, MF, PIADV, PPTERM, THV, PPTEN, PPI, PP3D, PPX, PPD, QK, PK1, PK2, MM, FPK, DIVH, HADVP,
  ELIM_C, ELIM_D, TRI_AA, TRI_BB, TRI_CC, TRI_DD, TRI_PIVOT, TRI_RESIDUAL, WTEN, WA, W3D, RRW, UA, U3D, UTEN, RRU,
  VA, V3D, VTEN, RRV, DTU0, DTV0, UF, VF, UH, VH, NSLOTS
};

struct Tab {
  float* p[NSLOTS];
};

constexpr int NZEROED = 15;  // QK .. TRI_RESIDUAL

GM1_DEV int64_t si(int k, int j, int i, int ni, int nj) { return ((int64_t)k * (nj + 2) + j) * (ni + 2) + i; }
GM1_DEV int64_t wi(int k, int j, int i, int ni, int nj) { return ((int64_t)k * nj + j) * ni + i; }
GM1_DEV int64_t ui(int k, int j, int f, int ni, int nj) { return ((int64_t)k * (nj + 2) + j) * (ni + 1) + f; }
GM1_DEV int64_t vi(int k, int f, int i, int ni, int nj) { return ((int64_t)k * (nj + 1) + f) * (ni + 2) + i; }

// :706-784.  One thread per word of the scalar family: diagnostics zeroed,
// ppd <- ppx and (nrk != 1) pp3d <- ppi on levels 1..nk, the stage
// coefficients qk, pk1, pk2, mm and the w carriers on physical cells.
// Also (:722-727) the face carriers, whose arrays hold fewer words: rru = rrv = 0,
// and (nrk != 1) u3d <- ua, v3d <- va.
__global__ void __launch_bounds__(256) k_sp_prepare(Tab t, Dims d, int nrk, float dts, float rdz, float cp,
                                                    float beta) {
  const int ni = d.ni, nj = d.nj, nk = d.nk;
  const int64_t total = (int64_t)(nk + 2) * (nj + 2) * (ni + 2);
  const int64_t nu = (int64_t)(nk + 2) * (nj + 2) * (ni + 1);
  const int64_t nv = (int64_t)(nk + 2) * (nj + 1) * (ni + 2);
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= total) return;
  if (q < nu) {
    t.p[RRU][q] = 0.0f;
    if (nrk != 1) t.p[U3D][q] = t.p[UA][q];
  }
  if (q < nv) {
    t.p[RRV][q] = 0.0f;
    if (nrk != 1) t.p[V3D][q] = t.p[VA][q];
  }
  const int i = (int)(q % (ni + 2));
  const int j = (int)((q / (ni + 2)) % (nj + 2));
  const int k = (int)(q / ((int64_t)(ni + 2) * (nj + 2)));
  const bool level = k >= 1 && k <= nk;
  const bool phys = level && j >= 1 && j <= nj && i >= 1 && i <= ni;
#pragma unroll
  for (int s = QK; s < QK + NZEROED; ++s) {
    if (phys && s <= MM) continue;  // coefficients below
    // words that the stage's last small step writes: fpk, divh, hadvp and elim_c on
    // levels 1..nk, the tri_* on 2..nk, elim_d on 2..nk-1
    if (phys && (s == FPK || s == DIVH || s == HADVP || s == ELIM_C)) continue;
    if (phys && k >= 2 && (s == ELIM_D ? k < nk : s >= TRI_AA)) continue;
    t.p[s][q] = 0.0f;
  }
  if (level) {
    t.p[PPD][q] = t.p[PPX][q];
    if (nrk != 1) t.p[PP3D][q] = t.p[PPI][q];
  }
  if (!phys) return;
  const float* mh = t.p[MH];
  const float* rr0 = t.p[RR0];
  const float* rf0 = t.p[RF0];
  const float* c1 = t.p[C1];
  const float* c2 = t.p[C2];
  const float* piadv = t.p[PIADV];
  const float* thv = t.p[THV];
  const int64_t up = si(k + 1, j, i, ni, nj), dn = si(k - 1, j, i, ni, nj);
  const float dr = dts * rdz;
  const float tem = dr * mh[q];
  float r2 = dr * mh[q];
  r2 = r2 * rr0[q];
  r2 = r2 * rf0[up];
  float r1 = dr * mh[q];
  r1 = r1 * rr0[q];
  r1 = r1 * rf0[q];
  const float tem1 = (dr * cp) * t.p[MF][q];
  t.p[QK][q] = tem * t.p[PPTERM][q];
  t.p[PK2][q] = (k == nk) ? 0.0f : r2 * ((-c2[up]) * piadv[up] + (1.0f - c1[up]) * piadv[q]);
  t.p[PK1][q] = (k == 1) ? 0.0f : r1 * (c1[q] * piadv[dn] + (c2[q] - 1.0f) * piadv[q]);
  t.p[MM][q] = tem1 * (c2[q] * thv[q] + c1[q] * thv[dn]);
  const int64_t w = wi(k, j - 1, i - 1, ni, nj);
  const float wa = t.p[WA][w];
  t.p[RRW][w] = wa * beta;
  if (nrk != 1) t.p[W3D][w] = wa;
}

// :787-828 and :1013-1032.  Every live u face (k 1..nk, j 1..nj+1, f 0..ni)
// and v face (k 1..nk, f 0..nj, i 1..ni+1): u += dts*dtu0*(uten - pg), then
// the running sum rru (n < nloop) or the average (rru + u)*(1/nloop).  A face's
// word of the step before is read here, so the sums take two steps' words at
// every second step (`add` 2; an odd last step adds its own, `add` 1; 0 none).
// From the second step on (`wrap`) ppd's halo words are taken from the interior
// words the periodic fill copies, so no fill runs between steps.
__global__ void __launch_bounds__(256) k_sp_faces(Tab t, Dims d, float dts, float tem1, float tem2, float tavg,
                                                  int add, int wrap, int last) {
  const int ni = d.ni, nj = d.nj, nk = d.nk;
  const int64_t nu = (int64_t)nk * (nj + 1) * (ni + 1);
  const int64_t nv = (int64_t)nk * (nj + 1) * (ni + 1);
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const float* ppd = t.p[PPD];
  const float* thv = t.p[THV];
  auto wi_ = [&](int x, int n) { return !wrap ? x : (x == 0) ? n : (x == n + 1) ? 1 : x; };
  const bool u_face = q < nu;
  if (!u_face) q -= nu;
  if (q >= nv) return;
  const int a = (int)(q % (ni + 1)), b = (int)((q / (ni + 1)) % (nj + 1));
  const int k = (int)(q / ((int64_t)(ni + 1) * (nj + 1))) + 1;
  // the face's cells: (j, f+1) and (j, f) for u, (f+1, i) and (f, i) for v
  const int j1 = b + 1, i1 = a + 1, j0 = u_face ? j1 : b, i0 = u_face ? a : i1;
  float pg = (u_face ? tem1 : tem2) *
             (ppd[si(k, wi_(j1, nj), wi_(i1, ni), ni, nj)] - ppd[si(k, wi_(j0, nj), wi_(i0, ni), ni, nj)]);
  pg = pg * (u_face ? t.p[UF][i1] : t.p[VF][j1]);
  pg = pg * (thv[si(k, j1, i1, ni, nj)] + thv[si(k, j0, i0, ni, nj)]);
  const int64_t o = u_face ? ui(k, j1, a, ni, nj) : vi(k, b, i1, ni, nj);
  const float dt0 = u_face ? t.p[DTU0][(int64_t)j1 * (ni + 1) + a] : t.p[DTV0][(int64_t)b * (ni + 2) + i1];
  float* q3 = u_face ? t.p[U3D] : t.p[V3D];
  float* rr = u_face ? t.p[RRU] : t.p[RRV];
  const float old = q3[o];
  const float r0 = add ? rr[o] : 0.0f;
  const float now = old + (dts * dt0) * ((u_face ? t.p[UTEN][o] : t.p[VTEN][o]) - pg);
  q3[o] = now;
  if (add) {
    const float r = (add == 2 ? r0 + old : r0) + now;
    rr[o] = last ? r * tavg : r;
  }
}

struct ColumnScalars {
  float dts, rdx, rdy, temx, temy, alph, beta, asq, kdiv, smeps, tavg;
  int write_ppx, last;
  int add_w;  // small steps' words rrw takes in this step: 0, 1 or 2 (k_sp_faces' rule)
};

// :830-1010, staged: a workgroup owns CW columns of one row and all levels, its
// CS level slots a chunk of at most CH levels each.  Phase A forms fpk, the
// tridiagonal terms and the right-hand sides of every slot's levels at once (pp,
// fpk, dd, mm and the old w of a thread's own levels in registers), phase B runs
// the recurrence out of LDS with one lane a column, phase C updates the pressure.
// The diagnostics (divh, hadvp, fpk, tri_*, elim_*) are overwritten by every
// small step, so only the stage's last one writes them.  Bound by latency (the
// words of a slot's levels are all requested at once, then the recurrence): the
// three stages take 1580 -> 355 us at 64x64x40, 3055 -> 1052 at 128x128x64 and
// 7559 -> 5247 at 256x256x80 against one thread walking each column and writing
// every diagnostic every step.  32 columns a workgroup measured the same within
// 5 % at 64x64x40 and 256x256x80 and 2-20 % slower between.
constexpr int CW = 16, CS = 32;

template <int CH>
__global__ void __launch_bounds__(CS* CW) k_sp_column_staged(Tab t, Dims d, ColumnScalars c) {
  extern __shared__ float lds[];
  const int ni = d.ni, nj = d.nj, nk = d.nk;
  const int lane = threadIdx.x % CW, slot = threadIdx.x / CW;
  const int i = (int)blockIdx.x * CW + lane + 1, j = (int)blockIdx.y + 1;
  const bool phys = i <= ni;
  const int L = (nk + 1) * CW;
  float* Ls1 = lds;
  float* Ls2 = lds + L;
  float* Lmm = lds + 2 * L;  // then elim_c
  float* Ldd = lds + 3 * L;  // then elim_d, then w
  float* Lbp = lds + 4 * L;
  float* Lbf = Lbp + CS * CW;
  auto at = [&](int k) { return k * CW + lane; };
  const int chunk = (nk + CS - 1) / CS;
  const int kb = 1 + slot * chunk, ke = min(nk, kb + chunk - 1);
  const bool mine = phys && kb <= ke;
  float* w = t.p[W3D];
  const int64_t plane = (int64_t)(nj + 2) * (ni + 2), wplane = (int64_t)nj * ni;
  const int64_t s0 = si(0, j, i, ni, nj), w0 = wi(0, j - 1, i - 1, ni, nj);
  float rpp[CH], rfpk[CH], rdd[CH], rmm[CH], rwo[CH], rwt[CH];
  if (mine) {
    const float uh = t.p[UH][i], vh = t.p[VH][j];
    struct In {
      float uw, ue, vs, vn, pc, pe, pw, pn, ps, wk, wup, ppten, ppterm, pk1, pk2, qk, pp, mm, wt;
    } in[CH];
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int k = kb + q;
      if (k <= ke) {
        const int64_t s = s0 + k * plane, wk = w0 + k * wplane, u = ui(k, j, i, ni, nj), v = vi(k, j, i, ni, nj);
        in[q].ue = t.p[U3D][u];
        in[q].uw = t.p[U3D][u - 1];
        in[q].vn = t.p[V3D][v];
        in[q].vs = t.p[V3D][v - (ni + 2)];
        in[q].pc = t.p[PIADV][s];
        in[q].pe = t.p[PIADV][s + 1];
        in[q].pw = t.p[PIADV][s - 1];
        in[q].pn = t.p[PIADV][s + (ni + 2)];
        in[q].ps = t.p[PIADV][s - (ni + 2)];
        in[q].wk = w[wk];
        in[q].wup = w[wk + wplane];
        in[q].ppten = t.p[PPTEN][s];
        in[q].ppterm = t.p[PPTERM][s];
        in[q].pk1 = t.p[PK1][s];
        in[q].pk2 = t.p[PK2][s];
        in[q].qk = t.p[QK][s];
        in[q].pp = t.p[PP3D][s];
        in[q].mm = t.p[MM][s];
        in[q].wt = t.p[WTEN][wk];
      }
    }
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int k = kb + q;
      if (k <= ke) {
        const In& n = in[q];
        const int64_t s = s0 + k * plane;
        const float du = ((n.ue - n.uw) * c.rdx) * uh;
        const float dv = ((n.vn - n.vs) * c.rdy) * vh;
        float div = du + dv;
        if (fabsf(div) < c.smeps) div = 0.0f;
        const float gxw = n.pc - n.pw, gxe = n.pe - n.pc, gys = n.pc - n.ps, gyn = n.pn - n.pc;
        float hx = n.uw * gxw + n.ue * gxe;
        hx = ((-hx) * c.temx) * uh;
        float hy = n.vs * gys + n.vn * gyn;
        hy = ((-hy) * c.temy) * vh;
        const float hp = hx + hy;
        const float src = c.dts * (n.ppten - n.ppterm * div);
        const float s1 = n.pk1 + n.qk, s2 = n.pk2 - n.qk;
        const float vert = n.wk * s1 + n.wup * s2;
        const float fpk = (src + hp) + c.beta * vert;
        if (c.last) {
          t.p[DIVH][s] = div;
          t.p[HADVP][s] = hp;
          t.p[FPK][s] = fpk;
        }
        Ls1[at(k)] = s1;
        Ls2[at(k)] = s2;
        Lmm[at(k)] = n.mm;
        rpp[q] = n.pp;
        rfpk[q] = fpk;
        rmm[q] = n.mm;
        rwo[q] = n.wk;
        rwt[q] = n.wt;
        if (k == ke) {
          Lbp[slot * CW + lane] = n.pp;
          Lbf[slot * CW + lane] = fpk;
        }
      }
    }
  }
  __syncthreads();
  if (mine) {  // right-hand sides; a slot's first level takes the level below from the previous slot
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int k = kb + q;
      if (k >= 2 && k <= ke) {
        const float ppm = q ? rpp[q - 1] : Lbp[(slot - 1) * CW + lane];
        const float fm = q ? rfpk[q - 1] : Lbf[(slot - 1) * CW + lane];
        const float pd = rpp[q] - ppm;
        const float fwk = c.dts * rwt[q] + c.beta * ((-rmm[q]) * pd);
        const float upd = (rpp[q] + rfpk[q]) - (ppm + fm);
        rdd[q] = (rwo[q] + fwk) + c.alph * ((-rmm[q]) * upd);
        Ldd[at(k)] = rdd[q];
      }
    }
  }
  __syncthreads();
  auto row = [&](int k, float m, float s1m, float s2m, float s1, float s2, float& aa, float& bb, float& cc) {
    aa = (k >= 3) ? (-c.asq) * (m * s1m) : 0.0f;
    cc = (k < nk) ? (-c.asq) * ((-m) * s2) : 0.0f;
    const float diag = (-s1) + s2m;
    bb = 1.0f - c.asq * (m * diag);
  };
  if (phys && slot == 0) {
    float ec_prev = 0.0f, ed_prev = 0.0f, s1m = Ls1[at(1)], s2m = Ls2[at(1)], wtop = 0.0f;
    float mn = Lmm[at(2)], s1n = Ls1[at(2)], s2n = Ls2[at(2)], dn = Ldd[at(2)];
    for (int k = 2; k <= nk; ++k) {
      const float m = mn, s1 = s1n, s2 = s2n, dd = dn;
      if (k < nk) {
        mn = Lmm[at(k + 1)];
        s1n = Ls1[at(k + 1)];
        s2n = Ls2[at(k + 1)];
        dn = Ldd[at(k + 1)];
      }
      float aa, bb, cc;
      row(k, m, s1m, s2m, s1, s2, aa, bb, cc);
      const float pivot = (k < 3) ? bb : aa * ec_prev + bb;
      const float inv = 1.0f / pivot;
      if (c.last) t.p[TRI_PIVOT][s0 + k * plane] = pivot;
      if (k < nk) {
        ec_prev = (-cc) * inv;
        ed_prev = ((k < 3) ? dd : dd - aa * ed_prev) * inv;
        Lmm[at(k)] = ec_prev;
        Ldd[at(k)] = ed_prev;
        if (c.last) t.p[ELIM_D][s0 + k * plane] = ed_prev;
      } else {
        wtop = (dd - aa * ed_prev) * inv;
      }
      s1m = s1;
      s2m = s2;
    }
    Ldd[at(nk)] = wtop;
    for (int k = nk - 1; k >= 2; --k) {
      wtop = Lmm[at(k)] * wtop + Ldd[at(k)];
      Ldd[at(k)] = wtop;
    }
  }
  __syncthreads();
  if (mine) {
    const float wlid = w[w0 + (int64_t)(nk + 1) * wplane], w1 = w[w0 + wplane];
    float* rrw = t.p[RRW];
    float rw[CH];
#pragma unroll
    for (int q = 0; q < CH; ++q)
      if (c.add_w && kb + q <= ke) rw[q] = rrw[w0 + (kb + q) * wplane];
    auto wat = [&](int k) { return k == 1 ? w1 : k == nk + 1 ? wlid : Ldd[at(k)]; };
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int k = kb + q;
      if (k <= ke) {
        const int64_t s = s0 + k * plane, w_k = w0 + k * wplane;
        const float wk = wat(k), wu = wat(k + 1), s1 = Ls1[at(k)], s2 = Ls2[at(k)];
        if (k >= 2) w[w_k] = wk;
        const float vert = wk * s1 + wu * s2;
        float upd = (rpp[q] + rfpk[q]) + c.alph * vert;
        if (fabsf(upd) < c.smeps) upd = 0.0f;
        t.p[PP3D][s] = upd;
        const float filt = c.kdiv * (upd - rpp[q]);
        t.p[PPD][s] = upd + filt;
        if (c.write_ppx) t.p[PPX][s] = filt;
        if (c.add_w) {
          const float r = (c.add_w == 2 ? rw[q] + rwo[q] : rw[q]);
          rrw[w_k] = c.last ? (r + wk * c.alph) * c.tavg : r + wk;
        }
        if (c.last) {
          t.p[ELIM_C][s] = filt;
          if (k >= 2) {
            float aa, bb, cc;
            row(k, rmm[q], Ls1[at(k - 1)], Ls2[at(k - 1)], s1, s2, aa, bb, cc);
            t.p[TRI_AA][s] = aa;
            t.p[TRI_BB][s] = bb;
            t.p[TRI_CC][s] = cc;
            t.p[TRI_DD][s] = rdd[q];
            float lhs = aa * wat(k - 1);
            lhs = lhs + bb * wk;
            lhs = lhs + cc * wu;
            t.p[TRI_RESIDUAL][s] = lhs - rdd[q];
          }
        }
      }
    }
  }
}

void launch_column_staged(const Tab& t, const Dims& d, const ColumnScalars& c, hipStream_t st) {
  const dim3 grid((unsigned)((d.ni + CW - 1) / CW), (unsigned)d.nj), block(CS * CW);
  const int chunk = (d.nk + CS - 1) / CS;
  const int lds = (4 * (d.nk + 1) + 2 * CS) * CW * (int)sizeof(float);
  if (chunk <= 2) hipLaunchKernelGGL((k_sp_column_staged<2>), grid, block, lds, st, t, d, c);
  else if (chunk <= 3) hipLaunchKernelGGL((k_sp_column_staged<3>), grid, block, lds, st, t, d, c);
  else hipLaunchKernelGGL((k_sp_column_staged<4>), grid, block, lds, st, t, d, c);
}

// :830-1010 on columns too tall for the staged pass (more than 128 levels).  One
// thread per physical column; k runs serially.  Lanes of a wavefront take
// consecutive i, so every level's loads are row-contiguous.
__global__ void __launch_bounds__(256) k_sp_column(Tab t, Dims d, ColumnScalars c) {
  const int ni = d.ni, nj = d.nj, nk = d.nk;
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > ni || j > nj) return;
  const float* u = t.p[U3D];
  const float* v = t.p[V3D];
  const float* piadv = t.p[PIADV];
  const float* ppterm = t.p[PPTERM];
  const float* ppten = t.p[PPTEN];
  const float* qk = t.p[QK];
  const float* pk1 = t.p[PK1];
  const float* pk2 = t.p[PK2];
  const float* mm = t.p[MM];
  const float* wten = t.p[WTEN];
  float* w = t.p[W3D];
  float* pp3d = t.p[PP3D];
  float* fpk = t.p[FPK];
  float* ec = t.p[ELIM_C];
  float* ed = t.p[ELIM_D];
  const float uh = t.p[UH][i], vh = t.p[VH][j];
  const int64_t plane = (int64_t)(nj + 2) * (ni + 2);
  const int64_t wplane = (int64_t)nj * ni;
  const int64_t s0 = si(0, j, i, ni, nj);
  const int64_t w0 = wi(0, j - 1, i - 1, ni, nj);

  // fpk on every level (:830-880).
  for (int k = 1; k <= nk; ++k) {
    const int64_t s = s0 + k * plane, w_k = w0 + k * wplane;
    const float du = ((u[ui(k, j, i, ni, nj)] - u[ui(k, j, i - 1, ni, nj)]) * c.rdx) * uh;
    const float dv = ((v[vi(k, j, i, ni, nj)] - v[vi(k, j - 1, i, ni, nj)]) * c.rdy) * vh;
    float div = du + dv;
    if (fabsf(div) < c.smeps) div = 0.0f;
    t.p[DIVH][s] = div;
    const float pc = piadv[s];
    const float gxw = pc - piadv[s - 1];
    const float gxe = piadv[s + 1] - pc;
    const float gys = pc - piadv[s - (ni + 2)];
    const float gyn = piadv[s + (ni + 2)] - pc;
    float hx = u[ui(k, j, i - 1, ni, nj)] * gxw + u[ui(k, j, i, ni, nj)] * gxe;
    hx = ((-hx) * c.temx) * uh;
    float hy = v[vi(k, j - 1, i, ni, nj)] * gys + v[vi(k, j, i, ni, nj)] * gyn;
    hy = ((-hy) * c.temy) * vh;
    const float hp = hx + hy;
    t.p[HADVP][s] = hp;
    const float src = c.dts * (ppten[s] - ppterm[s] * div);
    const float vert = w[w_k] * (pk1[s] + qk[s]) + w[w_k + wplane] * (pk2[s] - qk[s]);
    fpk[s] = (src + hp) + c.beta * vert;
  }

  // Forward elimination (:881-953); level k-1's terms are carried.
  float ec_prev = 0.0f, ed_prev = 0.0f;
  float pp_prev = pp3d[s0 + plane], fpk_prev = fpk[s0 + plane];
  float s1_prev = pk1[s0 + plane] + qk[s0 + plane];
  float s2_prev = pk2[s0 + plane] - qk[s0 + plane];
  for (int k = 2; k <= nk; ++k) {
    const int64_t s = s0 + k * plane, w_k = w0 + k * wplane;
    const float m = mm[s];
    const float s1 = pk1[s] + qk[s];
    const float s2 = pk2[s] - qk[s];
    const float aa = (k >= 3) ? (-c.asq) * (m * s1_prev) : 0.0f;
    const float cc = (k < nk) ? (-c.asq) * ((-m) * s2) : 0.0f;
    const float diag = (-s1) + s2_prev;
    const float bb = 1.0f - c.asq * (m * diag);
    const float pk = pp3d[s];
    const float fk = fpk[s];
    const float pd = pk - pp_prev;
    const float fwk = c.dts * wten[w_k] + c.beta * ((-m) * pd);
    const float upd = (pk + fk) - (pp_prev + fpk_prev);
    const float dd = (w[w_k] + fwk) + c.alph * ((-m) * upd);
    const float pivot = (k < 3) ? bb : aa * ec_prev + bb;
    const float inv = 1.0f / pivot;
    t.p[TRI_AA][s] = aa;
    t.p[TRI_BB][s] = bb;
    t.p[TRI_CC][s] = cc;
    t.p[TRI_DD][s] = dd;
    t.p[TRI_PIVOT][s] = pivot;
    if (k < nk) {
      ec_prev = (-cc) * inv;
      ed_prev = ((k < 3) ? dd : dd - aa * ed_prev) * inv;
      ec[s] = ec_prev;
      ed[s] = ed_prev;
    } else {
      w[w_k] = (dd - aa * ed_prev) * inv;
    }
    pp_prev = pk;
    fpk_prev = fk;
    s1_prev = s1;
    s2_prev = s2;
  }
  // Back substitution (:954-959).
  float w_up = w[w0 + nk * wplane];
  for (int k = nk - 1; k >= 2; --k) {
    const int64_t s = s0 + k * plane;
    w_up = ec[s] * w_up + ed[s];
    w[w0 + k * wplane] = w_up;
  }
  // Residual (:960-968).
  for (int k = 2; k <= nk; ++k) {
    const int64_t s = s0 + k * plane, w_k = w0 + k * wplane;
    float lhs = t.p[TRI_AA][s] * w[w_k - wplane];
    lhs = lhs + t.p[TRI_BB][s] * w[w_k];
    lhs = lhs + t.p[TRI_CC][s] * w[w_k + wplane];
    t.p[TRI_RESIDUAL][s] = lhs - t.p[TRI_DD][s];
  }
  // Pressure update, filter, ppx and the w average (:969-1010).
  float* rrw = t.p[RRW];
  for (int k = 1; k <= nk; ++k) {
    const int64_t s = s0 + k * plane, w_k = w0 + k * wplane;
    const float old = pp3d[s];
    const float wk = w[w_k];
    const float vert = wk * (pk1[s] + qk[s]) + w[w_k + wplane] * (pk2[s] - qk[s]);
    float upd = (old + fpk[s]) + c.alph * vert;
    if (fabsf(upd) < c.smeps) upd = 0.0f;
    pp3d[s] = upd;
    const float filt = c.kdiv * (upd - old);
    ec[s] = filt;
    t.p[PPD][s] = upd + filt;
    if (c.write_ppx) t.p[PPX][s] = filt;
    rrw[w_k] = c.last ? (rrw[w_k] + wk * c.alph) * c.tavg : rrw[w_k] + wk;
  }
}

// :506-516.  Halo word (k, j, i) of levels 1..nk takes the interior word the
// x-then-y copy sequence leaves there: i' = ni for i = 0, 1 for i = ni+1, and
// likewise in j (corners therefore read (nj or 1, ni or 1)).  r: position on the
// ring, rows 0 and nj+1 first.
GM1_DEV void fill_ring_word(float* s, int k, int r, int ni, int nj) {
  int i, j;
  if (r < ni + 2) { j = 0; i = r; }
  else if (r < 2 * (ni + 2)) { j = nj + 1; i = r - (ni + 2); }
  else { r -= 2 * (ni + 2); j = 1 + r / 2; i = (r & 1) ? ni + 1 : 0; }
  const int is = (i == 0) ? ni : (i == ni + 1) ? 1 : i;
  const int js = (j == 0) ? nj : (j == nj + 1) ? 1 : j;
  s[si(k, j, i, ni, nj)] = s[si(k, js, is, ni, nj)];
}

__global__ void __launch_bounds__(256) k_sp_fill_scalar(float* s, Dims d) {
  const int64_t ring = 2 * (d.ni + 2) + 2 * d.nj;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < d.nk * ring) fill_ring_word(s, (int)(q / ring) + 1, (int)(q % ring), d.ni, d.nj);
}

// The stage's last fills: :519-532, u rows 0 and nj+1 and v columns 0 and ni+1 of
// levels 1..nk, and pp3d's halo where p is given (nrk < 3).
__global__ void __launch_bounds__(256) k_sp_fill_end(float* u, float* v, float* p, Dims d) {
  const int ni = d.ni, nj = d.nj, nk = d.nk;
  const int64_t nu = (int64_t)nk * 2 * (ni + 1);
  const int64_t nv = (int64_t)nk * (nj + 1) * 2;
  const int64_t ring = 2 * (ni + 2) + 2 * nj;
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nu) {
    const int f = (int)(q % (ni + 1));
    const int side = (int)((q / (ni + 1)) % 2);
    const int k = (int)(q / (2 * (int64_t)(ni + 1))) + 1;
    const int j = side ? nj + 1 : 0, js = side ? 1 : nj;
    u[ui(k, j, f, ni, nj)] = u[ui(k, js, f, ni, nj)];
    return;
  }
  q -= nu;
  if (q < nv) {
    const int side = (int)(q % 2);
    const int f = (int)((q / 2) % (nj + 1));
    const int k = (int)(q / (2 * (int64_t)(nj + 1))) + 1;
    const int i = side ? ni + 1 : 0, is = side ? 1 : ni;
    v[vi(k, f, i, ni, nj)] = v[vi(k, f, is, ni, nj)];
    return;
  }
  q -= nv;
  if (p && q < nk * ring) fill_ring_word(p, (int)(q / ring) + 1, (int)(q % ring), ni, nj);
}

unsigned blocks(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

extern "C" int gm1hip_sound3_periodic_stage(void* const* arrays, int ni, int nj, int nk, int nrk, int nloop,
                                            float dts, float rdx, float rdy, float rdz, float cp, float alph,
                                            float kdiv, void* stream) {
  if (!arrays || ni < 3 || nj < 3 || nk < 3 || nrk < 1 || nrk > 3 || nloop < 1) return (int)hipErrorInvalidValue;
  Tab t;
  for (int s = 0; s < NSLOTS; ++s) {
    t.p[s] = static_cast<float*>(arrays[s]);
    if (!t.p[s]) return (int)hipErrorInvalidValue;
  }
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const Dims d{ni, nj, nk};
  const float beta = 1.0f - alph;
  const float asq = alph * alph;
  constexpr int T = 256;
  const int64_t scalar_words = (int64_t)(nk + 2) * (nj + 2) * (ni + 2);
  const int64_t live_faces = 2 * (int64_t)nk * (nj + 1) * (ni + 1);
  const int64_t ring_words = (int64_t)nk * (2 * (ni + 2) + 2 * nj);
  const int64_t uv_halo = (int64_t)nk * 2 * (ni + 1) + (int64_t)nk * (nj + 1) * 2;

  hipLaunchKernelGGL(k_sp_prepare, dim3(blocks(scalar_words, T)), dim3(T), 0, st, t, d, nrk, dts, rdz, cp, beta);
  const float tem1 = (rdx * cp) * 0.5f;
  const float tem2 = (rdy * cp) * 0.5f;
  ColumnScalars c;
  c.dts = dts;
  c.rdx = rdx;
  c.rdy = rdy;
  c.temx = (dts * 0.5f) * rdx;
  c.temy = (dts * 0.5f) * rdy;
  c.alph = alph;
  c.beta = beta;
  c.asq = asq;
  c.kdiv = kdiv;
  c.smeps = 1.0e-30f;
  c.tavg = 1.0f / (float)nloop;
  const dim3 cblock(64, 4);
  const dim3 cgrid((unsigned)((ni + 63) / 64), (unsigned)((nj + 3) / 4));
  const bool staged = nk <= 4 * CS;
  for (int n = 1; n <= nloop; ++n) {
    const int last = n == nloop;
    const int add = (n % 2 == 0) ? 2 : last ? 1 : 0;
    hipLaunchKernelGGL(k_sp_faces, dim3(blocks(live_faces, T)), dim3(T), 0, st, t, d, dts, tem1, tem2, c.tavg,
                       add, (int)(n > 1), last);
    c.last = last;
    c.write_ppx = (nrk == 3 && last) ? 1 : 0;
    c.add_w = add;
    if (staged) launch_column_staged(t, d, c, st);
    else hipLaunchKernelGGL(k_sp_column, cgrid, cblock, 0, st, t, d, c);
    // (ppd's halo itself only as the stage leaves it)
    if (n == nloop - 1)
      hipLaunchKernelGGL(k_sp_fill_scalar, dim3(blocks(ring_words, T)), dim3(T), 0, st, t.p[PPD], d);
  }
  hipLaunchKernelGGL(k_sp_fill_end, dim3(blocks(uv_halo + ring_words, T)), dim3(T), 0, st, t.p[U3D], t.p[V3D],
                     nrk < 3 ? t.p[PP3D] : (float*)nullptr, d);
  return (int)hipGetLastError();
}
