// Mixed-precision sweep of one spin channel, up to 64 electrons of a spin, with the inverse updated
// panel by panel (FP32 LCAO; the arithmetic of qw_mixed.hpp's sweep, bit for bit).
//
//   k_sweep_mxp<NS, DEPTH, JP, STAGE, SHL>  single-electron moves (src/method/Split_sample.cpp:302-540,
//       src/program_utils/MatrixAlgebrac.cpp:766-838), one wavefront per walker, four walkers per
//       block sharing the system tables; SHL = false: one walker per block with the shell records in
//       device memory, for systems of so many shells that four walkers' tables and lists do not fit
//       (from about 2400 shells on, 1500 with a thousand atoms)
//
// Only the rows of the next 16 electrons are held (four lanes per row, each with every fourth
// value: the four partial sums of the update's dot product), and take every accepted move's
// Sherman-Morrison update at once.  The other rows take a panel's updates when it ends, one after
// the other in the order of the moves with the same FP32 operations, so every element sees exactly
// the updates a register-resident inverse would.  A launch that the FP64 recompute follows
// discards the inverse, so it updates only the rows of electrons still to move (SweepArgs::keep).
//
// What bounds it: vector issue (Jastrow pair terms, LCAO, the uniform FP64 of the acceptance) and
// the latencies of a move's serial chain.  With the whole inverse in registers (240) a SIMD held
// two waves and every update ran over all rows; now 128 registers and four waves.  Measured at 64
// electrons of a spin and 8192 walkers: 2.05 -> 1.26 ms per 32-move launch on average (three waves
// per SIMD: 1.49 ms).
#pragma once
#include "qw_mixed.hpp"
#include "qw_panel.hpp"

namespace qw {

// Rows of a panel, lanes per row, values per lane.
template <int NS>
struct PanelMx {
  static constexpr int P = NS <= 32 ? NS : 16;
  static constexpr int TPR = NS == 32 ? 2 : 4;
  static constexpr int EPT = NS / TPR;
};
// Place of column c in a broadcast row: a lane's values are contiguous.  Four lanes: lane c % 4;
// two lanes (NS = 32): lane (c % 4) / 2.
template <int NS>
__device__ inline int perm_col(int c) {
  typedef PanelMx<NS> D;
  return D::TPR == 4 ? (c & 3) * D::EPT + (c >> 2) : ((c >> 1) & 1) * D::EPT + (c >> 2) * 2 + (c & 1);
}
// Column of value i of lane q (the inverse of perm_col).
template <int NS>
__device__ inline int lane_col(int q, int i) {
  return PanelMx<NS>::TPR == 4 ? 4 * i + q : 4 * (i >> 1) + 2 * q + (i & 1);
}

// Basis functions per LDS tile.  The general form's shells may be F and G, each a long serial loop that
// every batch of shells repeats, so its tile takes twice the functions (six atoms of 29 functions, 7F
// and 9G among them, 1024 walkers: a spin's VMC moves 0.98 -> 0.79 ms; without such shells no slower).
__host__ __device__ constexpr int cap_mx(bool usual) { return usual ? 128 : 256; }
constexpr int kMxStage = 4;    // updates staged in LDS at a time when a panel ends

__host__ __device__ inline size_t panel_mx_shared_lds(int na, int nsh, int ntab, int stage_nb, int nsp) {
  return lds_round16(panel_shared_lds(na, nsh, ntab, 1)) + lds_round16((size_t)stage_nb * nsp * 4);
}
__host__ __device__ inline size_t panel_mx_walker_lds(int nsh, int ns, int depth, bool usual) {
  return (size_t)cap_mx(usual) * (5 * 4 + 4) + lds_round16((size_t)(nsh + 64) * 8) + (size_t)((ns <= 32 ? ns : 16) * depth * 4) * 8 +
         lds_round16((size_t)2 * ns * 4) + (ns > 32 ? (size_t)kMxStage * 2 * ns * 4 : 0) + 64;
}
// stage_nb: the basis size when the coefficients are staged in LDS, else 0.
__host__ __device__ inline size_t panel_mx_lds_bytes(int na, int nsh, int ntab, int ns, int depth, int stage_nb, int nsp,
                                                          bool usual, int wpb = kPanelWpb) {
  return panel_mx_shared_lds(na, nsh, ntab, stage_nb, nsp) + (size_t)wpb * panel_mx_walker_lds(nsh, ns, depth, usual);
}

// PolyEval with the like and unlike coefficients equal (no choice per lane), and CuspEval with the
// chosen coefficient given: their operations in their order.
__device__ inline void poly4_f32(const QW_CONST JRad<float>& o, float r, float ri, float& u, float& gfac) {
  const float zz = r * o.rcinv, zz2 = zz * zz;
  const float zpp = zz2 * (6.f - 8.f * zz + 3.f * zz2), zpp1 = 1.f - zpp;
  const float zppd = 12.f * zz * (1.f - 2.f * zz + zz2);
  float s0 = 0, s1 = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float b = o.beta[i];
    const float pz = rcp_nr(1.f + b * zpp);
    const float c = o.cl[i], cb = o.cbl[i];
    s0 += c * pz;
    const float t = cb * pz * pz;
    s1 += t;
  }
  const bool in = r < o.rcut;
  const float g = -zppd * ri * o.rcinv * s1;
  u += in ? zpp1 * s0 : 0.f;
  gfac += in ? g : 0.f;
}
__device__ inline void cusp_f32(const QW_CONST JRad<float>& o, float c, float r, float ri, float& u, float& gfac) {
  const float zz = r * o.rcinv, zz2 = zz * zz;
  const float pp = zz - zz2 + zz * zz2 * (float)(1.0 / 3.0);
  const float pade = rcp_nr(1.f + o.gamma * pp), pade2 = pade * pade;
  const float ppd = 1.f - 2.f * zz + zz2;
  const float dadr = ppd * pade2 * ri;
  const bool in = r < o.rcut;
  u += in ? c * (o.rcut * (pp * pade - o.pade0)) : 0.f;
  gfac += in ? c * dadr : 0.f;
}
// jastrow_e_freg for the usual Jastrow (DevSys::usual): the same terms in the same order without
// the loops over objects.  epos: 3 doubles per atom.
__device__ inline float jastrow_usual_f32(const DevSys& S, int e, const double p[3], const double (*pe)[3], float g[3],
                                          int lane, const double* epos) {
  float u = 0, gx = 0, gy = 0, gz = 0;
  const QW_CONST int* ea0 = cptr(S.eit_a0);
  const QW_CONST int* eo0 = cptr(S.eit_o0);
  for (int t = 0; t < S.n_eit; t++) {
    const int a0 = ea0[t], a1 = ea0[t + 1], o0 = eo0[t];
    for (int k = a0 + lane; k < a1; k += kWave) {
      const double* ap = epos + 3 * k;
      const float x = (float)(p[0] - ap[0]), y = (float)(p[1] - ap[1]), z = (float)(p[2] - ap[2]);
      float r, ri;
      dist_inv(x * x + y * y + z * z, r, ri);
      float gf = 0;
      poly4_f32(cptr(S.eitf)[o0], r, ri, u, gf);
      gx += gf * x;
      gy += gf * y;
      gz += gf * z;
    }
  }
  const bool eup = e < S.nup;
  const QW_CONST JRad<float>* ee = cptr(S.eef);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int j = lane + h * kWave;
    if (j < S.ne && j != e) {
      const float x = (float)(p[0] - pe[h][0]), y = (float)(p[1] - pe[h][1]), z = (float)(p[2] - pe[h][2]);
      float r, ri;
      dist_inv(x * x + y * y + z * z, r, ri);
      float gf = 0;
      cusp_f32(ee[0], ((j < S.nup) != eup) ? ee[0].cu[0] : ee[0].cl[0], r, ri, u, gf);
      poly4_f32(ee[1], r, ri, u, gf);
      gx += gf * x;
      gy += gf * y;
      gz += gf * z;
    }
  }
  u = wsumf(u);
  g[0] = wsumf(gx);
  g[1] = wsumf(gy);
  g[2] = wsumf(gz);
  return u;
}

// basis_batch_lap in FP32 from a list of (meta, f0) records.
template <bool FG>
__device__ inline int panel_basis_f32(const DevSys& S, const float* spline, const double* tabs, const double* apos,
                                      const double p[3], const int2* list, int i0, int nact, int n, float* chi, int* roff,
                                      int cap, int* nfun, int lane) {
  const int i = i0 + lane;
  int2 d = make_int2(0, 0);
  int nf = 0;
  if (i < nact) {
    d = list[i];
    nf = shl_nf(d.x);
  }
  int tot;
  const int at = wave_excl_scan(nf, lane, &tot);
  const bool fit = nf > 0 && at + nf <= cap;
  const int take = __popcll(__ballot(fit));
  *nfun = take ? __builtin_amdgcn_readlane(at + nf, take - 1) : 0;
  if (fit) {
    const int tab = shl_table(d.x);
    const double* ap = apos + 3 * shl_atom(d.x);
    const double x = p[0] - ap[0], y = p[1] - ap[1], z = p[2] - ap[2];
    const double r = sqrt(x * x + y * y + z * z);
    int iv = (int)(r * tabs[2 * tab]);
    iv = iv < 0 ? 0 : (iv >= S.nint ? S.nint - 1 : iv);
    const float* c = spline + ((size_t)tab * S.nint + iv) * 4;
    const float c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
    const float rf = (float)r, xf = (float)x, yf = (float)y, zf = (float)z;
    const float h = rf - iv * (float)tabs[2 * tab + 1];
    const float f = c0 + h * (c1 + h * (c2 + h * c3));
    const float fd = (c1 + h * (2.f * c2 + h * (3.f * c3))) / rf;
    const float f2 = 2.f * c2 + 6.f * h * c3;
    shell_lap<float, FG>(shl_sym(d.x), f, fd, f2, xf, yf, zf, chi + at, cap);
    for (int q = 0; q < nf; q++) roff[at + q] = (d.y + q) * n * (int)sizeof(float);
  }
  return take;
}
__device__ inline void panel_lcao_f32(const float* C, const int* roff, const float* chi, int cap, int nfun, float acc[5],
                                      int lane, int u) {
  if (u == 8) lcao_batch<float, 8>(C, roff, chi, cap, nfun, acc, lane);
  else if (u == 16) lcao_batch<float, 16>(C, roff, chi, cap, nfun, acc, lane);
  else lcao_batch<float, 4>(C, roff, chi, cap, nfun, acc, lane);
}

// One Sherman-Morrison update of a lane's part of a row: t = row . phi (four partial sums over the
// columns modulo 4), row += rowb * (t * nri), nri = -1/R.  phi, rowb: the lane's own values in LDS.
template <int NS>
__device__ inline void mx_update(float a[PanelMx<NS>::EPT], const float* phi, const float* rowb, float nri, bool own,
                                 float f) {
  constexpr int EPT = PanelMx<NS>::EPT, TPR = PanelMx<NS>::TPR;
  float tk;
  if constexpr (TPR == 4) {
    float t = 0;
#pragma unroll
    for (int i = 0; i < EPT; i++) t += a[i] * phi[i];
    t += dpp_f<kDppXor1>(t);
    tk = t + dpp_f<kDppXor2>(t);
  } else {
    float t0 = 0, t1 = 0;
#pragma unroll
    for (int i = 0; i < EPT; i += 2) {
      t0 += a[i] * phi[i];
      t1 += a[i + 1] * phi[i + 1];
    }
    const float t = t0 + t1;
    tk = t + dpp_f<kDppXor1>(t);
  }
  const float pk = tk * nri;
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const float rb = rowb[i];
    const float v = fmaf(rb, pk, a[i]);
    a[i] = own ? rb * f : v;
  }
}

template <int NS>
__device__ inline void mx_row_load(const float* row, int n, int q, float a[PanelMx<NS>::EPT]) {
#pragma unroll
  for (int i = 0; i < PanelMx<NS>::EPT; i++) {
    const int c = lane_col<NS>(q, i);
    a[i] = c < n ? row[c] : 0.f;
  }
}
template <int NS>
__device__ inline void mx_row_store(float* row, int n, int q, const float a[PanelMx<NS>::EPT]) {
#pragma unroll
  for (int i = 0; i < PanelMx<NS>::EPT; i++) {
    const int c = lane_col<NS>(q, i);
    if (c < n) row[c] = a[i];
  }
}

// The accepted updates (bits of accm) of the panel rows from kp applied to the 16 rows from 16 g,
// in order: phi_j from the MO cache's value rows (mo0: electron 0 of the spin), the inverse row
// that update j used from row kp + j of ig, -1/R_j in nri.
template <int NS>
__device__ inline void mx_flush(float* ig, const float* mo0, int nsp, int n, int g, int kp, unsigned accm, const float* nri,
                                float* stage, int lane) {
  keep_local(lane);
  typedef PanelMx<NS> D;
  const int r = lane / D::TPR, q = lane % D::TPR, row = 16 * g + r;
  float a[D::EPT];
#pragma unroll
  for (int i = 0; i < D::EPT; i++) a[i] = 0.f;
  if (row < n) mx_row_load<NS>(ig + (size_t)row * nsp, n, q, a);
  const int pc = perm_col<NS>(lane);
  unsigned left = accm;
  float fp[kMxStage], fr[kMxStage];
  auto fetch = [&]() {
    unsigned m = left;
#pragma unroll
    for (int s = 0; s < kMxStage; s++) {
      fp[s] = fr[s] = 0.f;
      if (m) {
        const int k = kp + __ffs((int)m) - 1;
        m &= m - 1;
        if (lane < n) {
          fp[s] = mo0[(size_t)k * 5 * nsp + lane];
          fr[s] = ig[(size_t)k * nsp + lane];
        }
      }
    }
  };
  fetch();
  while (left) {
    wave_sync();
#pragma unroll
    for (int s = 0; s < kMxStage; s++) {
      stage[(2 * s) * NS + pc] = fp[s];
      stage[(2 * s + 1) * NS + pc] = fr[s];
    }
    wave_sync();
    unsigned m = left;
#pragma unroll
    for (int s = 0; s < kMxStage; s++) left &= left - 1;
    if (left) fetch();
#pragma unroll
    for (int s = 0; s < kMxStage; s++)
      if (m) {
        const int j = __ffs((int)m) - 1;
        m &= m - 1;
        mx_update<NS>(a, stage + (2 * s) * NS + q * D::EPT, stage + (2 * s + 1) * NS + q * D::EPT, nri[j], false, 0.f);
      }
  }
  if (row < n) mx_row_store<NS>(ig + (size_t)row * nsp, n, q, a);
}

// The moves of walker w's spin A.s by one wavefront.  sh: the block's shared LDS, own: the
// walker's region, Cl: the spin's coefficients in LDS (STAGE).  u: coefficient loads in flight.
template <int NS, int DEPTH, bool JP, bool STAGE, bool SHL = true>
__device__ __forceinline__ void sweep_mxp_body(const DevSys& S, const MixedTables& M, const DevWalkers& W,
                                               const SweepArgs& A, int w, int lane, char* sh, const float* Cl, char* own,
                                               int u) {
  typedef PanelMx<NS> D;
  constexpr int P = D::P, TPR = D::TPR, EPT = D::EPT, cap = cap_mx(JP);
  const int ne = S.ne, s = A.s, n = s ? S.ndn : S.nup, nsp = S.nsp, off = s ? S.nup : 0;
  const double* apos = (const double*)sh;
  const double* epos = apos + 3 * S.na;
  const double* tabs = epos + 3 * S.na;
  const ShellLds* shl;
  if constexpr (SHL) shl = (const ShellLds*)(tabs + 2 * S.ntab);
  else shl = S.shl;
  float* chi = (float*)own;
  int* roff = (int*)(chi + 5 * cap);
  int2* list = (int2*)(roff + cap);
  double* rnd = (double*)((char*)list + lds_round16((size_t)(S.nsh + 64) * 8));
  float* phib = (float*)(rnd + P * DEPTH * 4);
  float* rowk = phib + NS;
  float* nri = (float*)((char*)phib + lds_round16((size_t)2 * NS * 4));
  float* stage = nri + 16;
  // electron positions of this lane's Jastrow partners (and of the electrons that move)
  double pe[2][3];
#pragma unroll
  for (int h = 0; h < 2; h++)
    for (int d = 0; d < 3; d++) {
      const int j = lane + h * kWave;
      pe[h][d] = j < ne ? W.pos[((size_t)w * ne + j) * 3 + d] : 0.0;
    }
  double logdet = W.logdet[2 * w + s], sgn = W.sgn[2 * w + s], dprod = 1.0;
  int nacc = 0;
  float* mog = W.mof + (size_t)w * ne * 5 * nsp;
  float* ig = W.invf + ((size_t)w * 2 + s) * nsp * nsp;
  const bool mine = lane < n, full = A.dets || A.keep;
  const double tau = A.tau, stau = sqrt(tau);
  float m1 = 0, m2 = 0, m3 = 0;
  if (mine && A.k0 < A.k1) {
    const float* mr = mog + (size_t)(off + A.k0) * 5 * nsp + lane;
    m1 = mr[nsp];
    m2 = mr[2 * nsp];
    m3 = mr[3 * nsp];
  }
  const int r = lane / TPR, q = lane % TPR, pc = perm_col<NS>(lane);
  const bool prow = lane < P * TPR;
  float a[EPT];
  for (int kp = A.k0 / P * P; kp < A.k1; kp += P) {
    const int ka = max(kp, A.k0), kb = min(kp + P, A.k1);
    unsigned accm = 0;
#pragma unroll
    for (int i = 0; i < EPT; i++) a[i] = 0;
    if (prow && kp + r < n) mx_row_load<NS>(ig + (size_t)(kp + r) * nsp, n, q, a);
    // whether rows outside the panel take its updates
    const bool flush = P < NS && (full || kb < A.k1);
    // random numbers of the panel's moves, one move and stage per lane (the streams of sweep_randoms)
    for (int i = lane; i < (kb - ka) * DEPTH; i += kWave) {
      const unsigned st = step_of(A.step, A.stepp), ke = (unsigned)(off + ka + i / DEPTH);
      const int d = i % DEPTH;
      double g[3];
      gauss3(A.seed, (unsigned)w, st, ke, (d ? TAG_GAUSS2 : TAG_GAUSS1) | (A.sweep << 8), g);
      double* o = rnd + 4 * i;
      o[0] = g[0];
      o[1] = g[1];
      o[2] = g[2];
      o[3] = uniform(A.seed, (unsigned)w, st, ke, (d ? TAG_ACC2 : TAG_ACC1) | (A.sweep << 8));
    }
    for (int k = ka; k < kb; k++) {
      const int e = off + k;
      if (prow && r == k - kp) {
#pragma unroll
        for (int i = 0; i < EPT; i++) rowk[q * EPT + i] = a[i];
      }
      wave_sync();
      const float rk = mine ? rowk[pc] : 0.f;
      double r0[3];
#pragma unroll
      for (int d = 0; d < 3; d++) r0[d] = e < kWave ? readlane_d(pe[0][d], e) : readlane_d(pe[1][d], e - kWave);
      float gj0[3];
      const float u0 = JP ? jastrow_usual_f32(S, e, r0, pe, gj0, lane, epos) : jastrow_e_freg(S, e, r0, pe, gj0, lane, epos, 3);
      const double d0[3] = {(double)(wsumf(rk * m1) + gj0[0]), (double)(wsumf(rk * m2) + gj0[1]),
                            (double)(wsumf(rk * m3) + gj0[2])};
      float phi[5];
      double r1[3], d1[3], ln1 = 0;
      float R = 0;
      bool accepted = false;
      double acc_first = 0, g2first = 0;
      for (int dep = 1; dep <= DEPTH && !accepted; dep++) {
        const double t = dep == 1 ? tau : tau * 0.5, st = dep == 1 ? stau : sqrt(tau * 0.5);
        const double* rq = rnd + 4 * ((k - ka) * DEPTH + (dep - 1));
        double dr[3], rn[3], dn[3];
        lim_drift(d0, t, dr);
        for (int d = 0; d < 3; d++) rn[d] = r0[d] + (rq[d] * st + dr[d]);
        for (int c = 0; c < 5; c++) phi[c] = 0.f;
        const int nact = panel_active<kWave>(S, shl, apos, rn, list, lane);
        wave_sync();
        for (int i0 = 0; i0 < nact;) {
          int nfun;
          const int take =
              panel_basis_f32<!JP>(S, M.spline, tabs, apos, rn, list, i0, nact, n, chi, roff, cap, &nfun, lane);
          wave_sync();
          if (mine) panel_lcao_f32(STAGE ? Cl : M.Cf[s], roff, chi, cap, nfun, phi, lane, u);
          wave_sync();
          i0 += take;
        }
        const float t0 = wsumf(rk * phi[0]);
        const float t1 = wsumf(rk * phi[1]), t2 = wsumf(rk * phi[2]), t3 = wsumf(rk * phi[3]);
        float gj[3];
        const float un = JP ? jastrow_usual_f32(S, e, rn, pe, gj, lane, epos) : jastrow_e_freg(S, e, rn, pe, gj, lane, epos, 3);
        const float it0 = 1.f / t0;
        dn[0] = (double)(t1 * it0 + gj[0]);
        dn[1] = (double)(t2 * it0 + gj[1]);
        dn[2] = (double)(t3 * it0 + gj[2]);
        const bool neg = t0 < 0;
        // the proposal's displacement from the drifted point is the drawn Gaussian: its own
        // Green's function exponent is -|g|^2 / 2
        const double g2 = -0.5 * (rq[0] * rq[0] + rq[1] * rq[1] + rq[2] * rq[2]);
        double acc;
        if constexpr (DEPTH == 1) {
          // |ratio|^2 exp(dtrans) as t0^2 exp(2 du + dtrans): one exponential, no logarithm
          const double td = (double)t0;
          acc = (A.restrict_nodes && neg)
                    ? 0.0
                    : fmin(1.0, td * td * exp(2.0 * (double)(un - u0) + (trans_fast(rn, dn, r0, t) - g2)));
        } else if (dep == 1) {
          const double lnn = log(fabs((double)t0)) + (double)(un - u0);
          const double rr = exp(lnn);
          acc = (A.restrict_nodes && neg) ? 0.0 : fmin(1.0, rr * rr * exp(trans_fast(rn, dn, r0, t) - g2));
          acc_first = acc;
          g2first = g2;
          for (int d = 0; d < 3; d++) r1[d] = rn[d], d1[d] = dn[d];
          ln1 = lnn;
        } else {
          // delayed rejection through the rejected first point (src/method/Split_sample.cpp:302-373)
          const double lnn = log(fabs((double)t0)) + (double)(un - u0);
          const double rr = exp(lnn);
          const double tn1 = trans_fast(rn, dn, r1, tau);
          const double pt = (tn1 - g2first) + (trans_fast(rn, dn, r0, t) - g2);
          const double r21 = exp(ln1 - lnn);
          const double a21 = fmin(1.0, r21 * r21 * exp(trans_fast(r1, d1, rn, tau) - tn1));
          const double num = 1 - a21, den = 1 - acc_first;
          if (A.restrict_nodes && neg) acc = 0;
          else if (fabs(den) < 1e-10) acc = fabs(num) < 1e-10 ? 0.0 : 1.0;
          else acc = fmin(1.0, rr * rr * exp(pt) * num / den);
        }
        if (acc + rq[3] > 1.0) {
          accepted = true;
          R = t0;
          for (int d = 0; d < 3; d++) r1[d] = rn[d];
        }
      }
      if (accepted) {
        if (lane < NS) phib[pc] = mine ? phi[0] : 0.f;
        wave_sync();
        const float f = 1.f / R, nr = -1.f / R;
        if (prow) mx_update<NS>(a, phib + q * EPT, rowk + q * EPT, nr, r == k - kp, f);
        if (mine) {
          float* mr = mog + (size_t)e * 5 * nsp + lane;
          for (int c = 0; c < 5; c++) mr[c * nsp] = phi[c];
          // the row this update used, kept in row k's own (already loaded) place
          if (flush) ig[(size_t)k * nsp + lane] = rk;
        }
        if constexpr (P < NS)
          if (lane == 0) nri[k - kp] = nr;
        // accepted ratios multiply into dprod, folded into log|det| before it could overflow
        dprod *= (double)R;
        if (!(fabs(dprod) < 0x1p+512 && fabs(dprod) > 0x1p-512)) {
          logdet += log(fabs(dprod));
          dprod = 1.0;
        }
        if (R < 0) sgn = -sgn;
        nacc++;
        accm |= 1u << (k - kp);
        if (lane == (e & (kWave - 1))) {
          if (e < kWave)
            for (int d = 0; d < 3; d++) pe[0][d] = r1[d];
          else
            for (int d = 0; d < 3; d++) pe[1][d] = r1[d];
        }
      }
      if (mine && k + 1 < A.k1) {
        const float* mr = mog + (size_t)(e + 1) * 5 * nsp + lane;
        m1 = mr[nsp];
        m2 = mr[2 * nsp];
        m3 = mr[3 * nsp];
      }
      wave_sync();
    }
    if constexpr (P < NS) {
      if (flush) {
        __threadfence_block();
        for (int g = 0; 16 * g < n; g++) {
          if (16 * g == kp || !accm) continue;
          if (full || (16 * g >= kb && 16 * g < A.k1))
            mx_flush<NS>(ig, mog + (size_t)off * 5 * nsp, nsp, n, g, kp, accm, nri, stage, lane);
        }
        __threadfence_block();
      }
    }
    if (full && prow && kp + r < n) mx_row_store<NS>(ig + (size_t)(kp + r) * nsp, n, q, a);
    wave_sync();
  }
  if (A.dets) {
    // determinant parts of the local energy (write_det_parts): lane = electron
    __threadfence_block();
    wave_sync();
    if (mine) {
      const int e = off + lane;
      const float* ir = ig + (size_t)lane * nsp;
      const float* mr = mog + (size_t)e * 5 * nsp;
      double t[4] = {0, 0, 0, 0};
      int j = 0;
      if (nsp % 4 == 0) {
        typedef float tv4 __attribute__((ext_vector_type(4)));
        for (; j + 4 <= n; j += 4) {
          const tv4 iv = *(const tv4*)(ir + j);
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const tv4 mv = *(const tv4*)(mr + (size_t)(c + 1) * nsp + j);
#pragma unroll
            for (int i = 0; i < 4; i++) t[c] += (double)mv[i] * (double)iv[i];
          }
        }
      }
      for (; j < n; j++)
#pragma unroll
        for (int c = 0; c < 4; c++) t[c] += (double)mr[(size_t)(c + 1) * nsp + j] * (double)ir[j];
      double* o = W.dgl + ((size_t)w * ne + e) * 4;
      for (int c = 0; c < 4; c++) o[c] = t[c];
    }
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int j = lane + h * kWave;
    if (j < ne)
      for (int d = 0; d < 3; d++) W.pos[((size_t)w * ne + j) * 3 + d] = pe[h][d];
  }
  logdet += log(fabs(dprod));
  if (lane == 0) {
    W.logdet[2 * w + s] = logdet;
    W.sgn[2 * w + s] = sgn;
    W.acc[w] += nacc;
  }
}

// The block's shared LDS: the tables of panel_stage, and with STAGE the spin's coefficients.
template <bool STAGE, bool SHL = true>
__device__ inline const float* panel_mx_stage(const DevSys& S, const MixedTables& M, int s, char* sh, int t, int nt) {
  panel_stage(S, sh, SHL ? 1 : 2, t, nt);
  float* Cl = (float*)(sh + lds_round16(panel_shared_lds(S.na, S.nsh, S.ntab, 1)));
  if constexpr (STAGE) {
    const int nc = S.nb * (s ? S.ndn : S.nup);
    const float4* src4 = reinterpret_cast<const float4*>(M.Cf[s]);
    float4* dst4 = reinterpret_cast<float4*>(Cl);
    for (int i = t; i < nc / 4; i += nt) dst4[i] = src4[i];
    for (int i = (nc / 4) * 4 + t; i < nc; i += nt) Cl[i] = M.Cf[s][i];
  }
  return Cl;
}

// Four waves per SIMD (128 registers, 8 spilled at 64 electrons of a spin) for the usual DMC sweep;
// the delayed-rejection and general forms would spill a hundred there and run three.
template <int NS, int DEPTH, bool JP, bool STAGE, bool SHL = true>
__global__ __launch_bounds__(64 * (SHL ? kPanelWpb : 1), DEPTH == 1 && JP ? 4 : 3) void k_sweep_mxp(
    DevSys S, MixedTables M, DevWalkers W, SweepArgs A, int u) {
  extern __shared__ double ldsp[];
  const int wpb = (int)blockDim.x >> 6;
  char* sh = (char*)ldsp;
  const float* Cl = panel_mx_stage<STAGE, SHL>(S, M, A.s, sh, (int)threadIdx.x, (int)blockDim.x);
  __syncthreads();
  const int wid = (int)threadIdx.x >> 6, w = (int)blockIdx.x * wpb + wid;
  if (w >= W.nw) return;
  char* own = sh + panel_mx_shared_lds(S.na, SHL ? S.nsh : 0, S.ntab, STAGE ? S.nb : 0, S.nsp) +
              (size_t)wid * panel_mx_walker_lds(S.nsh, NS, DEPTH, JP);
  sweep_mxp_body<NS, DEPTH, JP, STAGE, SHL>(S, M, W, A, w, (int)threadIdx.x & 63, sh, Cl, own, u);
}

}  // namespace qw
