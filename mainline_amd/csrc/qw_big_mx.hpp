// Mixed-precision sweep of one spin channel with 65 to 256 electrons (the arithmetic of one
// wavefront per walker over a device-memory inverse, bit for bit).
//
//   k_sweep_mxb<NW, DEPTH, JP>  moves of at most kBigPanel electrons (src/method/
//       Split_sample.cpp:302-540, src/program_utils/MatrixAlgebrac.cpp:766-838) by NW wavefronts
//       per walker: wavefront 0 evaluates the Jastrow while the others fill the basis tiles, all of
//       them contract the LCAO (64 orbitals each), wavefront 1 updates the panel's rows
//   k_flush_mx<NS>  the updates of a launch applied to the other rows, in order, a lane per row
//       with the row in registers, and the determinant parts of the local energy
//
// Only the rows of the launch's electrons are held (LDS) and updated per accepted move; each
// update's row and -1/R are kept (DevWalkers::pend, pnri).  The other rows are brought up to date
// by k_flush_mx only where they are still used: those of electrons that move before the next FP64
// recompute, and all of them at the end of a sweep, whose determinant parts are read.
//
// What bounds it: vector issue (6300 wave instructions a move at 192 electrons) with a serial chain
// of old Jastrow, drift, new Jastrow or basis, LCAO and ratio per move; LDS keeps six walkers of 192
// electrons (26 KB each) or two of 512 on a compute unit.  One wavefront per walker streaming its
// inverse from device memory on every accepted move left one such wave per SIMD waiting on memory.
// Measured, one DMC step of 1024 walkers (all kernels): 256 electrons 22.0 -> 12.8 ms, 512
// electrons 233 -> 98 ms (its sweeps and updates 195 -> 60 ms).
#pragma once
#include "qw_big.hpp"
#include "qw_panel_mx.hpp"

namespace qw {

constexpr int kBigPanel = 32;  // moves of one launch at most

// floats per panel row: 16-byte chunks, an odd number of them (a lane per row: no bank conflicts)
__host__ __device__ inline int big_ldp(int n) { return 4 * ((n + 3) / 4 | 1); }
// active-shell lists and, once they are used, the new value rows (4 x 64 NW) over them
__host__ __device__ inline size_t big_list_bytes(int nsh, int nw) {
  const size_t l = lds_round16((size_t)nsh * 8), v = (size_t)4 * 64 * nw * 4;
  return l > v ? l : v;
}
// LDS of one walker: positions, atoms, spacings | draws | panel rows | lists or value rows |
// basis tiles | sums exchanged between the wavefronts.  192 electrons: 26.3 KB, six walkers per
// compute unit.
__host__ __device__ inline size_t sweep_mxb_lds_bytes(int ne, int na, int nsh, int ntab, int nmax, int nw, int depth,
                                                           bool usual) {
  return lds_round16((size_t)(3 * ne + 6 * na + 2 * ntab) * 8) + (size_t)kBigPanel * 32 * depth +
         (size_t)kBigPanel * big_ldp(nmax) * 4 + big_list_bytes(nsh, nw) + (size_t)(nw - 1) * cap_mx(usual) * 24 + 128;
}

// jastrow_e_t<float, false> for the usual Jastrow: the same terms in the same order.
__device__ inline float jastrow_big_usual(const DevSys& S, int e, const double p[3], const double* pos, float g[3],
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
  for (int j = lane; j < S.ne; j += kWave) {
    if (j == e) continue;
    const float x = (float)(p[0] - pos[3 * j]), y = (float)(p[1] - pos[3 * j + 1]), z = (float)(p[2] - pos[3 * j + 2]);
    float r, ri;
    dist_inv(x * x + y * y + z * z, r, ri);
    float gf = 0;
    cusp_f32(ee[0], ((j < S.nup) != eup) ? ee[0].cu[0] : ee[0].cl[0], r, ri, u, gf);
    gx += gf * x;
    gy += gf * y;
    gz += gf * z;
  }
  for (int j = lane; j < S.ne; j += kWave) {
    if (j == e) continue;
    const float x = (float)(p[0] - pos[3 * j]), y = (float)(p[1] - pos[3 * j + 1]), z = (float)(p[2] - pos[3 * j + 2]);
    float r, ri;
    dist_inv(x * x + y * y + z * z, r, ri);
    float gf = 0;
    poly4_f32(ee[1], r, ri, u, gf);
    gx += gf * x;
    gy += gf * y;
    gz += gf * z;
  }
  u = wsumf(u);
  g[0] = wsumf(gx);
  g[1] = wsumf(gy);
  g[2] = wsumf(gz);
  return u;
}

// Active shells of [lo, hi) at p, in shell order, into the wavefront's list.
__device__ inline int big_active(const ShellLds* shl, const double* apos, const double p[3], int lo, int hi, int2* list,
                                 int lane) {
  int n = 0;
  for (int s0 = lo; s0 < hi; s0 += kWave) {
    const int sh = s0 + lane;
    bool act = false;
    ShellLds d;
    if (sh < hi) {
      d = shl[sh];
      const double* ap = apos + 3 * shl_atom(d.meta);
      const double x = p[0] - ap[0], y = p[1] - ap[1], z = p[2] - ap[2];
      act = x * x + y * y + z * z < d.rc2;
    }
    const unsigned long long m = __ballot(act);
    if (act)
      list[n + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
          make_int2(d.meta, d.f0);
    n += __popcll(m);
  }
  return n;
}

// The moves [A.k0, A.k1) (at most kBigPanel) of walker w's spin A.s by 64 NW threads.  C[s]:
// coefficients; nmax: electrons of the larger spin.  A.keep: k_flush_mx follows.
template <int NW, int DEPTH, bool JP>
__device__ __forceinline__ void sweep_mxb_body(const DevSys& S, const MixedTables& M, const DevWalkers& W,
                                               const SweepArgs& A, int w, int t, char* base) {
  static_assert(NW == 2 || NW == 4, "wavefronts per walker");
  constexpr int NR = NW, NB = NW - 1, cap = cap_mx(JP), NT = 64 * NW;
  const int lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ne = S.ne, s = A.s, n = s ? S.ndn : S.nup, nsp = S.nsp, off = s ? S.nup : 0;
  const int ldp = big_ldp(S.nup > S.ndn ? S.nup : S.ndn), np = A.k1 - A.k0;
  double* pos = (double*)base;
  double* apos = pos + 3 * ne;
  double* epos = apos + 3 * S.na;
  double* tabs = epos + 3 * S.na;
  double* draw = (double*)(base + lds_round16((size_t)(3 * ne + 6 * S.na + 2 * S.ntab) * 8));  // [np][DEPTH][4]
  float* prow = (float*)(draw + kBigPanel * 4 * DEPTH);
  // [4][64 NW], over the lists: every wavefront reads the values of a stage, so a block barrier lies
  // between those reads and the next stage's (or move's) lists
  float* ph = prow + kBigPanel * ldp;
  int2* list0 = (int2*)ph;
  float* chi0 = (float*)((char*)ph + big_list_bytes(S.nsh, NW));
  int* roff0 = (int*)(chi0 + (size_t)NB * 5 * cap);
  double* gdl = (double*)(roff0 + NB * cap);  // [3]
  float* jl = (float*)(gdl + 4);  // Jastrow value and gradient: old point, each stage's new one
  int* cnt = (int*)(jl + 4 + 4 * DEPTH);  // [NB][2] functions in a tile, shells left
  for (int i = t; i < 3 * ne; i += NT) pos[i] = W.pos[(size_t)w * ne * 3 + i];
  for (int i = t; i < 3 * S.na; i += NT) {
    apos[i] = S.atom_pos[i];
    epos[i] = S.eit_pos[i];
  }
  for (int i = t; i < 2 * S.ntab; i += NT) tabs[i] = S.tabs[i];
  float* ig = W.invf + ((size_t)w * 2 + s) * nsp * nsp;
  float* mog = W.mof + (size_t)w * ne * 5 * nsp;
  float* pend = A.keep ? W.pend + (size_t)w * kBigPanel * nsp : nullptr;
  for (int r = 0; r < np; r++)
    for (int j = t; j < n; j += NT) prow[r * ldp + j] = ig[(size_t)(A.k0 + r) * nsp + j];
  const unsigned sp = step_of(A.step, A.stepp);
  // every move's Gaussians and uniform, a lane per move
  for (int r = t; r < np * DEPTH; r += NT) {
    const int d = r % DEPTH;
    const unsigned e = (unsigned)(off + A.k0 + r / DEPTH);
    double g[3];
    gauss3(A.seed, (unsigned)w, sp, e, (d ? TAG_GAUSS2 : TAG_GAUSS1) | (A.sweep << 8), g);
    for (int c = 0; c < 3; c++) draw[4 * r + c] = g[c];
    draw[4 * r + 3] = uniform(A.seed, (unsigned)w, sp, e, (d ? TAG_ACC2 : TAG_ACC1) | (A.sweep << 8));
  }
  double logdet = W.logdet[2 * w + s], sgn = W.sgn[2 * w + s];
  int nacc = 0;
  const double tau = A.tau, stau = sqrt(tau);
  // basis wavefronts 1..NW-1 take consecutive shares of the shells
  const int bw = wv - 1, lo = bw >= 0 ? S.nsh * bw / NB : 0, hi = bw >= 0 ? S.nsh * (bw + 1) / NB : 0;
  const int b0 = bw > 0 ? bw : 0;
  float* chi = chi0 + (size_t)b0 * 5 * cap;
  int* roff = roff0 + b0 * cap;
  int2* list = list0 + lo;
  const bool mine = t < n;
  __syncthreads();
  for (int k = A.k0; k < A.k1; k++) {
    const int e = off + k;
    const float* rowk = prow + (k - A.k0) * ldp;
    const double r0[3] = {pos[3 * e], pos[3 * e + 1], pos[3 * e + 2]};
    if (wv == 0) {
      float g[3];
      const float u = JP ? jastrow_big_usual(S, e, r0, pos, g, lane, epos)
                         : jastrow_e_t<float, false>(S, S.eef, S.eitf, e, r0, pos, g, nullptr, lane, epos, 3);
      if (lane == 0) {
        jl[0] = u;
        jl[1] = g[0];
        jl[2] = g[1];
        jl[3] = g[2];
      }
    } else if (wv == 1) {
      double gd[3] = {0, 0, 0};
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const int j = lane + kWave * r;
        if (j < n)
          for (int c = 0; c < 3; c++) gd[c] += (double)rowk[j] * (double)mog[((size_t)e * 5 + 1 + c) * nsp + j];
      }
      for (int c = 0; c < 3; c++) gd[c] = wsum(gd[c]);
      if (lane == 0)
        for (int c = 0; c < 3; c++) gdl[c] = gd[c];
    }
    __syncthreads();
    const double u0 = (double)jl[0];
    const double d0[3] = {gdl[0] + (double)jl[1], gdl[1] + (double)jl[2], gdl[2] + (double)jl[3]};
    double rk[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) rk[r] = lane + kWave * r < n ? (double)rowk[lane + kWave * r] : 0.0;
    float acc[5];
    double r1[3], d1[3], ln1 = 0, Rt = 0;
    bool accepted = false;
    double acc_first = 0, g2first = 0;
    for (int dep = 1; dep <= DEPTH && !accepted; dep++) {
      if (dep > 1) __syncthreads();  // the first stage's values are read (accepted is the block's)
      const double tt = dep == 1 ? tau : tau * 0.5, st = dep == 1 ? stau : sqrt(tau * 0.5);
      double dr[3], rn[3], dn[3];
      const double* dw = draw + 4 * ((k - A.k0) * DEPTH + dep - 1);
      const double g[3] = {dw[0], dw[1], dw[2]};
      lim_drift(d0, tt, dr);
      for (int d = 0; d < 3; d++) rn[d] = r0[d] + (g[d] * st + dr[d]);
      for (int c = 0; c < 5; c++) acc[c] = 0.f;
      int nact = 0, i0 = 0;
      if (wv == 0) {
        float g2[3];
        const float u = JP ? jastrow_big_usual(S, e, rn, pos, g2, lane, epos)
                           : jastrow_e_t<float, false>(S, S.eef, S.eitf, e, rn, pos, g2, nullptr, lane, epos, 3);
        if (lane == 0) {
          jl[4 * dep] = u;
          jl[4 * dep + 1] = g2[0];
          jl[4 * dep + 2] = g2[1];
          jl[4 * dep + 3] = g2[2];
        }
      } else {
        nact = big_active(S.shl, apos, rn, lo, hi, list, lane);
        wave_sync();
        int nfun = 0;
        if (nact > 0) i0 = panel_basis_f32<!JP>(S, M.spline, tabs, apos, rn, list, 0, nact, n, chi, roff, cap, &nfun, lane);
        if (lane == 0) {
          cnt[2 * bw] = nfun;
          cnt[2 * bw + 1] = nact - i0;
        }
      }
      __syncthreads();
      // the tiles in shell order; a share that did not fit its tile is continued before the next
#pragma unroll
      for (int x = 0; x < NB; x++) {
        while (true) {
          const int nf = cnt[2 * x], left = cnt[2 * x + 1];
          if (mine)
            lcao_batch<float, 8>(M.Cf[s] + kWave * wv, roff0 + x * cap, chi0 + (size_t)x * 5 * cap, cap, nf, acc, lane);
          if (left <= 0) break;
          __syncthreads();
          if (bw == x) {
            int nfun = 0;
            i0 += panel_basis_f32<!JP>(S, M.spline, tabs, apos, rn, list, i0, nact, n, chi, roff, cap, &nfun, lane);
            if (lane == 0) {
              cnt[2 * bw] = nfun;
              cnt[2 * bw + 1] = nact - i0;
            }
          }
          __syncthreads();
        }
      }
      for (int c = 0; c < 4; c++) ph[c * NT + t] = mine ? acc[c] : 0.f;
      __syncthreads();
      double tv[4] = {0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < NR; r++)
        for (int c = 0; c < 4; c++) tv[c] += rk[r] * (double)ph[c * NT + lane + kWave * r];
      for (int c = 0; c < 4; c++) tv[c] = wsum(tv[c]);
      const double t0 = tv[0], un = (double)jl[4 * dep], it0 = 1.0 / t0;
      dn[0] = tv[1] * it0 + (double)jl[4 * dep + 1];
      dn[1] = tv[2] * it0 + (double)jl[4 * dep + 2];
      dn[2] = tv[3] * it0 + (double)jl[4 * dep + 3];
      const double lnn = log(fabs(t0)) + (un - u0);
      const bool neg = t0 < 0;
      const double gg = -0.5 * (g[0] * g[0] + g[1] * g[1] + g[2] * g[2]);
      double acc_p;
      if (dep == 1) {
        const double rr = exp(lnn);
        acc_p = (A.restrict_nodes && neg) ? 0.0 : fmin(1.0, rr * rr * exp(trans_fast(rn, dn, r0, tt) - gg));
        acc_first = acc_p;
        g2first = gg;
        for (int d = 0; d < 3; d++) r1[d] = rn[d], d1[d] = dn[d];
        ln1 = lnn;
      } else {
        const double rr = exp(lnn);
        const double tn1 = trans_fast(rn, dn, r1, tau);
        const double pt = (tn1 - g2first) + (trans_fast(rn, dn, r0, tt) - gg);
        const double r21 = exp(ln1 - lnn);
        const double a21 = fmin(1.0, r21 * r21 * exp(trans_fast(r1, d1, rn, tau) - tn1));
        const double num = 1 - a21, den = 1 - acc_first;
        if (A.restrict_nodes && neg) acc_p = 0;
        else if (fabs(den) < 1e-10) acc_p = fabs(num) < 1e-10 ? 0.0 : 1.0;
        else acc_p = fmin(1.0, rr * rr * exp(pt) * num / den);
      }
      if (acc_p + dw[3] > 1.0) {
        accepted = true;
        Rt = t0;
        for (int d = 0; d < 3; d++) r1[d] = rn[d];
      }
    }
    if (accepted) {
      if (mine)
        for (int c = 0; c < 5; c++) mog[((size_t)e * 5 + c) * nsp + t] = acc[c];
      if (wv == 1) {
        // Sherman-Morrison on the panel's rows (those still to move, or all when they are kept):
        // a lane per row for the dot products, then the wavefront over the columns
        const int r_lo = A.keep ? 0 : k - A.k0;
        const double nri = -1.0 / Rt;
        double pk = 0;
        if (lane >= r_lo && lane < np) {
          const float* row = prow + lane * ldp;
          double tk = 0;
          int j = 0;
          typedef float tv4 __attribute__((ext_vector_type(4)));
          for (; j + 4 <= n; j += 4) {
            const tv4 a = *(const tv4*)(row + j);
            const tv4 b = *(const tv4*)(ph + j);
#pragma unroll
            for (int q = 0; q < 4; q++) tk += (double)a[q] * (double)b[q];
          }
          for (; j < n; j++) tk += (double)row[j] * (double)ph[j];
          pk = tk * nri;
        }
        for (int r = r_lo; r < np; r++) {
          float* row = prow + r * ldp;
          if (r == k - A.k0) {
            const double f = 1.0 / Rt;
#pragma unroll
            for (int x = 0; x < NR; x++)
              if (lane + kWave * x < n) row[lane + kWave * x] = (float)(rk[x] * f);
          } else {
            const double p = readlane_d(pk, r);
#pragma unroll
            for (int x = 0; x < NR; x++) {
              const int j = lane + kWave * x;
              if (j < n) row[j] = (float)((double)row[j] + rk[x] * p);
            }
          }
        }
        if (pend) {
#pragma unroll
          for (int x = 0; x < NR; x++)
            if (lane + kWave * x < n) pend[(size_t)(k - A.k0) * nsp + lane + kWave * x] = (float)rk[x];
          if (lane == 0) W.pnri[(size_t)w * kBigPanel + k - A.k0] = nri;
        }
        wave_sync();
      }
      logdet += log(fabs(Rt));
      if (Rt < 0) sgn = -sgn;
      nacc++;
      if (t < 3) pos[3 * e + t] = r1[t];
    } else if (pend && wv == 1 && lane == 0) {
      W.pnri[(size_t)w * kBigPanel + k - A.k0] = 0.0;  // no update
    }
    if (wv == 0) wave_sync();
    // wavefront 0 goes on to the next old Jastrow with its own position write, wavefront 1 to the
    // next drift with its own rows; the next barrier shows both to the others
  }
  __syncthreads();
  if (A.keep)
    for (int r = 0; r < np; r++)
      for (int j = t; j < n; j += NT) ig[(size_t)(A.k0 + r) * nsp + j] = prow[r * ldp + j];
  for (int i = t; i < 3 * ne; i += NT) W.pos[(size_t)w * ne * 3 + i] = pos[i];
  if (t == 0) {
    W.logdet[2 * w + s] = logdet;
    W.sgn[2 * w + s] = sgn;
    W.acc[w] += nacc;
  }
}

template <int NW, int DEPTH, bool JP>
__global__ __launch_bounds__(64 * NW, 4) void k_sweep_mxb(DevSys S, MixedTables M, DevWalkers W, SweepArgs A) {
  extern __shared__ double ldsp[];
  sweep_mxb_body<NW, DEPTH, JP>(S, M, W, A, (int)blockIdx.x, (int)threadIdx.x, (char*)ldsp);
}

// Rows outside the panel that need the updates of a launch ending at move k1, for a spin with n
// electrons recomputed every rf moves: those that move before the next recompute, and all of them
// where the determinant parts are taken (dets: in this sweep) before one; *hi = 0 for none.
__host__ __device__ inline void flush_rows(int n, int k1, int rf, bool dets, int* lo, int* hi) {
  *lo = *hi = 0;
  if (k1 >= n) {
    if (dets) *hi = n;
  } else if (k1 % rf != 0) {
    const int end = (k1 / rf + 1) * rf;
    *lo = dets && end >= n ? 0 : k1;
    *hi = end < n ? end : n;
  }
}

// ---------------------------------------------------------------- k_flush_mx
constexpr int kFlushStage = 4;            // updates staged in LDS at a time
constexpr int kFlushW = 16, kFlushLd = 17;  // columns of a row tile, floats per row of it
template <int NS>
struct FlushLds {
  union {
    struct {
      alignas(16) double phi[kFlushStage][NS];
      alignas(16) double rowb[kFlushStage][NS];
    };
    float tile[NS * kFlushLd];
  };
};
// Columns [j0, j0 + 16) of nrow rows of `src` (stride floats apart) into the tile, zero from column
// n on: 64 consecutive bytes per row instead of a lane per row across the whole matrix.
template <int NS>
__device__ inline void flush_tile_in(const float* src, size_t stride, int nrow, int j0, int n, float* tile, int t) {
  const int j = j0 + (t & 15), r0 = t >> 4;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; i++) {  // all in flight
    const int r = r0 + i * (NS / 16);
    v[i] = r < nrow && j < n ? src[(size_t)r * stride + j] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 16; i++) tile[(r0 + i * (NS / 16)) * kFlushLd + (t & 15)] = v[i];
}
// The updates of the panel [k0, k0 + np) applied in order to the rows [lo, hi) outside it, a lane
// per row (t: thread of the walker, row lo + t) with the row in registers; dets (lo = 0, hi = n):
// then the determinant parts of every row.
template <int NS>
__device__ __forceinline__ void flush_mx_body(const DevSys& S, const DevWalkers& W, int s, int k0, int np, int lo, int hi,
                                              int dets, int w, int t, FlushLds<NS>& L) {
  constexpr int NC = NS / kFlushW;
  const int n = s ? S.ndn : S.nup, nsp = S.nsp, off = s ? S.nup : 0, nrow = hi - lo;
  float* ig = W.invf + ((size_t)w * 2 + s) * nsp * nsp + (size_t)lo * nsp;
  const float* mog = W.mof + (size_t)w * S.ne * 5 * nsp;
  const float* pend = W.pend + (size_t)w * kBigPanel * nsp;
  const int row = lo + t, nc = (n + kFlushW - 1) / kFlushW;
  const bool upd = t < nrow && (row < k0 || row >= k0 + np);
  const bool work = __any(upd);  // some row of this wavefront
  const double nriv = (t & 63) < np ? W.pnri[(size_t)w * kBigPanel + (t & 63)] : 0.0;
  float a[NC][kFlushW];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (c < nc) {
      __syncthreads();
      flush_tile_in<NS>(ig, nsp, nrow, kFlushW * c, n, L.tile, t);
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < kFlushW; j++) a[c][j] = c < nc && t < nrow ? L.tile[t * kFlushLd + j] : 0.f;
  }
  for (int p0 = 0; p0 < np; p0 += kFlushStage) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFlushStage; i++) {
      const bool on = p0 + i < np && t < n;
      L.phi[i][t] = on ? (double)mog[(size_t)(off + k0 + p0 + i) * 5 * nsp + t] : 0.0;
      L.rowb[i][t] = on ? (double)pend[(size_t)(p0 + i) * nsp + t] : 0.0;
    }
    __syncthreads();
    if (!work) continue;
    for (int i = 0; i < kFlushStage && p0 + i < np; i++) {
      const double nri = readlane_d(nriv, p0 + i);
      if (nri == 0.0) continue;  // rejected move
      double tk = 0;
#pragma unroll
      for (int c = 0; c < NC; c++)
        if (c < nc) {
#pragma unroll
          for (int j = 0; j < kFlushW; j++) tk += (double)a[c][j] * L.phi[i][kFlushW * c + j];
        }
      const double pk = tk * nri;
      if (upd) {
#pragma unroll
        for (int c = 0; c < NC; c++)
          if (c < nc) {
#pragma unroll
            for (int j = 0; j < kFlushW; j++)
              a[c][j] = (float)((double)a[c][j] + L.rowb[i][kFlushW * c + j] * pk);
          }
      }
    }
  }
  const int ob = t >> 4, oj = t & 15;  // coalesced: 16 threads per row
#pragma unroll
  for (int c = 0; c < NC; c++)
    if (c < nc) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kFlushW; j++) L.tile[t * kFlushLd + j] = a[c][j];
      __syncthreads();
      if (kFlushW * c + oj < n)
        for (int r = ob; r < nrow; r += NS / 16)
          if (lo + r < k0 || lo + r >= k0 + np) ig[(size_t)r * nsp + kFlushW * c + oj] = L.tile[r * kFlushLd + oj];
    }
  if (!dets) return;
  for (int d = 0; d < 4; d++) {
    double dv = 0;
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (c < nc) {
        __syncthreads();
        flush_tile_in<NS>(mog + ((size_t)off * 5 + d + 1) * nsp, (size_t)5 * nsp, n, kFlushW * c, n, L.tile, t);
        __syncthreads();
        if (t < n) {
#pragma unroll
          for (int j = 0; j < kFlushW; j++) dv += (double)L.tile[t * kFlushLd + j] * (double)a[c][j];
        }
      }
    if (t < n) W.dgl[((size_t)w * S.ne + off + t) * 4 + d] = dv;
  }
}
template <int NS>
__global__ __launch_bounds__(NS, NS == 128 ? 3 : 1) void k_flush_mx(DevSys S, DevWalkers W, int s, int k0, int np, int lo,
                                                                     int hi, int dets) {
  __shared__ FlushLds<NS> L;
  flush_mx_body<NS>(S, W, s, k0, np, lo, hi, dets, (int)blockIdx.x, (int)threadIdx.x, L);
}

}  // namespace qw
