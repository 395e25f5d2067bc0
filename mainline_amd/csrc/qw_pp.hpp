// Nonlocal pseudopotential energy of one walker by one wavefront
// (src/system/Pseudopotential.cpp:596-815).
//
// The ratio at a quadrature point of electron k is linear in the basis values there:
//   sum_j inv(k, j) phi_j(r) = sum_b chi_b(r) D_b,  D_b = sum_j C[b][j] inv(k, j),
// and D does not depend on the point.  So for each selected (atom, electron) pair D is formed
// once (in large bases for the shells near its points only), and a lane then takes one quadrature
// point (of several pairs at a time): it walks the shells near it adding chi_b D_b, and the Jastrow partners, with no sums over lanes and no
// orbital at all.  The pair's own unmoved position is one more point (its Jastrow value).
//
// What bounds it: the latency of the shells' table rows and coefficients at three wavefronts per
// SIMD (65 % of the vector issue slots are used); two shells' rows in flight together take 1.27 ms
// against 1.58 one at a time, three and four 1.56 and 1.75 (registers), eight coefficient loads
// instead of four 1.40.  Contracting the orbitals at every point instead, four points at a time with the
// wave over orbitals, partners and shells in turn, held 255 registers (two waves per SIMD; now
// 161, three) and waited on coefficient loads.  Measured: local energy of the 64-electron
// pseudopotential molecule, 4096 walkers 4.56 -> 1.27 ms, of N2 (10 electrons, 2048 walkers)
// 0.232 -> 0.046 ms; 500 configurations of the 64-electron molecule 1.89 -> 0.62 ms.  Several
// determinants: with every lane searching all occupations for its orbital, 60 determinants of 64 electrons and
// 50 orbitals took 1.75 times what contracting the points took; gathered by half-waves 0.7 times
// (128 evaluations 15.0 -> 5.9 ms).
#pragma once
#include "qw_jastrow.hpp"
#include "qw_kernels.hpp"

namespace qw {

constexpr int kPPShells = 2;  // shells whose table rows are in flight together

constexpr int kPPDets = 8;   // determinants whose rows are in flight together
constexpr int kPPPairs = 8;  // pairs whose points the lanes share at most
// Functions of a chunk up to which D is formed for all of them.  Above, only for those of shells that
// reach a point: 32 atoms of 40 functions, 256 walkers, rules of 4, 6 and 12 points, a step pair 13.9,
// 14.0 and 16.8 -> 9.6, 9.7 and 12.3 ms, 32 atoms of 13 8.7 -> 7.5 ms; 16 atoms of 13 functions, 4096
// walkers, were 7 % slower with the list.
constexpr int kPPAll = 256;

// chi . D of one shell (values of shell_val; src/basis_function/Cubic_spline_calc.cpp:25-140).
__device__ __attribute__((noinline)) double shell_poly_dot(int sym, double f, double x, double y, double z, const double* d) {
  double v = 0;
  const int nf = (sym == SK_7F || sym == SK_7FC) ? 7 : (sym == SK_15G ? 15 : 9);
  for (int i = 0; i < nf; i++) {
    const AngMono* m;
    const int nm = ang_monos(ang_fn(sym, i), &m);
    double P = 0;
    for (int k = 0; k < nm; k++) P += m[k].c * pw4(x, m[k].ex) * pw4(y, m[k].ey) * pw4(z, m[k].ez);
    v += P * d[i];
  }
  return v * f;
}
template <bool FG>
__device__ inline double shell_dot(int sym, double f, double x, double y, double z, const double* d) {
  switch (sym) {
    case SK_S: return f * d[0];
    case SK_P: return f * (x * d[0] + y * d[1] + z * d[2]);
    case SK_5D:
      return f * ((2. * z * z - x * x - y * y) * d[0] + x * z * d[1] + y * z * d[2] + (x * x - y * y) * d[3] + x * y * d[4]);
    case SK_6D:
      return f * (x * x * d[0] + y * y * d[1] + z * z * d[2] + x * y * d[3] + x * z * d[4] + y * z * d[5]);
    case SK_10F:
      return f * (x * x * x * d[0] + y * y * y * d[1] + z * z * z * d[2] + x * x * y * d[3] + x * x * z * d[4] +
                  y * y * x * d[5] + y * y * z * d[6] + z * z * x * d[7] + z * z * y * d[8] + x * y * z * d[9]);
    default:
      if constexpr (FG) return shell_poly_dot(sym, f, x, y, z, d);
      return 0.0;
  }
}

// Pairs a wavefront takes together, and the LDS doubles pp_energy uses.
__host__ __device__ inline int pp_pairs(int aip) {
  const int g = 64 / (aip + 1);
  return g < kPPPairs ? g : kPPPairs;
}
// (gmax: pp_pairs of the system's smallest quadrature, DevSys::pp_g).
__host__ __device__ inline size_t pp_lds_doubles(int gmax, int chunk_nf, int nsp) {
  return (size_t)gmax * (chunk_nf | 1) + (size_t)gmax * ((nsp + 2) & ~1) + 64 + (64 + kPPPairs) +
         (chunk_nf > kPPAll ? (chunk_nf + 3) / 4 : 0);
}

// The functions (from f0 on) of the shells [sh0, sh1) that reach a point of the pairs list[0..np-1] into
// fl, in order; returns their count.  reach: the pairs' smallest and largest distance of a point from
// its atom, so the points lie between two spheres about the atom.
__device__ inline int pp_reached(const DevSys& S, int sh0, int sh1, int f0, const int2* list, const double* reach, int np,
                                 unsigned short* fl, int lane) {
  int n = 0;
  for (int s0 = sh0; s0 < sh1; s0 += kWave) {
    const int sh = s0 + lane;
    int nf = 0, f = 0;
    if (sh < sh1) {
      const ShellDesc d = S.shells[sh];
      const double* b = S.atom_pos + 3 * d.atom;
      const double rc = fmin(d.rcut, d.objthr);
      f = d.f0 - f0;
      for (int p = 0; p < np; p++) {
        const double* a = S.atom_pos + 3 * list[p].x;
        const double x = a[0] - b[0], y = a[1] - b[1], z = a[2] - b[2], lo = reach[2 * p], hi = reach[2 * p + 1];
        const double r = sqrt(x * x + y * y + z * z);
        // (rounding of the points' own distances is far below the margin; a NaN reaches everything)
        if (!(fmax(r - hi, lo - r) >= rc + 1e-6 * (1.0 + r + hi))) nf = d.nf;
      }
    }
    int tot;
    const int at = n + wave_excl_scan(nf, lane, &tot);
    for (int i = 0; i < nf; i++) fl[at + i] = (unsigned short)(f + i);
    n += tot;
  }
  return n;
}

// Jastrow value of electron e at p, terms of every other electron and atom (this lane's own e, p).
template <bool JP>
__device__ inline double jastrow_at(const DevSys& S, int e, const double p[3], const double* pos) {
  double u = 0, gf = 0, l = 0;
  const QW_CONST int* ea0 = cptr(S.eit_a0);
  const QW_CONST int* eo0 = cptr(S.eit_o0);
  const QW_CONST double* epos = cptr(S.eit_pos);
  for (int t = 0; t < S.n_eit; t++) {
    const int o0 = eo0[t], o1 = eo0[t + 1];
    for (int k = ea0[t]; k < ea0[t + 1]; k++) {
      const double x = p[0] - epos[3 * k], y = p[1] - epos[3 * k + 1], z = p[2] - epos[3 * k + 2];
      double r, ri;
      dist_inv(x * x + y * y + z * z, r, ri);
      if constexpr (JP) {
        pair_ei64<false, false>(cptr(S.eit)[o0], r, ri, u, gf, l);
      } else {
        for (int o = o0; o < o1; o++)
          with_jrad<double, false>(cptr(S.eit)[o], [&](const auto& ev) { ev(0.0, r, ri, u, gf, l); });
      }
    }
  }
  const bool eup = e < S.nup;
  for (int j = 0; j < S.ne; j++) {
    const double x = p[0] - pos[3 * j], y = p[1] - pos[3 * j + 1], z = p[2] - pos[3 * j + 2];
    double r, ri, uj = 0;
    dist_inv(x * x + y * y + z * z, r, ri);
    const bool unlike = (j < S.nup) != eup;
    if constexpr (JP) {
      const QW_CONST JRad<double>* ee = cptr(S.ee);
      pair_ee64<false, false>(ee[0], ee[1], unlike ? ee[0].cu[0] : ee[0].cl[0], r, ri, uj, gf, l);
    } else {
      for (int o = 0; o < S.nee; o++)
        with_jrad<double, false>(cptr(S.ee)[o], [&](const auto& ev) { ev(unlike ? 1.0 : 0.0, r, ri, uj, gf, l); });
    }
    u += j == e ? 0.0 : uj;
  }
  return u;
}

// The terms of the g pairs list[0..g-1] (atom, electron) of pseudopotential P: returns this lane's
// share of the nonlocal energy and writes the pairs' negative sums.
template <typename TM, bool MD, bool JP>
__device__ inline double pp_pairs_energy(const DevSys& S, const DevWalkers& W, const LocalArgs& A, int w,
                                         const QW_CONST PPType& P, const double* pos, const double rot[9],
                                         const int2* list, int g, double* dl, double* rowl, double* vx,
                                         unsigned short* fl, const double* bw, double md_den, int lane) {
  const int nsp = S.nsp, ne = S.ne, ldd = S.chunk_nf | 1, ldr = (nsp + 2) & ~1, npt = P.aip + 1;
  __syncthreads();
  // the pairs' inverse rows
  if constexpr (MD) {
    // the determinants' rows weighted and gathered onto the spin's orbital list, one half-wave per
    // pair (at most 32 electrons of a spin): a determinant's orbitals are distinct, so its lanes add to
    // distinct places, determinant after determinant
    for (int i = lane; i < g * ldr; i += kWave) rowl[i] = 0.0;
    const int nd = S.ndet, ns = S.nsig, j = lane & 31;
    for (int p0 = 0; p0 < g; p0 += 2) {
      const int p = p0 + (lane >> 5), e = list[min(p, g - 1)].y, s = e < S.nup ? 0 : 1, k = e - (s ? S.nup : 0);
      const bool on = p < g && j < (s ? S.ndn : S.nup);
      const double* inv = W.invd + ((size_t)w * 2 + s) * nd * ns * ns + (size_t)k * ns + j;
      const int* oc = S.occ + (size_t)s * nd * ns + j;
      double* row = rowl + p * ldr;
      for (int d0 = 0; d0 < nd; d0 += kPPDets) {
        double v[kPPDets];
        int m[kPPDets];
#pragma unroll
        for (int i = 0; i < kPPDets; i++) {
          const int d = min(d0 + i, nd - 1);
          v[i] = on ? inv[(size_t)d * ns * ns] : 0.0;
          m[i] = on ? oc[d * ns] : 0;
        }
#pragma unroll
        for (int i = 0; i < kPPDets; i++) {
          wave_sync();
          if (on && d0 + i < nd) row[m[i]] += bw[d0 + i] * v[i];
        }
      }
    }
    __syncthreads();
    for (int i = lane; i < g * ldr; i += kWave) rowl[i] /= md_den;
  } else {
    for (int p = 0; p < g; p++) {
      const int e = list[p].y, s = e < S.nup ? 0 : 1, k = e - (s ? S.nup : 0), n = s ? S.ndn : S.nup;
      const TM* row = inv_store<TM>(W) + (((size_t)w * 2 + s) * nsp + k) * nsp;
      for (int j = lane; j < n; j += kWave) rowl[p * ldr + j] = (double)row[j];
    }
  }
  // this lane's point: q < aip a quadrature point of pair lane / npt, q = aip the unmoved electron
  const int p = lane / npt, q = lane - p * npt;
  const bool valid = p < g;
  const int2 ae = list[valid ? p : 0];
  const double* ap = S.atom_pos + 3 * ae.x;
  const double* re = pos + 3 * ae.y;
  const double od[3] = {re[0] - ap[0], re[1] - ap[1], re[2] - ap[2]};
  const double orr = sqrt(od[0] * od[0] + od[1] * od[1] + od[2] * od[2]);
  double pt[3] = {re[0], re[1], re[2]};
  double cs = 1.0, wq = 0.0;
  const bool quad = valid && q < P.aip;
  if (quad) {
    const QW_CONST double* pq = P.q[q];
    const double qx = pq[0] * rot[0] + pq[1] * rot[3] + pq[2] * rot[6];
    const double qy = pq[0] * rot[1] + pq[1] * rot[4] + pq[2] * rot[7];
    const double qz = pq[0] * rot[2] + pq[1] * rot[5] + pq[2] * rot[8];
    pt[0] += qx * orr - od[0];
    pt[1] += qy * orr - od[1];
    pt[2] += qz * orr - od[2];
    const double nd[3] = {pt[0] - ap[0], pt[1] - ap[1], pt[2] - ap[2]};
    const double nr = sqrt(nd[0] * nd[0] + nd[1] * nd[1] + nd[2] * nd[2]);
    cs = (nd[0] * od[0] + nd[1] * od[1] + nd[2] * od[2]) / (nr * orr);
    wq = P.w[q];
    if (S.chunk_nf > kPPAll) vx[lane] = nr;
  }
  if (S.chunk_nf > kPPAll) {
    __syncthreads();
    double lo = 0, hi = 0;
    if (lane < g) {
      lo = hi = vx[lane * npt];
      for (int i = 1; i < P.aip; i++) {
        lo = fmin(lo, vx[lane * npt + i]);
        hi = fmax(hi, vx[lane * npt + i]);
      }
    }
    __syncthreads();
    if (lane < g) {  // (read until the energies of the points take its place)
      vx[2 * lane] = lo;
      vx[2 * lane + 1] = hi;
    }
  }
  double R = 0;
  for (int ch = 0; ch < S.nchunk; ch++) {
    const int sh0 = cptr(S.chunk_sh0)[ch], sh1 = cptr(S.chunk_sh0)[ch + 1];
    const QW_CONST ShellDesc* shs = cptr(S.shells);
    const int f0 = shs[sh0].f0, f1 = shs[sh1 - 1].f0 + shs[sh1 - 1].nf;
    __syncthreads();
    // D of the chunk's functions, up to four pairs of one spin at a time (each coefficient load
    // serves them all); Ct: the coefficients with the functions contiguous.  In a large chunk only
    // those of shells that reach a point.
    const bool all = f1 - f0 <= kPPAll;
    for (int p0 = 0; p0 < g;) {
      const int s = list[p0].y < S.nup ? 0 : 1, n = S.nmo[s];
      int np = 1;
      while (np < 4 && p0 + np < g && (list[p0 + np].y < S.nup ? 0 : 1) == s) np++;
      const double* r0 = rowl + p0 * ldr;
      const double *r1 = r0 + (np > 1 ? ldr : 0), *r2 = r0 + (np > 2 ? 2 * ldr : 0), *r3 = r0 + (np > 3 ? 3 * ldr : 0);
      int nf = f1 - f0;
      if (!all) {
        __syncthreads();
        nf = pp_reached(S, sh0, sh1, f0, list + p0, vx + 2 * p0, np, fl, lane);
        __syncthreads();
      }
      for (int i = lane; i < nf; i += kWave) {
        const int f = all ? i : fl[i];
        const double* c = S.Ct[s] + f0 + f;
        double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
#pragma unroll 4
        for (int j = 0; j < n; j++) {
          const double v = c[(size_t)j * S.nb];
          a0 += v * r0[j];
          a1 += v * r1[j];
          a2 += v * r2[j];
          a3 += v * r3[j];
        }
        double* o = dl + p0 * ldd + f;
        o[0] = a0;
        if (np > 1) o[ldd] = a1;
        if (np > 2) o[2 * ldd] = a2;
        if (np > 3) o[3 * ldd] = a3;
      }
      p0 += np;
    }
    __syncthreads();
    const double* d = dl + (valid ? p : 0) * ldd;
    // two shells at a time: their records and spline rows are all in flight before the first use
    int atom = -1;
    double x = 0, y = 0, z = 0, r = 0;
    for (int sh = sh0; sh < sh1; sh += kPPShells) {
      double c[kPPShells][4], hx[kPPShells], xs[kPPShells][3];
      bool act[kPPShells];
#pragma unroll
      for (int i = 0; i < kPPShells; i++) {
        const bool in = sh + i < sh1;
        const QW_CONST ShellDesc& D = shs[in ? sh + i : sh];
        if (D.atom != atom) {
          atom = D.atom;
          const QW_CONST double* pa = cptr(S.atom_pos) + 3 * atom;
          x = pt[0] - pa[0];
          y = pt[1] - pa[1];
          z = pt[2] - pa[2];
          double ri;
          dist_inv(x * x + y * y + z * z, r, ri);
        }
        act[i] = quad && in && r < D.rcut && r < D.objthr;
        xs[i][0] = x;
        xs[i][1] = y;
        xs[i][2] = z;
        if (act[i]) {
          int iv = (int)(r * cptr(S.tab_inv)[D.table]);
          iv = iv < 0 ? 0 : (iv >= S.nint ? S.nint - 1 : iv);
          const double* cc = S.spline + ((size_t)D.table * S.nint + iv) * 4;
          hx[i] = r - iv * cptr(S.tab_sp)[D.table];
          for (int k = 0; k < 4; k++) c[i][k] = cc[k];
        }
      }
#pragma unroll
      for (int i = 0; i < kPPShells; i++) {
        if (!wave_any(act[i])) continue;
        const QW_CONST ShellDesc& D = shs[sh + i];
        if (act[i]) {
          const double f = c[i][0] + hx[i] * (c[i][1] + hx[i] * (c[i][2] + hx[i] * c[i][3]));
          R += shell_dot<!JP>(D.sym, f, xs[i][0], xs[i][1], xs[i][2], d + (D.f0 - f0));
        }
      }
    }
  }
  const double u = valid ? jastrow_at<JP>(S, ae.y, pt, pos) : 0.0;
  const double u_old = __shfl(u, (valid ? p : 0) * npt + P.aip);
  double vxx = 0;
  if (quad) {
    double v[kMaxPPL];
    pp_radial(P, S.atom_Z[ae.x], orr, v);
    if (A.pp_mode == 1) {
      double strength = 0;
      for (int l = 0; l < P.L - 1; l++) strength += 10.0 * (2 * l + 1) * fabs(v[l]);
      strength = fmin(1.0, strength);
      if (fabs(strength) > 0)
        for (int l = 0; l < P.L - 1; l++) v[l] /= strength;
    }
    double ts = 0;
    for (int l = 0; l < P.L - 1; l++) ts += (2 * l + 1) * v[l] * legendre(cs, l);
    vxx = ts * (R * exp(u - u_old) * wq);
  }
  vx[lane] = vxx;
  __syncthreads();
  double nl = 0, nneg = 0;
  if (lane < g) {
    for (int i = 0; i < P.aip; i++) {
      const double t = vx[lane * npt + i];
      nl += t;
      if (t < 0.0) nneg -= t;
    }
    if (A.tneg) A.tneg[((size_t)w * S.na + list[lane].x) * ne + list[lane].y] = nneg;
  }
  return nl;
}

// This lane's share of the walker's pseudopotential energy: the local channels, and the nonlocal
// terms of the pairs inside the cutoff (deterministic) or drawn by their strength (stochastic).
template <typename TM, bool MD, bool JP>
__device__ inline double pp_energy(const DevSys& S, const DevWalkers& W, const LocalArgs& A, int w, const double* pos,
                                   double* lds, const double* bw, double md_den, int lane) {
  const int ne = S.ne;
  double* dl = lds;
  double* rowl = dl + (size_t)S.pp_g * (S.chunk_nf | 1);
  double* vx = rowl + (size_t)S.pp_g * ((S.nsp + 2) & ~1);
  int2* list = (int2*)(vx + 64);
  unsigned short* fl = (unsigned short*)(list + 64 + kPPPairs);
  double rot[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  if (A.mode == 0) {
    if (A.rot)
      for (int i = 0; i < 9; i++) rot[i] = A.rot[i];
  } else {
    random_rotation(A.seed, (unsigned)w, step_of(A.step, A.stepp), rot);
  }
  double vnl = 0;
  // pairs wait in the list until a wavefront is full of points, or their pseudopotential ends
  int cnt = 0, type = -1, a = -1, e0 = ne;
  while (true) {
    bool last = false;
    e0 += kWave;
    if (e0 >= ne) {
      e0 = 0;
      do a++;
      while (a < S.na && cptr(S.atom_pp)[a] < 0);
      last = a >= S.na;
    }
    const int pk = last ? -1 : cptr(S.atom_pp)[a];
    const bool drain = pk != type;
    if (type >= 0) {
      const QW_CONST PPType& P = cptr(S.pp)[type];
      const int G = pp_pairs(P.aip);
      int done = 0;
      while (cnt - done >= G || (drain && cnt > done)) {
        const int g = min(G, cnt - done);
        vnl += pp_pairs_energy<TM, MD, JP>(S, W, A, w, P, pos, rot, list + done, g, dl, rowl, vx, fl, bw, md_den, lane);
        done += g;
      }
      if (done) {
        __syncthreads();
        const int left = cnt - done;  // < G <= kPPPairs
        const int2 keep = list[done + (lane < left ? lane : 0)];
        __syncthreads();
        if (lane < left) list[lane] = keep;
        cnt = left;
      }
    }
    if (last) break;
    type = pk;
    const QW_CONST PPType& P = cptr(S.pp)[pk];
    const QW_CONST double* ap = cptr(S.atom_pos) + 3 * a;
    const int e = e0 + lane;
    bool want = false;
    if (e < ne) {
      double vl[kMaxPPL];
      const double x = pos[3 * e] - ap[0], y = pos[3 * e + 1] - ap[1], z = pos[3 * e + 2] - ap[2];
      const double r = sqrt(x * x + y * y + z * z);
      pp_radial(P, cptr(S.atom_Z)[a], r, vl);
      if (A.pp_mode == 0) {
        want = r < P.cutoff;
      } else {
        double strength = 0;
        for (int l = 0; l < P.L - 1; l++) strength += 10.0 * (2 * l + 1) * fabs(vl[l]);
        strength = fmin(1.0, strength);
        const double rr = A.mode == 0 ? A.pp_rand[((size_t)w * S.na + a) * ne + e]
                                      : uniform(A.seed, (unsigned)w, step_of(A.step, A.stepp), (unsigned)(a * ne + e), TAG_PP);
        want = strength > rr;
      }
      vnl += vl[P.L - 1];  // local channel for every electron
      if (A.tneg && !want) A.tneg[((size_t)w * S.na + a) * ne + e] = 0.0;
    }
    const unsigned long long m = __ballot(want);
    if (want)
      list[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
          make_int2(a, e);
    cnt += __popcll(m);
  }
  return vnl;
}

}  // namespace qw
