// FP64 DMC sweep of one spin channel with the inverse updated panel by panel.
//
//   k_sweep_p<NW, NS, JP>  single-electron moves (src/method/Split_sample.cpp:302-540,
//       src/program_utils/MatrixAlgebrac.cpp:766-838) of up to NS = 64 NW electrons of a spin by
//       NW wavefronts per walker (NW = 1: NS = 4..64, several walkers per block)
//
// The electrons of a channel move in order, so the moves of kPanelRows consecutive electrons
// need only those rows of the transposed inverse: the rows are held in registers, spread over
// the walker's threads, and take every accepted move's Sherman-Morrison update at once.  The
// rest of the inverse stays in device memory and takes the panel's updates together when the
// panel ends.  With M the inverse before the panel, M' after it, phi_j the new orbital rows of
// the accepted electrons k_j, the rows i outside the panel obey
//     M'_i = M_i - sum_j (M_i . phi_j) M'_(k_j)
// (Woodbury's identity: the panel's own updated rows are what the rank-1 steps would have
// combined to), two products on the FP64 matrix cores.
//
// What bounds it: vector issue and the latencies of a move's serial chain (old Jastrow, drift,
// basis, LCAO, ratio, acceptance).  With the whole inverse in one wavefront's registers (64
// doubles a lane) a SIMD held two waves and spilled 141 registers, and with the inverse in
// device memory (more than 64 of a spin) every accepted move streamed all of it through one
// wavefront, one such wave per SIMD at 1024 walkers; now a lane holds 16 doubles of the panel,
// three waves share a SIMD, the inverse is read and written once per 16 moves, and above 64 of a
// spin 2 or 4 wavefronts share a walker's basis, LCAO and pair terms.  Measured per launch (one
// spin channel): 64 electrons, 8192 walkers 6.74 -> 4.0 ms; 32 electrons, 4096 walkers (pseudo-
// atoms) 1.24 -> 0.69 ms; 256 electrons, 1024 walkers 173 -> 24.5 ms.  Of that, splitting the LCAO's
// functions over lane groups gave 4.39 -> 4.0, 0.92 -> 0.69 and 27 -> 24.5 ms.  Two and four waves per SIMD
// measured 4 % and 18 % slower than three at 64 electrons (four spill).
#pragma once
#include "qw_jastrow.hpp"
#include "qw_kernels.hpp"

namespace qw {

typedef double f64x4 __attribute__((ext_vector_type(4)));
// two consecutive doubles that may start on any double (16-byte global accesses need only
// 4-byte alignment)
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// Rows of a panel, threads per row and values per thread: 16 rows above 32 electrons of a spin,
// the whole matrix (no flush) below.
template <int NW, int NS>
struct PanelDims {
  static constexpr int P = NS <= 32 ? NS : 16;
  static constexpr int TPR = NS == 4 ? 2 : NS <= 16 ? 4 : NS == 32 ? 2 : 4 * NW;
  static constexpr int EPT = NS / TPR;
  static_assert(P * TPR <= 64 * NW && TPR <= 16, "panel layout");
};

constexpr int kCapPanel = 128;  // basis functions per LDS tile, one wavefront per walker
constexpr int kCapPanelW = 64;  // per wavefront's tile, several wavefronts per walker

// Makes v opaque to the compiler here, so that what is computed from it (row addresses) is not
// hoisted out of the panel loop and kept in registers through all the moves.
__device__ inline void keep_local(int& v) { asm volatile("" : "+v"(v)); }

// ---------------------------------------------------------------- reductions
template <int CTRL>
__device__ inline double dpp_add(double v) { return v + dpp_d<CTRL>(v); }

// a' + b' after exchanging a's upper half-wave with b's lower one: lanes below 32 get the sum of
// a over both halves, the others that of b (swap16: the same between neighbouring 16-lane rows).
__device__ inline double swap32_add(double a, double b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  const double u = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  const double v = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
  return u + v;
}
__device__ inline double swap16_add(double a, double b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  const double u = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  const double v = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
  return u + v;
}
// Sums of eight values over the wavefront in one tree: each step halves the values a lane
// carries instead of repeating the whole butterfly for every value (50 instead of 184
// instructions).  The sum of v[i] ends in the eight lanes from kRed8[i] on.
constexpr int kDppRor8 = 0x128;
__device__ inline double wred8(const double v[8], int lane) {
  const double s0 = swap32_add(v[0], v[1]), s1 = swap32_add(v[2], v[3]);
  const double s2 = swap32_add(v[4], v[5]), s3 = swap32_add(v[6], v[7]);
  const double t0 = swap16_add(s0, s1), t1 = swap16_add(s2, s3);
  const bool up = (lane & 8) != 0;
  const double keep = up ? t1 : t0, give = up ? t0 : t1;
  double w = keep + dpp_d<kDppRor8>(give);
  w = dpp_add<kDppHalfMirror>(w);
  w = dpp_add<kDppXor1>(w);
  return dpp_add<kDppXor2>(w);
}
// lane that starts the group holding value i of wred8
__device__ constexpr int red8_lane(int i) { return (i & 4 ? 8 : 0) + (i & 2 ? 16 : 0) + (i & 1 ? 32 : 0); }

// Sums of v[0..7] over the walker's NW wavefronts, the same bits in every thread.  red: LDS,
// NW x 8 doubles; a barrier separates the writers from the readers (and, with `before`, the
// previous readers from the writers).
template <int NW>
__device__ inline void walker_sum8(double v[8], double* red, int lane, int wv) {
  const double w = wred8(v, lane);
  if constexpr (NW == 1) {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = readlane_d(w, red8_lane(i));
  } else {
    if ((lane & 7) == 0) {
      const int i = ((lane >> 3) & 1) * 4 + ((lane >> 4) & 1) * 2 + (lane >> 5);
      red[wv * 8 + i] = w;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) {
      double s = red[i];
#pragma unroll
      for (int k = 1; k < NW; k++) s += red[8 * k + i];
      v[i] = s;
    }
  }
}

// ---------------------------------------------------------------- Jastrow
// This thread's share (partners t, t + NT, ...) of the Jastrow terms of electron e at p: value
// and gradient.  pos: LDS positions; epos: atoms in e-i type order, 3 doubles each.
template <int NT, bool JP>
__device__ inline void jastrow_share(const DevSys& S, int e, const double p[3], const double* pos, const double* epos,
                                     double& u, double& gx, double& gy, double& gz, int t) {
  u = gx = gy = gz = 0;
  const QW_CONST int* ea0 = cptr(S.eit_a0);
  const QW_CONST int* eo0 = cptr(S.eit_o0);
  for (int ty = 0; ty < S.n_eit; ty++) {
    const int a0 = ea0[ty], a1 = ea0[ty + 1], o0 = eo0[ty], o1 = eo0[ty + 1];
    for (int k = a0 + t; k < a1; k += NT) {
      const double* ap = epos + 3 * k;
      const double x = p[0] - ap[0], y = p[1] - ap[1], z = p[2] - ap[2];
      double r, ri, gf = 0, l = 0;
      dist_inv(x * x + y * y + z * z, r, ri);
      if constexpr (JP) {
        pair_ei64<true, false>(cptr(S.eit)[o0], r, ri, u, gf, l);
      } else {
        for (int o = o0; o < o1; o++)
          with_jrad<double, false>(cptr(S.eit)[o], [&](const auto& ev) { ev(0.0, r, ri, u, gf, l); });
      }
      gx += gf * x;
      gy += gf * y;
      gz += gf * z;
    }
  }
  const bool eup = e < S.nup;
  for (int j = t; j < S.ne; j += NT) {
    if (j == e) continue;
    const double x = p[0] - pos[3 * j], y = p[1] - pos[3 * j + 1], z = p[2] - pos[3 * j + 2];
    double r, ri, gf = 0, l = 0;
    dist_inv(x * x + y * y + z * z, r, ri);
    const bool unlike = (j < S.nup) != eup;
    if constexpr (JP) {
      const QW_CONST JRad<double>* ee = cptr(S.ee);
      pair_ee64<true, false>(ee[0], ee[1], unlike ? ee[0].cu[0] : ee[0].cl[0], r, ri, u, gf, l);
    } else {
      for (int o = 0; o < S.nee; o++)
        with_jrad<double, false>(cptr(S.ee)[o], [&](const auto& ev) { ev(unlike ? 1.0 : 0.0, r, ri, u, gf, l); });
    }
    gx += gf * x;
    gy += gf * y;
    gz += gf * z;
  }
}

// ---------------------------------------------------------------- drift
// Drift limiter factor (lim_drift) as 2 tau / (1 + sqrt(1 + 2 tau d2)): the same value without
// the subtraction that loses digits for small drifts, and without its small-drift branch.
__device__ inline double drift_scale(const double v[3], double tau) {
  const double d2 = (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]) * 0.25;
  double s, si;
  dist_inv(fma(2.0 * tau, d2, 1.0), s, si);
  return 2.0 * tau * rcp_nr(1.0 + s);
}
// Exponent of the drift-diffusion Green's function from ra (drift da) to rb.
__device__ inline double trans_fast(const double ra[3], const double da[3], const double rb[3], double tau) {
  const double f = drift_scale(da, tau);
  double p = 0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double t = rb[d] - ra[d] - da[d] * f;
    p -= t * t;
  }
  return p * rcp_nr(2.0 * tau);
}

// ---------------------------------------------------------------- LDS
// Shared by a block's walkers: atom positions in shell order and in e-i type order, spline
// spacings, and (one wavefront per walker) the shell records.
__host__ __device__ inline size_t panel_shared_lds(int na, int nsh, int ntab, int nw) {
  return ((size_t)6 * na + 2 * ntab) * sizeof(double) + (nw == 1 ? (size_t)nsh * sizeof(ShellLds) : 0);
}
// Of one walker: positions, basis tiles, active-shell lists, new orbital values, inverse row,
// random numbers, reduction buffers.
__host__ __device__ inline size_t panel_walker_lds(int ne, int nsh, int ns, int nw) {
  const int cap = nw == 1 ? kCapPanel : kCapPanelW;
  return ((size_t)3 * ne * 8 + 8) / 16 * 16 + (size_t)nw * cap * (5 * 8 + 4) +
         ((size_t)(nsh + 64 * nw) * 8 + 15) / 16 * 16 + (size_t)2 * ns * 8 + (size_t)((ns <= 32 ? ns : 16) * 4) * 8 +
         (nw > 1 ? (size_t)(16 * nw) * 8 + 16 * 4 : 0);
}
__host__ __device__ inline size_t panel_lds_bytes(int ne, int na, int nsh, int ntab, int ns, int nw, int wpb) {
  return (panel_shared_lds(na, nsh, ntab, nw) + 15) / 16 * 16 + (size_t)wpb * panel_walker_lds(ne, nsh, ns, nw);
}
// Walkers per block: up to four wavefronts share the tables, fewer where four would leave compute units
// without a block (256 walkers of 8 electrons 286 -> 268 us a step pair, of 128 electrons 4.36 -> 4.11 ms;
// 512: 293 -> 286 us and 4.42 -> 4.29 ms; from 769 on the same).
constexpr int kPanelWpb = 4;
inline int panel_wpb(int nw) { return nw > 768 ? kPanelWpb : nw > 512 ? 3 : nw > 256 ? 2 : 1; }

// ---------------------------------------------------------------- basis
// Active shells of point p among this thread's shells t, t + NT, ...: (meta, f0) appended to the
// wavefront's list; returns their count.  Squared distances are compared (rc2 is the smallest
// number whose square root reaches the cutoff).
template <int NT>
__device__ inline int panel_active(const DevSys& S, const ShellLds* shl, const double* apos, const double p[3], int2* list,
                                   int t) {
  int n = 0;
  for (int s0 = 0; s0 < S.nsh; s0 += NT) {
    const int sh = s0 + t;
    bool act = false;
    ShellLds d;
    if (sh < S.nsh) {
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
// One batch of the wavefront's active shells into its tile (see basis_batch_lap); returns the
// shells consumed.
template <bool FG>
__device__ inline int panel_basis(const DevSys& S, const double* tabs, const double* apos, const double p[3],
                                  const int2* list, int i0, int nact, int n, double* chi, int* roff, int cap, int* nfun,
                                  int lane) {
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
    double r, ri;
    dist_inv(x * x + y * y + z * z, r, ri);
    int iv = (int)(r * tabs[2 * tab]);
    iv = iv < 0 ? 0 : (iv >= S.nint ? S.nint - 1 : iv);
    const double* c = S.spline + ((size_t)tab * S.nint + iv) * 4;
    const double c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
    const double h = r - iv * tabs[2 * tab + 1];
    const double f = c0 + h * (c1 + h * (c2 + h * c3));
    const double fd = (c1 + h * (2 * c2 + h * (3 * c3))) * ri;
    const double f2 = 2 * c2 + 6 * h * c3;
    shell_lap<double, FG>(shl_sym(d.x), f, fd, f2, x, y, z, chi + at, cap);
    for (int q = 0; q < nf; q++) roff[at + q] = (d.y + q) * n * (int)sizeof(double);
  }
  return take;
}

// ---------------------------------------------------------------- LCAO
// The wavefront's lanes form G groups of 64 / G; group g sums the functions 2g, 2g+1 of every 2G,
// a lane for the orbitals j, j + 64/G, ... (R of them), and the groups' sums meet at the end.  A
// function's five values read from LDS then serve R orbitals of a lane instead of one (with every
// lane reading them for one orbital, LDS took longer than the FMAs), and up to 32 electrons of a
// spin no lane is idle.
template <int NS>
struct PanelLcao {
  static constexpr int G = NS <= 8 ? 8 : NS <= 32 ? 4 : 2;
  static constexpr int R = NS <= 16 ? 1 : 2;
  static constexpr int unit = 2 * G;  // functions of a step
};
// Zero values after the nfun functions of a tile, up to a whole unit.
template <int UNIT>
__device__ inline void lcao_pad(double* chi, int* roff, int cap, int nfun, int lane) {
  static_assert(UNIT <= 16, "unit");
  const int i = lane & 15, c = lane >> 4;
  if (i < (UNIT - nfun % UNIT) % UNIT) {
    chi[c * cap + nfun + i] = 0.0;
    if (c == 0) chi[4 * cap + nfun + i] = 0.0;
    if (c == 1) roff[nfun + i] = 0;
  }
}
template <int G, int R, int K>
__device__ inline int lcao_units(const char* Cb, const unsigned lb[R], const int* roff, const double* chi, int cap, int b,
                                 int nfun, double acc[R][5]) {
  for (; b + 2 * G * (K - 1) < nfun; b += 2 * G * K) {
    double cv[K][2][R];
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int2 ro = *(const int2*)(roff + b + 2 * G * k);
#pragma unroll
      for (int r = 0; r < R; r++) {
        cv[k][0][r] = *reinterpret_cast<const double*>(Cb + ((unsigned)ro.x + lb[r]));
        cv[k][1][r] = *reinterpret_cast<const double*>(Cb + ((unsigned)ro.y + lb[r]));
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads issue before the first use
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
      for (int c = 0; c < 5; c++) {
        const f64x2 x = *(const f64x2*)(chi + c * cap + b + 2 * G * k);
#pragma unroll
        for (int r = 0; r < R; r++) {
          acc[r][c] += cv[k][0][r] * x[0];
          acc[r][c] += cv[k][1][r] * x[1];
        }
      }
  }
  return b;
}
// Adds a tile to the lane's partial sums; C: the wavefront's first orbital, nm of them.  2u
// loads in flight at most (the sums do not depend on it).
template <int G, int R>
__device__ inline void panel_lcao(const double* C, const int* roff, const double* chi, int cap, int nfun, int nm,
                                  double acc[R][5], int lane, int u) {
  constexpr int L = kWave / G;
  const char* Cb = reinterpret_cast<const char*>(C);
  unsigned lb[R];
#pragma unroll
  for (int r = 0; r < R; r++) {  // lanes past the last orbital repeat it
    const int j = lane % L + L * r;
    lb[r] = (unsigned)(j < nm ? j : nm - 1) * 8u;
  }
  const int g = lane / L;
  roff += 2 * g;
  chi += 2 * g;
  int b = 0;
  if (u == 8) b = lcao_units<G, R, 8 / R>(Cb, lb, roff, chi, cap, b, nfun, acc);
  else if (u == 4) b = lcao_units<G, R, 4 / R>(Cb, lb, roff, chi, cap, b, nfun, acc);
  lcao_units<G, R, 1>(Cb, lb, roff, chi, cap, b, nfun, acc);
}
// The groups' sums: orbital `lane` of the wavefront (below 32 orbitals, repeated).
template <int G, int R>
__device__ inline void lcao_join(const double acc[R][5], double phi[5]) {
#pragma unroll
  for (int c = 0; c < 5; c++) {
    if constexpr (G == 2 && R == 2) phi[c] = swap32_add(acc[0][c], acc[1][c]);
    else if constexpr (G == 4 && R == 2)
      phi[c] = swap16_add(swap32_add(acc[0][c], acc[0][c]), swap32_add(acc[1][c], acc[1][c]));
    else {
      static_assert(R == 1, "layout");
      double v = swap32_add(acc[0][c], acc[0][c]);
      if constexpr (G >= 4) v = swap16_add(v, v);
      if constexpr (G == 8) v = dpp_add<kDppRor8>(v);
      phi[c] = v;
    }
  }
}

// ---------------------------------------------------------------- panel rows
// Value ii, h (h = 0, 1) of a thread is column 2 (q + TPR ii) + h of its row: the threads of a
// row read LDS vectors and device memory contiguously, 16 bytes each.
template <int TPR, int EPT>
__device__ inline void row_load(const double* row, int n, int q, double a[EPT]) {
#pragma unroll
  for (int ii = 0; ii < EPT / 2; ii++) {
    const int c = 2 * (q + TPR * ii);
    if (c + 1 < n) {
      const f64x2u v = *(const f64x2u*)(row + c);
      a[2 * ii] = v[0];
      a[2 * ii + 1] = v[1];
    } else {
      a[2 * ii] = c < n ? row[c] : 0.0;
      a[2 * ii + 1] = 0.0;
    }
  }
}
template <int TPR, int EPT>
__device__ inline void row_store(double* row, int n, int q, const double a[EPT]) {
#pragma unroll
  for (int ii = 0; ii < EPT / 2; ii++) {
    const int c = 2 * (q + TPR * ii);
    if (c + 1 < n) {
      f64x2u v;
      v[0] = a[2 * ii];
      v[1] = a[2 * ii + 1];
      *(f64x2u*)(row + c) = v;
    } else if (c < n) {
      row[c] = a[2 * ii];
    }
  }
}
// Sum over the TPR consecutive lanes of a row, in each of them.
template <int TPR>
__device__ inline double row_sum(double v) {
  v = dpp_add<kDppXor1>(v);
  if constexpr (TPR >= 4) v = dpp_add<kDppXor2>(v);
  if constexpr (TPR >= 8) v = dpp_add<kDppHalfMirror>(v);
  if constexpr (TPR >= 16) v = dpp_add<kDppMirror>(v);
  return v;
}

// The updates of the panel rows kp..kp+15 (final in ig) applied to every other row of the
// n x n transposed inverse ig (row stride nsp): U_ij = M_i . phi_j over the accepted j (bit j of
// accm; phi_j is the electron's value row in the MO cache), M_i -= sum_j U_ij M'_(kp+j), both on
// v_mfma_f64_16x16x4 (A[i][k]: lane i + 16 k; B[k][j]: lane j + 16 k; D[i][j]: lane
// j + 16 (i % 4), register i / 4).  The first product is taken transposed, U^T = Phi M^T, so its
// registers are already the A operand of the second.  Wavefront wv takes the row groups
// 4 wv..4 wv+3 of 16 rows together: the phi and panel-row operands are loaded once for four.
__device__ inline void panel_flush(double* ig, const double* mo0, int nsp, int n, int kp, unsigned accm, int lane, int wv) {
  keep_local(lane);
  const int i = lane & 15, h = lane >> 4;
  const int g0 = 4 * wv, pg = kp >> 4;
  const int ng = (n + 15) >> 4;
  if (g0 >= ng || (ng == 1)) return;
  const bool on = (accm >> i) & 1;
  const double* ph = mo0 + (size_t)(on ? kp + i : kp) * 5 * nsp;
  const double* rw[4];
#pragma unroll
  for (int g = 0; g < 4; g++) rw[g] = ig + (size_t)min(16 * (g0 + g) + i, n - 1) * nsp;
  f64x4 U[4];
#pragma unroll
  for (int g = 0; g < 4; g++) U[g] = (f64x4){0, 0, 0, 0};
  int c0 = 0;
  for (; c0 + 8 <= n; c0 += 8) {
    const int c = c0 + 2 * h;
    const f64x2u av = *(const f64x2u*)(ph + c);
    f64x2u b[4];
#pragma unroll
    for (int g = 0; g < 4; g++) b[g] = *(const f64x2u*)(rw[g] + c);
    const double a0 = on ? av[0] : 0.0, a1 = on ? av[1] : 0.0;
#pragma unroll
    for (int g = 0; g < 4; g++) U[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[g][0], U[g], 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 4; g++) U[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[g][1], U[g], 0, 0, 0);
  }
  for (; c0 < n; c0 += 4) {
    const int c = c0 + h;
    const bool in = c < n;
    const double a0 = on && in ? ph[c] : 0.0;
#pragma unroll
    for (int g = 0; g < 4; g++)
      U[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, in ? rw[g][c] : 0.0, U[g], 0, 0, 0);
  }
  for (int ct = 0; ct < ng; ct++) {
    const int col = 16 * ct + i, cc = min(col, n - 1);
    double B[4];
    f64x4 C[4];
#pragma unroll
    for (int s = 0; s < 4; s++) B[s] = ig[(size_t)min(kp + 4 * s + h, n - 1) * nsp + cc];
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int r = 0; r < 4; r++) C[g][r] = ig[(size_t)min(16 * (g0 + g) + 4 * r + h, n - 1) * nsp + cc];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int g = 0; g < 4; g++) C[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(-U[g][s], B[s], C[g], 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = 16 * (g0 + g) + 4 * r + h;
        if (g0 + g != pg && row < n && col < n) ig[(size_t)row * nsp + col] = C[g][r];
      }
  }
}

// ---------------------------------------------------------------- sweep
template <int NW>
__device__ inline void panel_sync() {
  if constexpr (NW == 1)
    wave_sync();
  else
    __syncthreads();
}
// The moves of walker w's spin A.s by NW wavefronts (t: thread of the walker).  sh: the block's
// shared LDS tables, own: the walker's region.  u: half the coefficient loads in flight in the
// LCAO.
template <int NW, int NS, bool JP>
__device__ __forceinline__ void sweep_panel_body(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int w, int t,
                                                 char* sh, char* own, int u) {
  typedef PanelDims<NW, NS> D;
  constexpr int P = D::P, TPR = D::TPR, EPT = D::EPT, NT = 64 * NW;
  constexpr int cap = NW == 1 ? kCapPanel : kCapPanelW;
  const int lane = t & 63, wv = NW == 1 ? 0 : t >> 6;
  const int ne = S.ne, s = A.s, n = s ? S.ndn : S.nup, nsp = S.nsp, off = s ? S.nup : 0;
  const double* apos = (const double*)sh;
  const double* epos = apos + 3 * S.na;
  const double* tabs = epos + 3 * S.na;
  const ShellLds* shl = NW == 1 ? (const ShellLds*)(tabs + 2 * S.ntab) : S.shl;
  double* pos = (double*)own;
  double* phib = (double*)(own + ((size_t)3 * ne * 8 + 8) / 16 * 16);
  double* rowk = phib + NS;
  double* rnd = rowk + NS;
  double* chi0 = rnd + P * 4;
  double* red = chi0 + (size_t)NW * 5 * cap;
  int2* list0 = (int2*)(red + (NW > 1 ? 16 * NW : 0));
  int* roff0 = (int*)(list0 + S.nsh + 64 * NW);
  int* cnt = roff0 + NW * cap;  // NW > 1: functions in each wavefront's tile, and its shells left
  double* chi = chi0 + (size_t)wv * 5 * cap;
  int* roff = roff0 + wv * cap;
  int2* list = list0 + (size_t)wv * ((S.nsh + NT - 1) / NT * 64);
  for (int i = t; i < 3 * ne; i += NT) pos[i] = W.pos[(size_t)w * ne * 3 + i];
  double logdet = W.logdet[2 * w + s], sgn = W.sgn[2 * w + s], dprod = 1.0;
  int nacc = 0;
  double* mog = W.mo + (size_t)w * ne * 5 * nsp;
  double* ig = W.inv + ((size_t)w * 2 + s) * nsp * nsp;
  const double* Cw = S.C[s] + 64 * wv;
  const bool mine = t < n;
  const double tau = A.tau, stau = sqrt(tau);
  double m1 = 0, m2 = 0, m3 = 0;
  if (mine && A.k0 < A.k1) {
    const double* mr = mog + (size_t)(off + A.k0) * 5 * nsp + t;
    m1 = mr[nsp];
    m2 = mr[2 * nsp];
    m3 = mr[3 * nsp];
  }
  const int r = t / TPR, q = t % TPR;
  const bool prow = t < P * TPR;
  double a[EPT];
  for (int kp = A.k0 / P * P; kp < A.k1; kp += P) {
    const int ka = max(kp, A.k0), kb = min(kp + P, A.k1);
    unsigned accm = 0;
#pragma unroll
    for (int i = 0; i < EPT; i++) a[i] = 0;
    if (prow && kp + r < n) row_load<TPR, EPT>(ig + (size_t)(kp + r) * nsp, n, q, a);
    // random numbers of the panel's moves, one move per thread (the streams of sweep_randoms)
    for (int i = t; i < kb - ka; i += NT) {
      const unsigned st = step_of(A.step, A.stepp), ke = (unsigned)(off + ka + i);
      double g[3];
      gauss3(A.seed, (unsigned)w, st, ke, TAG_GAUSS1 | (A.sweep << 8), g);
      double* o = rnd + 4 * i;
      o[0] = g[0];
      o[1] = g[1];
      o[2] = g[2];
      o[3] = uniform(A.seed, (unsigned)w, st, ke, TAG_ACC1 | (A.sweep << 8));
    }
    for (int k = ka; k < kb; k++) {
      const int e = off + k;
      // row k of the inverse to every thread of the walker
      if (prow && r == k - kp) {
#pragma unroll
        for (int ii = 0; ii < EPT / 2; ii++) {
          f64x2 v;
          v[0] = a[2 * ii];
          v[1] = a[2 * ii + 1];
          *(f64x2*)(rowk + 2 * (q + TPR * ii)) = v;
        }
      }
      panel_sync<NW>();
      const double rk = mine ? rowk[t] : 0.0;
      const double r0[3] = {pos[3 * e], pos[3 * e + 1], pos[3 * e + 2]};
      // drift at the old position: determinant part from the cached MO row, Jastrow part fresh
      double v[8];
      jastrow_share<NT, JP>(S, e, r0, pos, epos, v[0], v[1], v[2], v[3], t);
      v[4] = rk * m1;
      v[5] = rk * m2;
      v[6] = rk * m3;
      v[7] = 0;
      walker_sum8<NW>(v, red, lane, wv);
      const double u0 = v[0];
      const double d0[3] = {v[4] + v[1], v[5] + v[2], v[6] + v[3]};
      // proposal
      const double* rq = rnd + 4 * (k - ka);
      const double fd = drift_scale(d0, tau);
      double rn[3];
      for (int d = 0; d < 3; d++) rn[d] = r0[d] + (rq[d] * stau + d0[d] * fd);
      typedef PanelLcao<NS> Lc;
      double phi[5], part[Lc::R][5];
#pragma unroll
      for (int x = 0; x < Lc::R; x++)
        for (int c = 0; c < 5; c++) part[x][c] = 0;
      const int nact = panel_active<NT>(S, shl, apos, rn, list, t);
      wave_sync();
      if constexpr (NW == 1) {
        for (int i0 = 0; i0 < nact;) {
          int nfun;
          const int take = panel_basis<!JP>(S, tabs, apos, rn, list, i0, nact, n, chi, roff, cap, &nfun, lane);
          lcao_pad<Lc::unit>(chi, roff, cap, nfun, lane);
          wave_sync();
          panel_lcao<Lc::G, Lc::R>(Cw, roff, chi, cap, nfun, n, part, lane, u);
          wave_sync();
          i0 += take;
        }
      } else {
        // every wavefront fills its own tile; all of them contract every tile
        for (int i0 = 0;;) {
          int nfun = 0;
          if (i0 < nact) i0 += panel_basis<!JP>(S, tabs, apos, rn, list, i0, nact, n, chi, roff, cap, &nfun, lane);
          lcao_pad<Lc::unit>(chi, roff, cap, nfun, lane);
          if (lane == 0) {
            cnt[2 * wv] = nfun;
            cnt[2 * wv + 1] = nact - i0;
          }
          __syncthreads();
          bool more = false;
#pragma unroll
          for (int x = 0; x < NW; x++) {
            const int nf = cnt[2 * x];
            more |= cnt[2 * x + 1] > 0;
            if (64 * wv < n)
              panel_lcao<Lc::G, Lc::R>(Cw, roff0 + x * cap, chi0 + (size_t)x * 5 * cap, cap, nf, n - 64 * wv, part, lane, u);
          }
          if (!more) break;
          __syncthreads();
        }
      }
      lcao_join<Lc::G, Lc::R>(part, phi);
      jastrow_share<NT, JP>(S, e, rn, pos, epos, v[0], v[1], v[2], v[3], t);
      for (int c = 0; c < 4; c++) v[4 + c] = mine ? rk * phi[c] : 0.0;
      if (t < NS) phib[t] = mine ? phi[0] : 0.0;
      walker_sum8<NW>(v, red + (NW > 1 ? 8 * NW : 0), lane, wv);
      const double un = v[0], R = v[4], it0 = 1.0 / R;
      const double dn[3] = {v[5] * it0 + v[1], v[6] * it0 + v[2], v[7] * it0 + v[3]};
      // |ratio|^2 exp(dtrans) as R^2 exp(2 du + dtrans): one exponential, no logarithm.  The
      // proposal's displacement from the drifted point is the drawn Gaussian, so its own
      // Green's function exponent is -|g|^2 / 2.
      const double g2 = -0.5 * (rq[0] * rq[0] + rq[1] * rq[1] + rq[2] * rq[2]);
      const double acc = (A.restrict_nodes && R < 0)
                             ? 0.0
                             : fmin(1.0, R * R * exp(2.0 * (un - u0) + (trans_fast(rn, dn, r0, tau) - g2)));
      const bool accepted = acc + rq[3] > 1.0;
      if (accepted) {
        // Sherman-Morrison on the panel's rows for the replaced row k (phib was written before
        // the last reduction's barrier; with one wavefront the fence orders it)
        if constexpr (NW == 1) wave_sync();
        if (prow) {
          double tq[2] = {0, 0};
#pragma unroll
          for (int ii = 0; ii < EPT / 2; ii++) {
            const f64x2 pv = *(const f64x2*)(phib + 2 * (q + TPR * ii));
            tq[0] += a[2 * ii] * pv[0];
            tq[1] += a[2 * ii + 1] * pv[1];
          }
          const double tk = row_sum<TPR>(tq[0] + tq[1]);
          const double f = 1.0 / R, pk = -tk * f;
          const bool me = r == k - kp;
#pragma unroll
          for (int ii = 0; ii < EPT / 2; ii++) {
            const f64x2 rv = *(const f64x2*)(rowk + 2 * (q + TPR * ii));
            a[2 * ii] = me ? rv[0] * f : fma(rv[0], pk, a[2 * ii]);
            a[2 * ii + 1] = me ? rv[1] * f : fma(rv[1], pk, a[2 * ii + 1]);
          }
        }
        if (mine) {
          double* mr = mog + (size_t)e * 5 * nsp + t;
          for (int c = 0; c < 5; c++) mr[c * nsp] = phi[c];
        }
        // accepted ratios multiply into dprod, folded into log|det| before it could overflow
        dprod *= R;
        if (!(fabs(dprod) < 0x1p+512 && fabs(dprod) > 0x1p-512)) {
          logdet += log(fabs(dprod));
          dprod = 1.0;
        }
        if (R < 0) sgn = -sgn;
        nacc++;
        accm |= 1u << (k - kp);
        if (t < 3) pos[3 * e + t] = rn[t];
      }
      if (mine && k + 1 < A.k1) {
        const double* mr = mog + (size_t)(e + 1) * 5 * nsp + t;
        m1 = mr[nsp];
        m2 = mr[2 * nsp];
        m3 = mr[3 * nsp];
      }
      panel_sync<NW>();
    }
    if (prow && kp + r < n) row_store<TPR, EPT>(ig + (size_t)(kp + r) * nsp, n, q, a);
    if constexpr (P < NS) {
      if (accm) {
        __threadfence_block();
        panel_sync<NW>();
        panel_flush(ig, mog + (size_t)off * 5 * nsp, nsp, n, kp, accm, lane, wv);
        __threadfence_block();
        panel_sync<NW>();
      }
    }
  }
  if (A.dets) {
    // determinant parts of the local energy (write_det_parts), P rows at a time
    __threadfence_block();
    panel_sync<NW>();
    for (int rp = 0; rp < n; rp += P) {
      const int row = rp + r;
      double tv[4] = {0, 0, 0, 0};
      if (prow && row < n) {
        if constexpr (P < NS) row_load<TPR, EPT>(ig + (size_t)row * nsp, n, q, a);
#pragma unroll
        for (int c = 0; c < 4; c++) {
          double b[EPT];
          row_load<TPR, EPT>(mog + ((size_t)(off + row) * 5 + c + 1) * nsp, n, q, b);
#pragma unroll
          for (int i = 0; i < EPT; i++) tv[c] += a[i] * b[i];
        }
      }
#pragma unroll
      for (int c = 0; c < 4; c++) tv[c] = row_sum<TPR>(tv[c]);
      if (prow && row < n && q == 0) {
        double* o = W.dgl + ((size_t)w * ne + off + row) * 4;
        for (int c = 0; c < 4; c++) o[c] = tv[c];
      }
    }
  }
  for (int i = t; i < 3 * ne; i += NT) W.pos[(size_t)w * ne * 3 + i] = pos[i];
  logdet += log(fabs(dprod));
  if (t == 0) {
    W.logdet[2 * w + s] = logdet;
    W.sgn[2 * w + s] = sgn;
    W.acc[w] += nacc;
  }
}

// Fills the block's shared tables (threads t of nt); a block barrier follows.
__device__ inline void panel_stage(const DevSys& S, char* sh, int nw, int t, int nt) {
  double* apos = (double*)sh;
  double* epos = apos + 3 * S.na;
  double* tabs = epos + 3 * S.na;
  for (int i = t; i < 3 * S.na; i += nt) {
    apos[i] = S.atom_pos[i];
    epos[i] = S.eit_pos[i];
  }
  for (int i = t; i < 2 * S.ntab; i += nt) tabs[i] = S.tabs[i];
  if (nw == 1) {
    ShellLds* shl = (ShellLds*)(tabs + 2 * S.ntab);
    for (int i = t; i < S.nsh; i += nt) shl[i] = S.shl[i];
  }
}

template <int NW, int NS, bool JP>
__global__ __launch_bounds__(NW == 1 ? 64 * kPanelWpb : 64 * NW, 3) void k_sweep_p(DevSys S, DevWalkers W, SweepArgs A,
                                                                                   int u) {
  extern __shared__ double ldsp[];
  char* sh = (char*)ldsp;
  const int nt = (int)blockDim.x, wpb = NW == 1 ? nt >> 6 : 1;
  panel_stage(S, sh, NW, (int)threadIdx.x, nt);
  __syncthreads();
  const int wid = NW == 1 ? (int)threadIdx.x >> 6 : 0, t = NW == 1 ? (int)threadIdx.x & 63 : (int)threadIdx.x;
  const int w = (int)blockIdx.x * wpb + wid;
  if (w >= W.nw) return;
  char* own = sh + (panel_shared_lds(S.na, S.nsh, S.ntab, NW) + 15) / 16 * 16 +
              (size_t)wid * panel_walker_lds(S.ne, S.nsh, NS, NW);
  sweep_panel_body<NW, NS, JP>(S, W, A, w, t, sh, own, u);
}

}  // namespace qw
