// k_local: local energy (kinetic, Coulomb, nonlocal pseudopotential), DMC weight and block sums of
// every walker (src/system/System.cpp:53-140, Molecular_system.cpp:209-284,
// src/method/Dmc_method.cpp:801-824).
#pragma once
#include "qw_jastrow.hpp"
#include "qw_kernels.hpp"
#include "qw_pp.hpp"

namespace qw {

// Dynamic LDS of k_local: positions, determinant gradients and laplacians; several determinants:
// their weights, logs and signs; with a pseudopotential the buffers of pp_energy.
__host__ __device__ inline size_t local_lds_bytes(const DevSys& S) {
  return ((size_t)7 * S.ne + (S.ndet > 1 ? 5 * (size_t)S.ndet : 0) + 1 + (S.has_pp ? pp_lds_doubles(S.pp_g, S.chunk_nf, S.nsp) : 0)) *
         sizeof(double);
}

// Jastrow of electron i for the local energy (jastrow_local) and its Coulomb terms (atoms, and
// electrons j < i), the usual FP64 Jastrow.
__device__ inline void jastrow_coulomb64(const DevSys& S, const double* pos, int i, double& u, double& gx, double& gy,
                                         double& gz, double& l, double& vei, double& vee) {
  const double px = pos[3 * i], py = pos[3 * i + 1], pz = pos[3 * i + 2];
  const QW_CONST int* ea0 = cptr(S.eit_a0);
  const QW_CONST int* eo0 = cptr(S.eit_o0);
  const QW_CONST double* epos = cptr(S.eit_pos);
  for (int t = 0; t < S.n_eit; t++) {
    const QW_CONST JRad<double>& o = cptr(S.eit)[eo0[t]];
    for (int k = ea0[t]; k < ea0[t + 1]; k++) {
      const double x = px - epos[3 * k], y = py - epos[3 * k + 1], z = pz - epos[3 * k + 2];
      double r, ri, gf = 0;
      dist_inv(x * x + y * y + z * z, r, ri);
      pair_ei64<true, true>(o, r, ri, u, gf, l);
      vei += cptr(S.eit_Z)[k] * ri;
      gx += gf * x;
      gy += gf * y;
      gz += gf * z;
    }
  }
  const bool iup = i < S.nup;
  const QW_CONST JRad<double>* ee = cptr(S.ee);
  for (int j = 0; j < S.ne; j++) {
    if (j == i) continue;
    const double x = px - pos[3 * j], y = py - pos[3 * j + 1], z = pz - pos[3 * j + 2];
    double r, ri, gf = 0, uj = 0;
    dist_inv(x * x + y * y + z * z, r, ri);
    pair_ee64<true, true>(ee[0], ee[1], ((j < S.nup) != iup) ? ee[0].cu[0] : ee[0].cl[0], r, ri, uj, gf, l);
    if (j > i) u += uj;
    if (j < i) vee += ri;
    gx += gf * x;
    gy += gf * y;
    gz += gf * z;
  }
}

// MD: several determinants (FP64): determinant parts and quadrature ratios are weighted sums
// over the determinants (md_contract), from their inverses in W.invd.
// PP = false compiles the nonlocal pseudopotential out (systems without one); JP: the usual trial
// function (DevSys::usual).
// The local energy of walker w by one 64-thread block (lds: the block's LDS).
template <typename TM, bool MD, bool PP, bool JP>
__device__ __forceinline__ void local_body(const DevSys& S, const DevWalkers& W, const LocalArgs& A, int w, int lane,
                                           double* lds) {
  if (w >= W.nw) return;
  const int ne = S.ne, nsp = S.nsp;
  double* pos = lds;
  double* gD = pos + 3 * ne;
  double* lD = gD + 3 * ne;
  // MD: determinant weights, their log/sign
  double* bw = lD + ne;
  double* mdl = bw + (MD ? S.ndet : 0);
  double* ppl = mdl + (MD ? 4 * S.ndet : 0) + (((MD ? S.ndet : 0) + ne) & 1);  // pseudopotential, 16-byte aligned
  for (int i = lane; i < 3 * ne; i += kWave) pos[i] = W.pos[(size_t)w * ne * 3 + i];
  const TM* mog = mo_cache<TM>(W) + (size_t)w * ne * 5 * nsp;
  double md_den = 1, md_l0 = 0, md_s0 = 1;
  const double* md_inv = nullptr;
  if constexpr (MD) {
    for (int i = lane; i < 2 * S.ndet; i += kWave) {
      mdl[i] = W.ldd[(size_t)w * 2 * S.ndet + i];
      mdl[2 * S.ndet + i] = W.sgd[(size_t)w * 2 * S.ndet + i];
    }
    __syncthreads();
    md_den = md_weights(S, mdl, mdl + 2 * S.ndet, bw, md_l0, md_s0, lane);
    md_inv = W.invd + (size_t)w * 2 * S.ndet * S.nsig * S.nsig;
    __syncthreads();
    for (int e = 0; e < ne; e++) {
      const int s = e < S.nup ? 0 : 1, k = e - (s ? S.nup : 0);
      double t[4];
      md_contract<4>(S, md_inv, s, k, (const double*)mog + ((size_t)e * 5 + 1) * nsp, nsp, bw, md_den, t, lane);
      if (lane == 0) {
        gD[3 * e] = t[0];
        gD[3 * e + 1] = t[1];
        gD[3 * e + 2] = t[2];
        lD[e] = t[3];
      }
    }
  }
  // determinant gradient / laplacian per electron: lane k owns row k of its spin's inverse
  if (A.use_dgl && !MD) {
    for (int e = lane; e < ne; e += kWave) {
      const double* d = W.dgl + ((size_t)w * ne + e) * 4;
      gD[3 * e] = d[0];
      gD[3 * e + 1] = d[1];
      gD[3 * e + 2] = d[2];
      lD[e] = d[3];
    }
  }
  // otherwise from the inverse and the MO cache: electron by electron, lanes over the MOs, so
  // every row is read coalesced
  for (int s = 0; s < 2 && !A.use_dgl && !MD; s++) {
    const int n = s ? S.ndn : S.nup, off = s ? S.nup : 0;
    const TM* ig = inv_store<TM>(W) + ((size_t)w * 2 + s) * nsp * nsp;
    for (int k = 0; k < n; k++) {
      const int e = off + k;
      double t1 = 0, t2 = 0, t3 = 0, t4 = 0;
      for (int j = lane; j < n; j += kWave) {
        const double iv = ig[(size_t)k * nsp + j];
        t1 += mog[((size_t)e * 5 + 1) * nsp + j] * iv;
        t2 += mog[((size_t)e * 5 + 2) * nsp + j] * iv;
        t3 += mog[((size_t)e * 5 + 3) * nsp + j] * iv;
        t4 += mog[((size_t)e * 5 + 4) * nsp + j] * iv;
      }
      t1 = wsum(t1);
      t2 = wsum(t2);
      t3 = wsum(t3);
      t4 = wsum(t4);
      if (lane == 0) {
        gD[3 * e] = t1;
        gD[3 * e + 1] = t2;
        gD[3 * e + 2] = t3;
        lD[e] = t4;
      }
    }
  }
  __syncthreads();
  // Jastrow per electron (lanes over electrons), kinetic energy, Coulomb
  constexpr bool fused = JP && sizeof(TM) == sizeof(double);
  double ke = 0, utot = 0, vei = 0, vee = 0;
  for (int i = lane; i < ne; i += kWave) {
    const double* pi = pos + 3 * i;
    double gx = 0, gy = 0, gz = 0, l = 0, u = 0;
    // the usual FP64 Jastrow with the Coulomb terms in one pass over atoms and electrons
    if constexpr (JP && sizeof(TM) == sizeof(double)) {
      jastrow_coulomb64(S, pos, i, u, gx, gy, gz, l, vei, vee);
    }
    // Coulomb (FP64)
    const QW_CONST double* epos = cptr(S.eit_pos);
    for (int k = 0; k < S.na && !fused; k++) {
      const QW_CONST double* ap = epos + 3 * k;
      double x = pi[0] - ap[0], y = pi[1] - ap[1], z = pi[2] - ap[2];
      double r, ri;
      dist_inv(x * x + y * y + z * z, r, ri);
      vei += cptr(S.eit_Z)[k] * ri;
    }
    for (int j = 0; j < i && !fused; j++) {
      double x = pi[0] - pos[3 * j], y = pi[1] - pos[3 * j + 1], z = pi[2] - pos[3 * j + 2];
      double r, ri;
      dist_inv(x * x + y * y + z * z, r, ri);
      vee += ri;
    }
    // Jastrow: FP64 on the FP64 path, FP32 pair terms on the mixed path
    if constexpr (fused) {
    } else if constexpr (sizeof(TM) == sizeof(double)) {
      jastrow_local<double>(S, S.ee, S.eit, pos, i, u, gx, gy, gz, l);
    } else {
      float uf = 0, gxf = 0, gyf = 0, gzf = 0, lf = 0;
      jastrow_local<float>(S, S.eef, S.eitf, pos, i, uf, gxf, gyf, gzf, lf);
      u = uf;
      gx = gxf;
      gy = gyf;
      gz = gzf;
      l = lf;
    }
    utot += u;
    double dot = gD[3 * i] * gx + gD[3 * i + 1] * gy + gD[3 * i + 2] * gz;
    double lap = lD[i] + (l + (gx * gx + gy * gy + gz * gz)) + 2 * dot;
    ke += -0.5 * lap;
    if (A.mode == 0) {
      double* og = A.out_grad + ((size_t)w * ne + i) * 3;
      og[0] = gD[3 * i] + gx;
      og[1] = gD[3 * i + 1] + gy;
      og[2] = gD[3 * i + 2] + gz;
      A.out_lap[(size_t)w * ne + i] = lap;
    }
  }
  ke = wsum(ke);
  utot = wsum(utot);
  double vloc = -wsum(vei) + S.vii + wsum(vee);

  double vnl = 0;
  if constexpr (PP) {
    if (S.has_pp) vnl = wsum(pp_energy<TM, MD, JP>(S, W, A, w, pos, ppl, bw, md_den, lane));
  }
  const double etot = ke + vloc + vnl;
  if (lane == 0) {
    double* el = W.elast + 4 * (size_t)w;
    el[0] = ke;
    el[1] = vloc;
    el[2] = vnl;
    el[3] = etot;
    if (A.mode == 0) {
      if constexpr (MD) {
        A.out_logpsi[w] = md_l0 + log(fabs(md_den)) + utot;
        A.out_sign[w] = md_s0 * (md_den < 0 ? -1.0 : 1.0);
      } else {
        A.out_logpsi[w] = W.logdet[2 * w] + W.logdet[2 * w + 1] + utot;
        A.out_sign[w] = W.sgn[2 * w] * W.sgn[2 * w + 1];
      }
      A.out_eparts[3 * w] = ke;
      A.out_eparts[3 * w + 1] = vloc;
      A.out_eparts[3 * w + 2] = vnl;
    } else if (A.mode == 3) {
      W.eold[w] = etot;
    } else {
      double wt = W.weight[w];
      if (A.mode == 2) {
        const DmcCtl& C = *A.ctl;
        double teffac = C.teff / 2.0;
        double eo = W.eold[w];
        double fbet = fmax(C.etrial - etot, C.etrial - eo);
        if (fbet > C.cut_stop) teffac = 0;
        else if (fbet > C.cut_start) teffac = teffac * (1. - (fbet - C.cut_start) / (C.cut_stop - C.cut_start));
        wt *= exp(teffac * (C.etrial * 2 - etot - eo));
        if (wt > C.max_weight) wt = C.max_weight;
        W.weight[w] = wt;
      }
      W.eold[w] = etot;
      double* bs = W.bsum + kBsum * (size_t)w;
      bs[0] += wt;
      bs[1] += wt * etot;
      bs[2] += wt * ke;
      bs[3] += wt * vloc;
      bs[4] += wt * vnl;
      bs[5] += 1;
      // unweighted first and second moments (per-point variances of the block log)
      bs[6] += etot;
      bs[7] += etot * etot;
      bs[8] += ke;
      bs[9] += ke * ke;
      bs[10] += vloc;
      bs[11] += vloc * vloc;
      bs[12] += vnl;
      bs[13] += vnl * vnl;
      bs[14] += wt * wt;
    }
  }
}

template <typename TM, bool MD, bool PP, bool JP>
__global__ __launch_bounds__(64, MD ? 3 : 1) void k_local(DevSys S, DevWalkers W, LocalArgs A) {
  extern __shared__ double lds[];
  local_body<TM, MD, PP, JP>(S, W, A, (int)blockIdx.x, (int)threadIdx.x, lds);
}

}  // namespace qw
