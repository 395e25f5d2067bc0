// FP64 pair terms of the usual Jastrow (DevSys::usual): one CUTOFF_CUSP and one POLYPADE object of
// up to four functions between electrons, one such POLYPADE object per atom type (the formulas of
// CuspEval and PolyEval).  Functions beyond an object's count have zero coefficients.  All the
// denominators of a pair share one reciprocal (1/a and 1/b are b/(ab) and a/(ab)): a double
// reciprocal costs a quarter-rate estimate and four multiply-adds, and a pair has five.  None of them
// vanishes where another object is inside its cutoff (the rule that sets DevSys::usual).
// GRAD: add (d/dr)/r to gf; LAP: add the laplacian to l.
#pragma once
#include "qw_device.hpp"

namespace qw {

// The POLYPADE part given the four reciprocals p of 1 + beta_i zpp.
template <bool GRAD, bool LAP>
__device__ inline void poly_terms64(const QW_CONST JRad<double>& o, double zz, double zz2, double zpp, const double p[4],
                                    double r, double ri, double& u, double& gf, double& l) {
  const double s0 = o.cl[0] * p[0] + o.cl[1] * p[1] + o.cl[2] * p[2] + o.cl[3] * p[3];
  const bool in = r < o.rcut;
  u += in ? (1.0 - zpp) * s0 : 0.0;
  if constexpr (GRAD) {
    const double t0 = o.cbl[0] * p[0] * p[0], t1 = o.cbl[1] * p[1] * p[1];
    const double t2 = o.cbl[2] * p[2] * p[2], t3 = o.cbl[3] * p[3] * p[3];
    const double s1 = t0 + t1 + t2 + t3;
    const double zppd = 12.0 * zz * (1.0 - 2.0 * zz + zz2);
    const double g = -zppd * ri * o.rcinv * s1;
    gf += in ? g : 0.0;
    if constexpr (LAP) {
      const double s2 = t0 * (o.beta[0] * p[0]) + t1 * (o.beta[1] * p[1]) + t2 * (o.beta[2] * p[2]) + t3 * (o.beta[3] * p[3]);
      const double zppdd2 = 6.0 - 24.0 * zz + 18.0 * zz2;
      const double d2 = -o.rcinv2 * (zppdd2 * s1 - zppd * zppd * s2);
      l += in ? 2.0 * (d2 + g) : 0.0;
    }
  }
}
// An electron pair: c the cusp object, cc its coefficient for this pair, o the POLYPADE object.
template <bool GRAD, bool LAP>
__device__ inline void pair_ee64(const QW_CONST JRad<double>& c, const QW_CONST JRad<double>& o, double cc, double r,
                                 double ri, double& u, double& gf, double& l) {
  const double yc = r * c.rcinv, yc2 = yc * yc;
  const double pp = yc - yc2 + yc * yc2 * (1.0 / 3.0);
  const double d4 = fma(c.gamma, pp, 1.0);
  const double zz = r * o.rcinv, zz2 = zz * zz;
  const double zpp = zz2 * (6.0 - 8.0 * zz + 3.0 * zz2);
  const double d0 = fma(o.beta[0], zpp, 1.0), d1 = fma(o.beta[1], zpp, 1.0);
  const double d2 = fma(o.beta[2], zpp, 1.0), d3 = fma(o.beta[3], zpp, 1.0);
  const double d01 = d0 * d1, d23 = d2 * d3, dp = d01 * d23;
  const double inv = rcp_nr(dp * d4);
  const double pade = inv * dp, ip = inv * d4;
  const double i01 = ip * d23, i23 = ip * d01;
  const double p[4] = {i01 * d1, i01 * d0, i23 * d3, i23 * d2};
  const bool in = r < c.rcut;
  u += in ? cc * (c.rcut * (pp * pade - c.pade0)) : 0.0;
  if constexpr (GRAD) {
    const double ppd = 1.0 - 2.0 * yc + yc2, pade2 = pade * pade;
    const double dadr = ppd * pade2 * ri;
    gf += in ? cc * dadr : 0.0;
    if constexpr (LAP) {
      const double ppdd = -2.0 + 2.0 * yc;
      const double d = (ppdd * pade2 - 2.0 * c.gamma * ppd * ppd * pade2 * pade) * c.rcinv + 2.0 * dadr;
      l += in ? cc * d : 0.0;
    }
  }
  poly_terms64<GRAD, LAP>(o, zz, zz2, zpp, p, r, ri, u, gf, l);
}
// An electron and an atom.
template <bool GRAD, bool LAP>
__device__ inline void pair_ei64(const QW_CONST JRad<double>& o, double r, double ri, double& u, double& gf, double& l) {
  const double zz = r * o.rcinv, zz2 = zz * zz;
  const double zpp = zz2 * (6.0 - 8.0 * zz + 3.0 * zz2);
  const double d0 = fma(o.beta[0], zpp, 1.0), d1 = fma(o.beta[1], zpp, 1.0);
  const double d2 = fma(o.beta[2], zpp, 1.0), d3 = fma(o.beta[3], zpp, 1.0);
  const double d01 = d0 * d1, d23 = d2 * d3;
  const double ip = rcp_nr(d01 * d23);
  const double i01 = ip * d23, i23 = ip * d01;
  const double p[4] = {i01 * d1, i01 * d0, i23 * d3, i23 * d2};
  poly_terms64<GRAD, LAP>(o, zz, zz2, zpp, p, r, ri, u, gf, l);
}

}  // namespace qw
