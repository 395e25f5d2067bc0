// Launches of the local energy (qw_local.hpp) and of the MO rows (qw_rows.hpp).
#include "qw_local.hpp"
#include "qw_rows.hpp"
#include "qw_sweep.hpp"

namespace qw {

void launch_local(const DevSys& S, const DevWalkers& W, const LocalArgs& A, bool f64, hipStream_t st) {
  const size_t lds = local_lds_bytes(S);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(W.nw), dim3(64), lds, st, S, W, A); };
  const bool u = S.usual != 0;
  if (S.ndet > 1) {
    if (u) go(k_local<double, true, true, true>);
    else go(k_local<double, true, true, false>);
  } else if (f64 && S.has_pp) {
    if (u) go(k_local<double, false, true, true>);
    else go(k_local<double, false, true, false>);
  } else if (f64) {
    if (u) go(k_local<double, false, false, true>);
    else go(k_local<double, false, false, false>);
  } else if (S.has_pp) {
    if (u) go(k_local<float, false, true, true>);
    else go(k_local<float, false, true, false>);
  } else {
    go(k_local<float, false, false, false>);
  }
}

void launch_rows_f64(const DevSys& S, const DevWalkers& W, hipStream_t st) {
  rows_go<RowsF64>(S, W.pos, S.C[0], S.C[1], nullptr, W.mo, W.nw, st);
}

void launch_rows_mx(const DevSys& S, const MixedTables& M, const DevWalkers& W, hipStream_t st) {
  if (std::max(S.nmo[0], S.nmo[1]) <= 64) rows_go<RowsMx>(S, W.pos, M.Cf[0], M.Cf[1], M.spline, W.mof, W.nw, st);
  else rows_go<RowsF32>(S, W.pos, M.Cf[0], M.Cf[1], nullptr, W.mof, W.nw, st);
}

}  // namespace qw
