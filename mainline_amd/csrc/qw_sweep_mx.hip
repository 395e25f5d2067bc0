// Launches of the mixed-precision sweeps, one kernel per size class, method depth and LCAO mode.
#include "qw_big.hpp"
#include "qw_mixed.hpp"
#include "qw_sweep.hpp"

namespace qw {

namespace {
template <int DEPTH, int MODE, int U, int WPB>
void mixed_u(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int ns, hipStream_t st) {
  const size_t lds = sweep_mx_lds_bytes(S.ne, S.na, S.nsh, S.ntab, ns, MODE, M.ldchi, DEPTH, S.nb, S.nsp, WPB);
  const unsigned grid = (unsigned)((W.nw + WPB - 1) / WPB);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WPB), lds, st, S, M, W, A); };
  switch (ns) {
    case 4: go(k_sweep_mx<4, DEPTH, MODE, U, WPB>); break;
    case 8: go(k_sweep_mx<8, DEPTH, MODE, U, WPB>); break;
    case 16: go(k_sweep_mx<16, DEPTH, MODE, U, WPB>); break;
    case 32: go(k_sweep_mx<32, DEPTH, MODE, U, WPB>); break;
    default: go(k_sweep_mx<64, DEPTH, MODE, U, WPB>); break;
  }
}
template <int DEPTH>
void mixed_mode(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int ns, int mode,
                int choice, hipStream_t st) {
  if (mode == LCAO_BF16X6) mixed_u<DEPTH, LCAO_BF16X6, 8, 1>(S, M, W, A, ns, st);
  else if (mode == LCAO_BF16X3) mixed_u<DEPTH, LCAO_BF16X3, 8, 1>(S, M, W, A, ns, st);
  else switch (choice) {
    case 4: mixed_u<DEPTH, LCAO_FP32, 4, 1>(S, M, W, A, ns, st); break;
    case 16: mixed_u<DEPTH, LCAO_FP32, 16, 1>(S, M, W, A, ns, st); break;
    case 104: mixed_u<DEPTH, LCAO_FP32, 4, kWpbCL>(S, M, W, A, ns, st); break;
    case 108: mixed_u<DEPTH, LCAO_FP32, 8, kWpbCL>(S, M, W, A, ns, st); break;
    case 116: mixed_u<DEPTH, LCAO_FP32, 16, kWpbCL>(S, M, W, A, ns, st); break;
    default: mixed_u<DEPTH, LCAO_FP32, 8, 1>(S, M, W, A, ns, st); break;
  }
}
}  // namespace

void launch_sweep_mx(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth, int ns,
                     int mode, int choice, hipStream_t st) {
  if (depth == 1) mixed_mode<1>(S, M, W, A, ns, mode, choice, st);
  else mixed_mode<2>(S, M, W, A, ns, mode, choice, st);
}

void launch_sweep_mx_big(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth,
                         hipStream_t st) {
  // one wavefront per walker, lanes over two (<= 128 per spin) or four rows
  const BigPtrs<float> P{W.invf, W.mof, {M.Cf[0], M.Cf[1]}, M.spline};
  const size_t lds = sweep_w_lds_bytes(S.ne, S.na, S.nsh, S.ntab, S.nsp, kCapF32, sizeof(float));
  const bool nr2 = (S.nup > S.ndn ? S.nup : S.ndn) <= 2 * kWave;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(W.nw), dim3(kWave), lds, st, S, W, P, A, kCapF32); };
  if (depth == 1) {
    if (nr2) go(k_sweep_w<float, float, 1, 2>);
    else go(k_sweep_w<float, float, 1, 4>);
  } else {
    if (nr2) go(k_sweep_w<float, float, 2, 2>);
    else go(k_sweep_w<float, float, 2, 4>);
  }
}

}  // namespace qw
