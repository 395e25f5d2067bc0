// Launches of the mixed-precision sweeps, one kernel per size class, method depth and LCAO mode.
#include "qw_big_mx.hpp"
#include "qw_mixed.hpp"
#include "qw_panel_mx.hpp"
#include "qw_sweep.hpp"

namespace qw {

namespace {
// FP32 LCAO (qw_panel_mx.hpp)
template <int NS, int DEPTH, bool JP, bool STAGE>
void go_p(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st) {
  const int wpb = STAGE ? kPanelWpb : panel_wpb(W.nw);  // (staged coefficients: always shared by four)
  const size_t lds = panel_mx_lds_bytes(S.na, S.nsh, S.ntab, NS, DEPTH, STAGE ? S.nb : 0, S.nsp, JP, wpb);
  hipLaunchKernelGGL((k_sweep_mxp<NS, DEPTH, JP, STAGE>), dim3((unsigned)((W.nw + wpb - 1) / wpb)),
                     dim3(64 * wpb), lds, st, S, M, W, A, u);
}
// the form for thousands of shells: one instantiation for every size and trial function
template <int DEPTH>
void go_shells(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st) {
  const size_t lds = panel_mx_shared_lds(S.na, 0, S.ntab, 0, S.nsp) + panel_mx_walker_lds(S.nsh, 64, DEPTH, false);
  hipLaunchKernelGGL((k_sweep_mxp<64, DEPTH, false, false, false>), dim3(W.nw), dim3(64), lds, st, S, M, W, A, u);
}
template <int NS, int DEPTH>
void panel(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int choice, hipStream_t st) {
  if (panel_mx_lds_bytes(S.na, S.nsh, S.ntab, NS, DEPTH, 0, S.nsp, S.usual) > kLdsMax) go_shells<DEPTH>(S, M, W, A, choice, st);
  else if (choice >= 100) {
    if (S.usual) go_p<NS, DEPTH, true, true>(S, M, W, A, choice - 100, st);
    else go_p<NS, DEPTH, false, true>(S, M, W, A, choice - 100, st);
  } else {
    if (S.usual) go_p<NS, DEPTH, true, false>(S, M, W, A, choice, st);
    else go_p<NS, DEPTH, false, false>(S, M, W, A, choice, st);
  }
}
// LCAO on the matrix cores
template <int NS, int DEPTH, int MODE>
void go_m(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, hipStream_t st) {
  const size_t lds = sweep_mx_lds_bytes(S.ne, S.na, S.nsh, S.ntab, NS, M.ldchi, DEPTH);
  hipLaunchKernelGGL((k_sweep_mx<NS, DEPTH, MODE>), dim3(W.nw), dim3(64), lds, st, S, M, W, A);
}
template <int NS, int DEPTH>
void by_mode(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int mode, int choice,
             hipStream_t st) {
  if (mode == LCAO_BF16X6) go_m<NS, DEPTH, LCAO_BF16X6>(S, M, W, A, st);
  else if (mode == LCAO_BF16X3) go_m<NS, DEPTH, LCAO_BF16X3>(S, M, W, A, st);
  else panel<NS, DEPTH>(S, M, W, A, choice, st);
}
template <int DEPTH>
void by_size(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int ns, int mode, int choice,
             hipStream_t st) {
  switch (ns) {
    case 4: by_mode<4, DEPTH>(S, M, W, A, mode, choice, st); break;
    case 8: by_mode<8, DEPTH>(S, M, W, A, mode, choice, st); break;
    case 16: by_mode<16, DEPTH>(S, M, W, A, mode, choice, st); break;
    case 32: by_mode<32, DEPTH>(S, M, W, A, mode, choice, st); break;
    default: by_mode<64, DEPTH>(S, M, W, A, mode, choice, st); break;
  }
}
}  // namespace

void launch_sweep_mx(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth, int ns,
                     int mode, int choice, hipStream_t st) {
  if (depth == 1) by_size<1>(S, M, W, A, ns, mode, choice, st);
  else by_size<2>(S, M, W, A, ns, mode, choice, st);
}

void launch_sweep_mx_big(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth,
                         hipStream_t st) {
  const int n = S.nup > S.ndn ? S.nup : S.ndn, nw = n <= 128 ? 2 : 4;
  const size_t lds = sweep_mxb_lds_bytes(S.ne, S.na, S.nsh, S.ntab, n, nw, depth, S.usual);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(W.nw), dim3(64 * nw), lds, st, S, M, W, A); };
  if (nw == 2) {
    if (depth == 1) S.usual ? go(k_sweep_mxb<2, 1, true>) : go(k_sweep_mxb<2, 1, false>);
    else S.usual ? go(k_sweep_mxb<2, 2, true>) : go(k_sweep_mxb<2, 2, false>);
  } else {
    if (depth == 1) S.usual ? go(k_sweep_mxb<4, 1, true>) : go(k_sweep_mxb<4, 1, false>);
    else S.usual ? go(k_sweep_mxb<4, 2, true>) : go(k_sweep_mxb<4, 2, false>);
  }
}

void launch_flush_mx(const DevSys& S, const DevWalkers& W, int s, int k0, int np, int lo, int hi, int dets,
                     hipStream_t st) {
  if ((S.nup > S.ndn ? S.nup : S.ndn) <= 128)
    hipLaunchKernelGGL(k_flush_mx<128>, dim3(W.nw), dim3(128), 0, st, S, W, s, k0, np, lo, hi, dets);
  else
    hipLaunchKernelGGL(k_flush_mx<256>, dim3(W.nw), dim3(256), 0, st, S, W, s, k0, np, lo, hi, dets);
}

}  // namespace qw
