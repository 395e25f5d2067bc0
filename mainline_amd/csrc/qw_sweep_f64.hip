// Launches of the FP64 DMC sweep (qw_panel.hpp), one kernel per size class and trial-function
// form.
#include <stdexcept>

#include "qw_panel.hpp"
#include "qw_sweep.hpp"

namespace qw {

namespace {
template <int NW, int NS, bool JP>
void go(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st) {
  const int wpb = NW == 1 ? panel_wpb(W.nw) : 1;
  const size_t lds = panel_lds_bytes(S.ne, S.na, S.nsh, S.ntab, NS, NW, wpb);
  hipLaunchKernelGGL((k_sweep_p<NW, NS, JP>), dim3((unsigned)((W.nw + wpb - 1) / wpb)), dim3(64 * NW * wpb), lds,
                     st, S, W, A, u);
}
template <int NW, int NS>
void by_form(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st) {
  if (S.usual) go<NW, NS, true>(S, W, A, u, st);
  else go<NW, NS, false>(S, W, A, u, st);
}
}  // namespace

void launch_sweep_f64(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st) {
  const int n = S.nup > S.ndn ? S.nup : S.ndn;
  // thousands of shells (from about 2400 on): the tables and lists of four walkers do not fit one
  // block, and the two-wavefront form, which leaves the shell records in device memory, takes any size
  if (n <= 64 && panel_lds_bytes(S.ne, S.na, S.nsh, S.ntab, pick_ns(n), 1, kPanelWpb) > kLdsMax) by_form<2, 128>(S, W, A, u, st);
  else if (n <= 4) by_form<1, 4>(S, W, A, u, st);
  else if (n <= 8) by_form<1, 8>(S, W, A, u, st);
  else if (n <= 16) by_form<1, 16>(S, W, A, u, st);
  else if (n <= 32) by_form<1, 32>(S, W, A, u, st);
  else if (n <= 64) by_form<1, 64>(S, W, A, u, st);
  else if (n <= 128) by_form<2, 128>(S, W, A, u, st);
  else by_form<4, 256>(S, W, A, u, st);
}

}  // namespace qw
