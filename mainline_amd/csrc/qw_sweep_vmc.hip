// Launches of the FP64 VMC sweep (delayed rejection).
#include "qw_big.hpp"
#include "qw_sweep.hpp"

namespace qw {

namespace {
template <int U>
void small(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int nsw, int ns, hipStream_t st) {
  const size_t lds = sweep_lds_bytes(S.ne, S.na, S.nsh, S.ntab, ns, kCapF64, sizeof(double), 2);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(W.nw), dim3(64), lds, st, S, W, A, nsw); };
  switch (ns) {
    case 4: go(k_sweeps<4, U>); break;
    case 8: go(k_sweeps<8, U>); break;
    case 16: go(k_sweeps<16, U>); break;
    case 32: go(k_sweeps<32, U>); break;
    default: go(k_sweeps<64, U>); break;
  }
}
}  // namespace

void launch_sweeps_vmc64(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int nsw, int ns, int u,
                         hipStream_t st) {
  if (u == 2) small<2>(S, W, A, nsw, ns, st);
  else if (u == 8) small<8>(S, W, A, nsw, ns, st);
  else small<4>(S, W, A, nsw, ns, st);
}

void launch_sweep_vmc64_big(const DevSys& S, const DevWalkers& W, const SweepArgs& A, hipStream_t st) {
  // one wavefront per walker, lanes over two (<= 128 per spin) or four rows
  const int n = S.nup > S.ndn ? S.nup : S.ndn;
  const size_t lds = sweep_w_lds_bytes(S.ne, S.na, S.nsh, S.ntab, S.nsp);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(W.nw), dim3(kWave), lds, st, S, W, A); };
  if (n <= 2 * kWave) go(k_sweep_w<2>);
  else go(k_sweep_w<4>);
}

}  // namespace qw
