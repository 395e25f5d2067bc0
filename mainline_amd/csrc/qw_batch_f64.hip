// Batched sweeps in FP64: each block runs the engine's own panel sweep (qw_panel.hpp) of its
// slot, four walkers per block up to 64 electrons of a spin, one above.
#include "qw_batch.hpp"
#include "qw_panel.hpp"

namespace qw {

template <bool JP>
__device__ __forceinline__ void batch_dmc(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int ns, int blk, int u,
                                           char* sh) {
  const int t = (int)threadIdx.x;
  const int n = S.nup > S.ndn ? S.nup : S.ndn;
  const size_t shared = (panel_shared_lds(S.na, S.nsh, S.ntab, ns ? 1 : 2) + 15) / 16 * 16;
  if (ns == 0) {
    // the wavefronts beyond the walker's own end here (barriers wait on the others only)
    if (t >= (n <= 128 ? 128 : 256)) return;
    panel_stage(S, sh, 2, t, n <= 128 ? 128 : 256);
    __syncthreads();
    if (n <= 128) sweep_panel_body<2, 128, JP>(S, W, A, blk, t, sh, sh + shared, u);
    else sweep_panel_body<4, 256, JP>(S, W, A, blk, t, sh, sh + shared, u);
    return;
  }
  panel_stage(S, sh, 1, t, 64 * kPanelWpb);
  __syncthreads();
  const int wid = t >> 6, w = blk * kPanelWpb + wid;
  if (w >= W.nw) return;
  char* own = sh + shared + (size_t)wid * panel_walker_lds(S.ne, S.nsh, ns, 1);
  switch (ns) {
    case 4: sweep_panel_body<1, 4, JP>(S, W, A, w, t & 63, sh, own, u); break;
    case 8: sweep_panel_body<1, 8, JP>(S, W, A, w, t & 63, sh, own, u); break;
    case 16: sweep_panel_body<1, 16, JP>(S, W, A, w, t & 63, sh, own, u); break;
    case 32: sweep_panel_body<1, 32, JP>(S, W, A, w, t & 63, sh, own, u); break;
    default: sweep_panel_body<1, 64, JP>(S, W, A, w, t & 63, sh, own, u); break;
  }
}

// VMC: the engine's own delayed-rejection sweeps.
__device__ __forceinline__ void batch_vmc(const QW_CONST BatchSlot& B, const SweepArgs& A, int blk, char* lds) {
  const int t = (int)threadIdx.x, lane = t & 63, wid = t >> 6;
  if (B.ns == 0) {
    if (wid >= B.wpb) return;
    char* base = lds + (size_t)wid * B.lds_w;
    const int w = blk * B.wpb + wid;
    if (B.nr == 2) sweep_w_body<2, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, base);
    else sweep_w_body<4, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, base);
    return;
  }
  const int w = blk * kBatchWpb + wid;
  // one choice of loads in flight serves the batch (every choice gives the same results)
  switch (B.ns) {
    case 4: sweep_fp64_body<4, 4, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, wid, lds); break;
    case 8: sweep_fp64_body<8, 4, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, wid, lds); break;
    case 16: sweep_fp64_body<16, 4, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, wid, lds); break;
    case 32: sweep_fp64_body<32, 4, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, wid, lds); break;
    default: sweep_fp64_body<64, 8, kBatchWpb>(gref(B.S), gref(B.W), A, w, lane, wid, lds); break;
  }
}

// DMC: three waves per SIMD, as the engine's own launches; VMC: two.
template <int DEPTH>
__global__ __launch_bounds__(256, DEPTH == 1 ? 3 : 2) void k_sweep_batch_f64(const BatchSlot* __restrict__ slots,
                                                                             int nslot, int s, int k0, int R, int sw) {
  extern __shared__ double ldsb[];
  const QW_CONST BatchSlot* sl = cptr(slots);
  int b0 = 0;
  const int i = batch_find(sl, nslot, s, k0, DEPTH, sw, (int)blockIdx.x, &b0);
  if (i < 0) return;
  const QW_CONST BatchSlot& B = sl[i];
  const int n = B.n[s];
  SweepArgs A{s, k0, min(n, k0 + R), B.tau, B.seed, 0u, (unsigned)sw, DEPTH == 1 ? 1 : 0, 0, B.stepp};
  A.dets = A.k1 == n && sw == B.ndecorr - 1;
  const int blk = (int)blockIdx.x - b0;
  if constexpr (DEPTH == 1) {
    if (B.S.usual) batch_dmc<true>(gref(B.S), gref(B.W), A, B.ns, blk, B.u, (char*)ldsb);
    else batch_dmc<false>(gref(B.S), gref(B.W), A, B.ns, blk, B.u, (char*)ldsb);
  } else {
    batch_vmc(B, A, blk, (char*)ldsb);
  }
}

void launch_sweep_batch_f64(int depth, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots, int nslot,
                            int s, int k0, int R, int sw) {
  if (depth == 1) hipLaunchKernelGGL(k_sweep_batch_f64<1>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
  else hipLaunchKernelGGL(k_sweep_batch_f64<2>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
}

}  // namespace qw
