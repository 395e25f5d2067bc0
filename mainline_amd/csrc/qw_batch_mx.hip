// Batched sweeps of the mixed path.
#include "qw_batch.hpp"
#include "qw_panel_mx.hpp"

namespace qw {

template <int DEPTH, bool JP>
__device__ __forceinline__ void batch_small(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A,
                                            int ns, int w, int lane, char* sh, char* own, int u) {
  switch (ns) {
    case 4: sweep_mxp_body<4, DEPTH, JP, false>(S, M, W, A, w, lane, sh, nullptr, own, u); break;
    case 8: sweep_mxp_body<8, DEPTH, JP, false>(S, M, W, A, w, lane, sh, nullptr, own, u); break;
    case 16: sweep_mxp_body<16, DEPTH, JP, false>(S, M, W, A, w, lane, sh, nullptr, own, u); break;
    case 32: sweep_mxp_body<32, DEPTH, JP, false>(S, M, W, A, w, lane, sh, nullptr, own, u); break;
    default: sweep_mxp_body<64, DEPTH, JP, false>(S, M, W, A, w, lane, sh, nullptr, own, u); break;
  }
}

// The mixed path (FP32 LCAO and inverse).
template <int DEPTH>
__global__ __launch_bounds__(256, 3) void k_sweep_batch_mx(const BatchSlot* __restrict__ slots, int nslot, int s, int k0,
                                                        int R, int sw) {
  extern __shared__ double ldsb[];
  const QW_CONST BatchSlot* sl = cptr(slots);
  int b0 = 0;
  const int i = batch_find(sl, nslot, s, k0, DEPTH, sw, (int)blockIdx.x, &b0);
  if (i < 0) return;
  const QW_CONST BatchSlot& B = sl[i];
  const int n = B.n[s];
  SweepArgs A{s, k0, min(n, k0 + R), B.tau, B.seed, 0u, (unsigned)sw, DEPTH == 1 ? 1 : 0, 0, B.stepp};
  A.dets = A.k1 == n && sw == B.ndecorr - 1;
  A.keep = !batch_recomputes(B.rf, n, k0, R);
  const int t = (int)threadIdx.x, blk = (int)blockIdx.x - b0;
  char* lds = (char*)ldsb;
  if (B.ns == 0) {
    // more than 64 electrons of a spin: B.wpb walkers per block, a wavefront each
    const int lane = t & 63, wid = t >> 6;
    if (wid >= B.wpb) return;
    const int w = blk * B.wpb + wid;
    char* base = lds + (size_t)wid * B.lds_w;
    if (B.nr == 2)
      sweep_w_body<float, float, DEPTH, 2, kBatchWpb>(gref(B.S), gref(B.W), gref(B.Pf), A, B.cap, w, lane, base);
    else
      sweep_w_body<float, float, DEPTH, 4, kBatchWpb>(gref(B.S), gref(B.W), gref(B.Pf), A, B.cap, w, lane, base);
    return;
  }
  // up to 64: four walkers per block share the tables
  panel_mx_stage<false>(gref(B.S), gref(B.M), s, lds, t, 64 * kBatchWpb);
  __syncthreads();
  const int wid = t >> 6, w = blk * kBatchWpb + wid;
  if (w >= B.W.nw) return;
  char* own = lds + panel_mx_shared_lds(B.S.na, B.S.nsh, B.S.ntab, 0, B.S.nsp) +
              (size_t)wid * panel_mx_walker_lds(B.S.nsh, B.ns, DEPTH);
  if (B.S.usual) batch_small<DEPTH, true>(gref(B.S), gref(B.M), gref(B.W), A, B.ns, w, t & 63, lds, own, B.u);
  else batch_small<DEPTH, false>(gref(B.S), gref(B.M), gref(B.W), A, B.ns, w, t & 63, lds, own, B.u);
}

void launch_sweep_batch_mx(int depth, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots, int nslot,
                           int s, int k0, int R, int sw) {
  if (depth == 1) hipLaunchKernelGGL(k_sweep_batch_mx<1>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
  else hipLaunchKernelGGL(k_sweep_batch_mx<2>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
}

}  // namespace qw
