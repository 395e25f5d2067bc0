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

// The mixed path (FP32 LCAO and inverse).  JP: every slot's Jastrow and shells are the usual ones;
// those bodies alone need at most 128 registers (four blocks per compute unit instead of three).
template <int DEPTH, bool JP>
__global__ __launch_bounds__(256, JP ? 4 : 3) void k_sweep_batch_mx(const BatchSlot* __restrict__ slots, int nslot, int s, int k0,
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
    // 65 to 128 electrons of a spin: one walker per block, two wavefronts (the others end here:
    // barriers wait on the remaining ones only)
    if (t >= 128) return;
    int lo, hi;
    flush_rows(n, A.k1, B.rf, sw == B.ndecorr - 1, &lo, &hi);
    A.keep = hi > 0;
    if (JP || B.S.usual) sweep_mxb_body<2, DEPTH, true>(gref(B.S), gref(B.M), gref(B.W), A, blk, t, lds);
    else sweep_mxb_body<2, DEPTH, false>(gref(B.S), gref(B.M), gref(B.W), A, blk, t, lds);
    return;
  }
  // up to 64: four walkers per block share the tables
  panel_mx_stage<false>(gref(B.S), gref(B.M), s, lds, t, 64 * kBatchWpb);
  __syncthreads();
  const int wid = t >> 6, w = blk * kBatchWpb + wid;
  if (w >= B.W.nw) return;
  char* own = lds + panel_mx_shared_lds(B.S.na, B.S.nsh, B.S.ntab, 0, B.S.nsp) +
              (size_t)wid * panel_mx_walker_lds(B.S.nsh, B.ns, DEPTH, JP || B.S.usual);
  if (JP || B.S.usual) batch_small<DEPTH, true>(gref(B.S), gref(B.M), gref(B.W), A, B.ns, w, t & 63, lds, own, B.u);
  else batch_small<DEPTH, false>(gref(B.S), gref(B.M), gref(B.W), A, B.ns, w, t & 63, lds, own, B.u);
}

// The updates of the moves [k0, k0 + R) applied to the rows still used (k_flush_mx), for the slots
// above 64 electrons of a spin that need it; a block per walker.
__global__ __launch_bounds__(128, 3) void k_flush_batch(const BatchSlot* __restrict__ slots, int nslot, int s, int k0, int R,
                                                        int depth, int sw) {
  __shared__ FlushLds<128> L;
  const QW_CONST BatchSlot* sl = cptr(slots);
  int b0 = 0;
  for (int i = 0; i < nslot; i++) {
    int lo, hi;
    if (!batch_flushes(sl[i], s, k0, R, depth, sw, &lo, &hi)) continue;
    if ((int)blockIdx.x < b0 + sl[i].W.nw) {
      const QW_CONST BatchSlot& B = sl[i];
      const int n = B.n[s], k1 = min(n, k0 + R), dets = k1 == n && sw == B.ndecorr - 1;
      flush_mx_body<128>(gref(B.S), gref(B.W), s, k0, k1 - k0, lo, hi, dets, (int)blockIdx.x - b0, (int)threadIdx.x, L);
      return;
    }
    b0 += sl[i].W.nw;
  }
}

void launch_sweep_batch_mx(int depth, bool usual, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots,
                           int nslot, int s, int k0, int R, int sw) {
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw); };
  if (depth == 1) usual ? go(k_sweep_batch_mx<1, true>) : go(k_sweep_batch_mx<1, false>);
  else usual ? go(k_sweep_batch_mx<2, true>) : go(k_sweep_batch_mx<2, false>);
}

void launch_flush_batch(unsigned grid, hipStream_t st, const BatchSlot* slots, int nslot, int s, int k0, int R, int depth,
                        int sw) {
  hipLaunchKernelGGL(k_flush_batch, dim3(grid), dim3(128), 0, st, slots, nslot, s, k0, R, depth, sw);
}

}  // namespace qw
