// Batched sweeps of the mixed path.
#include "qw_batch.hpp"

namespace qw {

// The mixed path (FP32 LCAO and inverse).
template <int DEPTH>
__global__ __launch_bounds__(256, 2) void k_sweep_batch_mx(const BatchSlot* __restrict__ slots, int nslot, int s, int k0,
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
  const int lane = t & 63, wid = t >> 6, w = blk * kBatchWpb + wid;
#define QW_MX(NS, U) \
  sweep_mx_body<NS, DEPTH, LCAO_FP32, U, kBatchWpb, false>(gref(B.S), gref(B.M), gref(B.W), A, w, lane, wid, lds)
#define QW_CASES(X, U0, U1, U2)                 \
  switch (B.ns * 100 + B.u) {                   \
    case 400 + U0: X(4, U0); break;             \
    case 400 + U1: X(4, U1); break;             \
    case 400 + U2: X(4, U2); break;             \
    case 800 + U0: X(8, U0); break;             \
    case 800 + U1: X(8, U1); break;             \
    case 800 + U2: X(8, U2); break;             \
    case 1600 + U0: X(16, U0); break;           \
    case 1600 + U1: X(16, U1); break;           \
    case 1600 + U2: X(16, U2); break;           \
    case 3200 + U0: X(32, U0); break;           \
    case 3200 + U1: X(32, U1); break;           \
    case 3200 + U2: X(32, U2); break;           \
    case 6400 + U0: X(64, U0); break;           \
    case 6400 + U1: X(64, U1); break;           \
    default: X(64, U2); break;                  \
  }
  QW_CASES(QW_MX, 4, 8, 16)
#undef QW_CASES
#undef QW_MX
}

void launch_sweep_batch_mx(int depth, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots, int nslot,
                           int s, int k0, int R, int sw) {
  if (depth == 1) hipLaunchKernelGGL(k_sweep_batch_mx<1>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
  else hipLaunchKernelGGL(k_sweep_batch_mx<2>, dim3(grid), dim3(256), lds, st, slots, nslot, s, k0, R, sw);
}

}  // namespace qw
