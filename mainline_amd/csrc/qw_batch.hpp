// The slot table of launches covering several systems (qw_batch.hip), and the batched sweeps'
// launchers (translation units of their own).
#pragma once
#include "qw_big_mx.hpp"
#include "qw_kernels.hpp"
#include "qw_mixed.hpp"

namespace qw {

// One system of a batched launch.
struct BatchSlot {
  DevSys S;
  MixedTables M;
  DevWalkers W;
  DmcCtl* ctl;
  unsigned long long* keys;
  int* vals;
  int* psrc;
  int* pdst;
  unsigned* stepp;
  unsigned long long seed;
  int n[2];     // electrons of each spin
  int ns;       // register tile of the inverse (4..64); 0 = more than 64 electrons of a spin
  int u;        // LCAO coefficient loads in flight (per size bucket, tuned)
  int inv_rows; // 33..64 electrons of a spin: row-per-lane inversion instead of 8x8 blocks
  // the slot's method: DMC (depth 1, node-crossing moves rejected, weights and branching)
  // or VMC (depth 2 with delayed rejection, ndecorr sweeps per step)
  int depth, ndecorr, lmode, pp_mode;
  int branch_np;  // branching after this step: the feedback interval's steps (0 = none)
  double tau;
  // walkers per 256-thread block; FP64 VMC above 64 electrons of a spin: LDS bytes of each walker
  // and rows per lane of the one-wavefront sweep (2 or 4)
  int wpb, lds_w, nr;
  // the slot's FP64 recompute interval (mixed path): a multiple of the batch's launch interval
  // R, or at least n (once per sweep); the recompute launch after moves [k0, k0 + R) covers
  // the slot when k0 + R is a multiple of rf or ends the sweep
  int rf;
};

constexpr int kBatchWpb = 4;  // walkers (wavefronts) per 256-thread block for <= 64 per spin

// A field of the slot table (constant address space) as the generic reference the kernel
// bodies take.
template <typename T>
__device__ inline const T& gref(const QW_CONST T& r) {
  return *(const T*)&r;
}

// Blocks of a slot in a sweep launch (wpb walkers each), and in a recompute launch (a
// wavefront per walker up to 64 electrons of a spin, a whole block per walker above).
__device__ inline int batch_blocks(const QW_CONST BatchSlot& B) { return (B.W.nw + B.wpb - 1) / B.wpb; }
__device__ inline int batch_blocks_inv(const QW_CONST BatchSlot& B) {
  return B.ns ? (B.W.nw + kBatchWpb - 1) / kBatchWpb : B.W.nw;
}

// Whether slot B recomputes spin s after the moves [k0, k0 + R) (host and device).
__host__ __device__ inline bool batch_recomputes(int rf, int n, int k0, int R) {
  return (k0 + R) % rf == 0 || k0 + R >= n;
}

// The slot of block `blk` among the slots of method depth `depth` with a sweep `sw` and moves
// k0.. of spin s (INV: and a recompute after the R moves from k0), and the slot's first block
// (*b0).  Uniform over the block; nslot is small.
template <bool INV = false>
__device__ inline int batch_find(const QW_CONST BatchSlot* sl, int nslot, int s, int k0, int depth, int sw, int blk,
                                 int* b0, int R = 0) {
  int acc = 0;
  for (int i = 0; i < nslot; i++) {
    if (sl[i].n[s] <= k0 || sl[i].depth != depth || sw >= sl[i].ndecorr) continue;
    if (INV && !batch_recomputes(sl[i].rf, sl[i].n[s], k0, R)) continue;
    const int nb = INV ? batch_blocks_inv(sl[i]) : batch_blocks(sl[i]);
    if (blk < acc + nb) {
      *b0 = acc;
      return i;
    }
    acc += nb;
  }
  return -1;
}

// Whether slot B (above 64 electrons of a spin, mixed path) applies the updates of the moves
// [k0, k0 + R) of spin s to other rows, and to which (host and device).
template <typename SLOT>
__host__ __device__ inline bool batch_flushes(const SLOT& B, int s, int k0, int R, int depth, int sw, int* lo, int* hi) {
  if (B.ns != 0 || B.n[s] <= k0 || B.depth != depth || sw >= B.ndecorr) return false;
  const int n = B.n[s], k1 = n < k0 + R ? n : k0 + R;
  flush_rows(n, k1, B.rf, sw == B.ndecorr - 1, lo, hi);
  return *hi > 0;
}

// Moves k0 .. min(n_s, k0 + R) of spin s, in sweep `sw` of the step, of every slot of method
// depth `depth` (1 DMC, 2 VMC) with more than k0 electrons of that spin: grid blocks of 256
// threads with lds bytes each.
void launch_sweep_batch_f64(int depth, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots, int nslot,
                            int s, int k0, int R, int sw);
void launch_sweep_batch_mx(int depth, bool usual, unsigned grid, size_t lds, hipStream_t st, const BatchSlot* slots,
                           int nslot, int s, int k0, int R, int sw);
void launch_flush_batch(unsigned grid, hipStream_t st, const BatchSlot* slots, int nslot, int s, int k0, int R, int depth,
                        int sw);

}  // namespace qw
