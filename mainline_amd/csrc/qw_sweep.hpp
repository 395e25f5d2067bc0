// Sweep and local-energy launches compiled in translation units of their own.
#pragma once
#include "qw_kernels.hpp"
#include "qw_mixed.hpp"

namespace qw {

// The DMC moves A of every walker in FP64 (up to 256 electrons of a spin); u: coefficient loads in
// flight in the LCAO, halved (2, 4 or 8; every choice gives the same results).
void launch_sweep_f64(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int u, hipStream_t st);
// The VMC moves in FP64: nsw sweeps of both spins (A: their common arguments) up to 64 electrons of
// a spin (ns: register tile of the inverse), and one spin's sweep above.
void launch_sweeps_vmc64(const DevSys& S, const DevWalkers& W, const SweepArgs& A, int nsw, int ns, int u,
                         hipStream_t st);
void launch_sweep_vmc64_big(const DevSys& S, const DevWalkers& W, const SweepArgs& A, hipStream_t st);

// The same on the mixed path: up to 64 electrons of a spin (ns: register tile, mode: LcaoMode,
// choice: 100 * (coefficients staged in LDS) + loads in flight), and above.
void launch_sweep_mx(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth, int ns,
                     int mode, int choice, hipStream_t st);
void launch_sweep_mx_big(const DevSys& S, const MixedTables& M, const DevWalkers& W, const SweepArgs& A, int depth,
                         hipStream_t st);
// ... of at most 32 moves, whose updates this launch then applies to the rows [lo, hi) outside the
// moved ones (dets: and writes the determinant parts).
void launch_flush_mx(const DevSys& S, const DevWalkers& W, int s, int k0, int np, int lo, int hi, int dets, hipStream_t st);

// The local energy of every walker (f64: FP64 caches).
void launch_local(const DevSys& S, const DevWalkers& W, const LocalArgs& A, bool f64, hipStream_t st);

// MO value, gradient and laplacian rows of every electron at W.pos, in FP64 and on the mixed path
// (FP32 LCAO).
void launch_rows_f64(const DevSys& S, const DevWalkers& W, hipStream_t st);
void launch_rows_mx(const DevSys& S, const MixedTables& M, const DevWalkers& W, hipStream_t st);

}  // namespace qw
