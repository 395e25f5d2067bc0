// MO value, gradient and laplacian rows of every electron of every walker (walker refresh,
// fixed-configuration evaluation; src/orbitals/MO_matrix_cutoff.h:480-560), all size classes.
//
//   k_rows<KIND, NR, G, FG>  a wavefront takes G electrons at a time (1, 2 or 4 of up to 64 / G
//       orbitals, so that small systems fill the lanes) or one electron of up to 64 NR orbitals.
//       Shells in windows of kRowsWin: the active ones are compacted in shell order (no table of a
//       window's size per walker), their functions evaluated a batch at a time into a tile in LDS,
//       and the batch is contracted with eight coefficient loads in flight.
//
// KIND: RowsF64; RowsMx (FP32 distances, table and tile: up to 64 electrons of a spin on the mixed
// path); RowsF32 (FP64 basis values rounded to an FP32 tile: above 64 electrons on the mixed path).
// Every orbital sums its functions in shell order (RowsF64 with NR = 1: per shell chunk of the
// system, then over the chunks).
//
// What bounds it: vector issue of the contraction, five FMAs per active function, electron and 64
// orbitals, with the coefficients coming from L2.  One electron per 64- or 256-thread block with a
// tile for 640 functions left five such blocks on a compute unit, one wavefront each evaluating.
// Measured: RowsMx, 2048 walkers of 128 electrons 1.19 -> 0.79 ms; RowsF64, 256 of 128 0.275 ->
// 0.185 ms; RowsF32, 1024 of 192 3.16 -> 1.17 ms and 1024 of 512 30.2 -> 14.7 ms.
#pragma once
#include "qw_mixed.hpp"
#include "qw_move.hpp"

namespace qw {

enum RowsKind { RowsF64 = 0, RowsMx = 1, RowsF32 = 2 };
constexpr int kRowsWin = 512;  // shells of a window
constexpr int kRowsWaves = 4;  // wavefronts of a block
template <int KIND>
struct RowsT {
  typedef float T;
};
template <>
struct RowsT<RowsF64> {
  typedef double T;
};
// Functions of a tile.  FG: F and G shells, each a long serial loop that every batch of shells repeats:
// a large tile (no larger than the basis, so that small systems keep four wavefronts per SIMD) and one
// electron per wavefront.  Six atoms of 29 functions with 7F and 9G shells, 24 electrons: 512
// configurations 276 -> 146 us, 1024 walkers 696 -> 268 us.
template <int KIND, bool FG>
__host__ __device__ inline int rows_cap(int nb) {
  if constexpr (FG) return nb < 256 ? (nb + 1) & ~1 : 256;
  else return KIND == RowsF64 ? 96 : 128;
}

// LDS of a wavefront: G tiles of values and coefficient offsets, G lists.
template <int KIND, int G, bool FG>
__host__ __device__ inline size_t rows_wave_lds(int nb, int nsh) {
  return G * ((size_t)rows_cap<KIND, FG>(nb) * (5 * sizeof(typename RowsT<KIND>::T) + 4) +
              (size_t)((nsh < kRowsWin ? nsh : kRowsWin) + 3) / 4 * 16);
}

// Active shells of [sh0, sh1) (at most kRowsWin) at p, in order, into the list.
template <int KIND>
__device__ inline int rows_active(const DevSys& S, const double p[3], int sh0, int sh1, int* list, int lane) {
  int n = 0;
  for (int s0 = sh0; s0 < sh1; s0 += kWave) {
    const int sh = s0 + lane;
    bool act = false;
    if (sh < sh1) {
      if constexpr (KIND == RowsMx) {
        const ShellDesc& d = S.shells[sh];
        const double* ap = S.atom_pos + 3 * d.atom;
        const float x = (float)(p[0] - ap[0]), y = (float)(p[1] - ap[1]), z = (float)(p[2] - ap[2]);
        const float r = sqrtf(x * x + y * y + z * z);
        act = r < (float)d.rcut && r < (float)d.objthr;
      } else {
        const ShellLds d = S.shl[sh];
        const double* ap = S.atom_pos + 3 * shl_atom(d.meta);
        const double x = p[0] - ap[0], y = p[1] - ap[1], z = p[2] - ap[2];
        act = x * x + y * y + z * z < d.rc2;
      }
    }
    const unsigned long long m = __ballot(act);
    if (act) list[n + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = sh;
    n += __popcll(m);
  }
  return n;
}

// One batch of the list from i0 on into the tile; n: orbitals per coefficient row.  Returns the
// shells taken.
template <int KIND, bool FG>
__device__ inline int rows_batch(const DevSys& S, const float* splf, const double p[3], const int* list, int i0, int nact,
                                 int n, typename RowsT<KIND>::T* chi, int* roff, int* nfun, int lane) {
  typedef typename RowsT<KIND>::T T;
  const int cap = rows_cap<KIND, FG>(S.nb);
  const int i = i0 + lane;
  ShellLds d;
  int nf = 0;
  if (i < nact) {
    d = S.shl[list[i]];
    nf = shl_nf(d.meta);
  }
  int tot;
  const int at = wave_excl_scan(nf, lane, &tot);
  const bool fit = nf > 0 && at + nf <= cap;
  const int take = __popcll(__ballot(fit));
  *nfun = take ? __builtin_amdgcn_readlane(at + nf, take - 1) : 0;
  if (fit) {
    const int tab = shl_table(d.meta);
    const double* ap = S.atom_pos + 3 * shl_atom(d.meta);
    if constexpr (KIND == RowsMx) {
      const float x = (float)(p[0] - ap[0]), y = (float)(p[1] - ap[1]), z = (float)(p[2] - ap[2]);
      const float r = sqrtf(x * x + y * y + z * z);
      int iv = (int)(r * (float)S.tab_inv[tab]);
      iv = iv < 0 ? 0 : (iv >= S.nint ? S.nint - 1 : iv);
      const float4 c = *(const float4*)(splf + ((size_t)tab * S.nint + iv) * 4);
      const float h = r - iv * (float)S.tab_sp[tab];
      const float f = c.x + h * (c.y + h * (c.z + h * c.w));
      const float fd = (c.y + h * (2.f * c.z + h * (3.f * c.w))) / r;
      const float f2 = 2.f * c.z + 6.f * h * c.w;
      shell_lap<T, FG>(shl_sym(d.meta), f, fd, f2, x, y, z, chi + at, cap);
    } else {
      const double x = p[0] - ap[0], y = p[1] - ap[1], z = p[2] - ap[2];
      const double r = sqrt(x * x + y * y + z * z);
      int iv = (int)(r * S.tab_inv[tab]);
      iv = iv < 0 ? 0 : (iv >= S.nint ? S.nint - 1 : iv);
      const double* c = S.spline + ((size_t)tab * S.nint + iv) * 4;
      const double c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
      const double h = r - iv * S.tab_sp[tab];
      const double f = c0 + h * (c1 + h * (c2 + h * c3));
      const double fd = (c1 + h * (2 * c2 + h * (3 * c3))) / r;
      const double f2 = 2 * c2 + 6 * h * c3;
      shell_lap<T, FG>(shl_sym(d.meta), f, fd, f2, x, y, z, chi + at, cap);
    }
    for (int q = 0; q < nf; q++) roff[at + q] = (d.f0 + q) * n * (int)sizeof(T);
  }
  return take;
}

// lcao_batch for orbitals j, j + 64, ... (NR of them, those below n) of one electron.
template <typename T, int NR>
__device__ inline void rows_lcao(const T* __restrict__ C, const int* roff, const T* chi, int ld, int nfun, T acc[NR][5],
                                 int n, int lane) {
  if constexpr (NR == 1) {
    if (lane < n) lcao_batch<T, 8>(C, roff, chi, ld, nfun, acc[0], lane);
  } else {
    constexpr int U = 4;
    const char* Cb = reinterpret_cast<const char*>(C);
    unsigned lb[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {  // lanes past the end repeat the last orbital
      const int j = lane + kWave * r;
      lb[r] = (unsigned)(j < n ? j : n - 1) * (unsigned)sizeof(T);
    }
    int b = 0;
    for (; b + U <= nfun; b += U) {
      T cv[U][NR];
#pragma unroll
      for (int q = 0; q < U; q++)
#pragma unroll
        for (int r = 0; r < NR; r++) cv[q][r] = *reinterpret_cast<const T*>(Cb + ((unsigned)roff[b + q] + lb[r]));
      __builtin_amdgcn_sched_barrier(0);  // all loads issue before the first use
#pragma unroll
      for (int q = 0; q < U; q++)
#pragma unroll
        for (int c = 0; c < 5; c++) {
          const T x = chi[c * ld + b + q];
#pragma unroll
          for (int r = 0; r < NR; r++) acc[r][c] += cv[q][r] * x;
        }
    }
    for (; b < nfun; b++)
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const T cv = *reinterpret_cast<const T*>(Cb + ((unsigned)roff[b] + lb[r]));
#pragma unroll
        for (int c = 0; c < 5; c++) acc[r][c] += cv * chi[c * ld + b];
      }
  }
}

template <int KIND, int NR, int G, bool FG>
__global__ __launch_bounds__(64 * kRowsWaves, 3) void k_rows(DevSys S, const double* wpos,
                                                             const typename RowsT<KIND>::T* C0,
                                                             const typename RowsT<KIND>::T* C1, const float* splf,
                                                             typename RowsT<KIND>::T* mo_out, int nw) {
  static_assert(NR == 1 || G == 1, "several electrons or several orbitals per lane");
  typedef typename RowsT<KIND>::T T;
  constexpr int LE = kWave / G;
  const int cap = rows_cap<KIND, FG>(S.nb);
  extern __shared__ double ldsr[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  char* own = (char*)ldsr + (size_t)wid * rows_wave_lds<KIND, G, FG>(S.nb, S.nsh);
  T* chi0 = (T*)own;
  int* roff0 = (int*)(chi0 + (size_t)G * 5 * cap);
  int* list0 = roff0 + G * cap;
  const int ll = ((S.nsh < kRowsWin ? S.nsh : kRowsWin) + 3) / 4 * 4;
  const size_t total = (size_t)nw * S.ne;
  const int el = lane / LE, lj = lane % LE;  // this lane's electron of the group and orbital
  for (size_t g = ((size_t)blockIdx.x * kRowsWaves + wid) * G; g < total; g += (size_t)gridDim.x * kRowsWaves * G) {
    double p[G][3];
    int n[G], i0[G], nact[G], nfun[G];
#pragma unroll
    for (int x = 0; x < G; x++) {
      const size_t ge = g + x < total ? g + x : total - 1;  // past the end: the last electron again
      n[x] = (int)(ge % S.ne) < S.nup ? S.nmo[0] : S.nmo[1];
      for (int d = 0; d < 3; d++) p[x][d] = wpos[ge * 3 + d];
    }
    const size_t mye = g + el < total ? g + el : total - 1;
    const int mys = (int)(mye % S.ne) < S.nup ? 0 : 1, myn = S.nmo[mys];
    const T* C = mys ? C1 : C0;
    T acc[NR][5];
#pragma unroll
    for (int r = 0; r < NR; r++)
      for (int c = 0; c < 5; c++) acc[r][c] = 0;
    constexpr bool parts = KIND == RowsF64 && NR == 1;
    const int nchunk = parts ? S.nchunk : 1;
    for (int ch = 0; ch < nchunk; ch++) {
      const int sh0 = parts ? S.chunk_sh0[ch] : 0, sh1 = parts ? S.chunk_sh0[ch + 1] : S.nsh;
      T a[NR][5];
#pragma unroll
      for (int r = 0; r < NR; r++)
        for (int c = 0; c < 5; c++) a[r][c] = 0;
      for (int w0 = sh0; w0 < sh1; w0 += kRowsWin) {
        const int w1 = w0 + kRowsWin < sh1 ? w0 + kRowsWin : sh1;
#pragma unroll
        for (int x = 0; x < G; x++) {
          nact[x] = rows_active<KIND>(S, p[x], w0, w1, list0 + x * ll, lane);
          i0[x] = 0;
        }
        wave_sync();
        while (true) {
          bool more = false;
          int myf = 0;
#pragma unroll
          for (int x = 0; x < G; x++) {
            nfun[x] = 0;
            if (i0[x] < nact[x])
              i0[x] += rows_batch<KIND, FG>(S, splf, p[x], list0 + x * ll, i0[x], nact[x], n[x],
                                            chi0 + (size_t)x * 5 * cap, roff0 + x * cap, &nfun[x], lane);
            more |= i0[x] < nact[x];
            if (x == el) myf = nfun[x];
          }
          wave_sync();
          rows_lcao<T, NR>(C, roff0 + el * cap, chi0 + (size_t)el * 5 * cap, cap, myf, a, myn, lj);
          wave_sync();
          if (!more) break;
        }
      }
#pragma unroll
      for (int r = 0; r < NR; r++)
        for (int c = 0; c < 5; c++) acc[r][c] += a[r][c];
    }
    if (g + el < total) {
      T* row = mo_out + mye * 5 * S.nsp;
#pragma unroll
      for (int r = 0; r < NR; r++)
        if (lj + kWave * r < myn)
          for (int c = 0; c < 5; c++) row[(size_t)c * S.nsp + lj + kWave * r] = acc[r][c];
    }
  }
}

template <int KIND>
inline void rows_go(const DevSys& S, const double* pos, const typename RowsT<KIND>::T* C0,
                    const typename RowsT<KIND>::T* C1, const float* splf, typename RowsT<KIND>::T* out, int nw,
                    hipStream_t st) {
  const int n = S.nmo[0] > S.nmo[1] ? S.nmo[0] : S.nmo[1];
  const size_t total = (size_t)nw * S.ne;
  auto go = [&](auto kern, int G, size_t lds) {
    const size_t blocks = (total + kRowsWaves * G - 1) / (kRowsWaves * G);
    // whole rounds of four blocks per compute unit; with F and G shells (three) an electron per wavefront
    const size_t most = S.fg ? 65536 : 4096;
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min(blocks, most)), dim3(64 * kRowsWaves), kRowsWaves * lds, st,
                       S, pos, C0, C1, splf, out, nw);
  };
#define ROWS(NR, G, FG) go(k_rows<KIND, NR, G, FG>, G, rows_wave_lds<KIND, G, FG>(S.nb, S.nsh))
  if constexpr (KIND != RowsF32) {
    // several electrons per wavefront fill the lanes of small systems (32 orbitals, 32000 electrons:
    // 163 -> 112 us), as long as that leaves four wavefronts per SIMD (1024 electrons of a
    // 2-orbital system: 7 us one at a time, 12 us four at a time)
    constexpr size_t kFill = 4096;
    if (n <= 16 && total >= 4 * kFill && !S.fg) return ROWS(1, 4, false);
    if (n <= 32 && total >= 2 * kFill && !S.fg) return ROWS(1, 2, false);
    if (n <= 64) return S.fg ? ROWS(1, 1, true) : ROWS(1, 1, false);
  }
  if constexpr (KIND != RowsMx) {
    if (n <= 128) S.fg ? ROWS(2, 1, true) : ROWS(2, 1, false);
    else S.fg ? ROWS(4, 1, true) : ROWS(4, 1, false);
  }
#undef ROWS
}

}  // namespace qw
