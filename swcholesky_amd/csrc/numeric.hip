// MI355X (gfx950) numeric phase: supernodal Cholesky, triangular solves, residual,
// refinement and adjoint, behind the C ABI of include/swcholesky_amd.h.
//
// The factor is multifrontal (fronts.h, front_kernels.h): two launches per level of the
// supernode tree.  The left-looking path (plan.h and the tile and panel kernels here)
// serves structures without a front tree, arenas that do not fit and H-level schedules.
// The solves are one persistent launch per sweep (sweeps.h, sweep_kernels.h); the selected
// inverse is in selinv.h and selinv_kernels.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "analysis.h"
#include "capi_common.h"
#include "fronts.h"
#include "plan.h"
#include "selinv.h"

using swc::Panel;
using swc::Plan;
using swc::Task;
using swc::Tile;

namespace {

constexpr int kThreads = 256;
constexpr int kLdsLd = swc::TM + 1;  // padded column stride of LDS tiles (doubles)

#define SWC_HIP(call)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return swc_set_error(SWC_EDEVICE, std::string(#call ": ") + hipGetErrorString(e_));  \
  } while (0)

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------

__global__ void k_fill(double* __restrict__ x, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) x[i] = v;
}

// L[amap[q]] = vals[q]: copy-in of A into the supernodal storage
// (_pthread_inner.c:139-147, with the map lookup precomputed).
__global__ void k_assemble(double* __restrict__ L, const int64_t* __restrict__ amap,
                           const double* __restrict__ vals, int64_t nnz) {
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; q < nnz; q += stride) L[amap[q]] = vals[q];
}

__global__ void k_set_int(int* p, int v) { *p = v; }

// Workgroup barrier for LDS traffic only: it waits for this wave's LDS
// operations but not for its global loads, which stay in flight across it
// (__syncthreads() waits for every outstanding memory operation).  Used where no
// thread reads global data that another thread of the workgroup has written.
// The wait is explicit: behind a store in a branch of its own the compiler left out
// the one that the release fence stands for, and waves passed the barrier with the
// store still on its way.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), the other counters free
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Lane layout of the 16x16x4 MFMA builtins on gfx950 (fixed by an on-device
// probe of both): lane l feeds A[l%16][k0 + l/16] and B^T[k0 + l/16][l%16];
// v_mfma_f64_16x16x4f64 leaves D[l/16 + 4r][l%16] in component r, the f32
// variant D[4(l/16) + r][l%16].

// Raw buffer resource over [base, base + bytes) (gfx9 descriptor word 3): a
// buffer load whose byte offset falls outside returns zero.
__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  const int n = (int)(bytes < 0x7fffffffLL ? bytes : 0x7fffffffLL);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, 0x00020000);
}

// The whole offset goes in the VGPR operand: the range check covers only the
// VGPR offset (plus the instruction offset), not the SGPR one.
template <typename T>
__device__ inline T load_elem(__amdgpu_buffer_rsrc_t r, unsigned voff);
template <>
__device__ inline double load_elem<double>(__amdgpu_buffer_rsrc_t r, unsigned voff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, 0, 0));
}
template <>
__device__ inline float load_elem<float>(__amdgpu_buffer_rsrc_t r, unsigned voff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, 0, 0));
}

// Byte offset of the source row feeding tile position p (a tile row or a panel
// column), elements of es bytes: the e-th set bit of mask receives source row
// base + e.  Positions receiving nothing get an offset past every buffer, so
// their loads read zero.
__device__ inline unsigned landing_off(uint64_t mask, int p, int base, unsigned es) {
  return ((mask >> p) & 1ull) ? (unsigned)(base + __popcll(mask & ((1ull << p) - 1ull))) * es
                              : 0x80000000u;
}

// acc += A B^T for one task, A = source rows landing on the tile's rows, B =
// source rows landing on the panel's columns, both placed at their landing
// positions, over this wave's share of the inner dimension: the 16-column
// chunks starting at 16 w + 64 g.  acc[bi][bj] is the 16x16 block (bi, bj) of
// the 64x64 tile in the f64 output layout.  A block is computed only if the
// task lands rows in block row bi and columns in block column bj (uniform over
// the wave) and, on the diagonal tile, bi >= bj (blocks above the diagonal are
// never stored).  Operands come through buffer loads over the chunk's columns,
// so rows that land nowhere (all rows of an inactive block) and columns past k
// read as zero without branches: a branch around a load would make the
// compiler wait for it at the join instead of overlapping all of them.
// T = float reads the FP32 copy of L and multiplies on v_mfma_f32_16x16x4f32,
// whose A rows are fed in the order pi(x) = x/4 + 4(x%4) so that its output
// (D[4(l/16) + r][l%16]) lands in the f64 layout; each 16-column chunk is
// accumulated in FP32 and then added to the FP64 accumulator.
template <typename T, int NBJ = 4, int KSTEP = 64>
__device__ inline void task_update(const T* __restrict__ src, int ld, int k, int ra, int ca,
                                   uint64_t rmask, uint64_t cmask, bool diag, int wave, int lane,
                                   d4 (&acc)[4][NBJ]) {
  constexpr bool kF32 = sizeof(T) == 4;
  const int lr = lane & 15, lk = lane >> 4;
  const int arow = kF32 ? (lr >> 2) + 4 * (lr & 3) : lr;
  const unsigned kstep = (unsigned)ld * sizeof(T);  // bytes between source columns
  unsigned ao[4], bo[NBJ];
  bool ab[4], bb[NBJ];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    ao[b] = landing_off(rmask, 16 * b + arow, ra, sizeof(T)) + lk * kstep;
    ab[b] = ((rmask >> (16 * b)) & 0xffffull) != 0;
  }
#pragma unroll
  for (int b = 0; b < NBJ; ++b) {
    bo[b] = landing_off(cmask, 16 * b + lr, ca, sizeof(T)) + lk * kstep;
    bb[b] = ((cmask >> (16 * b)) & 0xffffull) != 0;
  }
  for (int kb = 16 * wave; kb < k; kb += KSTEP) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc((const char*)src + (int64_t)kb * kstep,
                                                (int64_t)(k - kb) * kstep);
    T a[4][4], bv[NBJ][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int b = 0; b < 4; ++b) a[b][u] = load_elem<T>(rs, ao[b] + 4 * u * kstep);
#pragma unroll
      for (int b = 0; b < NBJ; ++b) bv[b][u] = load_elem<T>(rs, bo[b] + 4 * u * kstep);
    }
    if constexpr (!kF32) {
#pragma unroll
      for (int bi = 0; bi < 4; ++bi)
#pragma unroll
        for (int bj = 0; bj < NBJ; ++bj)
          if (ab[bi] && bb[bj] && !(diag && bi < bj)) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[bi][u], bv[bj][u], acc[bi][bj], 0, 0, 0);
          }
    } else {
#pragma unroll
      for (int bi = 0; bi < 4; ++bi) {
        if (!ab[bi]) continue;
        f4 c[NBJ];
#pragma unroll
        for (int bj = 0; bj < NBJ; ++bj) c[bj] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int bj = 0; bj < NBJ; ++bj)
          if (bb[bj] && !(diag && bi < bj)) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              c[bj] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[bi][u], bv[bj][u], c[bj], 0, 0, 0);
          }
#pragma unroll
        for (int bj = 0; bj < NBJ; ++bj)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[bi][bj][r] += (double)c[bj][r];
      }
    }
  }
}

// acc (f64 MFMA layout) -> a 64x64 LDS tile (column j at buf[j * kLdsLd])
__device__ inline void acc_store(const d4 (&acc)[4][4], double* buf, int lane) {
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int bj = 0; bj < 4; ++bj)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        buf[(16 * bj + (lane & 15)) * kLdsLd + 16 * bi + (lane >> 4) + 4 * r] = acc[bi][bj][r];
}

// the LDS tile += acc, element by element
__device__ inline void acc_add(const d4 (&acc)[4][4], double* buf, int lane) {
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int bj = 0; bj < 4; ++bj)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        buf[(16 * bj + (lane & 15)) * kLdsLd + 16 * bi + (lane >> 4) + 4 * r] += acc[bi][bj][r];
}

// Tile kernel: applies all source updates of one tile, in task order.  Every
// wave accumulates the products of a fixed share of each task's inner
// dimension over the whole 64x64 tile in MFMA registers; the four partial sums
// are combined in a fixed order, (w0 + w2) + (w1 + w3), through LDS and
// subtracted from the tile, so results do not depend on scheduling.  The
// factorization of panels completed by this level follows in the panel factor kernels.
// MODE 0: FP64 throughout; 1: descendant (kind 0) tiles on the FP32 copy,
// intra-supernode tiles in FP64 (a tile's tasks all have one kind); 2: FP32
// for every tile.
// The body of one tile (a workgroup of kThreads threads; red: 2 x PW x kLdsLd
// doubles of LDS), shared by k_tile_update and the dependency-driven kernel.
template <int MODE>
__device__ inline void tile_update_body(double* __restrict__ L, const Tile& tl,
                                        const Task* __restrict__ tasks,
                                        double* __restrict__ dscratch,
                                        const float* __restrict__ Lf, double* red_lds,
                                        int tid) {
  double(*red)[swc::PW * kLdsLd] = reinterpret_cast<double(*)[swc::PW * kLdsLd]>(red_lds);
  // the wave index is uniform over the wave: say so, so that the per-chunk
  // buffer resources stay in scalar registers
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nr = tl.nr, nc = tl.ncol, ld = tl.ld;
  const bool diag = tl.r0 == 0;
  double* gtile = L + tl.vbase + tl.r0;
  d4 acc[4][4];
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int bj = 0; bj < 4; ++bj) acc[bi][bj] = d4{0.0, 0.0, 0.0, 0.0};
  const bool f32 = MODE == 2 || (MODE == 1 && tl.task_end > tl.task_begin &&
                                   tasks[tl.task_begin].kind == 0);
  if (f32) {
    for (int t = tl.task_begin; t < tl.task_end; ++t) {
      const Task tk = tasks[t];
      task_update<float>(Lf + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask, tk.cmask, diag,
                         wave, lane, acc);
    }
  } else {
    for (int t = tl.task_begin; t < tl.task_end; ++t) {
      const Task tk = tasks[t];
      task_update<double>(L + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask, tk.cmask, diag,
                          wave, lane, acc);
    }
  }
  // the tile's current values, loaded before the reduction so that their
  // latency overlaps it: thread t owns elements t, t + 256, ... of the
  // column-major tile
  double cur[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int e = tid + q * kThreads, i = e & 63, j = e >> 6;
    cur[q] = (i < nr && j < nc) ? gtile[(int64_t)j * ld + i] : 0.0;
  }
  // partial sums (w0 + w2) and (w1 + w3) in LDS, added element-wise by all
  // threads below
  if (wave < 2) acc_store(acc, red[wave], lane);
  lds_barrier();
  if (wave >= 2) acc_add(acc, red[wave - 2], lane);
  lds_barrier();
  // write back tile - sum; rows 0..nc-1 of a tile at row offset 0 are the
  // panel's diagonal block, whose strict upper part stays untouched (zero).
  // When this level factors the panel, the diagonal block also goes to the
  // launch-invariant copy that every factor-kernel tile of the panel reads.
  const bool copy = tl.kind == 0 && tl.slot >= 0;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int e = tid + q * kThreads, i = e & 63, j = e >> 6;
    if (i < nr && j < nc) {
      if (!(diag && i < j)) {
        const double v = cur[q] - (red[0][j * kLdsLd + i] + red[1][j * kLdsLd + i]);
        gtile[(int64_t)j * ld + i] = v;
        if (copy && i < nc) dscratch[tl.slot + j * nc + i] = v;
      } else if (copy) {
        dscratch[tl.slot + j * nc + i] = 0.0;
      }
    }
  }
}

template <int MODE>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
k_tile_update(double* __restrict__ L, const Tile* __restrict__ tiles,
              const Task* __restrict__ tasks, int tile0, double* __restrict__ dscratch,
              const float* __restrict__ Lf) {
  __shared__ double red[2 * swc::PW * kLdsLd];
  const Tile tl = tiles[tile0 + blockIdx.x];
  tile_update_body<MODE>(L, tl, tasks, dscratch, Lf, red, threadIdx.x);
}

// Tiles of panels of at most 16 columns with a short total inner dimension: one
// wave per tile over the whole inner dimension, a 64x16 accumulator (four 16x16
// blocks), written back from the registers.  Same tasks, modes and write-back
// rules as k_tile_update.
template <int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
k_tile_narrow(double* __restrict__ L, const Tile* __restrict__ tiles,
              const Task* __restrict__ tasks, int tile0, double* __restrict__ dscratch,
              const float* __restrict__ Lf) {
  const Tile tl = tiles[tile0 + blockIdx.x];
  const int lane = threadIdx.x;
  const int nr = tl.nr, nc = tl.ncol, ld = tl.ld;
  const bool diag = tl.r0 == 0;
  double* gtile = L + tl.vbase + tl.r0;
  d4 acc[4][1];
#pragma unroll
  for (int bi = 0; bi < 4; ++bi) acc[bi][0] = d4{0.0, 0.0, 0.0, 0.0};
  const bool f32 = MODE == 2 || (MODE == 1 && tl.task_end > tl.task_begin &&
                                   tasks[tl.task_begin].kind == 0);
  if (f32) {
    for (int t = tl.task_begin; t < tl.task_end; ++t) {
      const Task tk = tasks[t];
      task_update<float, 1, 16>(Lf + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask, tk.cmask,
                                diag, 0, lane, acc);
    }
  } else {
    for (int t = tl.task_begin; t < tl.task_end; ++t) {
      const Task tk = tasks[t];
      task_update<double, 1, 16>(L + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask, tk.cmask,
                                 diag, 0, lane, acc);
    }
  }
  const bool copy = tl.kind == 0 && tl.slot >= 0;
  const int j = lane & 15;
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * bi + (lane >> 4) + 4 * r;
      if (i < nr && j < nc) {
        if (!(diag && i < j)) {
          const double v = gtile[(int64_t)j * ld + i] - acc[bi][0][r];
          gtile[(int64_t)j * ld + i] = v;
          if (copy && i < nc) dscratch[tl.slot + j * nc + i] = v;
        } else if (copy) {
          dscratch[tl.slot + j * nc + i] = 0.0;
        }
      }
    }
}

// Broadcast of lane src's value (src uniform over the wave).
__device__ inline double bcast(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
}

// Lane C of every 16 lanes' own group, in all of them (v_mov_b64_dpp, row_newbcast): half
// the instructions of bcast, and the value stays in vector registers.
extern "C" __device__ __attribute__((const)) double swc_update_dpp(double, double, int, int, int,
                                                                   bool) __asm("llvm.amdgcn.update.dpp.f64");
template <int C>
__device__ inline double group_bcast(double v) {
  return swc_update_dpp(0.0, v, 0x150 + C, 0xf, 0xf, true);
}

template <int N>
struct Index {
  static constexpr int value = N;
};
// f(Index<LO>) ... f(Index<HI - 1>): loops whose index is a template argument inside
template <int LO, int HI, class F>
__device__ inline void unrolled(F&& f) {
  if constexpr (LO < HI) {
    f(Index<LO>{});
    unrolled<LO + 1, HI>(f);
  }
}

// POTRF of a block of nc <= NC columns held by one wave, lane = row (y[c]: column c),
// and the same column operations on the rows of x (X): x <- x L11^{-T}.  Bound: the chain
// of nc pivots.  Pivot j + 1 is formed from column j's raw entries, read from their lanes
// while the reciprocal square root of pivot j runs, so the chain is reciprocal square
// root, product, fma; the same operations on the same values give the lanes' own copies,
// bitwise.  Reading it from the updated lane instead puts two lane reads and a select on
// the chain.  Columns past nc are checked four at a time: what their entries become is
// not used.  Returns 1 + the first column with a non-positive pivot, else 0; such a
// pivot continues as 1, so no NaNs spread.
template <int NC, bool X>
__device__ inline int factor_rows(double (&y)[NC], double (&x)[NC], int nc, int lane) {
  int badcol = 0;
  double d = bcast(y[0], 0);
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    if (j < nc) {
      const double b1 = j + 1 < NC ? bcast(y[j], j + 1) : 0.0;
      const double c1 = j + 1 < NC ? bcast(y[j + 1 < NC ? j + 1 : j], j + 1) : 0.0;
      // 1/sqrt(d) once, then a multiply per entry (dpotf2 scales the column by 1/ajj)
      double r = rsqrt(d);
      asm volatile("" : "+v"(r));  // computed whatever d is: a select, not a branch
      const bool ok = d > 0.0;
      badcol = ok || badcol != 0 ? badcol : j + 1;
      const double rs = ok ? r : 1.0;
      const double m1 = b1 * rs;  // entry (j+1, j)
      y[j] = ok ? y[j] * rs : (lane == j ? 1.0 : y[j]);
      if constexpr (X) x[j] *= rs;
      if (j + 1 < NC) {
        d = fma(-m1, m1, c1);
        y[j + 1] = fma(-y[j], m1, y[j + 1]);
        if constexpr (X) x[j + 1] = fma(-x[j], m1, x[j + 1]);
      }
#pragma unroll
      for (int g = (j + 2) & ~3; g < NC; g += 4) {
        if (g <= j + 2 || g < nc) {
#pragma unroll
          for (int c = g; c < g + 4; ++c) {
            if (c < j + 2) continue;
            const double m = bcast(y[j], c);
            y[c] = fma(-y[j], m, y[c]);
            if constexpr (X) x[c] = fma(-x[j], m, x[c]);
          }
        }
      }
    }
  }
  return badcol;
}

// Panel factorization for panels of at most 16 columns (NC), one wave per tile
// and registers only, for levels with many narrow panels (the leaves, batched
// instances), where how many workgroups fit on a CU matters more than one
// tile's latency: POTRF of the panel's nc x nc
// diagonal block (dpotrf 'L', sw_parallel_PB_Cholesky_05.c:430) in registers --
// lane i holds row i, the pivot and the multipliers of column j are read from
// their lanes -- then B <- B L11^{-T} for the tile's rows below the diagonal
// block (dtrsm 'R','L','T','N', .c:461-467), lane i substituting its own row.
// Both apply the updates of an entry in increasing column order, as the
// left-looking loops of the reference do.  Every tile of a panel computes the
// same L11 from the same launch-invariant copy (bitwise identical), so no tile
// waits for another; the diagonal tile stores it and reports info.  Entries
// above the diagonal of the register copy are never read by lanes on or below
// it, so they are left unmasked.
template <int NC, class TileT>
__device__ inline void panel_factor_regs_core(double* __restrict__ L, const TileT& tl,
                                              int* __restrict__ info_out, float* __restrict__ Lf,
                                              int lane, double (&y)[NC], double (&x)[NC]) {
  // y: row `lane` of the diagonal block, 0 past it; x: row `lane` of the tile
  const int nr = tl.nr, nc = tl.ncol;
  const int badcol = factor_rows<NC, true>(y, x, nc, lane);
  double* gtile = L + tl.vbase + tl.r0;
  float* ftile = Lf ? Lf + tl.vbase + tl.r0 : nullptr;
  if (tl.kind == 0) {
    if (badcol && lane == 0) atomicMin(info_out, tl.c0 + badcol);
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (lane < nc && c <= lane) {
        gtile[(int64_t)c * tl.ld + lane] = y[c];
        if (ftile) ftile[(int64_t)c * tl.ld + lane] = (float)y[c];
      }
  }
  // rows of this tile below the diagonal block: tile rows [first, nr)
  const int first = tl.kind == 0 ? nc : 0;
  const bool mine = lane >= first && lane < nr;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (mine && c < nc) {
      gtile[(int64_t)c * tl.ld + lane] = x[c];
      if (ftile) ftile[(int64_t)c * tl.ld + lane] = (float)x[c];
    }
}

template <int NC>
__device__ inline void panel_factor_regs_body(double* __restrict__ L, const Tile& tl,
                                              const double* __restrict__ dscratch,
                                              int* __restrict__ info_out, float* __restrict__ Lf,
                                              int lane) {
  const int nc = tl.ncol, first = tl.kind == 0 ? nc : 0;
  const double* gdiag = dscratch + tl.slot;  // updated diagonal block, ld nc
  const double* gtile = L + tl.vbase + tl.r0;
  const bool mine = lane >= first && lane < tl.nr;
  double y[NC], x[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    y[c] = (lane < nc && c < nc && c <= lane) ? gdiag[c * nc + lane] : 0.0;
    x[c] = (mine && c < nc) ? gtile[(int64_t)c * tl.ld + lane] : 0.0;
  }
  panel_factor_regs_core<NC>(L, tl, info_out, Lf, lane, y, x);
}

template <int NC>
__global__ void __launch_bounds__(64)
k_panel_factor_regs(double* __restrict__ L, const Tile* __restrict__ ftiles, int list0,
                    const double* __restrict__ dscratch, int* __restrict__ info_out,
                    float* __restrict__ Lf) {
  const Tile tl = ftiles[list0 + blockIdx.x];
  panel_factor_regs_body<NC>(L, tl, dscratch, info_out, Lf, threadIdx.x);
}


// Fused narrow panels of a level: one persistent launch whose waves take chunks
// of consecutive panels from a device worklist (a counter claimed with a vector
// atomic, the next claim issued while the current chunk is worked on) until the
// level's list is exhausted.  A panel (<= 16 columns, a single-panel supernode whose tiles all
// have short updates) is done by one wave from start to finish: every tile's
// updates as k_tile_narrow applies them, the updated tile handed from the MFMA
// layout to row-per-lane registers through the wave's own LDS buffer, the
// diagonal block factored and the rows solved as k_panel_factor_regs does it
// (the same operations in the same order, so the result does not depend on
// which wave takes which panel), no copy of the diagonal block through global
// memory and no second launch.  MODE as k_tile_update; Lf: the FP32 copy of L,
// read by FP32 updates and written with the factor when write_f32 is set.
template <int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
k_narrow_fused(double* __restrict__ L, const Tile* __restrict__ tiles,
               const Task* __restrict__ tasks, const swc::FusedPanel* __restrict__ items,
               int nitems, int chunk, int* __restrict__ counter, int* __restrict__ info_out,
               float* Lf, int write_f32) {
  constexpr int NC = 16;
  __shared__ double T[swc::TM * (NC + 1)];  // updated tile, row i at T[i * (NC + 1)]
  __shared__ double L11[NC * (NC + 1)];     // the panel's factored diagonal block, row-major
  const int lane = threadIdx.x;
  // the worklist hands out chunks of `chunk` consecutive panels
  int claim = 0;
  if (lane == 0) claim = atomicAdd(counter, 1);
  int item = __builtin_amdgcn_readfirstlane(claim) * chunk;
  int end = min(item + chunk, nitems);
  if (lane == 0) claim = atomicAdd(counter, 1);  // the next chunk, used after this one
  while (item < nitems) {
    if (item == end) {
      item = __builtin_amdgcn_readfirstlane(claim) * chunk;
      if (item >= nitems) break;
      end = min(item + chunk, nitems);
      if (lane == 0) claim = atomicAdd(counter, 1);
    }
    const swc::FusedPanel it = items[item];
    for (int t = 0; t < it.ntile; ++t) {
      const Tile tl = tiles[it.tile0 + t];
      const int nr = tl.nr, nc = tl.ncol, ld = tl.ld;
      const bool diag = tl.r0 == 0;
      double* gtile = L + tl.vbase + tl.r0;
      // (1) the tile's updates (k_tile_narrow)
      d4 acc[4][1];
#pragma unroll
      for (int bi = 0; bi < 4; ++bi) acc[bi][0] = d4{0.0, 0.0, 0.0, 0.0};
      const bool f32 = MODE == 2 || (MODE == 1 && tl.task_end > tl.task_begin &&
                                       tasks[tl.task_begin].kind == 0);
      if (f32) {
        for (int q = tl.task_begin; q < tl.task_end; ++q) {
          const Task tk = tasks[q];
          task_update<float, 1, 16>(Lf + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask,
                                    tk.cmask, diag, 0, lane, acc);
        }
      } else {
        for (int q = tl.task_begin; q < tl.task_end; ++q) {
          const Task tk = tasks[q];
          task_update<double, 1, 16>(L + tk.src_base, tk.ld, tk.k, tk.ra, tk.ca, tk.rmask,
                                     tk.cmask, diag, 0, lane, acc);
        }
      }
      {
        const int j = lane & 15;
#pragma unroll
        for (int bi = 0; bi < 4; ++bi)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * bi + (lane >> 4) + 4 * r;
            const bool in = i < nr && j < nc && !(diag && i < j);
            const double g = gtile[in ? (int64_t)j * ld + i : 0];
            T[i * (NC + 1) + j] = in ? g - acc[bi][0][r] : 0.0;
          }
      }
      float* ftile = write_f32 ? Lf + tl.vbase + tl.r0 : nullptr;
      if (t == 0) {
        // (2) POTRF of the diagonal block (k_panel_factor_regs), kept in LDS
        double y[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c)
          y[c] = (lane < nc && c < nc && c <= lane) ? T[lane * (NC + 1) + c] : 0.0;
        int badcol = 0;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          if (j < nc) {
            const double d = bcast(y[j], j);
            const bool ok = d > 0.0;
            if (!ok && badcol == 0) badcol = j + 1;
            double r = rsqrt(d);
            asm volatile("" : "+v"(r));  // a select, not a branch
            const double rs = ok ? r : 1.0;
            if (lane == j) y[j] = ok ? d * rs : 1.0;
            else if (lane > j) y[j] *= rs;
#pragma unroll
            for (int c = j + 1; c < NC; ++c)
              if (c < nc) y[c] -= y[j] * bcast(y[j], c);
          }
        }
        if (badcol && lane == 0) atomicMin(info_out, tl.c0 + badcol);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (lane < nc && c <= lane) {
            gtile[(int64_t)c * ld + lane] = y[c];
            if (ftile) ftile[(int64_t)c * ld + lane] = (float)y[c];
          }
          if (lane < NC) L11[lane * (NC + 1) + c] = y[c];
        }
      }
      // (3) the tile's rows below the diagonal block: x <- x L11^{-T}
      const int first = t == 0 ? nc : 0;
      const bool mine = lane >= first && lane < nr;
      double x[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c] = (mine && c < nc) ? T[lane * (NC + 1) + c] : 0.0;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        if (j < nc) {
          x[j] *= 1.0 / L11[j * (NC + 1) + j];
#pragma unroll
          for (int c = j + 1; c < NC; ++c)
            if (c < nc) x[c] -= x[j] * L11[c * (NC + 1) + j];
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (mine && c < nc) {
          gtile[(int64_t)c * ld + lane] = x[c];
          if (ftile) ftile[(int64_t)c * ld + lane] = (float)x[c];
        }
    }
    ++item;
  }
}

__global__ void k_fill_int(int* __restrict__ x, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

// Column stride (doubles) of the LDS working matrix of k_panel_factor_blk: rows
// 0..63 hold the panel's diagonal block, rows 64..127 the tile rows being solved.
// An odd stride spreads the 16 columns an MFMA output block touches over all
// LDS banks.
constexpr int kWld = 2 * swc::TM + 1;

// acc (16x16 block of the f64 MFMA output layout: lane l holds rows l/16 + 4r,
// column l%16) -= A B^T over 16 columns, A = W rows [16 ra, 16 ra + 16),
// B = W rows [16 rb, 16 rb + 16), both from columns [kb, kb + 16) of W.  The
// MFMA accumulates its products one after another, as a chain of FMAs would.
__device__ inline d4 lds_block_update(const double* __restrict__ W, d4 acc, int ra, int rb, int kb,
                                      int lane) {
  const int lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const double* col = W + (kb + lk + 4 * u) * kWld;
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-col[16 * ra + lr], col[16 * rb + lr], acc, 0, 0, 0);
  }
  return acc;
}

// One sweep over 16 columns: the 16x16 pivot block is factored, z holding its rows in
// every group of 16 lanes, and each lane's row x solved with it (x <- x L11^{-T}).  Every
// entry takes its updates in increasing column order.  A wave alone on its SIMD issues an
// instruction every 4 to 5 cycles, so the sweep costs its instructions, about 36 a
// column: a multiplier is one move within the lane group (group_bcast) for two fmas, the
// pivot of column j + 1 is formed from column j's raw entries beside the others' updates,
// and nothing is selected: a pivot that is not a positive finite number is noticed at the
// end and the sweep done again with a test in every column (SAFE).  Cycles a column, the
// kernel's own: multipliers through LDS and selects 328, by readlane 377, this 238.
// Returns 1 + the first column whose pivot is not positive, else 0; such a pivot
// continues as 1, so no NaNs spread.
template <bool SAFE>
__device__ inline int sweep_columns_as(double (&x)[16], double (&z)[16], int lane, int self, bool* redo) {
  double d = group_bcast<0>(z[0]);
  uint64_t ok = ~0ull;
  int bad = 0;
  unrolled<0, 16>([&](auto J) {
    constexpr int j = decltype(J)::value, jn = j < 15 ? j + 1 : 15;
    const double b1 = group_bcast<jn>(z[j]), c1 = group_bcast<jn>(z[jn]);  // (j+1, j), (j+1, j+1)
    double r;
    if constexpr (SAFE) {
      // 1/sqrt(d) once, then a multiply per entry (dpotf2 scales the column by 1/ajj)
      r = rsqrt(d);
      if (!(d > 0.0)) {
        r = 1.0;
        if (bad == 0) bad = j + 1;
        if (self == j) x[j] = 1.0;
        if ((lane & 15) == j) z[j] = 1.0;
      }
    } else {
      // 1/sqrt(d) = y / sqrt(1 - e), y within 2^-25 of it and e = 1 - d y^2, by the
      // first terms of the binomial series
      const double y = __builtin_amdgcn_rsq(d), e = fma(-d * y, y, 1.0);
      r = fma(y * e, fma(e, 0.375, 0.5), y);
      ok &= __ballot(__builtin_amdgcn_class(d, 0x180));  // positive, finite
    }
    const double m1 = b1 * r;
    d = fma(-m1, m1, c1);
    z[j] *= r;
    x[j] *= r;
    unrolled<j + 1, 16>([&](auto C) {
      constexpr int c = decltype(C)::value;
      const double m = group_bcast<c>(z[j]);
      z[c] = fma(-z[j], m, z[c]);
      x[c] = fma(-x[j], m, x[c]);
    });
    __builtin_amdgcn_sched_barrier(0);  // the columns' moves hoisted together spill
  });
  *redo = ok != ~0ull;
  return bad;
}
// self: the pivot row that this lane's x is, if any
__device__ inline int sweep_columns(double (&x)[16], double (&z)[16], int lane, int self) {
  double x0[16], z0[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    x0[c] = x[c];
    z0[c] = z[c];
  }
  bool redo;
  sweep_columns_as<false>(x, z, lane, self, &redo);
  // used here: not to be computed behind the branch, with every multiplier kept for it
#pragma unroll
  for (int c = 0; c < 16; ++c) asm volatile("" : "+v"(x[c]));
  if (!redo) return 0;
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    x[c] = x0[c];
    z[c] = z0[c];
    // opaque: the first pass's values are not kept for this one
    asm volatile("" : "+v"(x[c]), "+v"(z[c]));
  }
  return sweep_columns_as<true>(x, z, lane, self, &redo);
}

// Panel factorization of the panels completed at this level for panels of
// 17..64 columns, one workgroup of four waves per tile: POTRF of the panel's
// nc x nc diagonal block (dpotrf 'L', sw_parallel_PB_Cholesky_05.c:430) and
// B <- B L11^{-T} for the tile's rows below it (dtrsm 'R','L','T','N',
// .c:461-467), blocked in 16 columns and right-looking, as the reference's
// dpotrf_cluster_master blocks its POTRF (BLAS-sw/dpotrf_cluster_master.c:11-63).
// The diagonal block (from the launch-invariant copy, identity past nc) and the
// tile rows sit in LDS (W) from the first load to the final store.  Per block
// column J:
//  (1) one sweep over the 16 columns (sweep_columns) factors the 16x16 diagonal block
//      and solves every row below it at once, lane = row: wave 0 takes the diagonal
//      block's rows, wave 1 the tile rows, each with its own copy of the pivot rows
//      (the same operations on the same values, so both have the same pivots bitwise);
//  (2) block column J+1 of the diagonal block (blocks on or below its diagonal) and of
//      the tile rows takes the rank-16 update on FP64 MFMA, the 16x16 output blocks
//      spread over the four waves;
//  (3) while waves 0 and 1 sweep block column J, waves 2 and 3 give block column J+1
//      the updates of the block columns before J, and wave 3 stores block column J-1,
//      which is final, to L, so that only the last block column is stored after the loop.
// Bound: latency, of the four sweeps above all (15,200 of a tile's 28,200 cycles at 64
// columns, loads 4,400; 20,800 of 34,500 with the multipliers through LDS and every
// block's update between two sweeps).
// Both apply each entry's updates in increasing column order, so the result is
// bitwise the one of a column-by-column right-looking factorization.  Every
// tile of a panel computes the same L11, so no tile waits for another; the
// diagonal tile stores it and reports info.
// LDS of k_panel_factor_blk: W
constexpr int kBlkLds = swc::PW * kWld;

struct FrontIn;
__device__ inline void front_assemble_blk(const double* L, const swc::FactorTile& tl,
                                          const FrontIn& in, double* W, int first, int nx, int nb,
                                          int wave, int lane);

// In: nothing for the left-looking tiles (Tile), what a first panel is assembled from
// for the multifrontal ones (FactorTile).
template <class TileT, class... In>
__device__ inline void panel_factor_blk_body(double* __restrict__ L, const TileT& tl,
                                             const double* __restrict__ dscratch,
                                             int* __restrict__ info_out, float* __restrict__ Lf,
                                             double* lds, int tid, const In&... in) {
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nc = tl.ncol;
  const int nb = (nc + 15) >> 4;              // 16-column blocks (2..4)
  double* W = lds;                            // 16 nb columns
  const int first = tl.kind == 0 ? nc : 0;    // tile rows [first, nr) are solved ...
  const int nx = tl.nr > first ? tl.nr - first : 0;  // ... into W rows 64 .. 64 + nx
  const int nxb = (nx + 15) >> 4;
  const double* gdiag = dscratch + tl.slot;  // updated diagonal block, ld nc
  double* gtile = L + tl.vbase + tl.r0;
  float* ftile = Lf ? Lf + tl.vbase + tl.r0 : nullptr;
  bool load = true;
  if constexpr (sizeof...(In) > 0) {
    if (tl.first) {
      front_assemble_blk(L, tl, in..., W, first, nx, nb, wave, lane);
      load = false;
    }
  }
  if (load) {
    // wave w moves columns 16w..16w+15 of diagonal-block row `lane` and of tile
    // row `lane`; every lane loads from an address inside both buffers and then
    // selects, so all its loads are in flight together
    const int c0 = 16 * wave;
    double y[16], x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const int col = c0 + c;
      const bool iny = lane < nc && col < nc && col <= lane, inx = lane < nx && col < nc;
      const double vy = gdiag[iny ? col * nc + lane : 0];
      const double vx = gtile[inx ? (int64_t)col * tl.ld + first + lane : 0];
      y[c] = iny ? vy : ((lane >= nc || col >= nc) && col == lane ? 1.0 : 0.0);
      x[c] = inx ? vx : 0.0;
    }
    if (c0 < 16 * nb) {
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        W[(c0 + c) * kWld + lane] = y[c];
        W[(c0 + c) * kWld + 64 + lane] = x[c];
      }
    }
  }
  // Final columns c0 + cstep c, c < ncols (<= 16), of W to L and to the FP32
  // copy: the diagonal tile's rows of L11 and the solved tile rows.  All LDS
  // reads are issued before the first store.
  auto write_back = [&](int c0, int cstep, int ncols) {
    double vd[16], vt[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      if (c < ncols) {
        const int col = c0 + cstep * c;  // < 64
        vd[c] = W[col * kWld + lane];
        vt[c] = W[col * kWld + 64 + lane];
      }
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const int col = c0 + cstep * c;
      if (c < ncols && col < nc) {
        if (tl.kind == 0 && lane < nc && col <= lane) {
          gtile[(int64_t)col * tl.ld + lane] = vd[c];
          if (ftile) ftile[(int64_t)col * tl.ld + lane] = (float)vd[c];
        }
        if (lane < nx) {
          gtile[(int64_t)col * tl.ld + first + lane] = vt[c];
          if (ftile) ftile[(int64_t)col * tl.ld + first + lane] = (float)vt[c];
        }
      }
    }
  };
  lds_barrier();
  int badcol = 0;
  // Every wave has read its rows before any is written back (wave 1 reads the pivot rows
  // that wave 0 rewrites): a barrier follows every read.
  double x[16], z[16];
  auto read_row = [&](int jb) {
    if (wave >= 2) return;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      z[c] = W[(jb + c) * kWld + jb + (lane & 15)];
      x[c] = W[(jb + c) * kWld + 64 * wave + lane];
    }
  };
  read_row(0);
  lds_barrier();
  for (int J = 0; J < nb; ++J) {
    const int jb = 16 * J;
    if (wave < 2) {
      const bool store = wave == 0 ? (lane >= jb && lane < 16 * nb) : lane < nx;
      const int bad = sweep_columns(x, z, lane, wave == 0 ? lane - jb : -1);
      badcol = badcol != 0 || bad == 0 ? badcol : jb + bad;
      if (store) {
#pragma unroll
        for (int c = 0; c < 16; ++c) W[(jb + c) * kWld + 64 * wave + lane] = x[c];
      }
    } else if (J > 0) {
      // beside the sweep, waves 2 and 3: the updates of block column J + 1 from the
      // block columns before J; then wave 3 writes block column J - 1, which is final,
      // to L
      if (J + 1 < nb) {
        const int C = J + 1, nrb = (nb - C) + nxb;
        for (int q = wave - 2; q < nrb; q += 2) {
          const int R = q < nb - C ? C + q : 4 + (q - (nb - C));
          double* out = W + (16 * C + (lane & 15)) * kWld + 16 * R + (lane >> 4);
          d4 acc = d4{out[0], out[4], out[8], out[12]};
          for (int kb = 0; kb < jb; kb += 16) acc = lds_block_update(W, acc, R, C, kb, lane);
          out[0] = acc[0];
          out[4] = acc[1];
          out[8] = acc[2];
          out[12] = acc[3];
        }
      }
      if (wave == 3) write_back(jb - 16, 1, 16);
    }
    lds_barrier();
    if (J + 1 < nb) {
      // (2) block column C = J + 1: rows of the diagonal block from C on, then the
      // tile rows (W row blocks 4 .. 4 + nxb)
      const int C = J + 1, nrb = (nb - C) + nxb;
      for (int q = wave; q < nrb; q += 4) {
        const int R = q < nb - C ? C + q : 4 + (q - (nb - C));
        double* out = W + (16 * C + (lane & 15)) * kWld + 16 * R + (lane >> 4);
        d4 acc = d4{out[0], out[4], out[8], out[12]};
        acc = lds_block_update(W, acc, R, C, jb, lane);
        out[0] = acc[0];
        out[4] = acc[1];
        out[8] = acc[2];
        out[12] = acc[3];
      }
      lds_barrier();
      read_row(jb + 16);
      lds_barrier();
    }
  }
  if (tl.kind == 0 && badcol && badcol <= nc && tid == 0) atomicMin(info_out, tl.c0 + badcol);
  // the last block column, four columns per wave
  write_back(16 * (nb - 1) + wave, 4, 4);
}

// The tiles of a level's panels of at most 16 columns, four to a workgroup (one
// wave each, as k_panel_factor_regs<16>), in a launch of 256-thread workgroups
// whose first ceil(nregs / 4) workgroups take them: the level's panels of both
// width classes are then factored in one launch.  Returns false for the
// workgroups after those.
__device__ inline bool regs_tiles_in_block(double* __restrict__ L,
                                           const Tile* __restrict__ ftiles, int rlist0,
                                           int nregs, const double* __restrict__ dscratch,
                                           int* __restrict__ info_out, float* __restrict__ Lf) {
  if ((int)blockIdx.x >= (nregs + 3) >> 2) return false;
  const int t = 4 * (int)blockIdx.x + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (t < nregs) {
    const Tile tl = ftiles[rlist0 + t];
    panel_factor_regs_body<16>(L, tl, dscratch, info_out, Lf, threadIdx.x & 63);
  }
  return true;
}

// Workgroups [0, ceil(nregs / 4)): the level's panels of at most 16 columns
// (ftiles[rlist0 ..]); the others: one tile of a 17..64-column panel each
// (ftiles[list0 ..]).
__global__ void __launch_bounds__(256)
k_panel_factor_blk(double* __restrict__ L, const Tile* __restrict__ ftiles, int list0,
                   const double* __restrict__ dscratch, int* __restrict__ info_out,
                   float* __restrict__ Lf, int rlist0, int nregs) {
  __shared__ double lds[kBlkLds];
  if (regs_tiles_in_block(L, ftiles, rlist0, nregs, dscratch, info_out, Lf)) return;
  const Tile tl = ftiles[list0 + blockIdx.x - ((nregs + 3) >> 2)];
  panel_factor_blk_body(L, tl, dscratch, info_out, Lf, lds, threadIdx.x);
}

// ---- dependency-driven factorization ----------------------------------------
// One persistent launch for the plan's levels from dag_level0 on (swc::DagItem):
// as many workgroups as the device holds at once claim work items from a ticket
// counter, in the plan's item order.  An item applies one level's updates to one
// tile with tile_update_body and, when that level completes the tile's panel,
// factors the tile's rows with the panel factor bodies; the arithmetic is that of
// the per-level launches, so the factor is bitwise the same.  Before it starts, an
// item waits for the tile's previous writer and for every panel its updates read
// to be factored (all of the panel's tiles); a factoring tile below the diagonal
// also waits for its panel's diagonal tile to be updated (the copy of the
// diagonal block it factors from).  Item order is a topological order of these
// waits, so an item only waits for items claimed earlier by running workgroups
// that wait for nothing later: the launch cannot deadlock.  Every wait is also
// bounded (kDagWaitTicks of the constant 100 MHz clock); a wait that runs out
// sets the abort flag, every workgroup then stops, and the host reports the
// failure.  Publication: every wave waits for its stores to complete, a barrier,
// then one thread's agent-scope release store of the flag (which writes the
// XCD's cache back first: the device's L2 caches are per XCD); the waiting side
// polls with relaxed agent-scope loads, then the polling wave takes an
// agent-scope acquire fence (invalidating the CU's and the XCD's caches) before
// the barrier after which the workgroup loads.
// sync: [0] ticket counter, [1] abort flag, [2, 2 + nitems) item states (1: the
// tile's updates are written), then per panel the count of its factored tiles.
constexpr int kDagLds = kBlkLds > 2 * swc::PW * kLdsLd ? kBlkLds : 2 * swc::PW * kLdsLd;
constexpr uint64_t kDagWaitTicks = 500000000ull;  // 5 s

__device__ inline int ld_agent(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wave polls until the tile's previous writer (prev >= 0) has written it
// and the panels deps[dep0, dep1) are factored; false when the launch aborts.
__device__ bool dag_poll(const int* __restrict__ state, const int* __restrict__ pdone,
                         const swc::DagDep* __restrict__ deps, int prev, int dep0, int dep1,
                         int* __restrict__ abort_flag, int lane) {
  const uint64_t t0 = wall_clock64();
  for (;;) {
    bool ok = !(lane == 0 && prev >= 0) || ld_agent(state + prev) >= 1;
    for (int e = dep0 + lane; e < dep1; e += 64) {
      const swc::DagDep dp = deps[e];
      ok = ok && ld_agent(pdone + dp.panel) >= dp.count;
    }
    if (__builtin_amdgcn_ballot_w64(!ok) == 0) return true;
    if (ld_agent(abort_flag) != 0) return false;
    if (wall_clock64() - t0 > kDagWaitTicks) {
      if (lane == 0) __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

template <int MODE>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
k_dag_factor(double* __restrict__ L, const Tile* __restrict__ tiles,
             const Task* __restrict__ tasks, const swc::DagItem* __restrict__ items, int nitems,
             const swc::DagDep* __restrict__ deps, int* __restrict__ sync,
             double* __restrict__ dscratch, int* __restrict__ info_out, float* Lf, int write_f32) {
  __shared__ double lds[kDagLds];
  __shared__ int s_claim, s_ok;
  int* const ticket = sync;
  int* const abort_flag = sync + 1;
  int* const state = sync + 2;
  int* const pdone = sync + 2 + nitems;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const lf = write_f32 ? Lf : nullptr;
  for (;;) {
    if (tid == 0) {
      const int c = atomicAdd(ticket, 1);
      s_claim = ld_agent(abort_flag) != 0 ? nitems : c;
    }
    __syncthreads();
    const int k = s_claim;
    if (k >= nitems) break;
    {
      const swc::DagItem d = items[k];
      if (wave == 0) {
        const bool ok = dag_poll(state, pdone, deps, d.prev, d.dep0, d.dep1, abort_flag, lane);
        // one acquire for the workgroup: it invalidates the CU's and the XCD's
        // caches, and the other waves load only after the barrier below
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (lane == 0) s_ok = ok;
      }
      __syncthreads();
      if (!s_ok) break;
      // the thread index is made opaque per item, so that the compiler does not
      // hoist the bodies' per-lane address arithmetic out of the loop and keep it
      // in registers across items
      int t1 = tid;
      asm volatile("" : "+v"(t1));
      tile_update_body<MODE>(L, tiles[d.tile], tasks, dscratch, Lf, lds, t1);
    }
    // every wave's stores complete before the barrier; the one release below then
    // writes them back from the XCD's cache before the flag is set
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // the item and its tile are read again rather than kept in registers over the
    // updates (an index the compiler cannot see through)
    int k2 = k;
    asm volatile("" : "+s"(k2));
    const swc::DagItem d = items[k2];
    const Tile tl = tiles[d.tile];
    if (d.fclass < 0 || tl.kind == 0) {  // someone waits for these updates
      if (tid == 0) __hip_atomic_store(state + k2, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (d.fclass >= 0) {
      if (wave == 0) {
        const bool ok = d.diag < 0 || dag_poll(state, pdone, deps, d.diag, 0, 0, abort_flag, lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (lane == 0) s_ok = ok;
      }
      __syncthreads();
      if (!s_ok) break;
      int t2 = tid;
      asm volatile("" : "+v"(t2));
      if (d.fclass == 0) {
        if (wave == 0) panel_factor_regs_body<16>(L, tl, dscratch, info_out, lf, t2 & 63);
      } else {
        panel_factor_blk_body(L, tl, dscratch, info_out, lf, lds, t2);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (tid == 0)
        __hip_atomic_fetch_add(pdone + tl.panel, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
  }
}

// A level's panel factorization (panels of at most 16 columns in the first
// ceil(nregs / 4) workgroups, four tiles each; then panels of 17..64 columns,
// nfac workgroups: k_panel_factor_blk) in the same launch as the level's updates
// of tiles whose panels it does not factor (the remaining workgroups:
// k_tile_update), so that those updates, which nothing of this level waits for,
// overlap the factorization instead of delaying it.  Same bodies, same results.
template <int MODE>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
k_factor_and_update(double* __restrict__ L, const Tile* __restrict__ ftiles, int list0, int nfac,
                    const Tile* __restrict__ tiles, const Task* __restrict__ tasks, int tile0,
                    double* __restrict__ dscratch, int* __restrict__ info_out, float* Lf_factor,
                    const float* __restrict__ Lf_update, int rlist0, int nregs) {
  __shared__ double lds[kDagLds];
  if (regs_tiles_in_block(L, ftiles, rlist0, nregs, dscratch, info_out, Lf_factor)) return;
  const int b = (int)blockIdx.x - ((nregs + 3) >> 2);
  if (b < nfac) {
    const Tile tl = ftiles[list0 + b];
    panel_factor_blk_body(L, tl, dscratch, info_out, Lf_factor, lds, threadIdx.x);
  } else {
    const Tile tl = tiles[tile0 + (b - nfac)];
    tile_update_body<MODE>(L, tl, tasks, dscratch, Lf_update, lds, threadIdx.x);
  }
}

#include "front_kernels.h"

// CSC export of the factor (the layout of the reference's bcsc2csc,
// common/Util.h:311-338): column j's entries are its supernode's rows from its
// own diagonal down.  col[j] = {value offset of L(j, j), offset in Ls of row j,
// entry count, offset in the output}; one wave per column.
struct CscColumn {
  int64_t v0, r0, len, c0;
};

__global__ void k_factor_csc(const double* __restrict__ L, const int* __restrict__ Ls,
                             const CscColumn* __restrict__ col, int n, int64_t* __restrict__ Cp,
                             int* __restrict__ Ci, double* __restrict__ Cx) {
  const int j = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (j >= n) return;
  const CscColumn c = col[j];
  for (int64_t e = lane; e < c.len; e += 64) {
    Cx[c.c0 + e] = L[c.v0 + e];
    Ci[c.c0 + e] = Ls[c.r0 + e];
  }
  if (lane == 0) {
    Cp[j + 1] = c.c0 + c.len;
    if (j == 0) Cp[0] = 0;
  }
}

#include "sweep_kernels.h"

// y[k] = b[perm[k]] (to the factor's ordering) or x[perm[k]] = y[k] (back).
__global__ void k_permute(const double* __restrict__ in, double* __restrict__ out,
                          const int* __restrict__ perm, int n, int nrhs, int64_t ldin,
                          int64_t ldout, int inverse) {
  const int64_t total = (int64_t)n * nrhs;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int k = (int)(e % n);
    const int r = (int)(e / n);
    if (!inverse) out[r * ldout + k] = in[r * ldin + perm[k]];
    else out[r * ldout + perm[k]] = in[r * ldin + k];
  }
}

}  // namespace

// ---- residual, norms and vector updates (FP64) ---------------------------

constexpr int kRedBlocks = 512;
constexpr int kSetupBlocks = 2048;
// Elements behind L and its FP32 copy: an update tile's staged loads read up to three rows
// past its last.
constexpr int kLoadPad = 16;

// Workspace of swc_solve_noalloc, the entry point that allocates nothing: one
// copy of this array per GPU, held from the library's load until the process
// ends.  Host code never uses its name as an address: swc_create looks up each
// device's copy once (scratch_ptr) and everything else uses that pointer.
constexpr int64_t kScratchDoubles = (int64_t)16 << 20;  // 128 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];

// What kernels report to the host, in pinned memory (a kernel's store is on the host when
// the stream is, without a copy command and its gap, 14 to 45 us each): one per handle,
// taken in swc_create and given back in swc_destroy, in blocks that are kept for later
// handles.
struct HostRecord {
  int abort;      // set when one of a sweep's waits ran out
  int info;       // of the factor
  double norm;    // ||A||_inf
  double logdet;  // sum of log L_jj
  HostRecord* next;  // of the free ones
};
std::mutex g_record_mu;
HostRecord* g_record_free = nullptr;

// Free records are linked through themselves: handles come and go without an allocation
// that could fail.
HostRecord* take_record() {
  std::lock_guard<std::mutex> lock(g_record_mu);
  if (!g_record_free) {
    constexpr int kRecords = 256;
    HostRecord* block = nullptr;
    if (hipHostMalloc((void**)&block, kRecords * sizeof(HostRecord), hipHostMallocPortable) != hipSuccess)
      return nullptr;
    for (int i = 0; i < kRecords; ++i) {
      block[i].next = g_record_free;
      g_record_free = block + i;
    }
  }
  HostRecord* r = g_record_free;
  g_record_free = r->next;
  *r = HostRecord{};
  return r;
}

void give_record(HostRecord* r) {
  if (!r) return;
  std::lock_guard<std::mutex> lock(g_record_mu);
  r->next = g_record_free;
  g_record_free = r;
}

// Per-device address of `scratch`, looked up once per device with that device
// current (hipGetSymbolAddress); null until then.
std::mutex g_scratch_mu;
std::vector<double*> g_scratch_ptr;

int bind_scratch(int device) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize(device + 1, nullptr);
  if (g_scratch_ptr[device]) return SWC_OK;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return swc_set_error(SWC_EDEVICE, std::string("no-alloc workspace: hipGetSymbolAddress: ") +
                                          hipGetErrorString(e));
  g_scratch_ptr[device] = (double*)ptr;
  return SWC_OK;
}

double* scratch_ptr(int device) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return device < (int)g_scratch_ptr.size() ? g_scratch_ptr[device] : nullptr;
}

// Y = A X, or R = B - A X when B is given, for all nrhs columns (CSR): a group
// of 8 lanes per row, lane k taking the row's entries k, k+8, ... (consecutive
// lanes read consecutive entries), right-hand sides 4 at a time against the
// same entries, each sum completed by a fixed butterfly over the group.  Whole
// waves step through the rows together (the butterfly needs every lane).
constexpr int kMvGroup = 8;
__global__ void __launch_bounds__(kThreads)
k_csr_mv(const int* __restrict__ rp, const int* __restrict__ ci, const double* __restrict__ av,
         const double* __restrict__ X, const double* __restrict__ B, double* __restrict__ Y, int n,
         int64_t ld, int nrhs) {
  constexpr int G = kMvGroup, RPW = 64 / G;  // rows per wave
  const int lane = threadIdx.x & 63, k = lane % G;
  const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
  const int64_t nw = (int64_t)gridDim.x * blockDim.x / 64;
  for (int64_t base = wid * RPW; base < n; base += nw * RPW) {
    const int64_t i = base + lane / G;
    const bool valid = i < n;
    const int e0 = valid ? rp[i] : 0, e1 = valid ? rp[i + 1] : 0;
    for (int c0 = 0; c0 < nrhs; c0 += 4) {
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
      for (int e = e0 + k; e < e1; e += G) {
        const double a = av[e];
        const int64_t col = ci[e];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c0 + q < nrhs) acc[q] = fma(a, X[(int64_t)(c0 + q) * ld + col], acc[q]);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int off = G / 2; off >= 1; off /= 2) acc[q] += __shfl_xor(acc[q], off, G);
      if (valid && k < 4 && c0 + k < nrhs) {
        // lane k of the group writes right-hand side c0 + k
        const double t = k == 0 ? acc[0] : k == 1 ? acc[1] : k == 2 ? acc[2] : acc[3];
        const int64_t o = (int64_t)(c0 + k) * ld + i;
        Y[o] = B ? B[o] - t : t;
      }
    }
  }
}

// First launch of a factorization: the values into the handle's copy (keep, unless they
// are there already), the full symmetric matrix in CSR for the residuals (both triangles,
// entry e from value vmap[e]) and its row sums' maxima, part[block] (||A||_inf), and a
// clean info word.  G lanes a row, as its length asks (setup_group).  Bound: HBM and the
// latency of vmap -> value.  A 1100-row dense matrix took 222 us for the norm alone with a
// thread per row; the whole launch is 15 us.
template <int G>
__global__ void __launch_bounds__(kThreads)
k_factor_setup(const double* __restrict__ vals, double* __restrict__ keep, int64_t nvals,
               const int* __restrict__ rp, const int64_t* __restrict__ vmap, int n,
               double* __restrict__ af, double* __restrict__ part, int* __restrict__ info) {
  __shared__ double red[kThreads / 64];
  const int64_t t0 = (int64_t)blockIdx.x * kThreads + threadIdx.x, nt = (int64_t)gridDim.x * kThreads;
  if (t0 == 0) *info = 0x7fffffff;
  if (keep)
    for (int64_t q = t0; q < nvals; q += nt) keep[q] = vals[q];
  const int k = (int)(t0 % G);
  double m = 0.0;
  for (int64_t i0 = t0 / G; i0 < n; i0 += nt / G) {
    const int e1 = rp[i0 + 1];
    double t = 0.0;
#pragma unroll 4
    for (int e = rp[i0] + k; e < e1; e += G) {
      const double v = vals[vmap[e]];
      af[e] = v;
      t += fabs(v);
    }
#pragma unroll
    for (int w = G / 2; w > 0; w >>= 1) t += __shfl_xor(t, w, G);
    m = fmax(m, t);
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) m = fmax(m, __shfl_xor(m, w, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// Last launch of a factorization: its info and ||A||_inf to the host's record.
__global__ void __launch_bounds__(kThreads)
k_factor_report(const double* __restrict__ part, int npart, const int* __restrict__ info,
                HostRecord* __restrict__ rec) {
  __shared__ double red[kThreads / 64];
  double m = 0.0;
  for (int i = threadIdx.x; i < npart; i += kThreads) m = fmax(m, part[i]);
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) m = fmax(m, __shfl_xor(m, w, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    rec->norm = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    rec->info = *info;
  }
}

// Per-column partial reductions over a fixed grid (deterministic): op 0 max|x|,
// op 1 dot(x, y).  part[c * kRedBlocks + block].
__global__ void k_reduce_partial(const double* __restrict__ X, const double* __restrict__ Y,
                                 int n, int64_t ld, int op, double* __restrict__ part) {
  __shared__ double red[kThreads];
  const int64_t c = blockIdx.y;
  const double* x = X + c * ld;
  const double* y = Y ? Y + c * ld : nullptr;
  double acc = 0.0;
  for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += kRedBlocks * kThreads)
    acc = op == 0 ? fmax(acc, fabs(x[i])) : fma(x[i], y[i], acc);
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      red[threadIdx.x] = op == 0 ? fmax(red[threadIdx.x], red[threadIdx.x + w])
                                 : red[threadIdx.x] + red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[c * kRedBlocks + blockIdx.x] = red[0];
}

__global__ void k_reduce_final(const double* __restrict__ part, int op, double* __restrict__ out) {
  __shared__ double red[kThreads];
  const int c = blockIdx.x;
  double acc = 0.0;
  for (int i = threadIdx.x; i < kRedBlocks; i += kThreads) {
    const double v = part[(int64_t)c * kRedBlocks + i];
    acc = op == 0 ? fmax(acc, v) : acc + v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      red[threadIdx.x] = op == 0 ? fmax(red[threadIdx.x], red[threadIdx.x + w])
                                 : red[threadIdx.x] + red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = red[0];
}

// Y[:, c] += alpha[c] * X[:, c]   (sign folded into alpha by the caller)
__global__ void k_axpy_cols(double* __restrict__ Y, const double* __restrict__ X,
                            const double* __restrict__ alpha, int n, int64_t ld) {
  const int64_t c = blockIdx.y;
  const double a = alpha[c];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    Y[c * ld + i] = fma(a, X[c * ld + i], Y[c * ld + i]);
}

// P[:, c] = Z[:, c] + beta[c] * P[:, c]
__global__ void k_xpby_cols(double* __restrict__ P, const double* __restrict__ Z,
                            const double* __restrict__ beta, int n, int64_t ld) {
  const int64_t c = blockIdx.y;
  const double b = beta[c];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    P[c * ld + i] = fma(b, P[c * ld + i], Z[c * ld + i]);
}

// ---- adjoint: selected inverse on the pattern of L ------------------------
// Z = A^{-1} restricted to the pattern of L (in L's BCSC layout): the reverse sweep of
// the blocked Cholesky adjoint for d logdet(A) / dA = A^{-1} (no reference counterpart).
#include "selinv_kernels.h"
constexpr int kSelLists = 8;

// logdet partials: sum of log L_jj over the diagonal entries (fixed grid).
__global__ void k_logdet_partial(const double* __restrict__ L, const int64_t* __restrict__ diag,
                                 int n, double* __restrict__ part) {
  __shared__ double red[kThreads];
  double acc = 0.0;
  for (int j = blockIdx.x * kThreads + threadIdx.x; j < n; j += kRedBlocks * kThreads)
    acc += log(L[diag[j]]);
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Gradient w.r.t. the input values of A (each stored lower entry a_q stands for
// a_ij and a_ji):  g_q = w_q (alpha Z_ij - beta x_i x_j),  w_q = 1 on the
// diagonal, 2 off it; Z at zpos[q] (offset in L's layout), x in factor order.
__global__ void k_grad_values(const double* __restrict__ Zv, const int64_t* __restrict__ zpos,
                              const int* __restrict__ qi, const int* __restrict__ qj,
                              const double* __restrict__ x, double alpha, double beta,
                              int64_t nvals, double* __restrict__ g) {
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nvals;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int i = qi[q], j = qj[q];
    const double w = i == j ? 1.0 : 2.0;
    double v = 0.0;
    if (alpha != 0.0) v += alpha * Zv[zpos[q]];
    if (beta != 0.0) v -= beta * x[i] * x[j];
    g[q] = w * v;
  }
}

// ---------------------------------------------------------------------------
// handle
// ---------------------------------------------------------------------------

struct swc_handle {
  int device = 0;
  hipStream_t stream = nullptr;
  Plan plan;
  swc::PlanParams params;  // shape parameters of the next structure upload
  swc::HLevelSchedule hlevel;  // non-empty: factor levels follow this schedule
  bool multifrontal = false;   // the factor runs the front plan, else the left-looking one
  swc::FrontPlan fronts;
  swc::PlanParams up_params;   // the parameters of the uploaded structure's plan
  bool uploading = false;      // an upload is under way: it sees to a refused allocation itself
  bool no_room = false;        // one was refused in it
  int n = 0, nsuper = 0;
  int64_t nvals = 0;  // number of values swc_factor expects
  std::vector<int> super, Ls;
  std::vector<int64_t> pi, px;
  std::vector<int> perm;  // perm[new] = old, empty if not set
  std::vector<int> pruneptr, pruneset;
  // device buffers
  double* dL = nullptr;
  double* dU = nullptr;  // the front plan's arena
  float* dLf = nullptr;  // FP32 shadow of L, written with it when FP32 updates are on
  int64_t lf_cap = 0;    // elements allocated at dLf
  int* dLs = nullptr;
  Tile* dTiles = nullptr;
  Task* dTasks = nullptr;
  int64_t* dGptr = nullptr;  // forward gathers: per column, offsets into dGidx
  int64_t* dGidx = nullptr;
  swc::SweepSmall* dSweepSmall = nullptr;  // the solves' work lists (sweeps.h)
  swc::SweepItem* dSweepFwd = nullptr;
  swc::SweepItem* dSweepBwd = nullptr;
  int* dSweepSync = nullptr;  // tickets of the two sweeps, abort flag
  HostRecord* rec = nullptr;  // pinned
  double* dV = nullptr;   // contribution vectors, vsize * work_cols
  double* dPb = nullptr;  // backward partial sums, max_lvl_fblk * SPW * work_cols
  double* dY = nullptr;   // forward solutions, n * work_cols
  Tile* dFtiles = nullptr;  // factor-kernel tiles (copies), by level and width class
  swc::FusedPanel* dFused = nullptr;  // fused narrow panels, by level
  swc::Gather* dGathers = nullptr;    // the front plan's lists (fronts.h)
  swc::AEntry* dAents = nullptr;
  swc::FactorTile* dFactorTiles = nullptr;
  swc::SmallFront* dSmall = nullptr;
  swc::FrontTile* dFrontTiles = nullptr;
  int* dCounters = nullptr;  // per level: the fused kernel's worklist counter
  int fused_cap[3] = {0, 0, 0};  // per precision mode: fused-kernel workgroups resident at once
  swc::DagItem* dDagItems = nullptr;  // dependency-driven launch: work items, dependencies,
  swc::DagDep* dDagDeps = nullptr;    // and its ticket / abort / per-item / per-panel flags
  int* dDagSync = nullptr;
  int dag_cap[3] = {0, 0, 0};  // per precision mode: its workgroups resident at once
  double* dDiag = nullptr;  // per-level copies of the diagonal blocks being factored
  int64_t* dAmap = nullptr;
  int* dPerm = nullptr;
  double* dVals = nullptr;  // staging for host values
  double* dWork = nullptr;  // solve workspace, n * work_cols doubles
  int work_cols = 0;
  int* dInfo = nullptr;
  // full P A P^T (factor ordering) for residuals: CSR pattern, value map, values
  int* dRp = nullptr;
  int* dCi = nullptr;
  int64_t* dVmap = nullptr;
  double* dAf = nullptr;
  int64_t nnz_full = 0;
  double* dScal = nullptr;   // reductions and coefficients of the refinement, 4 * work_cols
                             // (eager launches only)
  double* dNormPart = nullptr;  // kSetupBlocks partial maxima of ||A||_inf, kRedBlocks partial
                                // sums of the log determinant
  double* dPart = nullptr;   // reduction partials, kRedBlocks * work_cols
  double* dRef = nullptr;    // refinement vectors, 5 * n * work_cols
  double normA = 0;
  // adjoint (selected inverse) state, built on first use
  double* dZ = nullptr;          // selected inverse, xsize
  double* dArena = nullptr;      // Z(R,R) of a level's supernodes
  double* dSelM = nullptr;       // [T; U] of a chunk of levels
  swc::SelNode* dNodes = nullptr;
  swc::SelRun* dSelRuns = nullptr;
  int* dSelJrun = nullptr;
  int* dSelRel = nullptr;
  swc::SelItem* dSelItems = nullptr;  // the plan's item lists
  size_t sel_items[kSelLists] = {};   // and where each begins
  swc::SelPlan sel;                   // offsets per chunk and level
  int64_t* dDiagPos = nullptr;   // offset of L(j,j), j in factor order
  int* dQi = nullptr;            // factor-order row / column of every input value
  int* dQj = nullptr;
  bool zvalid = false;
  int precision = 0;  // 0 FP64; 1 FP32 descendant updates; 2 FP32 for every update
  int fp32_mask = 0;  // bit k: tasks of kind k use FP32 MFMA
  int factored_precision = 0;
  bool factored = false;
  bool has_values = false;  // the A2 pattern (value map, residual CSR) is uploaded
  int last_info = 0;
  // captured launch sequences (hipGraph): factor per precision mode, solves per
  // (buffer, nrhs, ld); rebuilt when the structure changes
  bool use_graphs = true;
  hipGraphExec_t fgraph[3] = {nullptr, nullptr, nullptr};
  bool factor_seen[3] = {};  // a factorization of this structure in that mode has run
  struct SolveGraph {
    const double* x;
    int nrhs;
    int64_t ld;
    bool marked;
    hipGraphExec_t exec;
  };
  std::vector<SolveGraph> sgraphs;
  // timing (device events on `stream`)
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  bool profile = false;
  std::vector<hipEvent_t> pev;  // per-launch pairs when profiling
  double t_factor_ms = 0, t_solve_ms = 0, t_tile_ms = 0, t_trsm_ms = 0;
  std::vector<double> lvl_tile_ms;  // per level, when profiling
  int n_tile = 0, n_trsm = 0;

  int sweep_cap = 0;  // workgroups of a sweep's persistent launch

  ~swc_handle() {
    release();
    give_record(rec);
  }
  void drop_graphs() {
    for (auto& g : fgraph)
      if (g) (void)hipGraphExecDestroy(g);
    for (auto& g : fgraph) g = nullptr;
    for (auto& s : factor_seen) s = false;
    for (auto& g : sgraphs) (void)hipGraphExecDestroy(g.exec);
    sgraphs.clear();
  }
  void release() {
    drop_graphs();
    (void)hipFree(dL); (void)hipFree(dU); (void)hipFree(dLf); (void)hipFree(dLs); (void)hipFree(dTiles); (void)hipFree(dTasks);
    (void)hipFree(dGptr); (void)hipFree(dGidx); (void)hipFree(dSweepSmall); (void)hipFree(dSweepFwd); (void)hipFree(dSweepBwd); (void)hipFree(dSweepSync); (void)hipFree(dV); (void)hipFree(dPb); (void)hipFree(dY); (void)hipFree(dFtiles); (void)hipFree(dFused);
    (void)hipFree(dGathers); (void)hipFree(dAents); (void)hipFree(dFactorTiles); (void)hipFree(dSmall); (void)hipFree(dFrontTiles);
    (void)hipFree(dCounters); (void)hipFree(dDagItems); (void)hipFree(dDagDeps); (void)hipFree(dDagSync); (void)hipFree(dDiag); (void)hipFree(dAmap); (void)hipFree(dPerm);
    (void)hipFree(dVals); (void)hipFree(dWork); (void)hipFree(dInfo);
    (void)hipFree(dRp); (void)hipFree(dCi); (void)hipFree(dVmap); (void)hipFree(dAf); (void)hipFree(dScal); (void)hipFree(dPart); (void)hipFree(dNormPart);
    (void)hipFree(dRef);
    (void)hipFree(dZ); (void)hipFree(dArena); (void)hipFree(dNodes); (void)hipFree(dSelM); (void)hipFree(dSelRuns);
    (void)hipFree(dSelJrun); (void)hipFree(dSelRel); (void)hipFree(dSelItems); (void)hipFree(dDiagPos); (void)hipFree(dQi); (void)hipFree(dQj);
    dL = nullptr; dU = nullptr; dLf = nullptr; dLs = nullptr; dTiles = nullptr; dTasks = nullptr;
    dGptr = nullptr; dGidx = nullptr; dSweepSmall = nullptr; dSweepFwd = nullptr; dSweepBwd = nullptr; dSweepSync = nullptr; dV = nullptr; dPb = nullptr; dY = nullptr; dFtiles = nullptr; dFused = nullptr; dGathers = nullptr; dAents = nullptr; dFactorTiles = nullptr; dSmall = nullptr; dFrontTiles = nullptr; dCounters = nullptr; dDagItems = nullptr; dDagDeps = nullptr; dDagSync = nullptr; dDiag = nullptr; dAmap = nullptr; dPerm = nullptr;
    dVals = nullptr; dWork = nullptr; dInfo = nullptr;
    dRp = nullptr; dCi = nullptr; dVmap = nullptr; dAf = nullptr; dScal = nullptr; dPart = nullptr; dNormPart = nullptr;
    lf_cap = 0;
    dRef = nullptr;
    dZ = nullptr; dArena = nullptr; dNodes = nullptr; dSelM = nullptr; dSelRuns = nullptr;
    dSelJrun = nullptr; dSelRel = nullptr; dSelItems = nullptr; dDiagPos = nullptr; dQi = nullptr; dQj = nullptr;
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : pev) (void)hipEventDestroy(e);
    pev.clear();
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
  }
};

namespace {

// Device allocations of the calling thread until one is refused (0: none is); for tests.
thread_local int refuse_allocation = 0;

bool give_up_arena(swc_handle* h);

// Device memory for a handle.  The front plan's arena is as large as L, and only
// factorizations use it: where there is no room beside it, it is given back, and the
// handle's later factorizations run left-looking.
template <class Alloc>
hipError_t with_room(swc_handle* h, Alloc&& alloc) {
  auto attempt = [&] {
    if (refuse_allocation > 0 && --refuse_allocation == 0) return hipErrorOutOfMemory;
    return alloc();
  };
  hipError_t e = attempt();
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  if (h->uploading) h->no_room = true;
  else if (give_up_arena(h)) e = attempt();
  return e;
}
hipError_t device_malloc(swc_handle* h, void** p, size_t bytes) {
  return with_room(h, [&] { return hipMalloc(p, bytes); });
}

template <class T>
int upload(T** dst, const T* src, size_t count, swc_handle* h) {
  (void)hipFree(*dst);
  *dst = nullptr;
  const size_t alloc = count == 0 ? 1 : count;
  SWC_HIP(device_malloc(h, (void**)dst, alloc * sizeof(T)));
  if (src && count)
    SWC_HIP(hipMemcpyAsync(*dst, src, count * sizeof(T), hipMemcpyHostToDevice, h->stream));
  return SWC_OK;
}

int grid_for(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + kThreads - 1) / kThreads, 65536)); }

// Position of every entry of tril(P A P^T), given as CSC (a2p, a2i), in the row list of
// its column's supernode; false for bad pointers or an entry outside the structure.
bool a2_positions(const swc_handle* h, const int* a2p, const int* a2i, std::vector<int>& pos) {
  if (!a2p || !a2i || a2p[0] != 0) return false;
  for (int j = 0; j < h->n; ++j)
    if (a2p[j + 1] < a2p[j]) return false;
  pos.resize((size_t)a2p[h->n]);
  for (int s = 0; s < h->nsuper; ++s) {
    const int* rows = h->Ls.data() + h->pi[s];
    const int len = (int)(h->pi[s + 1] - h->pi[s]);
    for (int j = h->super[s]; j < h->super[s + 1]; ++j) {
      int k = j - h->super[s];  // row j
      for (int64_t q = a2p[j]; q < a2p[j + 1]; ++q) {
        const int v = a2i[q];
        if (v < j) return false;
        // the row after the last entry's, for most of a dense column, else a search
        if (rows[k] != v && !(k + 1 < len && rows[++k] == v)) {
          k = int(std::lower_bound(rows, rows + len, v) - rows);
          if (k >= len || rows[k] != v) return false;
        }
        pos[q] = k;
      }
    }
  }
  return true;
}

// Value offset inside L of every entry of A2 (at row positions pos).  With src != null,
// entry e of A2 came from input entry src[e] and the map is indexed by input entries (so
// swc_factor takes values in the caller's order).
int build_amap(const swc_handle* h, const int* a2p, const std::vector<int>& pos,
               const int64_t* src, int64_t nvals, std::vector<int64_t>& amap) {
  const int n = h->n;
  const int64_t nnz = a2p[n];
  amap.assign(src ? nvals : nnz, -1);
  for (int s = 0; s < h->nsuper; ++s) {
    const int64_t len = h->pi[s + 1] - h->pi[s];
    for (int j = h->super[s]; j < h->super[s + 1]; ++j)
      for (int64_t q = a2p[j]; q < a2p[j + 1]; ++q) {
        const int64_t dst = src ? src[q] : q;
        if (dst < 0 || dst >= (int64_t)amap.size())
          return swc_set_error(SWC_EINVAL, "value map index out of range");
        amap[dst] = h->px[s] + (j - h->super[s]) * len + pos[q];
      }
  }
  for (int64_t v : amap)
    if (v < 0) return swc_set_error(SWC_EINVAL, "value map does not cover every value");
  return SWC_OK;
}

int ensure_work(swc_handle* h, int cols) {
  if (h->work_cols >= cols) return SWC_OK;
  for (auto& g : h->sgraphs) (void)hipGraphExecDestroy(g.exec);  // they captured the old buffers
  h->sgraphs.clear();
  (void)hipFree(h->dWork);
  (void)hipFree(h->dV);
  (void)hipFree(h->dY);
  (void)hipFree(h->dPb);
  (void)hipFree(h->dPart);
  (void)hipFree(h->dRef);
  h->dWork = h->dV = h->dY = h->dPb = h->dPart = h->dRef = nullptr;
  h->work_cols = 0;
  const Plan& P = h->plan;
  SWC_HIP(device_malloc(h, (void**)&h->dPart, sizeof(double) * (size_t)kRedBlocks * cols));
  (void)hipFree(h->dScal);
  h->dScal = nullptr;
  SWC_HIP(device_malloc(h, (void**)&h->dScal, sizeof(double) * (size_t)(4 * cols)));
  SWC_HIP(device_malloc(h, (void**)&h->dRef, sizeof(double) * (size_t)5 * h->n * cols));
  SWC_HIP(device_malloc(h, (void**)&h->dWork, sizeof(double) * (size_t)h->n * cols));
  SWC_HIP(device_malloc(h, (void**)&h->dV, sizeof(double) * (size_t)std::max<int64_t>(P.vsize, 1) * cols));
  SWC_HIP(device_malloc(h, (void**)&h->dY, sizeof(double) * (size_t)h->n * cols));
  SWC_HIP(device_malloc(h, (void**)&h->dPb, sizeof(double) * (size_t)std::max(P.max_lvl_fblk, 1) * swc::SPW * cols));
  h->work_cols = cols;
  return SWC_OK;
}

// The multifrontal factorization's levels (fronts.h): F_l, then U_l.
template <int MODE>
void enqueue_fronts(swc_handle* h, bool profile) {
  hipStream_t st = h->stream;
  const swc::FrontPlan& F = h->fronts;
  const FrontIn in{h->dGathers, h->dAents, h->dVals};
  float* lf = MODE ? h->dLf : nullptr;
  const swc::SmallFront* sm = h->dSmall;
  const swc::FactorTile* ft = h->dFactorTiles;
  const swc::FrontTile* ut = h->dFrontTiles;
  for (int l = 0; l < F.nlevel; ++l) {
    hipEvent_t* pe = profile ? &h->pev[(size_t)4 * l] : nullptr;
    const int s0 = F.lvl_small[l], ns = F.lvl_small[l + 1] - s0;
    const int f0 = F.lvl_f[l], nf = F.lvl_f[l + 1] - f0, nn = F.lvl_fn[l], nw = nf - nn;
    const int nd = l > 0 && !profile ? F.lvl_ud[l - 1] : 0;
    if (pe) (void)hipEventRecord(pe[1], st);
    // many one-wave items keep their own launch, where more of them fit on a CU.  From 512 /
    // 2048 / 8192 items on (ms): 500^2 GMRF 0.996 / 0.970 / 0.968, 600 2D instances 0.775 / 0.755 /
    // 0.746, larger grids the same; in between, so that LDS does not bound larger levels
    const bool lean = nw + nd == 0 || ns + nn > 2048;
    if (lean && ns + nn > 0)
      hipLaunchKernelGGL(k_front_narrow<MODE>, dim3(ns + nn), dim3(64), 0, st, h->dL, sm, s0, ns,
                         ft, f0, in, (const double*)h->dDiag, h->dInfo, lf);
    if (nw + nd > 0) {
      const int s1 = lean ? 0 : ns, n1 = lean ? 0 : nn;
      hipLaunchKernelGGL(k_front_factor<MODE>, dim3((s1 + 3) / 4 + (n1 + 3) / 4 + nw + nd),
                         dim3(kThreads), front_factor_lds(s1 + n1, F.lvl_widest[l], nd), st, h->dL,
                         sm, s0, s1, ft, f0 + nn - n1, n1, nw, ut,
                         F.lvl_u[l] - nd, in, (const double*)h->dDiag, h->dDiag,
                         h->dInfo, lf, (const float*)h->dLf);
    }
    if (pe) (void)hipEventRecord(pe[2], st);
    const int u0 = F.lvl_u[l], nu = F.lvl_u[l + 1] - u0 - (profile ? 0 : F.lvl_ud[l]);
    if (nu > 0)
      hipLaunchKernelGGL((F.lvl_kmax[l] >= kStageMin ? k_front_update<MODE, true> : k_front_update<MODE, false>),
                         dim3(nu), dim3(kThreads), 0, st, h->dL, ut, u0, in, h->dDiag,
                         (const float*)h->dLf);
    if (pe) (void)hipEventRecord(pe[3], st);
  }
}

// Lanes per row of k_factor_setup, and its workgroups.  8 lanes take rows of a grid or a
// mesh (5 to 30 entries, vector operators up to 81) in a few steps; a row of more than 64
// on average gets a wave.  8 against 64 lanes: 100^2 grid 3.2 us against 5.4, 32^3 4.4
// against 10.5, vector 20^3 6.4 against 9.3, a 1100-row dense matrix 46 against 15.
int setup_group(const swc_handle* h) { return h->nnz_full > (int64_t)64 * h->n ? 64 : 8; }
int setup_blocks(const swc_handle* h) {
  return (int)std::min<int64_t>(((int64_t)h->n * setup_group(h) + kThreads - 1) / kThreads, kSetupBlocks);
}

// The launch before the factor's graph: it reads the caller's values, whose address the
// graph does not know.
void launch_setup(swc_handle* h, const double* dvals) {
  auto kern = setup_group(h) == 64 ? k_factor_setup<64> : k_factor_setup<8>;
  hipLaunchKernelGGL(kern, dim3(setup_blocks(h)), dim3(kThreads), 0, h->stream, dvals,
                     dvals != h->dVals ? h->dVals : nullptr, h->nvals, (const int*)h->dRp,
                     (const int64_t*)h->dVmap, h->n, h->dAf, h->dNormPart, h->dInfo);
}
void launch_report(swc_handle* h) {
  hipLaunchKernelGGL(k_factor_report, dim3(1), dim3(kThreads), 0, h->stream, (const double*)h->dNormPart,
                     setup_blocks(h), (const int*)h->dInfo, h->rec);
}

// Enqueues the whole numeric factorization of the staged values h->dVals.
void enqueue_factor(swc_handle* h, bool profile) {
  hipStream_t st = h->stream;
  const Plan& P = h->plan;
  const double* dvals = h->dVals;
  if (h->multifrontal) {
    // L needs no clearing: every entry on and below a diagonal block's diagonal is
    // written by a factor launch, and what lies above is cleared at upload
    if (h->precision == 0) enqueue_fronts<0>(h, profile);
    else if (h->precision == 1) enqueue_fronts<1>(h, profile);
    else enqueue_fronts<2>(h, profile);
    launch_report(h);
    return;
  }
  hipLaunchKernelGGL(k_fill, dim3(grid_for(P.xsize)), dim3(kThreads), 0, st, h->dL, P.xsize, 0.0);
  hipLaunchKernelGGL(k_assemble, dim3(grid_for(h->nvals)), dim3(kThreads), 0, st, h->dL,
                     (const int64_t*)h->dAmap, dvals, h->nvals);
  hipLaunchKernelGGL(k_fill_int, dim3((std::max(P.nlevel, 1) + kThreads - 1) / kThreads),
                     dim3(kThreads), 0, st, h->dCounters, std::max(P.nlevel, 1), 0);
  // the levels from dag_level0 on run as one dependency-driven launch (per-level
  // launches when profiling, so that each level can be timed)
  const bool dag = !profile && !P.dag_items.empty();
  const int nsync = 2 + (int)P.dag_items.size() + P.npanel;
  if (dag)
    hipLaunchKernelGGL(k_fill_int, dim3((nsync + kThreads - 1) / kThreads), dim3(kThreads), 0, st,
                       h->dDagSync, nsync, 0);
  for (int l = 0; l < (dag ? P.dag_level0 : P.nlevel); ++l) {
    const int t0 = P.lvl_tiles[l], nt = P.lvl_tiles[l + 1] - t0;
    const int s0 = P.lvl_trsm[l], ns = P.lvl_trsm[l + 1] - s0;
    hipEvent_t* pe = profile ? &h->pev[(size_t)4 * l] : nullptr;
    if (pe) (void)hipEventRecord(pe[0], st);
    // the level's tiles: fused narrow panels first, then one-wave tiles, then the rest
    const int ntf = P.lvl_tiles_fused[l], ntn = P.lvl_tiles_narrow[l];
    const int f0 = P.lvl_fused[l], nf = P.lvl_fused[l + 1] - f0;
    if (nf > 0) {
      auto kern = h->precision == 0 ? k_narrow_fused<0> : (h->precision == 1 ? k_narrow_fused<1>
                                                                              : k_narrow_fused<2>);
      // about four chunks per workgroup: few claims on the one counter, and the
      // last chunks still balance the waves' loads
      const int grid = std::min(nf, h->fused_cap[h->precision]);
      const int chunk = std::max(1, (nf + 4 * grid - 1) / (4 * grid));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(64), 0, st, h->dL, (const Tile*)h->dTiles,
                         (const Task*)h->dTasks, (const swc::FusedPanel*)h->dFused + f0, nf, chunk,
                         h->dCounters + l, h->dInfo, h->dLf, h->fp32_mask ? 1 : 0);
    }
    if (ntn > 0) {
      auto kern = h->precision == 0 ? k_tile_narrow<0> : (h->precision == 1 ? k_tile_narrow<1>
                                                                             : k_tile_narrow<2>);
      hipLaunchKernelGGL(kern, dim3(ntn), dim3(64), 0, st, h->dL, (const Tile*)h->dTiles,
                         (const Task*)h->dTasks, t0 + ntf, h->dDiag, (const float*)h->dLf);
    }
    // tiles of the panels this level factors, then (last in the level's list) the
    // others, which run beside the panel factorization unless profiling times the
    // update launches on their own
    const int ntd = profile ? 0 : P.lvl_tiles_deferred[l];
    const int tc0 = t0 + ntf + ntn, ntc = nt - ntf - ntn - ntd;
    if (ntc > 0) {
      auto kern = h->precision == 0 ? k_tile_update<0> : (h->precision == 1 ? k_tile_update<1>
                                                                             : k_tile_update<2>);
      hipLaunchKernelGGL(kern, dim3(ntc), dim3(kThreads), 0, st, h->dL, (const Tile*)h->dTiles,
                         (const Task*)h->dTasks, tc0, h->dDiag, (const float*)h->dLf);
    }
    if (pe) (void)hipEventRecord(pe[1], st);
    {
      // the level's panels by width class: <= 16, <= 32, <= 64 columns
      const int* cls = &P.lvl_trsm_cls[(size_t)4 * l];
      float* lf = h->fp32_mask ? h->dLf : nullptr;
      const Tile* ft = (const Tile*)h->dFtiles;
      const int nblk = ns > 0 ? cls[3] - cls[1] : 0, nreg = ns > 0 ? cls[1] - cls[0] : 0;
      // the narrow panels go into the launch of the wider ones when there is one
      // (four tiles to a workgroup), else into their own launch
      const int nrw = (nreg + 3) / 4;
      if (ntd > 0) {
        auto kern = h->precision == 0
                        ? k_factor_and_update<0>
                        : (h->precision == 1 ? k_factor_and_update<1> : k_factor_and_update<2>);
        hipLaunchKernelGGL(kern, dim3(nrw + nblk + ntd), dim3(kThreads), 0, st, h->dL, ft,
                           ns > 0 ? cls[1] : 0, nblk, (const Tile*)h->dTiles,
                           (const Task*)h->dTasks, tc0 + ntc, h->dDiag, h->dInfo, lf,
                           (const float*)h->dLf, ns > 0 ? cls[0] : 0, nreg);
      } else if (nblk > 0) {
        hipLaunchKernelGGL(k_panel_factor_blk, dim3(nrw + nblk), dim3(256), 0, st, h->dL, ft,
                           cls[1], (const double*)h->dDiag, h->dInfo, lf, cls[0], nreg);
      } else if (nreg > 0) {
        hipLaunchKernelGGL(k_panel_factor_regs<16>, dim3(nreg), dim3(64), 0, st, h->dL, ft,
                           cls[0], (const double*)h->dDiag, h->dInfo, lf);
      }
    }
    if (pe) (void)hipEventRecord(pe[2], st);
  }
  if (dag) {
    auto kern = h->precision == 0 ? k_dag_factor<0> : (h->precision == 1 ? k_dag_factor<1>
                                                                          : k_dag_factor<2>);
    const int nitems = (int)P.dag_items.size();
    const int grid = std::min(nitems, h->dag_cap[h->precision]);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), 0, st, h->dL, (const Tile*)h->dTiles,
                       (const Task*)h->dTasks, (const swc::DagItem*)h->dDagItems, nitems,
                       (const swc::DagDep*)h->dDagDeps, h->dDagSync, h->dDiag, h->dInfo, h->dLf,
                       h->fp32_mask ? 1 : 0);
  }
  launch_report(h);
}

// Numeric factorization from values on the device (in upload order).
int factor_device(swc_handle* h, const double* dvals) {
  hipStream_t st = h->stream;
  const Plan& P = h->plan;
  const int nlevel = h->multifrontal ? h->fronts.nlevel : P.nlevel;
  if (h->profile && h->pev.size() < (size_t)4 * nlevel) {
    for (auto& e : h->pev) (void)hipEventDestroy(e);
    h->pev.assign((size_t)4 * nlevel, nullptr);
    for (auto& e : h->pev) SWC_HIP(hipEventCreate(&e));
  }
  // the first factorization is launched kernel by kernel: capturing and instantiating
  // its graph costs a call that is not repeated more than the graph saves it
  bool& again = h->factor_seen[h->precision];
  const bool graph = h->use_graphs && !h->profile && again;
  again = true;
  hipGraphExec_t& gx = h->fgraph[h->precision];
  if (graph && !gx) {
    hipGraph_t g = nullptr;
    SWC_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    enqueue_factor(h, false);
    SWC_HIP(hipStreamEndCapture(st, &g));
    hipError_t e = hipGraphInstantiate(&gx, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) {
      gx = nullptr;
      return swc_set_error(SWC_EDEVICE, std::string("factor graph: ") + hipGetErrorString(e));
    }
  }
  SWC_HIP(hipEventRecord(h->ev[0], st));
  launch_setup(h, dvals);
  if (graph) SWC_HIP(hipGraphLaunch(gx, st));
  else enqueue_factor(h, h->profile);
  SWC_HIP(hipEventRecord(h->ev[1], st));
  SWC_HIP(hipGetLastError());
  const int big = 0x7fffffff;
  hipError_t ce = hipSuccess;
  int dag_abort = 0;
  const bool dag = !h->profile && !P.dag_items.empty();
  if (ce == hipSuccess && dag)
    ce = hipMemcpyAsync(&dag_abort, h->dDagSync + 1, sizeof(int), hipMemcpyDeviceToHost, st);
  SWC_HIP(hipStreamSynchronize(st));
  SWC_HIP(ce);
  const int info = h->rec->info;
  h->normA = h->rec->norm;
  if (dag_abort) {
    h->factored = false;
    return swc_set_error(SWC_EDEVICE, "factor: a dependency wait of the factor launch timed out");
  }
  float ms = 0;
  SWC_HIP(hipEventElapsedTime(&ms, h->ev[0], h->ev[1]));
  h->t_factor_ms = ms;
  if (h->profile) {
    h->t_tile_ms = h->t_trsm_ms = 0;
    h->n_tile = h->n_trsm = 0;
    h->lvl_tile_ms.assign(nlevel, 0.0);
    for (int l = 0; l < nlevel; ++l) {
      // the events around the level's update launch and around its factor launches
      const swc::FrontPlan& F = h->fronts;
      const bool mf = h->multifrontal;
      const int nt = mf ? F.lvl_u[l + 1] - F.lvl_u[l] : P.lvl_tiles[l + 1] - P.lvl_tiles[l];
      const int ns = mf ? 1 : P.lvl_trsm[l + 1] - P.lvl_trsm[l];
      hipEvent_t* pe = &h->pev[(size_t)4 * l];
      if (nt > 0) {
        SWC_HIP(hipEventElapsedTime(&ms, mf ? pe[2] : pe[0], mf ? pe[3] : pe[1]));
        h->t_tile_ms += ms;
        h->lvl_tile_ms[l] = ms;
        h->n_tile++;
      }
      if (ns > 0) {
        SWC_HIP(hipEventElapsedTime(&ms, pe[1], pe[2]));
        h->t_trsm_ms += ms;
        h->n_trsm++;
      }
    }
  }
  h->last_info = info == big ? 0 : info;
  h->factored = true;
  h->factored_precision = h->precision;
  h->zvalid = false;
  return SWC_OK;
}

// One persistent launch of a sweep; the ticket was cleared before.
template <bool FORWARD, int GROUP>
void launch_sweep(swc_handle* h, const SweepRun& a) {
  if (a.nitems == 0) return;
  const int ngroups = (a.nrhs + GROUP - 1) / GROUP;
  // tickets are ints: very many right-hand sides go in several launches
  const int step = (int)std::max<int64_t>(1, std::min<int64_t>(ngroups, (1 << 30) / a.nitems));
  for (int g0 = 0; g0 < ngroups; g0 += step) {
    const int ng = std::min(step, ngroups - g0);
    if (g0 > 0)
      hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, h->stream, a.ticket, 0);
    const int64_t total = (int64_t)a.nitems * ng;
    hipLaunchKernelGGL((k_sweep<FORWARD, GROUP>), dim3((unsigned)std::min<int64_t>(total, h->sweep_cap)),
                       dim3(kThreads), 0, h->stream, a, g0, ng);
  }
}

template <bool FORWARD>
void launch_small(swc_handle* h, const SweepRun& a, int level) {
  const std::vector<int>& ls = h->plan.sweeps.lvl_small;
  const int s0 = ls[level], ns = ls[level + 1] - s0;
  // the packed ones and the others wait for nothing of the level: any order
  const int n16 = h->plan.sweeps.lvl_small16[level], nw = ns - n16;
  if (n16 > 0)
    hipLaunchKernelGGL((k_sweep_small16<FORWARD>), dim3((n16 + 15) / 16, a.nrhs), dim3(kThreads), 0,
                       h->stream, a, s0, n16);
  if (nw > 0 && a.nrhs == 1)
    hipLaunchKernelGGL((k_sweep_small<FORWARD, 1>), dim3((nw + 3) / 4, 1), dim3(kThreads), 0,
                       h->stream, a, s0 + n16, nw);
  else if (nw > 0)
    hipLaunchKernelGGL((k_sweep_small<FORWARD, 4>), dim3((nw + 3) / 4, (a.nrhs + 3) / 4),
                       dim3(kThreads), 0, h->stream, a, s0 + n16, nw);
}

SweepRun sweep_run(swc_handle* h, double* dX, int nrhs, int64_t ldx, double* dY, double* dV,
                   double* dPb) {
  const Plan& P = h->plan;
  SweepRun a{};
  a.L = h->dL;
  a.Ls = h->dLs;
  a.gptr = h->dGptr;
  a.gidx = h->dGidx;
  a.small = h->dSweepSmall;
  a.abort_flag = h->dSweepSync + 2;
  a.abort_host = &h->rec->abort;
  a.X = dX;
  a.Y = dY;
  a.V = dV;
  a.P = dPb;
  a.ldx = ldx;
  a.ldy = h->n;
  a.ldv = std::max<int64_t>(P.vsize, 1);
  a.ldp = std::max<int64_t>(P.sweeps.psize, 1);
  a.nrhs = nrhs;
  return a;
}

// The marks that the sweeps of `a` start from; X = P in on the way when `in` is given.
void enqueue_marks(swc_handle* h, const SweepRun& a, const double* in, int64_t ldin) {
  const int64_t ny = a.ldy * a.nrhs, nv = a.ldv * a.nrhs, np = a.ldp * a.nrhs;
  hipLaunchKernelGGL(k_sweep_init, dim3(std::min(grid_for(std::max(ny, nv)), 4096)), dim3(kThreads),
                     0, h->stream, a.Y, ny, a.V, nv, a.P, np, h->dSweepSync, in, ldin, a.X, a.ldx,
                     (const int*)h->dPerm, h->n, a.nrhs);
}

// Forward sweep L Y = X (X is left marked for the backward sweep); marked: its
// enqueue_marks has been launched.
void enqueue_forward(swc_handle* h, SweepRun a, bool marked = false) {
  const swc::SweepPlan& W = h->plan.sweeps;
  if (!marked) enqueue_marks(h, a, nullptr, 0);
  for (int l = 0; l + 1 < (int)W.lvl_small.size(); ++l) launch_small<true>(h, a, l);
  a.items = h->dSweepFwd;
  a.nitems = (int)W.fwd.size();
  a.ticket = h->dSweepSync;
  if (!swc::sweep_by_16(W, a.nrhs)) launch_sweep<true, 1>(h, a);
  else launch_sweep<true, 16>(h, a);
}

// Backward sweep L^T X = Y.
void enqueue_backward(swc_handle* h, SweepRun a) {
  const swc::SweepPlan& W = h->plan.sweeps;
  a.items = h->dSweepBwd;
  a.nitems = (int)W.bwd.size();
  a.ticket = h->dSweepSync + 1;
  if (!swc::sweep_by_16(W, a.nrhs)) launch_sweep<false, 1>(h, a);
  else launch_sweep<false, 16>(h, a);
  for (int l = (int)W.lvl_small.size() - 2; l >= 0; --l) launch_small<false>(h, a, l);
}

// dY (n x nrhs), dV (max(vsize, 1) x nrhs) and dPb (max(max_lvl_fblk, 1) SPW x nrhs, which
// holds the backward partials) are the sweeps' workspace.
void enqueue_solve_bufs(swc_handle* h, double* dX, int nrhs, int64_t ldx, double* dY, double* dV,
                        double* dPb, bool marked = false) {
  const SweepRun a = sweep_run(h, dX, nrhs, ldx, dY, dV, dPb);
  enqueue_forward(h, a, marked);
  enqueue_backward(h, a);
}

// Waits for the handle's stream; an error where a sweep's wait ran out.
int sync_stream(swc_handle* h) {
  SWC_HIP(hipStreamSynchronize(h->stream));
  if (__atomic_exchange_n(&h->rec->abort, 0, __ATOMIC_RELAXED) != 0)
    return swc_set_error(SWC_EDEVICE, "solve: a wait inside a sweep ran out of time");
  return SWC_OK;
}

void enqueue_solve(swc_handle* h, double* dX, int nrhs, int64_t ldx, bool marked) {
  enqueue_solve_bufs(h, dX, nrhs, ldx, h->dY, h->dV, h->dPb, marked);
}

// In-place solve of L L^T X = B on device columns X (factor ordering); needs
// ensure_work(h, nrhs).  marked: enqueue_marks has been launched, after ev[2].
int solve_device(swc_handle* h, double* dX, int nrhs, int64_t ldx, bool marked) {
  hipStream_t st = h->stream;
  hipGraphExec_t gx = nullptr;
  if (h->use_graphs) {
    for (auto& g : h->sgraphs)
      if (g.x == dX && g.nrhs == nrhs && g.ld == ldx && g.marked == marked) gx = g.exec;
    if (!gx) {
      if (h->sgraphs.size() >= 8) {
        (void)hipGraphExecDestroy(h->sgraphs.front().exec);
        h->sgraphs.erase(h->sgraphs.begin());
      }
      hipGraph_t g = nullptr;
      SWC_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      enqueue_solve(h, dX, nrhs, ldx, marked);
      SWC_HIP(hipStreamEndCapture(st, &g));
      hipError_t e = hipGraphInstantiate(&gx, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (e != hipSuccess) return swc_set_error(SWC_EDEVICE, std::string("solve graph: ") + hipGetErrorString(e));
      h->sgraphs.push_back({dX, nrhs, ldx, marked, gx});
    }
  }
  if (!marked) SWC_HIP(hipEventRecord(h->ev[2], st));
  if (gx) SWC_HIP(hipGraphLaunch(gx, st));
  else enqueue_solve(h, dX, nrhs, ldx, marked);
  SWC_HIP(hipEventRecord(h->ev[3], st));
  SWC_HIP(hipGetLastError());
  return SWC_OK;
}

// ---- vectors in and out of the factor ordering ----------------------------

// dOut (n x nrhs, ld n, factor ordering) = P B; B host or device with ld ldb.
int to_factor(swc_handle* h, const double* B, int on_device, int64_t ldb, double* dOut, int nrhs) {
  const int n = h->n;
  hipStream_t st = h->stream;
  const double* src = B;
  int64_t lds = ldb;
  if (!on_device) {
    SWC_HIP(hipMemcpy2DAsync(h->dWork, sizeof(double) * n, B, sizeof(double) * ldb,
                             sizeof(double) * n, nrhs, hipMemcpyHostToDevice, st));
    src = h->dWork;
    lds = n;
  }
  if (!h->perm.empty())
    hipLaunchKernelGGL(k_permute, dim3(grid_for((int64_t)n * nrhs)), dim3(kThreads), 0, st, src,
                       dOut, (const int*)h->dPerm, n, nrhs, lds, (int64_t)n, 0);
  else
    SWC_HIP(hipMemcpy2DAsync(dOut, sizeof(double) * n, src, sizeof(double) * lds,
                             sizeof(double) * n, nrhs, hipMemcpyDeviceToDevice, st));
  return SWC_OK;
}

// X (host or device, ld ldx) = P^T dIn.
int from_factor(swc_handle* h, const double* dIn, double* X, int on_device, int64_t ldx, int nrhs) {
  const int n = h->n;
  hipStream_t st = h->stream;
  double* dst = on_device ? X : h->dWork;
  const int64_t ldd = on_device ? ldx : n;
  if (!h->perm.empty())
    hipLaunchKernelGGL(k_permute, dim3(grid_for((int64_t)n * nrhs)), dim3(kThreads), 0, st, dIn,
                       dst, (const int*)h->dPerm, n, nrhs, (int64_t)n, ldd, 1);
  else
    SWC_HIP(hipMemcpy2DAsync(dst, sizeof(double) * ldd, dIn, sizeof(double) * n,
                             sizeof(double) * n, nrhs, hipMemcpyDeviceToDevice, st));
  if (!on_device)
    SWC_HIP(hipMemcpy2DAsync(X, sizeof(double) * ldx, h->dWork, sizeof(double) * n,
                             sizeof(double) * n, nrhs, hipMemcpyDeviceToHost, st));
  return sync_stream(h);
}

// ---- refinement -------------------------------------------------------------

// Column reductions (op 0 max|x|, 1 dot(x, y)) into slot `slot` of dScal, and slots
// [0, nslots) to the host: what one decision needs is waited for once.
void launch_reduce(swc_handle* h, const double* X, const double* Y, int ncol, int op, int slot) {
  hipStream_t st = h->stream;
  hipLaunchKernelGGL(k_reduce_partial, dim3(kRedBlocks, ncol), dim3(kThreads), 0, st, X, Y, h->n,
                     (int64_t)h->n, op, h->dPart);
  hipLaunchKernelGGL(k_reduce_final, dim3(ncol), dim3(kThreads), 0, st, (const double*)h->dPart, op,
                     h->dScal + (int64_t)slot * ncol);
}
int fetch_reduced(swc_handle* h, int ncol, int nslots, double* out) {
  SWC_HIP(hipMemcpyAsync(out, h->dScal, sizeof(double) * ncol * nslots, hipMemcpyDeviceToHost, h->stream));
  return sync_stream(h);
}
int reduce_cols(swc_handle* h, const double* X, const double* Y, int ncol, int op, double* out) {
  launch_reduce(h, X, Y, ncol, op, 0);
  return fetch_reduced(h, ncol, 1, out);
}

// Y = A X, or R = B - A X when B is given, on n x nrhs device columns of
// leading dimension ld (A = the full P A P^T in CSR, uploaded with the pattern).
void launch_csr_mv(swc_handle* h, const double* X, const double* B, double* Y, int n, int64_t ld,
                   int nrhs) {
  const int64_t rows_per_block = kThreads / kMvGroup;
  const int64_t blocks = std::min<int64_t>((n + rows_per_block - 1) / rows_per_block, 2048);
  hipLaunchKernelGGL(k_csr_mv, dim3((unsigned)std::max<int64_t>(blocks, 1)), dim3(kThreads), 0,
                     h->stream, (const int*)h->dRp, (const int*)h->dCi, (const double*)h->dAf, X, B,
                     Y, n, ld, nrhs);
}

int put_coeffs(swc_handle* h, const std::vector<double>& c) {
  SWC_HIP(hipMemcpyAsync(h->dScal + 2 * c.size(), c.data(), sizeof(double) * c.size(),
                         hipMemcpyHostToDevice, h->stream));
  return SWC_OK;
}

int solve_device(swc_handle* h, double* dX, int nrhs, int64_t ldx, bool marked = false);

// Refines X for A X = B (both n x nrhs, factor ordering, ld n) until every
// column's eta = ||b - A x||_inf / (||A||_inf ||x||_inf + ||b||_inf) <= tol.
// method 0: classical refinement x += M^{-1} r; method 1: conjugate gradients
// preconditioned with M = L L^T.  Starts from x = M^{-1} b.
int refine_device(swc_handle* h, const double* Bt, double* Xt, int nrhs, double tol, int maxiter,
                  int method, double* eta, int* iters) {
  const int n = h->n;
  const int64_t ld = n;
  hipStream_t st = h->stream;
  double* R = h->dRef + (int64_t)2 * n * nrhs;
  double* Z = h->dRef + (int64_t)3 * n * nrhs;
  double* Pv = h->dRef + (int64_t)4 * n * nrhs;
  const dim3 g(std::min(grid_for(n), 2048), nrhs);
  std::vector<double> bn, red(3 * (size_t)nrhs), rz(nrhs), pq(nrhs), co(nrhs);
  std::vector<char> conv(nrhs, 0);
  auto copy = [&](double* dst, const double* src) {
    return hipMemcpyAsync(dst, src, sizeof(double) * n * nrhs, hipMemcpyDeviceToDevice, st);
  };
  auto evaluate = [&](double* Rbuf, bool& done) -> int {
    launch_csr_mv(h, (const double*)Xt, Bt, Rbuf, n, ld, nrhs);
    launch_reduce(h, Rbuf, nullptr, nrhs, 0, 0);
    launch_reduce(h, Xt, nullptr, nrhs, 0, 1);
    // the first evaluation fetches max|b| too (slot 2, which put_coeffs uses later)
    if (int rc = fetch_reduced(h, nrhs, bn.empty() ? 3 : 2, red.data())) return rc;
    if (bn.empty()) bn.assign(red.begin() + 2 * nrhs, red.end());
    done = true;
    for (int c = 0; c < nrhs; ++c) {
      const double den = h->normA * red[nrhs + c] + bn[c];
      eta[c] = den > 0 ? red[c] / den : 0.0;
      conv[c] = eta[c] <= tol;
      done = done && conv[c];
    }
    return SWC_OK;
  };
  launch_reduce(h, Bt, nullptr, nrhs, 0, 2);
  SWC_HIP(copy(Xt, Bt));
  if (int rc = solve_device(h, Xt, nrhs, ld)) return rc;
  int it = 0;
  bool done = false;
  if (int rc = evaluate(R, done)) return rc;
  if (method == 0) {
    for (; !done && it < maxiter; ++it) {
      SWC_HIP(copy(Z, R));
      if (int rc = solve_device(h, Z, nrhs, ld)) return rc;
      for (int c = 0; c < nrhs; ++c) co[c] = conv[c] ? 0.0 : 1.0;
      if (int rc = put_coeffs(h, co)) return rc;
      hipLaunchKernelGGL(k_axpy_cols, g, dim3(kThreads), 0, st, Xt, (const double*)Z,
                         (const double*)(h->dScal + 2 * nrhs), n, ld);
      if (int rc = evaluate(R, done)) return rc;
    }
  } else {
    if (!done) {
      SWC_HIP(copy(Z, R));
      if (int rc = solve_device(h, Z, nrhs, ld)) return rc;
      SWC_HIP(copy(Pv, Z));
      if (int rc = reduce_cols(h, R, Z, nrhs, 1, rz.data())) return rc;
    }
    for (; !done && it < maxiter; ++it) {
      launch_csr_mv(h, (const double*)Pv, nullptr, Z, n, ld, nrhs);
      if (int rc = reduce_cols(h, Pv, Z, nrhs, 1, pq.data())) return rc;
      for (int c = 0; c < nrhs; ++c) {
        if (!conv[c] && !(pq[c] > 0))
          return swc_set_error(SWC_ENOTPOS, "swc_refine: conjugate gradients broke down");
        co[c] = conv[c] ? 0.0 : rz[c] / pq[c];
      }
      if (int rc = put_coeffs(h, co)) return rc;
      hipLaunchKernelGGL(k_axpy_cols, g, dim3(kThreads), 0, st, Xt, (const double*)Pv,
                         (const double*)(h->dScal + 2 * nrhs), n, ld);
      for (int c = 0; c < nrhs; ++c) co[c] = -co[c];
      if (int rc = put_coeffs(h, co)) return rc;
      hipLaunchKernelGGL(k_axpy_cols, g, dim3(kThreads), 0, st, R, (const double*)Z,
                         (const double*)(h->dScal + 2 * nrhs), n, ld);
      if (int rc = evaluate(Z, done)) return rc;  // true residual, for eta only
      if (done) {
        ++it;
        break;
      }
      SWC_HIP(copy(Z, R));
      if (int rc = solve_device(h, Z, nrhs, ld)) return rc;
      std::vector<double> rzn(nrhs);
      if (int rc = reduce_cols(h, R, Z, nrhs, 1, rzn.data())) return rc;
      for (int c = 0; c < nrhs; ++c) {
        co[c] = (conv[c] || rz[c] == 0) ? 0.0 : rzn[c] / rz[c];
        rz[c] = rzn[c];
      }
      if (int rc = put_coeffs(h, co)) return rc;
      hipLaunchKernelGGL(k_xpby_cols, g, dim3(kThreads), 0, st, Pv, (const double*)Z,
                         (const double*)(h->dScal + 2 * nrhs), n, ld);
    }
  }
  SWC_HIP(hipGetLastError());
  if (iters) *iters = it;
  return SWC_OK;
}

// ---- adjoint ---------------------------------------------------------------

int build_selinv_arrays(swc_handle* h) {
  hipStream_t st = h->stream;
  h->sel = swc::build_selinv(h->n, h->nsuper, h->super.data(), h->pi.data(), h->px.data(), h->Ls.data());
  swc::SelPlan& S = h->sel;
  // the item lists, one after the other
  std::vector<swc::SelItem> items;
  const std::vector<swc::SelItem>* lists[kSelLists] = {&S.diag,   &S.cols,  &S.u,   &S.gather,
                                                        &S.small, &S.z21, &S.z11, &S.diag16};
  size_t total = 0;
  for (int q = 0; q < kSelLists; ++q) total += lists[q]->size();
  items.reserve(total);
  for (int q = 0; q < kSelLists; ++q) {
    h->sel_items[q] = items.size();
    items.insert(items.end(), lists[q]->begin(), lists[q]->end());
  }
  int rc = upload(&h->dSelRuns, S.runs.data(), S.runs.size(), h);
  if (!rc) rc = upload(&h->dSelJrun, S.jrun.data(), S.jrun.size(), h);
  if (!rc) rc = upload(&h->dSelRel, (const int*)nullptr, (size_t)S.nrel, h);
  if (!rc) rc = upload(&h->dSelItems, items.data(), items.size(), h);
  if (!rc) rc = upload(&h->dSelM, (const double*)nullptr, (size_t)S.msize, h);
  if (!rc) rc = upload(&h->dArena, (const double*)nullptr, (size_t)S.zsize, h);
  if (!rc) rc = upload(&h->dZ, (const double*)nullptr, (size_t)h->plan.xsize, h);
  if (!rc) rc = upload(&h->dNodes, S.nodes.data(), S.nodes.size(), h);
  if (rc) {
    (void)hipStreamSynchronize(st);  // the uploads read vectors of this frame
    return rc;
  }
  // the strict upper triangles of the diagonal blocks are not written
  hipError_t e = hipMemsetAsync(h->dZ, 0, sizeof(double) * (size_t)h->plan.xsize, st);
  if (e == hipSuccess && !S.runs.empty()) {
    hipLaunchKernelGGL(k_selinv_rel, dim3((unsigned)S.runs.size()), dim3(kThreads), 0, st,
                       (const int*)h->dLs, (const swc::SelNode*)h->dNodes,
                       (const swc::SelRun*)h->dSelRuns, h->dSelRel);
    e = hipGetLastError();
  }
  const hipError_t es = hipStreamSynchronize(st);
  if (e == hipSuccess) e = es;
  if (e != hipSuccess) {  // the next call starts over
    (void)hipFree(h->dNodes);
    h->dNodes = nullptr;
    SWC_HIP(e);
  }
  // the lists are on the device: only the offsets stay
  for (auto* v : {&S.diag, &S.cols, &S.u, &S.gather, &S.small, &S.z21, &S.z11, &S.diag16})
    std::vector<swc::SelItem>().swap(*v);
  std::vector<swc::SelNode>().swap(S.nodes);
  std::vector<swc::SelRun>().swap(S.runs);
  std::vector<int>().swap(S.jrun);
  return SWC_OK;
}

int selinv_setup(swc_handle* h) {
  if (h->dNodes) return SWC_OK;
  try {
    return build_selinv_arrays(h);
  } catch (const std::bad_alloc&) {  // thrown before anything is uploaded
    return swc_set_error(SWC_ENOMEM, "selected inverse: out of host memory");
  }
}

int selinv_device(swc_handle* h) {
  if (h->zvalid) return SWC_OK;
  if (int rc = selinv_setup(h)) return rc;
  hipStream_t st = h->stream;
  const swc::SelPlan& S = h->sel;
  const swc::SelNode* nd = h->dNodes;
  const double* L = h->dL;
  double* M = h->dSelM;
  auto list = [&](int q, int first) { return (const swc::SelItem*)h->dSelItems + h->sel_items[q] + first; };
  for (size_t c = 0; c + 1 < S.chunk_lvl.size(); ++c) {
    const int d0 = S.chunk_diag[c], nd0 = S.chunk_diag[c + 1] - d0;
    const int h0 = S.chunk_diag16[c], nh = S.chunk_diag16[c + 1] - h0;
    const int t0 = S.chunk_cols[c], nt = S.chunk_cols[c + 1] - t0;
    const int u0 = S.chunk_u[c], nu = S.chunk_u[c + 1] - u0;
    if (nd0) hipLaunchKernelGGL(k_selinv_diag, dim3(nd0), dim3(64), 0, st, L, nd, list(0, d0), M);
    if (nh)
      hipLaunchKernelGGL(k_selinv_diag16, dim3((nh + 15) / 16), dim3(kThreads), 0, st, L, nd, list(7, h0), nh, M);
    if (nt) hipLaunchKernelGGL(k_selinv_cols, dim3(nt), dim3(kThreads), 0, st, L, nd, list(1, t0), M);
    if (nu) hipLaunchKernelGGL(k_selinv_U, dim3(nu), dim3(kThreads), 0, st, L, nd, list(2, u0), M);
    for (int l = S.chunk_lvl[c]; l < S.chunk_lvl[c + 1]; ++l) {
      const int g0 = S.lvl_gather[l], ng = S.lvl_gather[l + 1] - g0;
      const int s0 = S.lvl_small[l], nsm = S.lvl_small[l + 1] - s0;
      const int z0 = S.lvl_z21[l], nz = S.lvl_z21[l + 1] - z0;
      const int y0 = S.lvl_z11[l], ny = S.lvl_z11[l + 1] - y0;
      const int ldz = S.lvl_m[l] | 1;
      const size_t lds = nsm ? sizeof(double) * (size_t)ldz * (2 * 17 + S.lvl_m[l]) : 0;
      if (nsm + ng)
        hipLaunchKernelGGL(k_selinv_gather, dim3(nsm + ng), dim3(kThreads), lds, st, h->dZ, (const double*)M,
                           (const int*)h->dLs, nd, (const swc::SelRun*)h->dSelRuns, (const int*)h->dSelJrun,
                           (const int*)h->dSelRel, list(4, s0), nsm, ldz, list(3, g0), h->dArena);
      if (nz)
        hipLaunchKernelGGL(k_selinv_Z21, dim3(nz), dim3(kThreads), 0, st, h->dZ, (const double*)M,
                           (const double*)h->dArena, nd, list(5, z0));
      if (ny)
        hipLaunchKernelGGL(k_selinv_Z11, dim3(ny), dim3(kThreads), 0, st, h->dZ, (const double*)M, nd, list(6, y0));
    }
  }
  SWC_HIP(hipGetLastError());
  SWC_HIP(hipStreamSynchronize(st));
  h->zvalid = true;
  return SWC_OK;
}

int check_handle(const swc_handle* h) {
  if (!h) return swc_set_error(SWC_EINVAL, "null handle");
  return SWC_OK;
}

// The BCSC structure the kernels index: every supernode's row list holds its
// own columns first, then strictly increasing rows below them, all in [0, n);
// its value block (ld = row count) lies at a non-negative offset.
int validate_structure(int n, const int* blockSet, int supNo, const size_t* lC, const int* Ls,
                       const size_t* Li_ptr) {
  if (n <= 0 || supNo <= 0 || !blockSet || !lC || !Ls || !Li_ptr)
    return swc_set_error(SWC_EINVAL, "structure: bad argument");
  if (blockSet[0] != 0 || blockSet[supNo] != n)
    return swc_set_error(SWC_EINVAL, "structure: blockSet must span 0..n");
  for (int s = 0; s < supNo; ++s) {
    const int c0 = blockSet[s], c1 = blockSet[s + 1];
    if (c1 <= c0) return swc_set_error(SWC_EINVAL, "structure: empty supernode");
    const size_t p0 = Li_ptr[c0], p1 = Li_ptr[c1];
    if (p1 < p0 + (size_t)(c1 - c0) || p1 - p0 > 0x7fffffffu)
      return swc_set_error(SWC_EINVAL, "structure: row list shorter than the supernode");
    if (lC[c0] > ((size_t)1 << 62)) return swc_set_error(SWC_EINVAL, "structure: bad value offset");
    for (int c = c0; c < c1; ++c)
      if (Ls[p0 + (c - c0)] != c)
        return swc_set_error(SWC_EINVAL, "structure: a supernode's rows must start with its columns");
    for (size_t i = p0 + (c1 - c0); i < p1; ++i)
      if (Ls[i] <= Ls[i - 1] || Ls[i] >= n)
        return swc_set_error(SWC_EINVAL, "structure: rows must increase and stay below n");
  }
  return SWC_OK;
}

// What a factorization needs of A2: its pattern, and its entries' row positions.
struct A2Pattern {
  const int* p;
  const int* i;
  const int64_t* src;
  int64_t nvals;
  std::vector<int> pos;
  bool ok = false;  // pos is valid
};

// Every input value is used once: the condition under which the entry lists of the front
// plan and the value map agree (build_amap refuses the rest).
bool covers_values(const A2Pattern& a, int n) {
  if (!a.src) return true;
  if (a.nvals != a.p[n]) return false;
  std::vector<char> seen((size_t)a.nvals, 0);
  for (int e = 0; e < a.p[n]; ++e) {
    if (a.src[e] < 0 || a.src[e] >= a.nvals || seen[a.src[e]]) return false;
    seen[a.src[e]] = 1;
  }
  return true;
}

// The plan counts the arena's offsets as if it followed L (rounded up); it is an allocation
// of its own, `shift` values further on.
void place_arena(swc::FrontPlan& F, int64_t shift) {
  for (swc::Gather& g : F.gathers) g.src += shift;
  for (swc::SmallFront& f : F.small)
    if (f.R > f.w) f.ubase += shift;
  for (swc::FrontTile& u : F.utiles)
    if (u.upd) u.vbase += shift;
}

void free_all(std::initializer_list<void**> ps) {
  for (void** p : ps) {
    (void)hipFree(*p);
    *p = nullptr;
  }
}

// Work lists of the left-looking factorization.
int upload_left_looking(swc_handle* h) {
  const Plan& P = h->plan;
  int rc = upload(&h->dTiles, P.tiles.data(), P.tiles.size(), h);
  if (!rc) rc = upload(&h->dTasks, P.tasks.data(), P.tasks.size(), h);
  if (!rc) rc = upload(&h->dFtiles, P.ftiles.data(), P.ftiles.size(), h);
  if (!rc) rc = upload(&h->dFused, P.fused.data(), P.fused.size(), h);
  if (!rc) rc = upload(&h->dCounters, (const int*)nullptr, (size_t)std::max(P.nlevel, 1), h);
  if (!rc) rc = upload(&h->dDagItems, P.dag_items.data(), P.dag_items.size(), h);
  if (!rc) rc = upload(&h->dDagDeps, P.dag_deps.data(), P.dag_deps.size(), h);
  if (!rc)
    rc = upload(&h->dDagSync, (const int*)nullptr, 2 + P.dag_items.size() + (size_t)P.npanel, h);
  return rc;
}

// Leaves the multifrontal plan: its lists and arena are freed.
void drop_fronts(swc_handle* h) {
  (void)hipStreamSynchronize(h->stream);  // uploads read the lists
  free_all({(void**)&h->dU, (void**)&h->dGathers, (void**)&h->dAents, (void**)&h->dFactorTiles,
            (void**)&h->dSmall, (void**)&h->dFrontTiles});
  h->multifrontal = false;
  h->fronts = swc::FrontPlan();
}

void plan_structure(swc_handle* h, bool left_looking) {
  swc::build_plan(h->n, h->nsuper, h->super.data(), h->pi.data(), h->px.data(), h->Ls.data(),
                  h->pruneptr.data(), h->pruneset.data(), h->plan, left_looking, h->up_params,
                  h->hlevel.level_ptr.empty() ? nullptr : &h->hlevel);
}

// After an upload: gives the arena's memory back and prepares the left-looking
// factorization.  The factor in L and the solves stay as they are.  False where there is
// no arena or no room even so; swc_factor then refuses until the next upload.
bool give_up_arena(swc_handle* h) {
  if (!h->multifrontal || !h->dU) return false;
  for (auto& g : h->fgraph) {
    if (g) (void)hipGraphExecDestroy(g);
    g = nullptr;
  }
  for (auto& f : h->factor_seen) f = false;
  drop_fronts(h);
  h->lvl_tile_ms.clear();
  int rc = SWC_ENOMEM;
  try {
    swc::Plan left;
    // an H-level schedule set since the upload belongs to the next one
    swc::build_plan(h->n, h->nsuper, h->super.data(), h->pi.data(), h->px.data(), h->Ls.data(),
                    h->pruneptr.data(), h->pruneset.data(), left, true, h->up_params, nullptr);
    h->plan = std::move(left);
    rc = upload_left_looking(h);
    if (!rc)
      rc = upload(&h->dDiag, (const double*)nullptr, (size_t)std::max<int64_t>(h->plan.diag_scratch, 1), h);
  } catch (const std::exception&) {
  }
  if (rc) h->has_values = false;
  return rc == SWC_OK && hipStreamSynchronize(h->stream) == hipSuccess;
}

// L, its FP32 copy, the row lists and the plans' arrays on the device.
int upload_arrays(swc_handle* h, bool factor) {
  hipStream_t st = h->stream;
  const Plan& P = h->plan;
  swc::FrontPlan& F = h->fronts;
  int rc = upload(&h->dL, (const double*)nullptr, (size_t)(P.xsize + kLoadPad), h);
  if (!rc && h->multifrontal) {
    // above the diagonal blocks' diagonals L is never written
    hipLaunchKernelGGL(k_fill, dim3(grid_for(P.xsize)), dim3(kThreads), 0, st, h->dL, P.xsize, 0.0);
    const int64_t ubase = (P.xsize + 31) & ~(int64_t)31;  // where the plan has the arena
    if (F.usize > 0) rc = upload(&h->dU, (const double*)nullptr, (size_t)(P.xsize + F.usize - ubase), h);
    if (!rc && F.usize > 0) place_arena(F, ((intptr_t)h->dU - (intptr_t)h->dL) / (intptr_t)sizeof(double) - ubase);
  }
  if (h->multifrontal) {
    if (!rc) rc = upload(&h->dGathers, F.gathers.data(), F.gathers.size(), h);
    if (!rc) rc = upload(&h->dAents, F.aents.data(), F.aents.size(), h);
    if (!rc) rc = upload(&h->dFactorTiles, F.ftiles.data(), F.ftiles.size(), h);
    if (!rc) rc = upload(&h->dSmall, F.small.data(), F.small.size(), h);
    if (!rc) rc = upload(&h->dFrontTiles, F.utiles.data(), F.utiles.size(), h);
  } else if (!rc) {
    rc = upload_left_looking(h);
  }
  // the FP32 shadow follows the structure's size whatever the current mode: a
  // later switch to a mixed mode finds it sized for this structure
  (void)hipFree(h->dLf);
  h->dLf = nullptr;
  h->lf_cap = 0;
  if (!rc && h->precision > 0 && factor) {
    rc = upload(&h->dLf, (const float*)nullptr, (size_t)(P.xsize + kLoadPad), h);
    if (!rc) h->lf_cap = P.xsize;
  }
  if (!rc) rc = upload(&h->dLs, h->Ls.data(), h->Ls.size(), h);
  if (!rc) rc = upload(&h->dGptr, P.gptr.data(), P.gptr.size(), h);
  if (!rc) rc = upload(&h->dGidx, P.gidx.data(), P.gidx.size(), h);
  if (!rc) rc = upload(&h->dSweepSmall, P.sweeps.small.data(), P.sweeps.small.size(), h);
  if (!rc) rc = upload(&h->dSweepFwd, P.sweeps.fwd.data(), P.sweeps.fwd.size(), h);
  if (!rc) rc = upload(&h->dSweepBwd, P.sweeps.bwd.data(), P.sweeps.bwd.size(), h);
  if (!rc) rc = upload(&h->dSweepSync, (const int*)nullptr, 4, h);
  if (!rc && h->sweep_cap == 0) {
    // two workgroups to a CU (what the sweeps' registers allow); any number is safe
    int ncu = 0;
    const hipError_t e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device);
    if (e != hipSuccess)
      rc = swc_set_error(SWC_EDEVICE, std::string("upload: device query: ") + hipGetErrorString(e));
    else
      h->sweep_cap = 2 * std::max(ncu, 1);
  }
  if (!rc && h->fused_cap[0] == 0) {
    // a persistent grid: as many workgroups as the device holds at once
    int ncu = 0, per[3] = {0, 0, 0};
    hipError_t e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[0], k_narrow_fused<0>, 64, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[1], k_narrow_fused<1>, 64, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[2], k_narrow_fused<2>, 64, 0);
    if (e != hipSuccess)
      rc = swc_set_error(SWC_EDEVICE, std::string("upload: occupancy query: ") + hipGetErrorString(e));
    else
      for (int m = 0; m < 3; ++m) h->fused_cap[m] = std::max(1, per[m]) * std::max(ncu, 1);
  }
  if (!rc && h->dag_cap[0] == 0) {
    int ncu = 0, per[3] = {0, 0, 0};
    hipError_t e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[0], k_dag_factor<0>, kThreads, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[1], k_dag_factor<1>, kThreads, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[2], k_dag_factor<2>, kThreads, 0);
    if (e != hipSuccess)
      rc = swc_set_error(SWC_EDEVICE, std::string("upload: occupancy query: ") + hipGetErrorString(e));
    else
      for (int m = 0; m < 3; ++m) h->dag_cap[m] = std::max(1, per[m]) * std::max(ncu, 1);
  }
  if (!rc)
    rc = upload(&h->dDiag, (const double*)nullptr,
                (size_t)std::max(P.diag_scratch, F.diag_scratch), h);
  if (!rc) rc = upload(&h->dNormPart, (const double*)nullptr, kSetupBlocks, h);
  return rc;
}

// Structure part of an upload: the plan (solve part only without A2), L and its FP32
// copy, the row lists and the plan arrays on the device.  The factorization runs the
// multifrontal plan (fronts.h) where the structure has one and its arena fits the
// device beside everything else, else, and for an H-level schedule, the left-looking one
// (plan.h).
int upload_structure(swc_handle* h, int n, const int* blockSet, int supNo, const size_t* lC,
                     const int* Ls, const size_t* Li_ptr, const int* prunePtr,
                     const int* pruneSet, A2Pattern* a2) {
  const bool factor = a2 != nullptr;
  if (int rc = validate_structure(n, blockSet, supNo, lC, Ls, Li_ptr)) return rc;
  // pruneSet may be null when it is empty (no supernode has descendants)
  if (!prunePtr || (!pruneSet && prunePtr[supNo] != 0) || prunePtr[0] != 0)
    return swc_set_error(SWC_EINVAL, "structure: bad descendant sets");
  for (int s = 0; s < supNo; ++s)
    if (prunePtr[s + 1] < prunePtr[s]) return swc_set_error(SWC_EINVAL, "structure: bad descendant sets");
  h->factored = false;
  h->has_values = false;
  h->drop_graphs();
  h->work_cols = 0;  // the solve buffers are sized by the structure: rebuilt on next use
  // the old structure's L goes first: if this upload fails part way, no buffer
  // sized for the old structure is left beside the new plan, and swc_factor
  // refuses to run until an upload completes
  (void)hipFree(h->dL);
  h->dL = nullptr;
  drop_fronts(h);
  free_all({(void**)&h->dTiles, (void**)&h->dTasks, (void**)&h->dFtiles, (void**)&h->dFused, (void**)&h->dCounters,
            (void**)&h->dDagItems, (void**)&h->dDagDeps, (void**)&h->dDagSync});
  h->up_params = h->params;
  h->n = n;
  h->nsuper = supNo;
  h->nvals = 0;
  h->super.assign(blockSet, blockSet + supNo + 1);
  h->pi.resize(supNo + 1);
  h->px.resize(supNo);
  for (int s = 0; s <= supNo; ++s) h->pi[s] = (int64_t)Li_ptr[blockSet[s]];
  for (int s = 0; s < supNo; ++s) h->px[s] = (int64_t)lC[blockSet[s]];
  const int64_t ssize = h->pi[supNo];
  h->Ls.assign(Ls, Ls + ssize);
  h->pruneptr.assign(prunePtr, prunePtr + supNo + 1);
  h->pruneset.assign(pruneSet, pruneSet + prunePtr[supNo]);
  h->uploading = true;
  h->no_room = false;
  hipStream_t st = h->stream;
  int rc = SWC_OK;
  try {
    if (factor) a2->ok = a2_positions(h, a2->p, a2->i, a2->pos);
    int64_t xsize = 0;
    for (int s = 0; s < supNo; ++s)
      xsize = std::max(xsize, h->px[s] + (h->pi[s + 1] - h->pi[s]) * (h->super[s + 1] - h->super[s]));
    h->multifrontal =
        factor && a2->ok && h->hlevel.level_ptr.empty() && covers_values(*a2, n) &&
        swc::build_fronts(n, supNo, h->super.data(), h->pi.data(), h->px.data(), xsize,
                          h->Ls.data(), prunePtr, pruneSet, a2->p, a2->src, a2->pos.data(),
                          h->params.rlb, h->fronts);
    if (!h->multifrontal) h->fronts = swc::FrontPlan();
    plan_structure(h, factor && !h->multifrontal);
    rc = upload_arrays(h, factor);
    if (rc && h->fronts.usize > 0 && h->no_room) {
      drop_fronts(h);
      plan_structure(h, true);
      rc = upload_arrays(h, factor);
    }
  } catch (const std::bad_alloc&) {
    rc = swc_set_error(SWC_ENOMEM, "upload: out of host memory");
  } catch (const std::exception& e) {
    rc = swc_set_error(SWC_EINVAL, std::string("upload: ") + e.what());
  }
  h->uploading = false;
  h->zvalid = false;
  free_all({(void**)&h->dZ, (void**)&h->dArena, (void**)&h->dNodes, (void**)&h->dSelM, (void**)&h->dSelRuns,
            (void**)&h->dSelJrun, (void**)&h->dSelRel, (void**)&h->dSelItems});
  const hipError_t se = hipStreamSynchronize(st);
  if (rc) {
    (void)hipFree(h->dL);
    h->dL = nullptr;
    return rc;
  }
  SWC_HIP(se);
  return SWC_OK;
}

}  // namespace

extern "C" {

int swc_create(swc_handle** out) {
  if (!out) return swc_set_error(SWC_EINVAL, "swc_create: null argument");
  *out = nullptr;
  auto* h = new (std::nothrow) swc_handle;
  if (!h) return swc_set_error(SWC_ENOMEM, "swc_create: out of host memory");
  hipError_t e = hipGetDevice(&h->device);
  if (e == hipSuccess && bind_scratch(h->device) != SWC_OK) {
    delete h;
    return SWC_EDEVICE;  // bind_scratch recorded why
  }
  if (e == hipSuccess && !(h->rec = take_record())) e = hipErrorOutOfMemory;
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc((void**)&h->dInfo, sizeof(int));
  for (auto& ev : h->ev)
    if (e == hipSuccess) e = hipEventCreate(&ev);
  if (e != hipSuccess) {
    delete h;
    return swc_set_error(SWC_EDEVICE, std::string("swc_create: ") + hipGetErrorString(e));
  }
  *out = h;
  return SWC_OK;
}

int swc_destroy(swc_handle* h) {
  delete h;
  return SWC_OK;
}

int swc_upload(swc_handle* h, int n, const int* blockSet, int supNo, const size_t* lC,
               const int* Ls, const size_t* Li_ptr, const int* prunePtr, const int* pruneSet,
               const int* A2p, const int* A2i, const int64_t* a2src, int64_t nvals) {
  if (int rc = check_handle(h)) return rc;
  if (!A2p || !A2i) return swc_set_error(SWC_EINVAL, "swc_upload: bad argument");
  A2Pattern a2{A2p, A2i, a2src, nvals, {}};
  if (int rc = upload_structure(h, n, blockSet, supNo, lC, Ls, Li_ptr, prunePtr, pruneSet, &a2))
    return rc;
  if (A2p[0] != 0 || A2p[n] < 0) return swc_set_error(SWC_EINVAL, "swc_upload: bad A2 pointers");
  for (int j = 0; j < n; ++j)
    if (A2p[j + 1] < A2p[j]) return swc_set_error(SWC_EINVAL, "swc_upload: bad A2 pointers");
  h->nvals = a2src ? nvals : (int64_t)A2p[n];
  if (!a2.ok) return swc_set_error(SWC_EINVAL, "A2 entry outside the structure of L");
  std::vector<int64_t> amap;
  if (int rc = build_amap(h, A2p, a2.pos, a2src, nvals, amap)) return rc;
  // full CSR of P A P^T from its lower triangle, each entry mapped to its value
  std::vector<int> frp(n + 1, 0), fci;
  std::vector<int64_t> fvm;
  for (int j = 0; j < n; ++j)
    for (int q = A2p[j]; q < A2p[j + 1]; ++q) {
      frp[A2i[q] + 1]++;
      if (A2i[q] != j) frp[j + 1]++;
    }
  for (int i = 0; i < n; ++i) frp[i + 1] += frp[i];
  fci.resize(frp[n]);
  fvm.resize(frp[n]);
  {
    std::vector<int> fill(frp.begin(), frp.end() - 1);
    // row i: first the lower-triangle entries (columns j <= i, ascending j) ...
    for (int j = 0; j < n; ++j)
      for (int q = A2p[j]; q < A2p[j + 1]; ++q) {
        const int i = A2i[q];
        fci[fill[i]] = j;
        fvm[fill[i]++] = a2src ? a2src[q] : q;
      }
    // ... then the mirrored strictly-upper entries (columns > i, ascending)
    for (int j = 0; j < n; ++j)
      for (int q = A2p[j]; q < A2p[j + 1]; ++q) {
        const int i = A2i[q];
        if (i == j) continue;
        fci[fill[j]] = i;
        fvm[fill[j]++] = a2src ? a2src[q] : q;
      }
  }
  h->nnz_full = frp[n];
  // factor-order coordinates of every input value, and the diagonal positions
  std::vector<int> qi(h->nvals, 0), qj(h->nvals, 0);
  for (int j = 0; j < n; ++j)
    for (int q = A2p[j]; q < A2p[j + 1]; ++q) {
      const int64_t dst = a2src ? a2src[q] : q;
      qi[dst] = A2i[q];
      qj[dst] = j;
    }
  std::vector<int64_t> dpos(n);
  for (int s = 0; s < supNo; ++s) {
    const int64_t R = h->pi[s + 1] - h->pi[s];
    for (int c = blockSet[s]; c < blockSet[s + 1]; ++c)
      dpos[c] = h->px[s] + (int64_t)(c - blockSet[s]) * R + (c - blockSet[s]);
  }
  hipStream_t st = h->stream;
  int rc = SWC_OK;
  if (!rc) rc = upload(&h->dAmap, amap.data(), amap.size(), h);
  if (!rc) rc = upload(&h->dVals, (const double*)nullptr, (size_t)h->nvals, h);
  if (!rc) rc = upload(&h->dRp, frp.data(), frp.size(), h);
  if (!rc) rc = upload(&h->dCi, fci.data(), fci.size(), h);
  if (!rc) rc = upload(&h->dVmap, fvm.data(), fvm.size(), h);
  if (!rc) rc = upload(&h->dAf, (const double*)nullptr, fci.size(), h);
  if (!rc) rc = upload(&h->dQi, qi.data(), qi.size(), h);
  if (!rc) rc = upload(&h->dQj, qj.data(), qj.size(), h);
  if (!rc) rc = upload(&h->dDiagPos, dpos.data(), dpos.size(), h);
  // the copies above read this frame's vectors: wait for them on every path
  const hipError_t se = hipStreamSynchronize(st);
  if (rc) {
    // a partial upload leaves no usable structure: factor calls are refused
    (void)hipFree(h->dL);
    h->dL = nullptr;
    return rc;
  }
  SWC_HIP(se);
  h->has_values = true;
  return SWC_OK;
}

int swc_upload_symbolic(swc_handle* h, const swc_symbolic* sym) {
  if (int rc = check_handle(h)) return rc;
  if (!sym) return swc_set_error(SWC_EINVAL, "swc_upload_symbolic: null symbolic");
  int64_t sz[8];
  double fl;
  if (int rc = swc_symbolic_sizes(sym, sz, &fl)) return rc;
  const int n = (int)sz[0], ns = (int)sz[1];
  std::vector<int> super(ns + 1), Ls(sz[2]), pp(ns + 1), ps(sz[7]), a2p(n + 1), a2i(sz[6]), perm(n);
  std::vector<int64_t> iptr(n + 1), p(n + 1), a2src(sz[6]);
  swc_symbolic_copy(sym, SWC_SYM_SUPER, super.data());
  swc_symbolic_copy(sym, SWC_SYM_S, Ls.data());
  swc_symbolic_copy(sym, SWC_SYM_PRUNEPTR, pp.data());
  swc_symbolic_copy(sym, SWC_SYM_PRUNESET, ps.data());
  swc_symbolic_copy(sym, SWC_SYM_A2P, a2p.data());
  swc_symbolic_copy(sym, SWC_SYM_A2I, a2i.data());
  swc_symbolic_copy(sym, SWC_SYM_A2SRC, a2src.data());
  swc_symbolic_copy(sym, SWC_SYM_I_PTR, iptr.data());
  swc_symbolic_copy(sym, SWC_SYM_P, p.data());
  swc_symbolic_copy(sym, SWC_SYM_PERM, perm.data());
  int rc = swc_upload(h, n, super.data(), ns, (const size_t*)p.data(), Ls.data(),
                      (const size_t*)iptr.data(), pp.data(), ps.data(), a2p.data(), a2i.data(),
                      a2src.data(), (int64_t)a2src.size());
  if (rc) return rc;
  return swc_set_perm(h, perm.data());
}

int swc_set_perm(swc_handle* h, const int* perm) {
  if (int rc = check_handle(h)) return rc;
  if (!perm) {
    h->perm.clear();
    return SWC_OK;
  }
  std::vector<char> seen(h->n, 0);
  for (int k = 0; k < h->n; ++k) {
    if (perm[k] < 0 || perm[k] >= h->n || seen[perm[k]])
      return swc_set_error(SWC_EINVAL, "swc_set_perm: not a permutation");
    seen[perm[k]] = 1;
  }
  h->perm.assign(perm, perm + h->n);
  return upload(&h->dPerm, h->perm.data(), h->perm.size(), h);
}

int swc_factor(swc_handle* h, const double* values, int values_on_device, int* info) {
  if (int rc = check_handle(h)) return rc;
  if (!values) return swc_set_error(SWC_EINVAL, "swc_factor: null values");
  if (!h->dL || !h->has_values) return swc_set_error(SWC_ESTATE, "swc_factor: no structure uploaded");
  const double* dv = values;
  if (!values_on_device) {
    SWC_HIP(hipMemcpyAsync(h->dVals, values, sizeof(double) * h->nvals, hipMemcpyHostToDevice,
                           h->stream));
    dv = h->dVals;
  }
  if (int rc = factor_device(h, dv)) return rc;
  if (info) *info = h->last_info;
  if (h->last_info)
    return swc_set_error(SWC_ENOTPOS, "swc_factor: matrix is not positive definite (column " +
                                          std::to_string(h->last_info - 1) + ")");
  return SWC_OK;
}

int swc_get_factor(swc_handle* h, double* lValues, int on_device) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_get_factor: not factored");
  SWC_HIP(hipMemcpyAsync(lValues, h->dL, sizeof(double) * h->plan.xsize,
                         on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, h->stream));
  SWC_HIP(hipStreamSynchronize(h->stream));
  return SWC_OK;
}

int swc_solve(swc_handle* h, double* B, int nrhs, int64_t ldb, int on_device) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_solve: not factored");
  if (h->last_info) return swc_set_error(SWC_ENOTPOS, "swc_solve: factorization failed");
  if (!B || nrhs <= 0 || nrhs > 65535 || ldb < h->n)
    return swc_set_error(SWC_EINVAL, "swc_solve: bad argument");
  if (int rc = ensure_work(h, nrhs)) return rc;
  double* dY = h->dRef;
  // with an ordering, B goes into factor order in the launch that marks the vectors
  const bool marked = !h->perm.empty();
  if (marked) {
    const double* src = B;
    if (!on_device) {
      SWC_HIP(hipMemcpy2DAsync(h->dWork, sizeof(double) * h->n, B, sizeof(double) * ldb,
                               sizeof(double) * h->n, nrhs, hipMemcpyHostToDevice, h->stream));
      src = h->dWork;
    }
    SWC_HIP(hipEventRecord(h->ev[2], h->stream));  // the marks are part of the solve
    enqueue_marks(h, sweep_run(h, dY, nrhs, h->n, h->dY, h->dV, h->dPb), src, on_device ? ldb : h->n);
  } else if (int rc = to_factor(h, B, on_device, ldb, dY, nrhs)) {
    return rc;
  }
  if (int rc = solve_device(h, dY, nrhs, h->n, marked)) return rc;
  if (int rc = from_factor(h, dY, B, on_device, ldb, nrhs)) return rc;
  float ms = 0;
  SWC_HIP(hipEventElapsedTime(&ms, h->ev[2], h->ev[3]));
  h->t_solve_ms = ms;
  return SWC_OK;
}

// swc_solve on device columns with every buffer the sweeps need taken from the
// static `scratch` array (through this device's looked-up address): no device
// allocation, no captured graph (eager launches on the handle's stream).
// Layout, each part starting on a 256-byte boundary: the permuted right-hand
// sides (n x nrhs), the forward solutions (n x nrhs), the contribution vectors
// (max(vsize,1) x nrhs, marked pending before the forward sweep) and the
// backward partials.  Calls on one GPU share the array: overlapping calls race.
int swc_solve_noalloc(swc_handle* h, double* B, int nrhs, int64_t ldb) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_solve_noalloc: not factored");
  if (h->last_info) return swc_set_error(SWC_ENOTPOS, "swc_solve_noalloc: factorization failed");
  if (!B || nrhs <= 0 || nrhs > 65535 || ldb < h->n)
    return swc_set_error(SWC_EINVAL, "swc_solve_noalloc: bad argument");
  double* base = scratch_ptr(h->device);
  if (!base) return swc_set_error(SWC_ESTATE, "swc_solve_noalloc: workspace not bound to this device");
  const Plan& P = h->plan;
  auto up = [](int64_t x) { return (x + 31) & ~(int64_t)31; };  // 32 doubles = 256 bytes
  const int64_t n = h->n;
  const int64_t vld = std::max<int64_t>(P.vsize, 1);
  const int64_t pld = (int64_t)std::max(P.max_lvl_fblk, 1) * swc::SPW;
  const int64_t oX = 0, oY = oX + up(n * nrhs), oV = oY + up(n * nrhs), oP = oV + up(vld * nrhs);
  const int64_t need = oP + up(pld * nrhs);
  if (need > kScratchDoubles)
    return swc_set_error(SWC_EINVAL, "swc_solve_noalloc: needs " + std::to_string(need * 8) +
                                         " bytes of workspace for " + std::to_string(nrhs) +
                                         " right-hand sides; the fixed workspace holds " +
                                         std::to_string(kScratchDoubles * 8));
  double* Xt = base + oX;
  if (int rc = to_factor(h, B, 1, ldb, Xt, nrhs)) return rc;
  SWC_HIP(hipEventRecord(h->ev[2], h->stream));
  enqueue_solve_bufs(h, Xt, nrhs, n, base + oY, base + oV, base + oP);
  SWC_HIP(hipEventRecord(h->ev[3], h->stream));
  SWC_HIP(hipGetLastError());
  if (int rc = from_factor(h, Xt, B, 1, ldb, nrhs)) return rc;
  float ms = 0;
  SWC_HIP(hipEventElapsedTime(&ms, h->ev[2], h->ev[3]));
  h->t_solve_ms = ms;
  return SWC_OK;
}

int swc_refine(swc_handle* h, const double* B, double* X, int nrhs, int64_t ld, int on_device,
               double tol, int maxiter, int method, double* eta, int* iters) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_refine: not factored");
  if (h->last_info) return swc_set_error(SWC_ENOTPOS, "swc_refine: factorization failed");
  if (!B || !X || nrhs <= 0 || nrhs > 65535 || ld < h->n || !eta)
    return swc_set_error(SWC_EINVAL, "swc_refine: bad argument");
  if (method < 0) method = h->factored_precision ? 1 : 0;
  if (method > 1) return swc_set_error(SWC_EINVAL, "swc_refine: method must be -1, 0 or 1");
  if (int rc = ensure_work(h, nrhs)) return rc;
  double* Bt = h->dRef;
  double* Xt = h->dRef + (int64_t)h->n * nrhs;
  if (int rc = to_factor(h, B, on_device, ld, Bt, nrhs)) return rc;
  if (int rc = refine_device(h, Bt, Xt, nrhs, tol, maxiter, method, eta, iters)) return rc;
  return from_factor(h, Xt, X, on_device, ld, nrhs);
}

int swc_residual(swc_handle* h, const double* B, const double* X, int nrhs, int64_t ld,
                 int on_device, double* eta) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_residual: no values (factor first)");
  if (!B || !X || nrhs <= 0 || nrhs > 65535 || ld < h->n || !eta)
    return swc_set_error(SWC_EINVAL, "swc_residual: bad argument");
  if (int rc = ensure_work(h, nrhs)) return rc;
  const int n = h->n;
  double* Bt = h->dRef;
  double* Xt = h->dRef + (int64_t)n * nrhs;
  double* R = h->dRef + (int64_t)2 * n * nrhs;
  if (int rc = to_factor(h, B, on_device, ld, Bt, nrhs)) return rc;
  if (int rc = to_factor(h, X, on_device, ld, Xt, nrhs)) return rc;
  launch_csr_mv(h, (const double*)Xt, (const double*)Bt, R, n, (int64_t)n, nrhs);
  std::vector<double> red(3 * (size_t)nrhs);
  launch_reduce(h, R, nullptr, nrhs, 0, 0);
  launch_reduce(h, Xt, nullptr, nrhs, 0, 1);
  launch_reduce(h, Bt, nullptr, nrhs, 0, 2);
  if (int rc = fetch_reduced(h, nrhs, 3, red.data())) return rc;
  for (int c = 0; c < nrhs; ++c) {
    const double den = h->normA * red[nrhs + c] + red[2 * nrhs + c];
    eta[c] = den > 0 ? red[c] / den : 0.0;
  }
  return SWC_OK;
}

namespace {
// Per-column CSC descriptors of the uploaded structure and the factor's entry count.
std::vector<CscColumn> csc_columns(const swc_handle* h, int64_t* nnz) {
  std::vector<CscColumn> cols(h->n);
  int64_t off = 0;
  for (int s = 0; s < h->nsuper; ++s) {
    const int c0 = h->super[s], c1 = h->super[s + 1];
    const int64_t R = h->pi[s + 1] - h->pi[s];
    for (int j = c0; j < c1; ++j) {
      const int64_t d = j - c0;
      cols[j] = CscColumn{h->px[s] + d * R + d, h->pi[s] + d, R - d, off};
      off += R - d;
    }
  }
  *nnz = off;
  return cols;
}
}  // namespace

int swc_factor_nnz(swc_handle* h, int64_t* nnz) {
  if (int rc = check_handle(h)) return rc;
  if (!nnz) return swc_set_error(SWC_EINVAL, "swc_factor_nnz: null argument");
  if (h->n <= 0) return swc_set_error(SWC_ESTATE, "swc_factor_nnz: no structure");
  (void)csc_columns(h, nnz);
  return SWC_OK;
}

int swc_factor_csc(swc_handle* h, int64_t* Cp, int* Ci, double* Cx, int on_device) {
  if (int rc = check_handle(h)) return rc;
  if (!Cp || !Ci || !Cx) return swc_set_error(SWC_EINVAL, "swc_factor_csc: null argument");
  if (!h->factored) return swc_set_error(SWC_ESTATE, "swc_factor_csc: not factored");
  int64_t nnz = 0;
  const std::vector<CscColumn> cols = csc_columns(h, &nnz);
  hipStream_t st = h->stream;
  CscColumn* dcol = nullptr;
  int64_t* dCp = on_device ? Cp : nullptr;
  int* dCi = on_device ? Ci : nullptr;
  double* dCx = on_device ? Cx : nullptr;
  hipError_t e = device_malloc(h, (void**)&dcol, sizeof(CscColumn) * cols.size());
  if (e == hipSuccess && !on_device) e = device_malloc(h, (void**)&dCp, sizeof(int64_t) * (h->n + 1));
  if (e == hipSuccess && !on_device) e = device_malloc(h, (void**)&dCi, sizeof(int) * std::max<int64_t>(nnz, 1));
  if (e == hipSuccess && !on_device) e = device_malloc(h, (void**)&dCx, sizeof(double) * std::max<int64_t>(nnz, 1));
  if (e == hipSuccess)
    e = hipMemcpyAsync(dcol, cols.data(), sizeof(CscColumn) * cols.size(), hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    const int per = kThreads / 64;
    hipLaunchKernelGGL(k_factor_csc, dim3((h->n + per - 1) / per), dim3(kThreads), 0, st,
                       (const double*)h->dL, (const int*)h->dLs, (const CscColumn*)dcol, h->n, dCp,
                       dCi, dCx);
    e = hipGetLastError();
  }
  if (e == hipSuccess && !on_device) {
    e = hipMemcpyAsync(Cp, dCp, sizeof(int64_t) * (h->n + 1), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(Ci, dCi, sizeof(int) * nnz, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(Cx, dCx, sizeof(double) * nnz, hipMemcpyDeviceToHost, st);
  }
  const hipError_t se = hipStreamSynchronize(st);
  if (e == hipSuccess) e = se;
  (void)hipFree(dcol);
  if (!on_device) {
    (void)hipFree(dCp);
    (void)hipFree(dCi);
    (void)hipFree(dCx);
  }
  if (e != hipSuccess)
    return swc_set_error(SWC_EDEVICE, std::string("swc_factor_csc: ") + hipGetErrorString(e));
  return SWC_OK;
}

int swc_set_plan_params(swc_handle* h, const int* params, int count) {
  if (int rc = check_handle(h)) return rc;
  swc::PlanParams p;
  if (params && !swc::plan_params_from(params, count, p))
    return swc_set_error(SWC_EINVAL, "swc_set_plan_params: parameter out of range");
  // The dependency-driven launch is switched off: one run of it gave a wrong factor
  // (a non-positive pivot where the per-level launches give none) without a cause
  // found in its waits and fences.
  if (p.dag != 0)
    return swc_set_error(SWC_EINVAL,
                         "swc_set_plan_params: the dependency-driven launch (dag) is disabled");
  h->params = p;  // NULL: the defaults
  return SWC_OK;
}

int swc_set_schedule(swc_handle* h, int nLevels, const int* levelPtr, const int* parPtr,
                     const int* partition) {
  if (int rc = check_handle(h)) return rc;
  if (nLevels <= 0 || !levelPtr) {
    h->hlevel = swc::HLevelSchedule();
    return SWC_OK;
  }
  if (!parPtr || !partition || levelPtr[0] != 0 || levelPtr[nLevels] < 0)
    return swc_set_error(SWC_EINVAL, "swc_set_schedule: bad argument");
  const int npar = levelPtr[nLevels];
  if (parPtr[0] != 0 || parPtr[npar] < 0)
    return swc_set_error(SWC_EINVAL, "swc_set_schedule: bad partition pointers");
  swc::HLevelSchedule hl;
  hl.level_ptr.assign(levelPtr, levelPtr + nLevels + 1);
  hl.par_ptr.assign(parPtr, parPtr + npar + 1);
  hl.partition.assign(partition, partition + parPtr[npar]);
  h->hlevel = std::move(hl);  // checked against the structure at the next upload
  return SWC_OK;
}

int swc_set_precision(swc_handle* h, int mode) {
  if (int rc = check_handle(h)) return rc;
  if (mode < 0 || mode > 2) return swc_set_error(SWC_EINVAL, "swc_set_precision: mode must be 0, 1 or 2");
  if (mode > 0 && h->lf_cap < h->plan.xsize) {
    // a factor graph of a mixed mode captured the old shadow: drop it with the buffer
    for (int m = 1; m < 3; ++m)
      if (h->fgraph[m]) {
        (void)hipGraphExecDestroy(h->fgraph[m]);
        h->fgraph[m] = nullptr;
      }
    (void)hipFree(h->dLf);
    h->dLf = nullptr;
    h->lf_cap = 0;
    SWC_HIP(device_malloc(h, (void**)&h->dLf, sizeof(float) * (size_t)(h->plan.xsize + kLoadPad)));
    h->lf_cap = h->plan.xsize;
  }
  h->precision = mode;
  h->fp32_mask = mode == 0 ? 0 : (mode == 1 ? 1 : 3);
  return SWC_OK;
}

int swc_selected_inverse(swc_handle* h, double* Z, int on_device) {
  if (int rc = check_handle(h)) return rc;
  if (!h->factored || h->last_info) return swc_set_error(SWC_ESTATE, "swc_selected_inverse: no valid factor");
  if (int rc = selinv_device(h)) return rc;
  if (Z) {
    SWC_HIP(hipMemcpyAsync(Z, h->dZ, sizeof(double) * h->plan.xsize,
                           on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, h->stream));
    SWC_HIP(hipStreamSynchronize(h->stream));
  }
  return SWC_OK;
}

int swc_logdet(swc_handle* h, double* logdet) {
  if (int rc = check_handle(h)) return rc;
  if (!logdet) return swc_set_error(SWC_EINVAL, "swc_logdet: null argument");
  if (!h->factored || h->last_info) return swc_set_error(SWC_ESTATE, "swc_logdet: no valid factor");
  hipStream_t st = h->stream;
  hipLaunchKernelGGL(k_logdet_partial, dim3(kRedBlocks), dim3(kThreads), 0, st, (const double*)h->dL,
                     (const int64_t*)h->dDiagPos, h->n, h->dNormPart);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kThreads), 0, st, (const double*)h->dNormPart, 1,
                     &h->rec->logdet);
  SWC_HIP(hipGetLastError());
  SWC_HIP(hipStreamSynchronize(st));
  *logdet = 2.0 * h->rec->logdet;
  return SWC_OK;
}

int swc_gradient(swc_handle* h, const double* x, int x_on_device, double alpha, double beta,
                 double* grad, int grad_on_device) {
  if (int rc = check_handle(h)) return rc;
  if (!grad || (beta != 0.0 && !x)) return swc_set_error(SWC_EINVAL, "swc_gradient: null argument");
  if (!h->factored || h->last_info) return swc_set_error(SWC_ESTATE, "swc_gradient: no valid factor");
  if (alpha != 0.0)
    if (int rc = selinv_device(h)) return rc;
  if (int rc = ensure_work(h, 1)) return rc;
  hipStream_t st = h->stream;
  double* xt = h->dRef;
  if (beta != 0.0)
    if (int rc = to_factor(h, x, x_on_device, h->n, xt, 1)) return rc;
  double* g = grad_on_device ? grad : h->dRef + h->n;  // dRef holds >= 5 n doubles
  double* gbuf = nullptr;
  if (!grad_on_device) {
    SWC_HIP(with_room(h, [&] {
      return hipMallocAsync((void**)&gbuf, sizeof(double) * std::max<int64_t>(h->nvals, 1), st);
    }));
    g = gbuf;
  }
  hipLaunchKernelGGL(k_grad_values, dim3(grid_for(h->nvals)), dim3(kThreads), 0, st,
                     (const double*)h->dZ, (const int64_t*)h->dAmap, (const int*)h->dQi,
                     (const int*)h->dQj, (const double*)xt, alpha, beta, h->nvals, g);
  SWC_HIP(hipGetLastError());
  if (!grad_on_device) {
    SWC_HIP(hipMemcpyAsync(grad, gbuf, sizeof(double) * h->nvals, hipMemcpyDeviceToHost, st));
    SWC_HIP(hipFreeAsync(gbuf, st));
  }
  SWC_HIP(hipStreamSynchronize(st));
  return SWC_OK;
}

int swc_refuse_allocation(int nth) {
  if (nth < 0) return swc_set_error(SWC_EINVAL, "swc_refuse_allocation: negative count");
  refuse_allocation = nth;
  return SWC_OK;
}

int swc_set_graphs(swc_handle* h, int on) {
  if (int rc = check_handle(h)) return rc;
  h->use_graphs = on != 0;
  return SWC_OK;
}

int swc_set_profiling(swc_handle* h, int on) {
  if (int rc = check_handle(h)) return rc;
  h->profile = on != 0;
  return SWC_OK;
}

int swc_get_timings(const swc_handle* h, double* out) {
  if (int rc = check_handle(h)) return rc;
  if (!out) return swc_set_error(SWC_EINVAL, "swc_get_timings: null argument");
  const Plan& P = h->plan;
  out[0] = h->t_factor_ms;
  out[1] = h->t_solve_ms;
  out[2] = h->t_tile_ms;
  out[3] = h->n_tile;
  out[4] = h->t_trsm_ms;
  out[5] = h->n_trsm;
  out[6] = h->multifrontal ? h->fronts.update_flops : P.tile_kernel_flops;
  out[7] = h->multifrontal ? h->fronts.factor_flops : P.trsm_kernel_flops;
  return SWC_OK;
}

int swc_level_timings(const swc_handle* h, double* out, int cap, int* nlevel) {
  if (int rc = check_handle(h)) return rc;
  if (!nlevel) return swc_set_error(SWC_EINVAL, "swc_level_timings: null argument");
  const auto& flops = h->multifrontal ? h->fronts.lvl_flops : h->plan.lvl_tile_flops;
  *nlevel = h->multifrontal ? h->fronts.nlevel : h->plan.nlevel;
  if (!out) return SWC_OK;
  for (int l = 0; l < std::min(cap, *nlevel); ++l) {
    out[2 * l] = l < (int)h->lvl_tile_ms.size() ? h->lvl_tile_ms[l] : 0.0;
    out[2 * l + 1] = flops[l];
  }
  return SWC_OK;
}

int swc_plan_stats(const swc_handle* h, int64_t* out, double* flops) {
  if (int rc = check_handle(h)) return rc;
  const Plan& P = h->plan;
  out[0] = P.npanel;
  out[1] = (int64_t)P.tiles.size();
  out[2] = (int64_t)P.tasks.size();
  out[3] = P.nlevel;
  out[4] = P.xsize;
  out[5] = (int64_t)P.dag_items.size();
  out[6] = P.dag_items.empty() ? P.nlevel : P.dag_level0;
  if (flops) {
    flops[0] = P.update_flops;
    flops[1] = P.factor_flops;
    flops[2] = P.dag_flops;
    flops[3] = P.dag_sim_us;
    flops[4] = P.lvl_sim_us;
  }
  if (h->multifrontal) {  // update tiles, and the gathers and products they apply
    const swc::FrontPlan& F = h->fronts;
    out[0] = F.npanel;
    out[1] = (int64_t)F.utiles.size();
    out[2] = (int64_t)(F.utiles.size() + F.gathers.size());
    out[3] = out[6] = F.nlevel;
    if (flops) {
      flops[0] = F.update_flops;
      flops[1] = F.factor_flops;
    }
  }
  return SWC_OK;
}

// Reference entry point (sw_parallel_PB_Cholesky_05.h:52-66, PRUNE variant):
// uploads the structure, factors on the current GPU and writes lValues in place.
// The schedule arguments (levelPtr, parPtr, partition, chunk, threads, ...) are
// accepted and ignored: the GPU schedule is derived from prunePtr/pruneSet.
// Returns 1 on success and 0 on failure (the driver's convention,
// sw_choleskyTest01.cpp:240-244); swc_last_error() says why.
int sw_cholesky_left_par_05(int n, int* c, int* r, double* values, size_t* lC, int* Ls,
                            size_t* Li_ptr, double* lValues, int* blockSet, int supNo,
                            double* timing, int* prunePtr, int* pruneSet, int nLevels,
                            int* levelPtr, int* levelSet, int nPar, int* parPtr, int* partition,
                            int chunk, int threads, int super_max, int col_max, double* nodCost) {
  (void)nLevels; (void)levelPtr; (void)levelSet; (void)nPar; (void)parPtr; (void)partition;
  (void)chunk; (void)threads; (void)super_max; (void)col_max; (void)nodCost;
  swc_handle* h = nullptr;
  if (swc_create(&h)) return 0;
  std::unique_ptr<swc_handle> guard(h);
  int ok = 0;
  if (!swc_upload(h, n, blockSet, supNo, lC, Ls, Li_ptr, prunePtr, pruneSet, c, r, nullptr, 0)) {
    int info = 0;
    const int rc = swc_factor(h, values, 0, &info);
    if (rc == SWC_OK && swc_get_factor(h, lValues, 0) == SWC_OK) ok = 1;
    if (timing) timing[0] = h->t_factor_ms * 1e-3;  // device time of the factorization
  }
  return ok;
}

// Reference forward solve (triangularSolve/Triangular_BCSC.h:14-49, called as
// examples/triangularTest02.cpp:195): L y = x in place on the host vector x, for
// the BCSC factor (Lp = L->p, Li = L->s, Lx = values, Li_ptr = L->i_ptr, sup2col =
// L->super, supNo = L->nsuper), on the current GPU.  NNZ and col2sup are not used
// (the reference does not read them either).  The solve schedule comes from the
// row lists (the call carries no descendant sets); it is built on the first call
// for a structure and kept, with L's device buffer, for later calls with the
// same structure (the arrays are compared, not their addresses).  Returns 1, or
// 0 on failure (the reference's convention; swc_last_error() says why).
namespace {
std::mutex g_lsolve_mu;
swc_handle* g_lsolve = nullptr;  // held until the process ends

bool same_structure(const swc_handle* h, int n, const size_t* Lp, const int* Li,
                    const size_t* Li_ptr, const int* sup2col, int supNo) {
  if (!h || !h->dL || h->n != n || h->nsuper != supNo) return false;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev != h->device) return false;
  if (std::memcmp(h->super.data(), sup2col, sizeof(int) * (size_t)(supNo + 1)) != 0) return false;
  for (int s = 0; s <= supNo; ++s)
    if ((int64_t)Li_ptr[sup2col[s]] != h->pi[s]) return false;
  for (int s = 0; s < supNo; ++s)
    if ((int64_t)Lp[sup2col[s]] != h->px[s]) return false;
  return std::memcmp(h->Ls.data(), Li, sizeof(int) * h->Ls.size()) == 0;
}
}  // namespace

int blockedLsolve(int n, size_t* Lp, int* Li, double* Lx, int NNZ, size_t* Li_ptr, int* col2sup,
                  int* sup2col, int supNo, double* x) {
  (void)NNZ; (void)col2sup;
  if (!Lp || !Li || !x) return 0;  // the reference's own check
  if (!Lx) {
    swc_set_error(SWC_EINVAL, "blockedLsolve: null values");
    return 0;
  }
  std::lock_guard<std::mutex> lock(g_lsolve_mu);
  if (!same_structure(g_lsolve, n, Lp, Li, Li_ptr, sup2col, supNo)) {
    if (validate_structure(n, sup2col, supNo, Lp, Li, Li_ptr)) return 0;
    int dev = 0;
    if (g_lsolve && (hipGetDevice(&dev) != hipSuccess || dev != g_lsolve->device)) {
      delete g_lsolve;
      g_lsolve = nullptr;
    }
    if (!g_lsolve && swc_create(&g_lsolve)) return 0;
    std::vector<int> pp, ps;
    std::vector<int64_t> pi(supNo + 1);
    for (int s = 0; s <= supNo; ++s) pi[s] = (int64_t)Li_ptr[sup2col[s]];
    try {
      swc::descendant_sets(n, supNo, sup2col, pi.data(), Li, pp, ps);
    } catch (const std::exception& e) {
      swc_set_error(SWC_EINVAL, std::string("blockedLsolve: ") + e.what());
      return 0;
    }
    if (upload_structure(g_lsolve, n, sup2col, supNo, Lp, Li, Li_ptr, pp.data(), ps.data(), nullptr))
      return 0;
  }
  swc_handle* h = g_lsolve;
  if (ensure_work(h, 1)) return 0;
  hipStream_t st = h->stream;
  hipError_t e = hipMemcpyAsync(h->dL, Lx, sizeof(double) * (size_t)h->plan.xsize,
                                hipMemcpyHostToDevice, st);
  if (e == hipSuccess)
    e = hipMemcpyAsync(h->dWork, x, sizeof(double) * (size_t)n, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    enqueue_forward(h, sweep_run(h, h->dWork, 1, n, h->dY, h->dV, h->dPb));
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(x, h->dY, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost, st);
  const int rc = sync_stream(h);
  if (e != hipSuccess) {
    swc_set_error(SWC_EDEVICE, std::string("blockedLsolve: ") + hipGetErrorString(e));
    return 0;
  }
  return rc == SWC_OK ? 1 : 0;
}

}  // extern "C"
