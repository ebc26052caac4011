// Kernels of the triangular solves (work lists: sweeps.h).  Included by numeric.hip inside
// its anonymous namespace.
//
// Forward L y = b (blockedLsolve, Triangular_BCSC.h:14-49): row block of a supernode by row
// block, t = b - (descendants' contributions) - (earlier panels of the supernode), then the
// block's triangle; rows below give the supernode's contribution vector V_s = L21 y_s, which
// column c takes from all its descendants in increasing supernode order.  Backward
// L^T x = y: column panel by column panel, t = y - L21^T x - (later panels), then the
// transposed triangle.  Every sum has a fixed order, so results do not depend on timing.

#include "sweep_entries.h"

constexpr uint64_t kSweepTicks = 1000000000ull;  // 10 s of the 100 MHz clock

struct SweepRun {
  const double* L;
  const int* Ls;
  const int64_t* gptr;  // column c takes V[gidx[gptr[c] .. gptr[c + 1])]
  const int64_t* gidx;
  const swc::SweepSmall* small;
  const swc::SweepItem* items;
  int nitems;
  int* ticket;
  int* abort_flag;   // device: set when a wait ran out; every later wait then ends at once
  int* abort_host;   // the same for the host (pinned)
  double* X;         // right-hand sides / solutions, ld ldx
  double* Y;         // forward solutions, ld ldy
  double* V;         // contribution vectors, ld ldv
  double* P;         // backward partials, ld ldp
  int64_t ldx, ldy, ldv, ldp;
  int nrhs;
};

// Called by a whole wave: true while the wait may go on.
__device__ inline bool keep_waiting(const SweepRun& a, unsigned& spins, uint64_t& t0) {
  __builtin_amdgcn_s_sleep(1);
  if ((++spins & 255u) != 0) return true;
  if (__hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
  const uint64_t t = wall_clock64();
  if (t0 == 0) t0 = t;
  if (t - t0 < kSweepTicks) return true;
  __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(a.abort_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  return false;
}

// v[k] = the entry at p[k] once it is there, for lanes that need it (others 0).  `v` may
// hold an earlier load of the same entries.
template <int N>
__device__ inline void wait_entries(const SweepRun& a, const double* const (&p)[N], bool need,
                                    unsigned long long (&v)[N]) {
  unsigned spins = 0;
  uint64_t t0 = 0;
  for (;;) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < N; ++k) ok = ok && v[k] != kPending;
    if (__builtin_amdgcn_ballot_w64(need && !ok) == 0 || !keep_waiting(a, spins, t0)) break;
    if (need && !ok) {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = load_entry(p[k]);
    }
  }
}

__device__ inline double entry_value(unsigned long long b) {
  return __builtin_bit_cast(double, b == kPending ? kQuietNan : b);
}

// Sums of this lane's list V[q][gidx[e]], e = e0, e0 + step, ... < e1, in that order, for Q
// right-hand sides at once, N entries of each in flight.
template <int Q, int N>
__device__ inline void gather_sums(const SweepRun& a, const double* const (&V)[Q], int64_t e0,
                                   int64_t e1, int step, double (&sum)[Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) sum[q] = 0.0;
  for (int64_t e = e0; __builtin_amdgcn_ballot_w64(e < e1) != 0; e += N * step) {
    int64_t at[N];
    unsigned long long v[Q][N];
#pragma unroll
    for (int k = 0; k < N; ++k) at[k] = e + k * step < e1 ? a.gidx[e + k * step] : -1;
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int q = 0; q < Q; ++q) v[q][k] = at[k] >= 0 ? load_entry(V[q] + at[k]) : 0ull;
    unsigned spins = 0;
    uint64_t t0 = 0;
    for (;;) {
      bool ok = true;
#pragma unroll
      for (int k = 0; k < N; ++k)
#pragma unroll
        for (int q = 0; q < Q; ++q) ok = ok && v[q][k] != kPending;
      if (__builtin_amdgcn_ballot_w64(!ok) == 0 || !keep_waiting(a, spins, t0)) break;
#pragma unroll
      for (int k = 0; k < N; ++k)
#pragma unroll
        for (int q = 0; q < Q; ++q)
          if (v[q][k] == kPending) v[q][k] = load_entry(V[q] + at[k]);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int k = 0; k < N; ++k) sum[q] += entry_value(v[q][k]);
  }
}

// The triangle of an own block (n <= 64 columns) in LDS, column j of the block at T[kTriLd j],
// each row (forward) or column (backward, whose unknowns run the other way) scaled by the
// reciprocal of its diagonal entry, zeros wherever a lane does not depend on an unknown.  In
// LDS rather than in the substituting wave's registers it leaves them to the blocks of L in
// flight (64 entries are 128 registers).  Wave v brings columns 16 v .. 16 v + 15, lane =
// row; returns the reciprocal of diagonal entry `lane` (1 past n).
constexpr int kTriLd = 65;

template <bool FORWARD>
__device__ inline double stage_triangle(const double* __restrict__ D, int ld, int n, double* T,
                                        int wave, int lane) {
  const int l = min(lane, n - 1);
  double v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = D[(int64_t)min(16 * wave + k, n - 1) * ld + l];
  const double d = D[(int64_t)l * ld + l];
  const double rinv = lane < n ? 1.0 / d : 1.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int j = 16 * wave + k;
    const double s = FORWARD ? rinv : bcast(rinv, j);
    T[kTriLd * j + lane] = lane > j && lane < n ? v[k] * s : 0.0;
  }
  return rinv;
}

// Substitution for Q right-hand sides, lane i holding row i of each, t = t_i / L_ii on entry:
// x_i = t_i - sum of T_ij x_j over the unknowns before it (after it, backward).  One readlane
// and one FMA per step are on the chain: the scaled triangle keeps the multiply by 1 / L_ii
// off it.
template <bool FORWARD, int Q>
__device__ inline void sweep_triangle(const double* T, int lane, double (&t)[Q]) {
  double row[2][16];
  auto fetch = [&](int c, double(&r)[16]) {  // unknowns of chunk c, lane's coefficients
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int j = FORWARD ? 16 * c + s : 63 - (16 * c + s);
      r[s] = FORWARD ? T[kTriLd * j + lane] : T[kTriLd * lane + j];
    }
  };
  fetch(0, row[0]);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (c < 3) fetch(c + 1, row[(c + 1) & 1]);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int j = FORWARD ? 16 * c + s : 63 - (16 * c + s);
      if (j == (FORWARD ? 63 : 0)) continue;
      double xj[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) xj[q] = bcast(t[q], j);
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = fma(-row[c & 1][s], xj[q], t[q]);
    }
  }
}

// ---- narrow supernodes: one wave, right-hand sides r0 .. r0 + Q ------------------
template <int Q>
__device__ inline void small_forward(const SweepRun& a, const swc::SweepSmall& s, int r0, int nq,
                                     int lane) {
  const double* D = a.L + s.vbase;
  const int w = s.w, m = s.R - w, i = lane & 15, g = lane >> 4;
  double row[16], lv[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const double* col = D + (int64_t)min(c, w - 1) * s.R;
    const double v = col[min(i, w - 1)], b = col[min(w + lane, s.R - 1)];
    row[c] = i < w && c < i ? v : 0.0;
    lv[c] = c < w ? b : 0.0;
  }
  const double rinv = i < w ? 1.0 / D[(int64_t)min(i, w - 1) * (s.R + 1)] : 1.0;
  const int c = s.c0 + min(i, w - 1);
  const int64_t e0 = a.gptr[c], e1 = i < w ? a.gptr[c + 1] : e0;
#pragma unroll
  for (int k = 0; k < 16; ++k) row[k] *= rinv;
  // right-hand sides past nq repeat the last one's entries; all of a supernode's are
  // gathered and substituted together, so that their waits and chains overlap
  double b[Q], x[Q];
  const double* V[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int64_t r = r0 + min(q, nq - 1);
    b[q] = a.X[r * a.ldx + c];
    V[q] = a.V + r * a.ldv;
  }
  // four lanes share a column's list
  gather_sums<Q, Q == 1 ? 8 : 4>(a, V, e0 + g, e1, 4, x);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    x[q] += __shfl_xor(x[q], 16);
    x[q] += __shfl_xor(x[q], 32);
    x[q] = i < w ? (b[q] - x[q]) * rinv : 0.0;
  }
#pragma unroll
  for (int j = 0; j < 15; ++j)
#pragma unroll
    for (int q = 0; q < Q; ++q) x[q] = fma(-row[j], bcast(x[q], j), x[q]);
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (q < nq && lane < w) {
      publish(a.Y + (int64_t)(r0 + q) * a.ldy + c, x[q]);
      mark_pending(a.X + (int64_t)(r0 + q) * a.ldx + c);  // the backward sweep's entry
    }
  for (int r = 0; r < m; r += 64) {
    if (r > 0) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const double v = D[(int64_t)min(k, w - 1) * s.R + min(w + r + lane, s.R - 1)];
        lv[k] = k < w ? v : 0.0;
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (q >= nq) continue;
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc = fma(lv[k], bcast(x[q], k), acc);
      if (r + lane < m) publish(a.V + (int64_t)(r0 + q) * a.ldv + s.voff + r + lane, acc);
    }
  }
}

// Sums over the wave's 64 lanes of v[k], k < 16, for Q right-hand sides (the components of
// v): lane l ends up with the sums of v[l % 16] in v[0] (a fixed tree: halves exchanged, then
// the four lanes of one k).
template <int Q>
struct LaneSums {
  double v[16 * Q];  // v[Q k + q]
};
template <int Q, int H>
__device__ inline void fold_half(LaneSums<Q>& a, int lane) {
  const bool up = (lane & H) != 0;
#pragma unroll
  for (int k = 0; k < H * Q; ++k) {
    const double mine = up ? a.v[k + H * Q] : a.v[k], other = up ? a.v[k] : a.v[k + H * Q];
    a.v[k] = mine + __shfl_xor(other, H);
  }
}
template <int Q>
__device__ inline void fold16(LaneSums<Q>& a, int lane) {
  fold_half<Q, 8>(a, lane);
  fold_half<Q, 4>(a, lane);
  fold_half<Q, 2>(a, lane);
  fold_half<Q, 1>(a, lane);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    a.v[q] += __shfl_xor(a.v[q], 16);
    a.v[q] += __shfl_xor(a.v[q], 32);
  }
}

template <int Q>
__device__ inline void small_backward(const SweepRun& a, const swc::SweepSmall& s, int r0, int nq,
                                      int lane) {
  const double* D = a.L + s.vbase;
  const int w = s.w, m = s.R - w, i = lane & 15;
  double col[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const double v = D[(int64_t)min(i, w - 1) * s.R + min(j, w - 1)];
    col[j] = i < w && j > i && j < w ? v : 0.0;
  }
  const double rinv = i < w ? 1.0 / D[(int64_t)min(i, w - 1) * (s.R + 1)] : 1.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) col[k] *= rinv;
  const int c = s.c0 + min(i, w - 1);
  LaneSums<Q> acc;
#pragma unroll
  for (int k = 0; k < 16 * Q; ++k) acc.v[k] = 0.0;
  for (int r = 0; r < m; r += 64) {
    const bool in = r + lane < m;
    const int gr = a.Ls[s.rows_off + w + min(r + lane, m - 1)];
    double lv[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const double v = D[(int64_t)min(k, w - 1) * s.R + w + min(r + lane, m - 1)];
      lv[k] = in && k < w ? v : 0.0;
    }
    const double* p[Q];
    unsigned long long v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {  // past nq: the last one again
      p[q] = a.X + (int64_t)(r0 + min(q, nq - 1)) * a.ldx + gr;
      v[q] = load_entry(p[q]);
    }
    wait_entries<Q>(a, p, true, v);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const double x = in ? entry_value(v[q]) : 0.0;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc.v[Q * k + q] = fma(lv[k], x, acc.v[Q * k + q]);
    }
  }
  fold16<Q>(acc, lane);
  double t[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const double y = a.Y[(int64_t)(r0 + min(q, nq - 1)) * a.ldy + c];
    t[q] = i < w ? (y - acc.v[q]) * rinv : 0.0;
  }
#pragma unroll
  for (int j = 15; j >= 1; --j)
#pragma unroll
    for (int q = 0; q < Q; ++q) t[q] = fma(-col[j], bcast(t[q], j), t[q]);
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (lane < w && q < nq) publish(a.X + (int64_t)(r0 + q) * a.ldx + c, t[q]);
}

// ---- one right-hand side, a workgroup of four waves per item --------------------

constexpr int kTriLds = 64 * kTriLd;
constexpr int kSweepLds1 = kTriLds + 5 * 64;  // triangle, the waves' parts

// 16 columns of a 64-row block, lane = row (rows clamped into the block, columns into the
// supernode): column c0 + k at D + k ld.
__device__ inline void load_cols(const double* __restrict__ D, int ld, int ncol, double (&v)[16]) {
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = D[(int64_t)min(k, ncol - 1) * ld];
}

// Forward row block.  Wave v takes columns [16 v, 16 v + 16) of each panel (lane = row, its
// columns' unknowns in lanes 0..15) and every fourth entry of the contribution lists; the
// next panel's entries of L and unknowns are in flight while the current ones are applied.
__device__ inline void forward_item(const SweepRun& a, const swc::SweepItem& it, double* lds,
                                    int wave, int lane) {
  double* part = lds + kTriLds;
  const double* D = a.L + it.vbase + it.row0;  // row 0 of the block, column 0
  const int rl = min(lane, it.nr - 1);
  const bool own = it.kind == swc::kSweepOwn;
  auto cols = [&](int q, double(&v)[16]) {  // panel q clamped into the supernode
    const int c = min(64 * q + 16 * wave, it.w - 1);
    load_cols(D + (int64_t)c * it.ld + rl, it.ld, min(16, it.w - c), v);
  };
  auto unknowns = [&](int q) {  // where lane k < 16 finds unknown k of this wave's columns
    return a.Y + it.c0 + min(64 * q + 16 * wave + (lane & 15), it.w - 1);
  };
  double rinv = 1.0, b = 0.0;
  double l0[16], l1[16];
  double acc = 0.0;
  const double* p0[1];
  const double* p1[1];
  unsigned long long x0[1], x1[1];
  if (own) {
    const int c = it.c0 + it.row0 + rl;
    const int64_t e0 = a.gptr[c], e1 = lane < it.nr ? a.gptr[c + 1] : e0;
    b = a.X[c];
    rinv = stage_triangle<true>(D + (int64_t)it.row0 * it.ld, it.ld, it.nr, lds, wave, lane);
    const double* V[1] = {a.V};
    double sum[1];
    gather_sums<1, 8>(a, V, e0 + wave, e1, 4, sum);
    acc = sum[0];
  }
  if (it.nq > 0) {
    cols(0, l0);
    p0[0] = unknowns(0);
    x0[0] = load_entry(p0[0]);
  }
  auto apply = [&](int q, const double(&v)[16], const double* const (&p)[1],
                   unsigned long long(&x)[1]) {
    wait_entries<1>(a, p, true, x);
    const int n = it.w - 64 * q - 16 * wave;  // columns of this wave in the panel
    const double xv = (lane & 15) < n ? entry_value(x[0]) : 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) acc = fma(v[k], bcast(xv, k), acc);
  };
  for (int q = 0; q < it.nq; q += 2) {
    const int q1 = min(q + 1, it.nq - 1), q2 = min(q + 2, it.nq - 1);
    cols(q1, l1);
    p1[0] = unknowns(q1);
    x1[0] = load_entry(p1[0]);
    apply(q, l0, p0, x0);
    cols(q2, l0);
    p0[0] = unknowns(q2);
    x0[0] = load_entry(p0[0]);
    if (q + 1 < it.nq) apply(q + 1, l1, p1, x1);
  }
  part[64 * wave + lane] = acc;
  lds_barrier();
  if (wave == 0) {
    const double sum = ((acc + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
    if (own) {
      double t[1] = {lane < it.nr ? (b - sum) * rinv : 0.0};
      sweep_triangle<true, 1>(lds, lane, t);
      if (lane < it.nr) {
        publish(a.Y + it.c0 + it.row0 + lane, t[0]);
        mark_pending(a.X + it.c0 + it.row0 + lane);
      }
    } else if (lane < it.nr) {
      publish(a.V + it.out + lane, sum);
    }
  }
}

// Backward column panel or part of one.  Wave v takes columns [16 v, 16 v + 16) of the panel
// over all its rows, lane = row within each 64: products accumulate per lane and are folded
// over the lanes once, at the end.  Blocks go four at a time, their rows' positions, unknowns
// and entries of L in flight together (a block's position -> unknown is two dependent loads);
// the first group is the short one, so that the last blocks, which the chain of panels waits
// for, have their entries of L long before their unknowns.
__device__ inline void backward_item(const SweepRun& a, const swc::SweepItem& it, double* lds,
                                     int wave, int lane) {
  double* part = lds + kTriLds;
  const int col0 = 64 * it.p;
  const bool own = it.kind == swc::kSweepOwn;
  const double* D = a.L + it.vbase + (int64_t)col0 * it.ld;  // row 0, the panel's column 0
  double rinv = 1.0, y = 0.0;
  if (own) {
    y = a.Y[it.c0 + col0 + min(lane, it.nr - 1)];
    rinv = stage_triangle<false>(D + col0, it.ld, it.nr, lds, wave, lane);
  }
  const int cw = min(16 * wave, it.nr - 1), ncw = min(16, it.nr - cw);
  const double* Dw = D + (int64_t)cw * it.ld;
  LaneSums<1> acc;
#pragma unroll
  for (int k = 0; k < 16; ++k) acc.v[k] = 0.0;
  // row blocks: rows [row0, row1) below from the last 64 up (the nearest ancestors' unknowns
  // come last), then own blocks np - 1 .. p + 1
  const int np = (it.w + 63) / 64;
  const int nbelow = (it.row1 - it.row0 + 63) / 64, nown = own ? np - 1 - it.p : 0;
  const int nblk = nbelow + nown;
  constexpr int G = 4;
  for (int k0 = nblk > 0 ? -((G - nblk % G) % G) : 0; k0 < nblk; k0 += G) {
    int row[G], last[G], at[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int k = k0 + g;  // uniform; k < 0: nothing (no row passes `last`)
      const bool below = k < nbelow;
      const int r = below ? it.row0 + 64 * (nbelow - 1 - max(k, 0)) : 64 * (np - 1 - (k - nbelow));
      last[g] = below ? it.row1 - 1 : it.w - 1;
      row[g] = min(r + lane, last[g]);
      at[g] = below ? a.Ls[it.rows_off + row[g]] : it.c0 + row[g];
      if (k < 0 || r + lane > last[g]) last[g] = -1;
    }
    double l[G][16];
#pragma unroll
    for (int g = 0; g < G; ++g) load_cols(Dw + row[g], it.ld, ncw, l[g]);
    const double* p[G][1];
    unsigned long long x[G][1];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      p[g][0] = a.X + at[g];
      x[g][0] = load_entry(p[g][0]);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (k0 + g < 0) continue;  // uniform
      wait_entries<1>(a, p[g], true, x[g]);
      const double xv = last[g] >= 0 ? entry_value(x[g][0]) : 0.0;
#pragma unroll
      for (int k = 0; k < 16; ++k) acc.v[k] = fma(l[g][k], xv, acc.v[k]);
    }
  }
  fold16<1>(acc, lane);
  const double sum = acc.v[0];
  if (!own) {
    if (lane < 16 && 16 * wave + lane < it.nr) publish(a.P + it.out + 16 * wave + lane, sum);
    return;
  }
  if (lane < 16) part[16 * wave + lane] = sum;
  // the parts made by other items, wave v taking every fourth, in order
  double ps = 0.0;
  for (int c = wave; c < it.nq; c += 4) {
    const double* p[1] = {a.P + it.out + 64 * (int64_t)c + min(lane, it.nr - 1)};
    unsigned long long v[1] = {load_entry(p[0])};
    wait_entries<1>(a, p, true, v);
    ps += entry_value(v[0]);
  }
  part[64 + 64 * wave + lane] = ps;
  lds_barrier();
  if (wave == 0) {
    const double parts = ((ps + part[128 + lane]) + part[192 + lane]) + part[256 + lane];
    double t[1] = {lane < it.nr ? (y - (part[lane] + parts)) * rinv : 0.0};
    sweep_triangle<false, 1>(lds, lane, t);
    if (lane < it.nr) publish(a.X + it.c0 + col0 + lane, t[0]);
  }
}

// ---- up to 16 right-hand sides per item -----------------------------------------
// The products of a row block with the right-hand sides are 64 x 64 by 64 x 16 on FP64
// MFMA, so L is read once per 16 right-hand sides; unknowns come in through LDS, wave v
// fetching right-hand sides 4 v .. 4 v + 3 (lane = row); the triangle's chains run four to
// a wave, interleaved.

constexpr int kXLd = 17;                                  // LDS row stride of a 64 x 16 block
constexpr int kSweepLds16 = kTriLds + 3 * 64 * kXLd;      // triangle, two blocks of unknowns, sums

// A block of unknowns on its way: this wave's four right-hand sides, lane = row.
struct Unknowns {
  const double* p[4];
  unsigned long long v[4];
};
__device__ inline void stage_unknowns(const SweepRun& a, Unknowns& u, bool in, int nq, double* xs,
                                      int wave, int lane) {
  wait_entries<4>(a, u.p, true, u.v);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    xs[lane * kXLd + 4 * wave + q] = in && 4 * wave + q < nq ? entry_value(u.v[q]) : 0.0;
}

// One block's products, summed from zero: added to the running sum as a whole they round
// once per block at its size (||b - A x|| of 32 right-hand sides on the vector 48^3 operator
// was 3 times larger with one accumulator over all blocks).
__device__ inline d4 block_products(const double (&v)[16], const double* xs, int lr, int lk) {
  d4 s = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int x = 0; x < 16; ++x)
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(v[x], xs[(4 * x + lk) * kXLd + lr], s, 0, 0, 0);
  return s;
}

// t = (rhs - sums) / L_ii through the triangle for this wave's nw right-hand sides, to `out`
// (ld ldo); mark: entries of X to mark pending.
template <bool FORWARD, int Q>
__device__ inline void solve_triangles(const double* T, double rinv, const double (&b)[4], int n,
                                       int nw, double* out, int64_t ldo, double* mark, int64_t ldm,
                                       int lane) {
  double t[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) t[q] = lane < n ? b[q] * rinv : 0.0;
  sweep_triangle<FORWARD, Q>(T, lane, t);
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (q < nw && lane < n) {
      publish(out + q * ldo + lane, t[q]);
      if (FORWARD) mark_pending(mark + q * ldm + lane);
    }
}

__device__ inline void forward_item16(const SweepRun& a, const swc::SweepItem& it, int r0, int nq,
                                      double* lds, int wave, int lane) {
  double* xs0 = lds + kTriLds;
  const int lr = lane & 15, lk = lane >> 4;
  const double* D = a.L + it.vbase + it.row0;
  const bool own = it.kind == swc::kSweepOwn;
  const int nw = min(4, max(0, nq - 4 * wave));  // this wave's right-hand sides
  const int rl = min(lane, it.nr - 1);
  // right-hand sides past nq repeat the last one's addresses and are replaced by zero
  auto rhs = [&](int q) { return (int64_t)(r0 + min(4 * wave + q, nq - 1)); };
  // A fragments: rows 16 wave + lr of the block, columns 64 q + 4 x + lk
  const double* A = D + min(16 * wave + lr, it.nr - 1);
  auto frags = [&](int q, double(&v)[16]) {
#pragma unroll
    for (int x = 0; x < 16; ++x) v[x] = A[(int64_t)min(64 * q + 4 * x + lk, it.w - 1) * it.ld];
  };
  auto entries = [&](int q, Unknowns& u) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u.p[k] = a.Y + rhs(k) * a.ldy + it.c0 + min(64 * q + lane, it.w - 1);
      u.v[k] = load_entry(u.p[k]);
    }
  };
  double rinv = 1.0;
  double b[4] = {0.0, 0.0, 0.0, 0.0}, g[4] = {0.0, 0.0, 0.0, 0.0};
  if (own) {
    const int c = it.c0 + it.row0 + rl;
    const int64_t e0 = a.gptr[c], e1 = lane < it.nr ? a.gptr[c + 1] : e0;
    const double* V[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      b[q] = a.X[rhs(q) * a.ldx + c];
      V[q] = a.V + rhs(q) * a.ldv;
    }
    rinv = stage_triangle<true>(D + (int64_t)it.row0 * it.ld, it.ld, it.nr, lds, wave, lane);
    if (nw > 0) gather_sums<4, 8>(a, V, e0, e1, 1, g);
  }
  double f0[16], f1[16];
  Unknowns u0, u1;
  d4 acc = d4{0.0, 0.0, 0.0, 0.0};
  auto apply = [&](int q, const double(&v)[16], Unknowns& u) {
    double* xs = xs0 + (q & 1) * 64 * kXLd;
    stage_unknowns(a, u, 64 * q + lane < it.w, nq, xs, wave, lane);
    lds_barrier();  // the block is staged; the one two panels back has been read
    acc += block_products(v, xs, lr, lk);
  };
  if (it.nq > 0) {
    frags(0, f0);
    entries(0, u0);
  }
  for (int q = 0; q < it.nq; q += 2) {
    const int q1 = min(q + 1, it.nq - 1), q2 = min(q + 2, it.nq - 1);
    frags(q1, f1);
    entries(q1, u1);
    apply(q, f0, u0);
    frags(q2, f0);
    entries(q2, u0);
    if (q + 1 < it.nq) apply(q + 1, f1, u1);
  }
  // acc: rows 16 wave + lk + 4 r, right-hand side lr
  double* sums = xs0 + 2 * 64 * kXLd;
#pragma unroll
  for (int r = 0; r < 4; ++r) sums[(16 * wave + lk + 4 * r) * kXLd + lr] = acc[r];
  lds_barrier();
  if (own) {
#pragma unroll
    for (int q = 0; q < 4; ++q) b[q] -= g[q] + sums[lane * kXLd + 4 * wave + q];
    double* out = a.Y + (int64_t)(r0 + 4 * wave) * a.ldy + it.c0 + it.row0;
    double* mark = a.X + (int64_t)(r0 + 4 * wave) * a.ldx + it.c0 + it.row0;
    if (nw > 2) solve_triangles<true, 4>(lds, rinv, b, it.nr, nw, out, a.ldy, mark, a.ldx, lane);
    else if (nw == 2) solve_triangles<true, 2>(lds, rinv, b, it.nr, nw, out, a.ldy, mark, a.ldx, lane);
    else if (nw == 1) solve_triangles<true, 1>(lds, rinv, b, it.nr, nw, out, a.ldy, mark, a.ldx, lane);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < nw && lane < it.nr)
        publish(a.V + rhs(q) * a.ldv + it.out + lane, sums[lane * kXLd + 4 * wave + q]);
  }
}

__device__ inline void backward_item16(const SweepRun& a, const swc::SweepItem& it, int r0, int nq,
                                       double* lds, int wave, int lane) {
  double* xs0 = lds + kTriLds;
  const int lr = lane & 15, lk = lane >> 4;
  const int col0 = 64 * it.p;
  const bool own = it.kind == swc::kSweepOwn;
  const double* D = a.L + it.vbase + (int64_t)col0 * it.ld;
  const int nw = min(4, max(0, nq - 4 * wave));
  auto rhs = [&](int q) { return (int64_t)(r0 + min(4 * wave + q, nq - 1)); };
  double rinv = 1.0;
  double b[4] = {0.0, 0.0, 0.0, 0.0}, g[4] = {0.0, 0.0, 0.0, 0.0};
  if (own) {
#pragma unroll
    for (int q = 0; q < 4; ++q) b[q] = a.Y[rhs(q) * a.ldy + it.c0 + col0 + min(lane, it.nr - 1)];
    rinv = stage_triangle<false>(D + col0, it.ld, it.nr, lds, wave, lane);
  }
  const int np = (it.w + 63) / 64;
  const int nbelow = (it.row1 - it.row0 + 63) / 64, nown = own ? np - 1 - it.p : 0;
  const int nblk = nbelow + nown;
  auto place = [&](int k, int& r, int& last) {  // row block k
    const bool below = k < nbelow;
    r = below ? it.row0 + 64 * (nbelow - 1 - k) : 64 * (np - 1 - (k - nbelow));
    last = below ? it.row1 - 1 : it.w - 1;
  };
  auto position = [&](int k) {  // where this lane's row of block k has its unknown
    int r, last;
    place(k, r, last);
    const int row = min(r + lane, last);
    return k < nbelow ? a.Ls[it.rows_off + row] : it.c0 + row;
  };
  // A fragments: column 16 wave + lr, rows 4 x + lk of the block
  const double* A = D + (int64_t)min(16 * wave + lr, it.nr - 1) * it.ld;
  auto frags = [&](int k, double(&v)[16]) {
    int r, last;
    place(k, r, last);
#pragma unroll
    for (int x = 0; x < 16; ++x) v[x] = A[min(r + 4 * x + lk, last)];
  };
  auto entries = [&](int at, Unknowns& u) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u.p[q] = a.X + rhs(q) * a.ldx + at;
      u.v[q] = load_entry(u.p[q]);
    }
  };
  double f0[16], f1[16];
  Unknowns u0, u1;
  d4 acc = d4{0.0, 0.0, 0.0, 0.0};
  auto apply = [&](int k, const double(&v)[16], Unknowns& u) {
    int r, last;
    place(k, r, last);
    double* xs = xs0 + (k & 1) * 64 * kXLd;
    stage_unknowns(a, u, r + lane <= last, nq, xs, wave, lane);
    lds_barrier();
    acc += block_products(v, xs, lr, lk);
  };
  int at1 = 0, at2 = 0;  // positions are fetched two blocks ahead of their unknowns
  if (nblk > 0) {
    const int at0 = position(0);
    at1 = position(min(1, nblk - 1));
    frags(0, f0);
    entries(at0, u0);
  }
  for (int k = 0; k < nblk; k += 2) {
    const int k1 = min(k + 1, nblk - 1), k2 = min(k + 2, nblk - 1), k3 = min(k + 3, nblk - 1);
    at2 = position(k2);
    frags(k1, f1);
    entries(at1, u1);
    apply(k, f0, u0);
    at1 = position(k3);
    frags(k2, f0);
    entries(at2, u0);
    if (k + 1 < nblk) apply(k + 1, f1, u1);
  }
  double* sums = xs0 + 2 * 64 * kXLd;
#pragma unroll
  for (int r = 0; r < 4; ++r) sums[(16 * wave + lk + 4 * r) * kXLd + lr] = acc[r];
  lds_barrier();
  if (!own) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < nw && lane < it.nr)
        publish(a.P + rhs(q) * a.ldp + it.out + lane, sums[lane * kXLd + 4 * wave + q]);
    return;
  }
  for (int c = 0; c < it.nq; ++c) {
    Unknowns u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u.p[q] = a.P + rhs(q) * a.ldp + it.out + 64 * (int64_t)c + min(lane, it.nr - 1);
      u.v[q] = load_entry(u.p[q]);
    }
    wait_entries<4>(a, u.p, true, u.v);
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] += entry_value(u.v[q]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) b[q] -= sums[lane * kXLd + 4 * wave + q] + g[q];
  double* out = a.X + (int64_t)(r0 + 4 * wave) * a.ldx + it.c0 + col0;
  if (nw > 2) solve_triangles<false, 4>(lds, rinv, b, it.nr, nw, out, a.ldx, nullptr, 0, lane);
  else if (nw == 2) solve_triangles<false, 2>(lds, rinv, b, it.nr, nw, out, a.ldx, nullptr, 0, lane);
  else if (nw == 1) solve_triangles<false, 1>(lds, rinv, b, it.nr, nw, out, a.ldx, nullptr, 0, lane);
}

// ---- launches ---------------------------------------------------------------------

// The persistent launch of one sweep: GROUP right-hand sides (1 or 16) per item, the groups
// g0 .. g0 + ngroups of an item one after another in ticket order (they read the same L).
template <bool FORWARD, int GROUP>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
k_sweep(SweepRun a, int g0, int ngroups) {
  __shared__ double lds[GROUP == 1 ? kSweepLds1 : kSweepLds16];
  __shared__ int s_next[2];  // the item in work, and the next one: taken in turn
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int total = a.nitems * ngroups;
  if (tid == 0) s_next[0] = atomicAdd(a.ticket, 1);
  for (int turn = 0;; turn ^= 1) {
    lds_barrier();  // the next item is known, and everyone is done with the last one's LDS
    const int k = __builtin_amdgcn_readfirstlane(s_next[turn]);
    if (k >= total) break;
    int next = 0;
    if (tid == 0) next = atomicAdd(a.ticket, 1);  // on its way while this item is worked on
    const swc::SweepItem it = a.items[k / ngroups];
    const int r0 = (g0 + k % ngroups) * GROUP, nq = min(GROUP, a.nrhs - r0);
    if (it.kind == swc::kSweepSmall) {
      if constexpr (GROUP == 1) {
        for (int i = wave; i < it.count; i += 4) {
          const swc::SweepSmall s = a.small[it.first + i];
          if constexpr (FORWARD) small_forward<1>(a, s, r0, 1, lane);
          else small_backward<1>(a, s, r0, 1, lane);
        }
      } else {
        // four right-hand sides to a wave; waves that are left over take other supernodes
        const int quads = (nq + 3) >> 2, side = 4 / quads;
        const int q0 = 4 * (wave % quads);
        for (int i = wave / quads; i < it.count && wave < quads * side; i += side) {
          const swc::SweepSmall s = a.small[it.first + i];
          if constexpr (FORWARD) small_forward<4>(a, s, r0 + q0, min(4, nq - q0), lane);
          else small_backward<4>(a, s, r0 + q0, min(4, nq - q0), lane);
        }
      }
    } else if constexpr (GROUP == 1) {
      SweepRun b = a;  // one right-hand side: its columns
      b.X += (int64_t)r0 * a.ldx;
      b.Y += (int64_t)r0 * a.ldy;
      b.V += (int64_t)r0 * a.ldv;
      b.P += (int64_t)r0 * a.ldp;
      if constexpr (FORWARD) forward_item(b, it, lds, wave, lane);
      else backward_item(b, it, lds, wave, lane);
    } else {
      if constexpr (FORWARD) forward_item16(a, it, r0, nq, lds, wave, lane);
      else backward_item16(a, it, r0, nq, lds, wave, lane);
    }
    if (tid == 0) s_next[turn ^ 1] = next;
  }
}

// A leading level of narrow supernodes (their entries wait for nothing in this launch): one
// wave each, Q right-hand sides per wave.
template <bool FORWARD, int Q>
__global__ void __launch_bounds__(kThreads)
k_sweep_small(SweepRun a, int s0, int ns) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i = 4 * (int)blockIdx.x + wave;
  const int r0 = Q * (int)blockIdx.y;
  if (i >= ns) return;
  const swc::SweepSmall s = a.small[s0 + i];
  if constexpr (FORWARD) small_forward<Q>(a, s, r0, min(Q, a.nrhs - r0), lane);
  else small_backward<Q>(a, s, r0, min(Q, a.nrhs - r0), lane);
}

// A leading level's supernodes with at most 16 rows below (lvl_small16), one right-hand
// side: 16 lanes each, four to a wave.  The leaves of large forests: a wave a supernode
// leaves three lanes of four idle and pays its chain of 16 columns once a supernode (a
// solve of 4096 2D instances: 8.4 ms in its six leaf launches, 4.6 with this).  Same
// sums in the same order as small_forward and small_backward, bitwise.  What it reads has
// been published by earlier launches, so nothing is waited for.
template <bool FORWARD>
__global__ void __launch_bounds__(kThreads)
k_sweep_small16(SweepRun a, int s0, int ns) {
  a.X += (int64_t)blockIdx.y * a.ldx;
  a.Y += (int64_t)blockIdx.y * a.ldy;
  a.V += (int64_t)blockIdx.y * a.ldv;
  const int i = threadIdx.x & 15, lane = threadIdx.x & 63;
  const int k0 = (int)blockIdx.x * (kThreads / 16) + ((int)threadIdx.x >> 4);
  const bool have = k0 < ns;
  const swc::SweepSmall s = a.small[s0 + min(k0, ns - 1)];
  const int w = s.w, m = s.R - w;
  const double* D = a.L + s.vbase;
  int wmax = max(w, __shfl_xor(w, 16));
  wmax = __builtin_amdgcn_readfirstlane(max(wmax, __shfl_xor(wmax, 32)));
  const int ic = min(i, w - 1), c = s.c0 + ic;
  const double rinv = i < w ? 1.0 / D[(int64_t)ic * (s.R + 1)] : 1.0;
  double tri[16], lv[16];  // forward: row i of the triangle, backward: its column i
  const int below = min(w + i, s.R - 1);
#pragma unroll
  for (int g = 0; g < 16; g += 4) {
#pragma unroll
    for (int k = g; k < g + 4; ++k) tri[k] = lv[k] = 0.0;
    if (g < wmax) {
#pragma unroll
      for (int k = g; k < g + 4; ++k) {
        const int kc = min(k, w - 1);
        const double* col = D + (int64_t)kc * s.R;
        const double v = FORWARD ? col[ic] : D[(int64_t)ic * s.R + kc], b = col[below];
        tri[k] = (FORWARD ? i < w && k < i : i < w && k > i && k < w) ? v * rinv : 0.0;
        lv[k] = k < w && (FORWARD || i < m) ? b : 0.0;
      }
    }
  }
  if constexpr (FORWARD) {
    const int64_t e0 = a.gptr[c], e1 = i < w ? a.gptr[c + 1] : e0;
    double p[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t e = e0; __builtin_amdgcn_ballot_w64(e < e1) != 0; e += 8) {
      int64_t at[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) at[q] = e + q < e1 ? a.gidx[e + q] : -1;
#pragma unroll
      for (int q = 0; q < 8; ++q) p[q & 3] += at[q] >= 0 ? entry_value(load_entry(a.V + at[q])) : 0.0;
    }
    double t = i < w ? (a.X[c] - ((p[0] + p[1]) + (p[2] + p[3]))) * rinv : 0.0;
    unrolled<0, 15>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if (j + 1 < wmax) t = fma(-tri[j], group_bcast<j>(t), t);
    });
    if (have && i < w) {
      publish(a.Y + c, t);
      mark_pending(a.X + c);  // the backward sweep's entry
    }
    double acc = 0.0;
    unrolled<0, 16>([&](auto K) {
      constexpr int k = decltype(K)::value;
      if (k < wmax) acc = fma(lv[k], group_bcast<k>(t), acc);
    });
    if (have && i < m) publish(a.V + s.voff + i, acc);
  } else {
    const double x = i < m ? entry_value(load_entry(a.X + a.Ls[s.rows_off + below])) : 0.0;
    LaneSums<1> acc;
#pragma unroll
    for (int k = 0; k < 16; ++k) acc.v[k] = lv[k] * x;
    fold_half<1, 8>(acc, lane);
    fold_half<1, 4>(acc, lane);
    fold_half<1, 2>(acc, lane);
    fold_half<1, 1>(acc, lane);
    double t = i < w ? (a.Y[c] - acc.v[0]) * rinv : 0.0;
    unrolled<0, 15>([&](auto J) {
      constexpr int j = 15 - decltype(J)::value;
      if (j < wmax) t = fma(-tri[j], group_bcast<j>(t), t);
    });
    if (have && i < w) publish(a.X + c, t);
  }
}

// Marks every entry a sweep waits for as pending and resets the two tickets; with `in`
// given, out = P in (n x nrhs, factor order) in the same launch.
__global__ void __launch_bounds__(kThreads)
k_sweep_init(double* __restrict__ Y, int64_t ny, double* __restrict__ V, int64_t nv,
             double* __restrict__ P, int64_t np, int* __restrict__ sync,
             const double* __restrict__ in, int64_t ldin, double* __restrict__ out, int64_t ldout,
             const int* __restrict__ perm, int n, int nrhs) {
  const int64_t i0 = (int64_t)blockIdx.x * kThreads + threadIdx.x, st = (int64_t)gridDim.x * kThreads;
  if (in)
    for (int64_t e = i0; e < (int64_t)n * nrhs; e += st) {
      const int k = (int)(e % n), r = (int)(e / n);
      out[r * ldout + k] = in[r * ldin + perm[k]];
    }
  for (int64_t i = i0; i < ny; i += st) mark_pending(Y + i);
  for (int64_t i = i0; i < nv; i += st) mark_pending(V + i);
  for (int64_t i = i0; i < np; i += st) mark_pending(P + i);
  if (i0 < 4) sync[i0] = 0;
}
