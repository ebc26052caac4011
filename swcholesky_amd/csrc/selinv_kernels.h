// Kernels of the selected inverse (plan and recurrences: selinv.h).  Included by
// numeric.hip inside its anonymous namespace, after the device helpers.
//
// [T; U] of a supernode is kept row major (ld = w), L and Z are column major (ld = nrow):
// with these orders every product below reads both operands in runs of 16 consecutive
// values, or in runs of 16 along the inner dimension.

// Step of a product's inner dimension: 16, as four MFMA instructions of 4.  Instruction x
// takes k = 4 (l / 16) + x from lane l, so that an operand whose k is its contiguous
// index is read in 32-byte pieces.  KROW: element (k, i) at p[k ld + i], else p[i ld + k].
// Indexes past n repeat the last one (their results are not stored), k past k1 gives 0.
template <bool KROW>
__device__ inline void sel_load(double (&v)[2][4], const double* __restrict__ p, int64_t ld,
                                int n, int kb, int k1, int lane) {
  const int lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = min(16 * q + lr, n - 1);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int k = kb + 4 * lk + x, kc = min(k, k1 - 1);
      const double e = KROW ? p[(int64_t)kc * ld + i] : p[(int64_t)i * ld + kc];
      v[q][x] = k < k1 ? e : 0.0;
    }
  }
}

// acc[bi][bj] += A B over k in [k0, k1) in steps of `stride` (a multiple of 16), A(i, k) and
// B(k, j) as sel_load reads them (na, nb valid rows, columns).  Lane l, entry r: row
// 16 bi + l / 16 + 4 r, column 16 bj + l % 16; with SWAP rows and columns change places.
template <bool AK, bool BK, bool SWAP, bool NEG>
__device__ inline void sel_product(d4 (&acc)[2][2], const double* __restrict__ A, int64_t lda,
                                   int na, const double* __restrict__ B, int64_t ldb, int nb,
                                   int k0, int k1, int stride, int lane) {
  double a0[2][4], b0[2][4], a1[2][4], b1[2][4];
  auto multiply = [&](const double(&a)[2][4], const double(&b)[2][4]) {
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const double av = NEG ? -a[bi][x] : a[bi][x];
          acc[bi][bj] = SWAP ? __builtin_amdgcn_mfma_f64_16x16x4f64(b[bj][x], av, acc[bi][bj], 0, 0, 0)
                             : __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[bj][x], acc[bi][bj], 0, 0, 0);
        }
  };
  if (k0 >= k1) return;
  sel_load<AK>(a0, A, lda, na, k0, k1, lane);
  sel_load<BK>(b0, B, ldb, nb, k0, k1, lane);
  for (int k = k0; k < k1; k += 2 * stride) {
    const bool second = k + stride < k1;
    if (second) {
      sel_load<AK>(a1, A, lda, na, k + stride, k1, lane);
      sel_load<BK>(b1, B, ldb, nb, k + stride, k1, lane);
    }
    multiply(a0, b0);
    if (k + 2 * stride < k1) {
      sel_load<AK>(a0, A, lda, na, k + 2 * stride, k1, lane);
      sel_load<BK>(b0, B, ldb, nb, k + 2 * stride, k1, lane);
    }
    if (second) multiply(a1, b1);
  }
}

// Sum of the four waves' accumulators: wave b returns block (b / 2, b % 2).
__device__ inline d4 sel_reduce(const d4 (&acc)[2][2], double* part, int wave, int lane) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[((wave * 4 + b) * 4 + r) * 64 + lane] = acc[b >> 1][b & 1][r];
  lds_barrier();
  d4 sum;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double v = part[((0 * 4 + wave) * 4 + r) * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) v += part[((w * 4 + wave) * 4 + r) * 64 + lane];
    sum[r] = v;
  }
  return sum;
}

// Places of a run's rows in its ancestor's row list (once per structure).
__global__ void __launch_bounds__(kThreads)
k_selinv_rel(const int* __restrict__ Ls, const swc::SelNode* __restrict__ nodes,
             const swc::SelRun* __restrict__ runs, int* __restrict__ rel) {
  const swc::SelRun r = runs[blockIdx.x];
  const swc::SelNode nd = nodes[r.node];
  const int m = nd.nrow - nd.w;
  for (int i = r.j0 + (int)threadIdx.x; i < m; i += kThreads) {
    const int v = Ls[nd.rows_off + nd.w + i];
    int lo = 0, hi = r.ld - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (Ls[r.rows_off + mid] < v) lo = mid + 1;
      else hi = mid;
    }
    rel[r.rel + i] = lo;
  }
}

// Inverse of one 64 x 64 diagonal block of L11, a column per lane: T(i, j) = 0 above the
// diagonal, 1 / L(j, j) on it, below it -(sum_{k < i} L(i, k) T(k, j)) / L(i, i), L's block
// in LDS.  A chain of 64 rows; all blocks of all supernodes of a chunk are one launch.
__global__ void __launch_bounds__(64)
k_selinv_diag(const double* __restrict__ L, const swc::SelNode* __restrict__ nodes,
              const swc::SelItem* __restrict__ items, double* __restrict__ M) {
  __shared__ double lb[64][64];  // lb[c][r] = L(i0 + r, i0 + c)
  const swc::SelItem it = items[blockIdx.x];
  const swc::SelNode nd = nodes[it.node];
  const int lane = (int)threadIdx.x, i0 = it.a * 64, nb = min(64, nd.w - i0);
  const double* B = L + nd.vbase + (int64_t)i0 * nd.nrow + i0;
  double* T = M + nd.moff + (int64_t)i0 * nd.w + i0;
  const int lc = min(lane, nb - 1);
#pragma unroll 8
  for (int q = 0; q < nb; ++q) lb[q][lane] = B[(int64_t)q * nd.nrow + lc];
  __syncthreads();
  const double rd = 1.0 / lb[lc][lc];
  double x[64];
#pragma unroll
  for (int r = 0; r < 64; ++r) {
    if (r < nb) {  // uniform
      double sum = 0.0;
#pragma unroll
      for (int c = 0; c < r; ++c) {
        sum = fma(lb[c][r], x[c], sum);
        if (c % 16 == 15) __builtin_amdgcn_sched_barrier(0);  // 16 LDS reads in flight
      }
      __builtin_amdgcn_sched_barrier(0);
      const double rr = bcast(rd, r);
      x[r] = r < lane ? 0.0 : (r == lane ? rr : -sum * rr);
      if (lane < nb) T[(int64_t)r * nd.w + lane] = x[r];
    }
  }
}

// The same for blocks of at most 16 rows, 16 lanes each: most supernodes of a plane or a
// volume are that narrow, and at 256 registers and 32 KB a block the kernel above holds
// four of them on a CU.
__global__ void __launch_bounds__(kThreads)
k_selinv_diag16(const double* __restrict__ L, const swc::SelNode* __restrict__ nodes,
                const swc::SelItem* __restrict__ items, int nitems, double* __restrict__ M) {
  __shared__ double lb[kThreads / 16][16][16];  // lb[group][c][r]
  const int g = (int)threadIdx.x >> 4, lane = (int)threadIdx.x & 15;
  const int e = blockIdx.x * (kThreads / 16) + g;
  const swc::SelItem it = items[min(e, nitems - 1)];
  const swc::SelNode nd = nodes[it.node];
  const int i0 = it.a * 64, nb = nd.w - i0;
  const double* B = L + nd.vbase + (int64_t)i0 * nd.nrow + i0;
  double* T = M + nd.moff + (int64_t)i0 * nd.w + i0;
  const int lc = min(lane, nb - 1);
#pragma unroll
  for (int q = 0; q < 16; ++q) {  // past the block: the identity
    const double v = B[(int64_t)min(q, nb - 1) * nd.nrow + lc];
    lb[g][q][lane] = q < nb && lane < nb ? v : (q == lane ? 1.0 : 0.0);
  }
  __syncthreads();
  double x[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    double sum = 0.0;
#pragma unroll
    for (int c = 0; c < r; ++c) sum = fma(lb[g][c][r], x[c], sum);
    const double rr = 1.0 / lb[g][r][r];
    x[r] = r < lane ? 0.0 : (r == lane ? rr : -sum * rr);
  }
  if (e < nitems && lane < nb) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (r < nb) T[(int64_t)r * nd.w + lane] = x[r];
  }
}

// Block column jb of T below its diagonal block, 64 rows at a time:
//   T(ib, jb) = -T(ib, ib) sum_{jb <= k < ib} L(ib, k) T(k, jb)
// Four waves, a 32 x 32 quadrant each; the sum goes through LDS into the second product.
// The chain over ib is the only serial part of a wide supernode.
__global__ void __launch_bounds__(kThreads)
k_selinv_cols(const double* __restrict__ L, const swc::SelNode* __restrict__ nodes,
              const swc::SelItem* __restrict__ items, double* __restrict__ M) {
  __shared__ double S[64 * 65];
  const swc::SelItem it = items[blockIdx.x];
  const swc::SelNode nd = nodes[it.node];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4, r0 = 32 * (wave & 1), c0 = 32 * (wave >> 1);
  const int j0 = it.a * 64;  // a whole block: rows follow below it
  double* T = M + nd.moff;
  for (int i0 = j0 + 64; i0 < nd.w; i0 += 64) {
    const int nb = min(64, nd.w - i0);
    d4 acc[2][2] = {};
    sel_product<true, true, false, false>(acc, L + nd.vbase + i0 + min(r0, nb - 1), nd.nrow,
                                          max(min(32, nb - r0), 1), T + j0 + c0, nd.w, 32, j0, i0, 16, lane);
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[(r0 + 16 * bi + lk + 4 * r) * 65 + c0 + 16 * bj + lr] = acc[bi][bj][r];
    lds_barrier();
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = d4{0.0, 0.0, 0.0, 0.0};
    // T(ib, ib) is lower triangular: rows r0 .. r0 + 31 need k < r0 + 32
    sel_product<false, true, false, true>(acc, T + (int64_t)(i0 + min(r0, nb - 1)) * nd.w + i0, nd.w,
                                          max(min(32, nb - r0), 1), S + c0, 65, 32, 0,
                                          min(nb, r0 + 32), 16, lane);
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = r0 + 16 * bi + lk + 4 * r;
          if (i < nb) T[(int64_t)(i0 + i) * nd.w + j0 + c0 + 16 * bj + lr] = acc[bi][bj][r];
        }
    __syncthreads();  // the next rows read these, and S is written again
  }
}

// The three products by 32 x 32 tiles of their result, four waves sharing the inner
// dimension (16 columns each in turn): a level near the root has few tiles and a long
// inner dimension.  Bound: latency of the operand loads from L2 at the sizes of a
// plane's separators (w, m <= 400), 4 flops a byte of L2 traffic above that.

// U = L21 T: entry (i, c) is the sum over k >= c of L21(i, k) T(k, c).
__global__ void __launch_bounds__(kThreads)
k_selinv_U(const double* __restrict__ L, const swc::SelNode* __restrict__ nodes,
           const swc::SelItem* __restrict__ items, double* __restrict__ M) {
  __shared__ double part[4 * 4 * 4 * 64];
  const swc::SelItem it = items[blockIdx.x];
  const swc::SelNode nd = nodes[it.node];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nd.w, m = nd.nrow - W, i0 = it.a, c0 = it.b;
  d4 acc[2][2] = {};
  sel_product<true, true, false, false>(acc, L + nd.vbase + W + i0, nd.nrow, min(32, m - i0),
                                        M + nd.moff + c0, W, min(32, W - c0), c0 + 16 * wave, W, 64, lane);
  const d4 s = sel_reduce(acc, part, wave, lane);
  const int c = c0 + 16 * (wave & 1) + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 16 * (wave >> 1) + (lane >> 4) + 4 * r;
    if (i < m && c < W) M[nd.moff + (int64_t)(W + i) * W + c] = s[r];
  }
}

// Z(R,R), both triangles, from the ancestors' Z: a run's columns share the rows' places.
__device__ inline void sel_gather(const double* __restrict__ Z, const int* __restrict__ Ls,
                                  const swc::SelNode* __restrict__ nodes,
                                  const swc::SelRun* __restrict__ runs, const int* __restrict__ rel,
                                  const swc::SelItem& it, double* __restrict__ zrr) {
  const swc::SelRun r = runs[it.node];
  const swc::SelNode nd = nodes[r.node];
  const int m = nd.nrow - nd.w, i = it.b + (int)threadIdx.x;
  if (i >= m) return;
  const int j1 = min(r.j0 + r.nj, it.a + swc::kSelRunCols);
  const double* src = Z + r.zbase + rel[r.rel + i];
  const int* rows = Ls + nd.rows_off + nd.w;
  double* out = zrr + nd.zoff;
#pragma unroll 4
  for (int j = it.a; j < j1; ++j) {
    if (i < j) continue;
    const double z = src[(int64_t)rows[j] * r.ld];
    out[(int64_t)j * m + i] = z;
    out[(int64_t)i * m + j] = z;
  }
}

// A small supernode (w <= 16, m <= 64): Z(R,R), U and Z21 in LDS, a wave per 16 rows of
// Z21, then wave 0 forms Z11.  lds: 2 x ldz x 17 + m x ldz doubles, ldz = lvl_m | 1.
__device__ inline void sel_small(double* __restrict__ Z, const double* __restrict__ M,
                                 const int* __restrict__ Ls,
                                 const swc::SelNode& nd, const swc::SelRun* __restrict__ runs,
                                 const int* __restrict__ jrun, const int* __restrict__ rel,
                                 int ldz, double* lds) {
  __shared__ int64_t cb[swc::kSelSmallM], rb[swc::kSelSmallM];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int W = nd.w, m = nd.nrow - W;
  double* u = lds;             // u[j * 17 + c] = U(j, c)
  double* z21 = u + ldz * 17;  // z21[i * 17 + c]
  double* zr = z21 + ldz * 17;
  const double* T = M + nd.moff;
  if (tid < m) {
    const swc::SelRun r = runs[jrun[nd.rows_off + W + tid]];
    cb[tid] = r.zbase + (int64_t)Ls[nd.rows_off + W + tid] * r.ld;
    rb[tid] = r.rel;
  }
  for (int e = tid; e < m * 16; e += kThreads) {
    const int j = e >> 4, c = e & 15;
    u[j * 17 + c] = c < W ? T[(int64_t)(W + j) * W + c] : 0.0;
  }
  lds_barrier();
#pragma unroll 8
  for (int j = wave; j < m; j += 4) {
    if (lane >= j && lane < m) {
      const double z = Z[cb[j] + rel[rb[j] + lane]];
      zr[j * ldz + lane] = z;
      zr[lane * ldz + j] = z;
    }
  }
  lds_barrier();
  if (16 * wave < m) {
    d4 acc = d4{0.0, 0.0, 0.0, 0.0};
    const int i = min(16 * wave + lr, m - 1);
    for (int k = 0; k < m; k += 4) {
      const int kk = k + lk, kc = min(kk, m - 1);
      const double a = kk < m ? -zr[kc * ldz + i] : 0.0;
      const double b = kk < m ? u[kc * 17 + lr] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * wave + lk + 4 * r;
      if (row < m) z21[row * 17 + lr] = acc[r];
    }
  }
  lds_barrier();
  double* Zs = Z + nd.vbase;
  if (wave == 0) {
    d4 acc = d4{0.0, 0.0, 0.0, 0.0};
    const int cc = min(lr, W - 1);
#pragma unroll
    for (int k = 0; k < 16; k += 4) {
      const int kk = k + lk, kc = min(kk, W - 1);
      const double t = kk < W ? T[(int64_t)kc * W + cc] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(t, t, acc, 0, 0, 0);
    }
    for (int k = 0; k < m; k += 4) {
      const int kk = k + lk, kc = min(kk, m - 1);
      const double a = kk < m ? -u[kc * 17 + lr] : 0.0;
      const double b = kk < m ? z21[kc * 17 + lr] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = lk + 4 * r;
      if (i < W && lr <= i) Zs[(int64_t)lr * nd.nrow + i] = acc[r];
    }
  }
  for (int e = tid; e < W * 64; e += kThreads) {
    const int c = e >> 6, i = e & 63;
    if (i < m) Zs[(int64_t)c * nd.nrow + W + i] = z21[i * 17 + c];
  }
}

// First launch of a level: small supernodes from start to finish (workgroups [0, nsmall)),
// and the gathers of the others.
__global__ void __launch_bounds__(kThreads)
k_selinv_gather(double* Z, const double* __restrict__ M, const int* __restrict__ Ls, const swc::SelNode* __restrict__ nodes,
                const swc::SelRun* __restrict__ runs, const int* __restrict__ jrun,
                const int* __restrict__ rel, const swc::SelItem* __restrict__ small, int nsmall,
                int ldz, const swc::SelItem* __restrict__ gather, double* __restrict__ zrr) {
  extern __shared__ double lds_dyn[];
  if ((int)blockIdx.x < nsmall) {
    const swc::SelNode nd = nodes[small[blockIdx.x].node];
    sel_small(Z, M, Ls, nd, runs, jrun, rel, ldz, lds_dyn);
  } else {
    sel_gather(Z, Ls, nodes, runs, rel, gather[blockIdx.x - nsmall], zrr);
  }
}

// Z21 = -Z(R,R) U into Z.
__global__ void __launch_bounds__(kThreads)
k_selinv_Z21(double* __restrict__ Z, const double* __restrict__ M, const double* __restrict__ zrr,
             const swc::SelNode* __restrict__ nodes, const swc::SelItem* __restrict__ items) {
  __shared__ double part[4 * 4 * 4 * 64];
  const swc::SelItem it = items[blockIdx.x];
  const swc::SelNode nd = nodes[it.node];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nd.w, m = nd.nrow - W, i0 = it.a, c0 = it.b;
  d4 acc[2][2] = {};
  sel_product<true, true, true, true>(acc, zrr + nd.zoff + i0, m, min(32, m - i0),
                                      M + nd.moff + (int64_t)W * W + c0, W, min(32, W - c0),
                                      16 * wave, m, 64, lane);
  const d4 s = sel_reduce(acc, part, wave, lane);
  const int i = i0 + 16 * (wave >> 1) + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = c0 + 16 * (wave & 1) + (lane >> 4) + 4 * r;
    if (i < m && c < W) Z[nd.vbase + (int64_t)c * nd.nrow + W + i] = s[r];
  }
}

// Z11 = T^T T - U^T Z21, tiles of the lower triangle.
__global__ void __launch_bounds__(kThreads)
k_selinv_Z11(double* Z, const double* __restrict__ M, const swc::SelNode* __restrict__ nodes,
             const swc::SelItem* __restrict__ items) {
  __shared__ double part[4 * 4 * 4 * 64];
  const swc::SelItem it = items[blockIdx.x];
  const swc::SelNode nd = nodes[it.node];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nd.w, m = nd.nrow - W, i0 = it.a, c0 = it.b;
  const double* T = M + nd.moff;
  const double* U = T + (int64_t)W * W;
  double* Zs = Z + nd.vbase;
  const int ni = min(32, W - i0), nc = min(32, W - c0);
  d4 acc[2][2] = {};
  sel_product<true, true, true, false>(acc, T + i0, W, ni, T + c0, W, nc, i0 + 16 * wave, W, 64, lane);
  sel_product<true, false, true, true>(acc, U + i0, W, ni, Zs + (int64_t)c0 * nd.nrow + W, nd.nrow, nc,
                                       16 * wave, m, 64, lane);
  const d4 s = sel_reduce(acc, part, wave, lane);
  const int i = i0 + 16 * (wave >> 1) + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = c0 + 16 * (wave & 1) + (lane >> 4) + 4 * r;
    if (i < W && c <= i) Zs[(int64_t)c * nd.nrow + i] = s[r];
  }
}
