// Kernels of the multifrontal factorization (plan: fronts.h).  Included by numeric.hip
// inside its anonymous namespace, after the device helpers and the panel factor bodies.

// What an F or U launch assembles a tile from.
struct FrontIn {
  const swc::Gather* gathers;
  const swc::AEntry* aents;
  const double* vals;  // values of A in upload order
};

// Byte offset of the landing bit p of mask (elements `stride` bytes apart); a position
// receiving nothing gets kNoLand.  A row and a column offset add up: their sum passes
// the 1 GiB range of land_rsrc as soon as one of them is kNoLand, so the load reads 0.
constexpr unsigned kNoLand = 0x40000000u;
__device__ inline unsigned land_off(uint64_t mask, int p, unsigned stride) {
  return ((mask >> p) & 1ull) ? (unsigned)__popcll(mask & ((1ull << p) - 1ull)) * stride : kNoLand;
}
__device__ inline __amdgpu_buffer_rsrc_t land_rsrc(const double* base) {
  return make_rsrc(base, 0x3fffffff);
}

// The gathers of one tile, lane e holding gather g0 + e: one load for all descriptors of
// a tile (they would be a chain of dependent scalar loads inside the loop over children).
struct LaneGathers {
  int n;
  int4 a, b;  // {src, ld, pad}, {rmask, cmask}
};
__device__ inline LaneGathers lane_gathers(const FrontIn& in, int g0, int g1, int lane) {
  LaneGathers lg;
  lg.n = min(g1 - g0, 64);
  lg.a = lg.b = make_int4(0, 0, 0, 0);
  if (lane < lg.n) {
    const int4* p = reinterpret_cast<const int4*>(in.gathers + g0 + lane);
    lg.a = p[0];
    lg.b = p[1];
  }
  return lg;
}
__device__ inline uint64_t lane_u64(int lo, int hi, int e) {
  return (uint32_t)__builtin_amdgcn_readlane(lo, e) |
         (uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, e) << 32;
}
__device__ inline swc::Gather lane_gather(const LaneGathers& lg, int e) {  // e uniform, < n
  swc::Gather g;
  g.src = (int64_t)lane_u64(lg.a.x, lg.a.y, e);
  g.ld = __builtin_amdgcn_readlane(lg.a.z, e);
  g.pad = 0;
  g.rmask = lane_u64(lg.b.x, lg.b.y, e);
  g.cmask = lane_u64(lg.b.z, lg.b.w, e);
  return g;
}

// ---- U launch: one tile of <= 64 x 64, target -= A B^T ----------------------
// Four waves, a 32 x 32 quadrant each over the whole inner dimension (four 16x16 MFMA
// blocks, 32 accumulator registers), operands straight from global memory: the tile's
// rows and columns are consecutive rows of one supernode, so a 16-lane group of a load
// reads 128 consecutive bytes, and the two waves that share an operand find it in L1.
// The next 16 columns are in flight while the current ones are multiplied.  The column
// operand is the MFMA's first, so that a lane group holds 16 consecutive rows of one
// column of the result: target and gather accesses are 128-byte runs too.  The
// target (or, on first touch, the gathered children and entries of A) is loaded while
// the products accumulate from zero, and the sum is subtracted once: accumulating onto
// the target instead rounds every product at the target's size (||L - oracle|| / ||L||
// 1.2e-12 instead of 1.2e-13 on the vector 48^3 operator).  Bound: L2 operand traffic
// (8 flops a byte), and latency for the k = 64 steps of a wide supernode.
// T = float: operands from the FP32 copy, 16 columns accumulated in FP32 and added to
// the FP64 accumulator (task_update).
constexpr int kTileLd = swc::TM + 1;

template <typename T>
__device__ inline void front_products(const T* __restrict__ src, const swc::FrontTile& u, int wr,
                                      int wc, int lane, d4 (&acc)[2][2]) {
  constexpr bool kF32 = sizeof(T) == 4;
  const int lr = lane & 15, lk = lane >> 4;
  const int cr = kF32 ? (lr >> 2) + 4 * (lr & 3) : lr;  // f32 output order (task_update)
  const unsigned kstep = (unsigned)u.sld * sizeof(T);
  unsigned ao[2], bo[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int i = 32 * wr + 16 * b + lr, j = 32 * wc + 16 * b + cr;
    ao[b] = (i < u.nr ? (unsigned)i * sizeof(T) : 0x80000000u) + lk * kstep;
    bo[b] = (j < u.nc ? (unsigned)j * sizeof(T) : 0x80000000u) + lk * kstep;
  }
  const bool skip01 = u.diag && wr == wc;  // the block of rows 0..15, columns 16..31
  auto load = [&](T(&a)[2][4], T(&b)[2][4], int kb) {
    const int64_t bytes = (int64_t)max(u.k - kb, 0) * kstep;
    const int64_t at = (int64_t)min(kb, u.k) * u.sld;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(src + u.asrc + at, bytes);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(src + u.bsrc + at, bytes);
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        a[q][x] = load_elem<T>(ra, ao[q] + 4 * x * kstep);
        b[q][x] = load_elem<T>(rb, bo[q] + 4 * x * kstep);
      }
  };
  auto multiply = [&](const T(&a)[2][4], const T(&b)[2][4]) {
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int bi = 0; bi < 2; ++bi) {
        if (bj == 1 && bi == 0 && skip01) continue;
        if constexpr (!kF32) {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            acc[bj][bi] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[bj][x], a[bi][x], acc[bj][bi], 0, 0, 0);
        } else {
          f4 c = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < 4; ++x)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(b[bj][x], a[bi][x], c, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[bj][bi][r] += (double)c[r];
        }
      }
  };
  T a0[2][4], b0[2][4], a1[2][4], b1[2][4];
  load(a0, b0, 0);
  for (int kb = 0; kb < u.k; kb += 32) {
    load(a1, b1, kb + 16);
    multiply(a0, b0);
    load(a0, b0, kb + 32);
    if (kb + 16 < u.k) multiply(a1, b1);
  }
}

// Operands through LDS in steps of 16 columns, two buffers: a thread loads four
// consecutive rows of one column of each operand (the rows behind the tile's last are
// read, not used), two steps ahead of their use, so an element comes from L1 once a
// workgroup instead of twice and in 16-byte loads: straight from global memory L1's
// lookups are taken 75% of the time and the matrix cores 44%.  Same sums in the same
// order as front_products, bitwise.
// Levels with a tile of kStageMin columns or more stage all their tiles; below that the
// barriers cost more than L1 does.  Straight -> staged from 128 columns on: vector 48^3
// with FP32 updates 50.6 -> 46.6 ms (update launches 33.2 -> 28.9), 64^3 in FP64 17.55 ->
// 17.49; from 300 on 46.7 and 17.53; staging every level 46.4 and 17.47, but a mesh of
// 20,000 points 0.88 -> 0.98.
constexpr int kStageK = 16;
constexpr int kStageMin = 128;
template <typename T>
constexpr int kStageLd = swc::TM + 16 / (int)sizeof(T);
constexpr int kUpdateLds = 4 * kStageK * kStageLd<double>;  // doubles; >= PW * kTileLd
static_assert(kUpdateLds >= swc::PW * kTileLd);
typedef int i4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ inline void front_products_staged(const T* __restrict__ src, const swc::FrontTile& u, int wr,
                                             int wc, bool active, int tid, double* lds,
                                             d4 (&acc)[2][2]) {
  constexpr bool kF32 = sizeof(T) == 4;
  constexpr int ld = kStageLd<T>, NV = kF32 ? 1 : 2;
  const int lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int cr = kF32 ? (lr >> 2) + 4 * (lr & 3) : lr;  // f32 output order (task_update)
  const int kk = tid >> 4, r4 = 4 * (tid & 15);
  const unsigned at = ((unsigned)kk * (unsigned)u.sld + (unsigned)r4) * (unsigned)sizeof(T);
  T* stage = reinterpret_cast<T*>(lds);
  i4 ra[NV], rb[NV];
  auto load = [&](int kb) {
    const int64_t base = (int64_t)min(kb, u.k) * u.sld;
    const __amdgpu_buffer_rsrc_t qa = make_rsrc(src + u.asrc + base, 0x3fffffff);
    const __amdgpu_buffer_rsrc_t qb = make_rsrc(src + u.bsrc + base, 0x3fffffff);
    const bool in = kb + kk < u.k;
    const unsigned oa = in && r4 < u.nr ? at : kNoLand, ob = in && r4 < u.nc ? at : kNoLand;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      ra[v] = __builtin_bit_cast(i4, __builtin_amdgcn_raw_buffer_load_b128(qa, (int)(oa + 16 * v), 0, 0));
      rb[v] = __builtin_bit_cast(i4, __builtin_amdgcn_raw_buffer_load_b128(qb, (int)(ob + 16 * v), 0, 0));
    }
  };
  auto store = [&](int buf) {
    i4* a = reinterpret_cast<i4*>(stage + (2 * buf) * kStageK * ld + kk * ld + r4);
    i4* b = reinterpret_cast<i4*>(stage + (2 * buf + 1) * kStageK * ld + kk * ld + r4);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      a[v] = ra[v];
      b[v] = rb[v];
    }
  };
  const bool skip01 = u.diag && wr == wc;  // the block of rows 0..15, columns 16..31
  auto multiply = [&](int buf) {
    const T* A = stage + (2 * buf) * kStageK * ld + lk * ld + 32 * wr + lr;
    const T* B = stage + (2 * buf + 1) * kStageK * ld + lk * ld + 32 * wc + cr;
    T a[2][4], b[2][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        a[q][x] = A[4 * x * ld + 16 * q];
        b[q][x] = B[4 * x * ld + 16 * q];
      }
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int bi = 0; bi < 2; ++bi) {
        if (bj == 1 && bi == 0 && skip01) continue;
        if constexpr (!kF32) {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            acc[bj][bi] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[bj][x], a[bi][x], acc[bj][bi], 0, 0, 0);
        } else {
          f4 c = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < 4; ++x)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(b[bj][x], a[bi][x], c, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[bj][bi][r] += (double)c[r];
        }
      }
  };
  load(0);
  store(0);
  load(kStageK);
  lds_barrier();
  for (int kb = 0, buf = 0; kb < u.k; kb += kStageK, buf ^= 1) {
    if (active) multiply(buf);
    if (kb + kStageK < u.k) {
      store(buf ^ 1);
      load(kb + 2 * kStageK);
    }
    lds_barrier();
  }
}

template <int MODE, bool STAGED>
__device__ inline void front_update_body(double* __restrict__ L, const float* __restrict__ Lf,
                                         const swc::FrontTile& u, const FrontIn& in,
                                         double* __restrict__ dscratch, double* lds, int tid) {
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4, wr = wave & 1, wc = wave >> 1;
  const bool diag = u.diag != 0;
  if (u.a1 > u.a0) {  // uniform over the workgroup: entries of A by way of LDS
    for (int e = tid; e < swc::PW * kTileLd; e += kThreads) lds[e] = 0.0;
    lds_barrier();
    for (int e = u.a0 + tid; e < u.a1; e += kThreads) {
      const swc::AEntry ae = in.aents[e];
      lds[(ae.pos >> 6) * kTileLd + (ae.pos & 63)] = in.vals[ae.q];
    }
    lds_barrier();
  }
  // a wave with nothing of the tile only loads operands
  const bool active = !((diag && wr < wc) || 32 * wr >= u.nr || 32 * wc >= u.nc);
  double* tgt = L + u.vbase;
  // this lane's elements: row 32 wr + 16 bi + l % 16, column 32 wc + 16 bj + l / 16 + 4 r
  auto row_of = [&](int l, int bi) { return 32 * wr + 16 * bi + (l & 15); };
  auto col_of = [&](int l, int bj, int r) { return 32 * wc + 16 * bj + (l >> 4) + 4 * r; };
  auto inside = [&](int i, int j) { return active && i < u.nr && j < u.nc && !(diag && i < j); };
  const __amdgpu_buffer_rsrc_t rt = land_rsrc(tgt);
  d4 cur[2][2];
  if (!active) {
  } else if (!u.first) {
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = row_of(lane, bi), j = col_of(lane, bj, r);
          cur[bj][bi][r] = load_elem<double>(
              rt, inside(i, j) ? ((unsigned)j * (unsigned)u.ld + (unsigned)i) * 8u : kNoLand);
        }
  } else {
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          cur[bj][bi][r] = u.a1 > u.a0 ? lds[(32 * wc + 16 * bj + lk + 4 * r) * kTileLd +
                                             32 * wr + 16 * bi + lr]
                                       : 0.0;
    for (int g0 = u.g0; g0 < u.g1; g0 += 64) {
      const LaneGathers lg = lane_gathers(in, g0, u.g1, lane);
      for (int g = 0; g < lg.n; ++g) {
        const swc::Gather ga = lane_gather(lg, g);
        const __amdgpu_buffer_rsrc_t rg = land_rsrc(L + ga.src);
        unsigned ro[2], co[2][4];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          ro[b] = land_off(ga.rmask, 32 * wr + 16 * b + lr, 8u);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            co[b][r] = land_off(ga.cmask, 32 * wc + 16 * b + lk + 4 * r, (unsigned)ga.ld * 8u);
        }
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              // above the diagonal a child holds nothing: read as zero
              const bool below = inside(row_of(lane, bi), col_of(lane, bj, r));
              const unsigned off = below ? ro[bi] + co[bj][r] : kNoLand;
              cur[bj][bi][r] += load_elem<double>(rg, off);
            }
      }
    }
  }
  d4 acc[2][2];
#pragma unroll
  for (int bj = 0; bj < 2; ++bj)
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) acc[bj][bi] = d4{0.0, 0.0, 0.0, 0.0};
  const bool f32 = MODE == 2 || (MODE == 1 && u.upd);
  if constexpr (STAGED) {
    if (u.a1 > u.a0) lds_barrier();  // the entries have been read
    if (f32) front_products_staged<float>(Lf, u, wr, wc, active, tid, lds, acc);
    else front_products_staged<double>(L, u, wr, wc, active, tid, lds, acc);
  } else {
    if (!active) return;
    if (f32) front_products<float>(Lf, u, wr, wc, lane, acc);
    else front_products<double>(L, u, wr, wc, lane, acc);
  }
  if (!active) return;
  // element addresses are formed again from an opaque lane index: kept from the loads
  // above they would hold 16 registers through the products
  int l2 = lane;
  asm volatile("" : "+v"(l2));
#pragma unroll
  for (int bj = 0; bj < 2; ++bj)
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = row_of(l2, bi), j = col_of(l2, bj, r);
        if (inside(i, j)) {
          const double v = cur[bj][bi][r] - acc[bj][bi][r];
          tgt[(int64_t)j * u.ld + i] = v;
          if (u.slot >= 0 && i < u.nc) dscratch[u.slot + j * u.nc + i] = v;
        }
      }
}

template <int MODE, bool STAGED>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(STAGED ? 4 : 3)))
k_front_update(double* __restrict__ L, const swc::FrontTile* __restrict__ tiles, int tile0,
               FrontIn in, double* __restrict__ dscratch, const float* __restrict__ Lf) {
  __shared__ __align__(16) double lds[kUpdateLds];
  const swc::FrontTile u = tiles[tile0 + blockIdx.x];
  front_update_body<MODE, STAGED>(L, Lf, u, in, dscratch, lds, threadIdx.x);
}

// ---- F launch ----------------------------------------------------------------

// Orders the LDS accesses of one wave's lanes (its own LDS buffer, no workgroup barrier).
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Entries of A in LDS working matrix W (column stride ld): rows [0, ndiag) of the tile go
// to W rows 0.., the others to W rows row1.. ; a null range adds nothing.
__device__ inline void add_entries(const FrontIn& in, int a0, int a1, double* W, int ld, int ndiag,
                                   bool rows_too, int row1, int tid, int nthreads) {
  for (int e = a0 + tid; e < a1; e += nthreads) {
    const swc::AEntry ae = in.aents[e];
    const int i = ae.pos & 63, j = ae.pos >> 6;
    const double v = in.vals[ae.q];
    if (i < ndiag) W[j * ld + i] += v;
    else if (rows_too) W[j * ld + row1 + i - ndiag] += v;
  }
}

// What the children hold for tile row `row` and columns c0 .. c0 + 15 (lower: only
// columns up to the row), rows outside [0, nrow) getting nothing, added to x in child
// order; two children's loads are in flight together.
__device__ inline void add_children(const double* __restrict__ L, const LaneGathers& lg, int lane,
                                    int row, int nrow, int c0, bool lower, double (&x)[16]) {
  auto issue = [&](int e, double(&v)[16]) {
    const swc::Gather ga = lane_gather(lg, e);
    const __amdgpu_buffer_rsrc_t rg = land_rsrc(L + ga.src);
    const unsigned ro = row < nrow ? land_off(ga.rmask, row & 63, 8u) : kNoLand;
    const unsigned cov = land_off(ga.cmask, lane, (unsigned)ga.ld * 8u);  // lane = column
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const unsigned co = __builtin_amdgcn_readlane(cov, c0 + c);
      v[c] = load_elem<double>(rg, lower && c0 + c > row ? kNoLand : ro + co);
    }
  };
  for (int e = 0; e < lg.n; e += 2) {
    double v0[16], v1[16];
    issue(e, v0);
    const bool two = e + 1 < lg.n;  // uniform; the second child read again otherwise
    issue(two ? e + 1 : e, v1);
#pragma unroll
    for (int c = 0; c < 16; ++c) x[c] = two ? (x[c] + v0[c]) + v1[c] : x[c] + v0[c];
  }
}

// The assembled first panel of a front in W (k_panel_factor_blk's layout): diagonal block
// (identity past nc) in rows 0..63, tile rows in rows 64.. .
__device__ inline void front_assemble_blk(const double* __restrict__ L, const swc::FactorTile& tl,
                                          const FrontIn& in, double* W, int first, int nx, int nb,
                                          int wave, int lane) {
  const int nc = tl.ncol, c0 = 16 * wave, tid = 64 * wave + lane;
  // the first entries of A are on their way while the children are gathered
  const int ad = tl.da0 + tid, at = tl.a0 + tid;
  const bool ind = ad < tl.da1, int_ = tl.kind != 0 && at < tl.a1;
  swc::AEntry ed{0, 0}, et{0, 0};
  if (ind) ed = in.aents[ad];
  if (int_) et = in.aents[at];
  LaneGathers lg = lane_gathers(in, tl.dg0, tl.dg1, lane);
  LaneGathers lt = tl.kind == 0 ? lg : lane_gathers(in, tl.g0, tl.g1, lane);
  const double vd = ind ? in.vals[ed.q] : 0.0, vt = int_ ? in.vals[et.q] : 0.0;
  if (c0 < 16 * nb) {
    double y[16], x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      y[c] = (lane >= nc || c0 + c >= nc) && c0 + c == lane ? 1.0 : 0.0;
      x[c] = 0.0;
    }
    add_children(L, lg, lane, lane, nc, c0, true, y);
    add_children(L, lt, lane, first + lane, first + nx, c0, false, x);
    for (int g = tl.dg0 + 64; g < tl.dg1; g += 64) {  // more than 64 children
      lg = lane_gathers(in, g, tl.dg1, lane);
      add_children(L, lg, lane, lane, nc, c0, true, y);
      if (tl.kind == 0) add_children(L, lg, lane, first + lane, first + nx, c0, false, x);
    }
    for (int g = tl.g0 + 64; tl.kind != 0 && g < tl.g1; g += 64)
      add_children(L, lane_gathers(in, g, tl.g1, lane), lane, first + lane, first + nx, c0, false, x);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      W[(c0 + c) * kWld + lane] = y[c];
      W[(c0 + c) * kWld + 64 + lane] = x[c];
    }
  }
  lds_barrier();
  auto put = [&](const swc::AEntry& e, double v, bool own) {
    const int i = e.pos & 63, j = e.pos >> 6;
    if (own) W[j * kWld + 64 + i] += v;
    else if (i < nc) W[j * kWld + i] += v;
    else if (tl.kind == 0) W[j * kWld + 64 + i - nc] += v;
  };
  if (ind) put(ed, vd, false);
  if (int_) put(et, vt, true);
  for (int e = ad + kThreads; e < tl.da1; e += kThreads) put(in.aents[e], in.vals[in.aents[e].q], false);
  for (int e = at + kThreads; tl.kind != 0 && e < tl.a1; e += kThreads)
    put(in.aents[e], in.vals[in.aents[e].q], true);
}

// A front of <= 64 rows, <= 16 columns and <= 48 rows below them (more blocks of U would
// not leave registers for two waves per SIMD), one wave: assembled (lane = row), factored in
// registers as panel_factor_regs_body does it, its U formed on MFMA from the panel in LDS.
// T: 64 x 17 doubles of the wave's own LDS (row i at T[17 i]).
constexpr int kSmallLds = 80 * 17;

template <int MODE, int NB>
__device__ inline void small_front_nb(double* __restrict__ L, const swc::SmallFront& f,
                                      const FrontIn& in, int* __restrict__ info_out,
                                      float* __restrict__ Lf, double* T, int lane) {
  constexpr int NC = 16;
  constexpr int NP = NB * (NB + 1) / 2;  // 16x16 blocks of U on and below the diagonal
  const int w = f.w, R = f.R, m = R - w;
  const int lr = lane & 15, lk = lane >> 4;
  // A and the children: entries and descriptors first, then every child's part of the
  // panel and of U (in flight while the panel is factored)
  swc::AEntry ae{0, 0};
  const bool ina = f.a0 + lane < f.a1;
  if (ina) ae = in.aents[f.a0 + lane];
  LaneGathers lg = lane_gathers(in, f.g0, f.g1, lane);
  const double va = ina ? in.vals[ae.q] : 0.0;
#pragma unroll
  for (int c = 0; c < NC; ++c) T[lane * (NC + 1) + c] = 0.0;
  wave_lds_sync();
  if (ina) T[(ae.pos & 63) * (NC + 1) + (ae.pos >> 6)] = va;
  for (int e = f.a0 + 64 + lane; e < f.a1; e += 64) {
    const swc::AEntry x = in.aents[e];
    T[(x.pos & 63) * (NC + 1) + (x.pos >> 6)] = in.vals[x.q];
  }
  double y[NC];
  d4 u[NP > 0 ? NP : 1];
#pragma unroll
  for (int c = 0; c < NC; ++c) y[c] = 0.0;
#pragma unroll
  for (int b = 0; b < NP; ++b) u[b] = d4{0.0, 0.0, 0.0, 0.0};
  for (int g0 = f.g0; g0 < f.g1; g0 += 64) {
    if (g0 > f.g0) lg = lane_gathers(in, g0, f.g1, lane);
    for (int e = 0; e < lg.n; ++e) {
      const swc::Gather ga = lane_gather(lg, e);
      const __amdgpu_buffer_rsrc_t rg = land_rsrc(L + ga.src);
      const unsigned ro = land_off(ga.rmask, lane, 8u);
      const unsigned cov = land_off(ga.cmask, lane, (unsigned)ga.ld * 8u);  // lane = column
      double v[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const unsigned co = __builtin_amdgcn_readlane(cov, c);
        v[c] = load_elem<double>(rg, c > lane || c >= w ? kNoLand : ro + co);
      }
      unsigned ui[NB > 0 ? NB : 1];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const unsigned o = __shfl(ro, (w + 16 * b + lr) & 63);
        ui[b] = 16 * b + lr < m ? o : kNoLand;
      }
#pragma unroll
      for (int bj = 0, p = 0; bj < NB; ++bj) {
        unsigned uj[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * bj + lk + 4 * r;
          const unsigned o = __shfl(cov, (w + j) & 63);
          uj[r] = j < m ? o : kNoLand;
        }
#pragma unroll
        for (int bi = bj; bi < NB; ++bi, ++p)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            u[p][r] += load_elem<double>(rg, bi == bj && lr < lk + 4 * r ? kNoLand : ui[bi] + uj[r]);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) y[c] += v[c];
    }
  }
  wave_lds_sync();
#pragma unroll
  for (int c = 0; c < NC; ++c) y[c] += T[lane * (NC + 1) + c];
  const int badcol = factor_rows<NC, false>(y, y, w, lane);
  if (badcol && lane == 0) atomicMin(info_out, f.c0 + badcol);
  double* gl = L + f.vbase;
  float* fl = Lf ? Lf + f.vbase : nullptr;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c < w && lane < R && c <= lane) {
      gl[(int64_t)c * R + lane] = y[c];
      if (fl) fl[(int64_t)c * R + lane] = (float)y[c];
    }
    T[lane * (NC + 1) + c] = c < w && lane < R ? y[c] : 0.0;
  }
  wave_lds_sync();
  // U = children - L21 L21^T (the column operand first: front_update_body)
  double* gu = L + f.ubase;
#pragma unroll
  for (int bj = 0, p = 0; bj < NB; ++bj)
#pragma unroll
    for (int bi = bj; bi < NB; ++bi, ++p) {
      const int ia = min(w + 16 * bi + lr, 63), ib = min(w + 16 * bj + lr, 63);
      d4 acc = d4{0.0, 0.0, 0.0, 0.0};
      if constexpr (MODE == 0) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(T[ib * (NC + 1) + lk + 4 * x],
                                                     T[ia * (NC + 1) + lk + 4 * x], acc, 0, 0, 0);
      } else {
        const int ibf = min(w + 16 * bj + (lr >> 2) + 4 * (lr & 3), 63);
        f4 c = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 4; ++x)
          c = __builtin_amdgcn_mfma_f32_16x16x4f32((float)T[ibf * (NC + 1) + lk + 4 * x],
                                                   (float)T[ia * (NC + 1) + lk + 4 * x], c, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += (double)c[r];
      }
      const int i = 16 * bi + lr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * bj + lk + 4 * r;
        if (i < m && j <= i) gu[(int64_t)j * f.ldu + i] = u[p][r] - acc[r];
      }
    }
}

template <int MODE>
__device__ inline void small_front_body(double* __restrict__ L, const swc::SmallFront& f,
                                        const FrontIn& in, int* __restrict__ info_out,
                                        float* __restrict__ Lf, double* T, int lane) {
  const int m = f.R - f.w;  // uniform
  if (m > 32) small_front_nb<MODE, 3>(L, f, in, info_out, Lf, T, lane);
  else if (m > 16) small_front_nb<MODE, 2>(L, f, in, info_out, Lf, T, lane);
  else small_front_nb<MODE, 1>(L, f, in, info_out, Lf, T, lane);
}

// One tile of a panel of <= 16 columns (panel_factor_regs_body after assembling it).
// T: 80 x 17 doubles of the wave's own LDS: the diagonal block's rows, then the tile's.
__device__ inline void front_narrow_body(double* __restrict__ L, const swc::FactorTile& tl,
                                         const FrontIn& in, const double* __restrict__ dscratch,
                                         int* __restrict__ info_out, float* __restrict__ Lf,
                                         double* T, int lane) {
  constexpr int NC = 16;
  const int nc = tl.ncol, first = tl.kind == 0 ? nc : 0;
  const bool mine = lane >= first && lane < tl.nr;
  double y[NC], x[NC];
  if (tl.first) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (lane < 16) T[c * 81 + lane] = 0.0;
      T[c * 81 + 16 + lane] = 0.0;
      y[c] = x[c] = 0.0;
    }
    const LaneGathers lg = lane_gathers(in, tl.dg0, tl.dg1, lane);
    const LaneGathers lt = tl.kind == 0 ? lg : lane_gathers(in, tl.g0, tl.g1, lane);
    wave_lds_sync();
    add_entries(in, tl.da0, tl.da1, T, 81, nc, tl.kind == 0, 16 + nc, lane, 64);
    if (tl.kind != 0) add_entries(in, tl.a0, tl.a1, T, 81, 0, true, 16, lane, 64);
    add_children(L, lg, lane, lane, nc, 0, true, y);
    add_children(L, lt, lane, mine ? lane : 64, 64, 0, false, x);
    for (int g = tl.dg0 + 64; g < tl.dg1; g += 64) {  // more than 64 children
      const LaneGathers l2 = lane_gathers(in, g, tl.dg1, lane);
      add_children(L, l2, lane, lane, nc, 0, true, y);
      if (tl.kind == 0) add_children(L, l2, lane, mine ? lane : 64, 64, 0, false, x);
    }
    for (int g = tl.g0 + 64; tl.kind != 0 && g < tl.g1; g += 64)
      add_children(L, lane_gathers(in, g, tl.g1, lane), lane, mine ? lane : 64, 64, 0, false, x);
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (lane < nc) y[c] += T[c * 81 + lane];
      if (mine) x[c] += T[c * 81 + 16 + lane];
    }
  } else {
    const double* gdiag = dscratch + tl.slot;
    const double* gt = L + tl.vbase + tl.r0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      y[c] = (lane < nc && c < nc && c <= lane) ? gdiag[c * nc + lane] : 0.0;
      x[c] = (mine && c < nc) ? gt[(int64_t)c * tl.ld + lane] : 0.0;
    }
  }
  panel_factor_regs_core<NC>(L, tl, info_out, Lf, lane, y, x);
}

// Lean launch for levels without panels of more than 16 columns, or with many narrow
// ones: one wave per workgroup, [0, nsmall) small fronts, then narrow tiles.
template <int MODE>
__global__ void __launch_bounds__(64)
k_front_narrow(double* __restrict__ L, const swc::SmallFront* __restrict__ small, int s0,
               int nsmall, const swc::FactorTile* __restrict__ ftiles, int f0, FrontIn in,
               const double* __restrict__ dscratch, int* __restrict__ info_out,
               float* __restrict__ Lf) {
  __shared__ double T[kSmallLds];
  if ((int)blockIdx.x < nsmall) {
    const swc::SmallFront f = small[s0 + blockIdx.x];
    small_front_body<MODE>(L, f, in, info_out, Lf, T, threadIdx.x);
  } else {
    const swc::FactorTile tl = ftiles[f0 + blockIdx.x - nsmall];
    front_narrow_body(L, tl, in, dscratch, info_out, Lf, T, threadIdx.x);
  }
}

// F launch of a level with wider panels: workgroups [0, ceil(nsmall / 4)) four small
// fronts each, then ceil(nn / 4) four narrow tiles each, then nw tiles of 17..64-column
// panels, then the tiles that the previous level deferred (updates nothing of this
// level waits for, beside the latency-bound factorization).
template <int MODE>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
k_front_factor(double* __restrict__ L, const swc::SmallFront* __restrict__ small, int s0,
               int nsmall, const swc::FactorTile* __restrict__ ftiles, int f0, int nn, int nw,
               const swc::FrontTile* __restrict__ utiles, int u0, FrontIn in,
               const double* __restrict__ dscratch, double* __restrict__ dscratch_u,
               int* __restrict__ info_out, float* Lf_factor, const float* __restrict__ Lf_update) {
  extern __shared__ __align__(16) double lds[];  // front_factor_lds() doubles
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b = blockIdx.x;
  const int bs = (nsmall + 3) >> 2, bn = (nn + 3) >> 2;
  if (b < bs) {
    const int k = 4 * b + wave;
    if (k < nsmall) {
      const swc::SmallFront f = small[s0 + k];
      small_front_body<MODE>(L, f, in, info_out, Lf_factor, lds + wave * kSmallLds, lane);
    }
    return;
  }
  b -= bs;
  if (b < bn) {
    const int k = 4 * b + wave;
    if (k < nn) {
      const swc::FactorTile tl = ftiles[f0 + k];
      front_narrow_body(L, tl, in, dscratch, info_out, Lf_factor, lds + wave * kSmallLds, lane);
    }
    return;
  }
  b -= bn;
  if (b < nw) {
    const swc::FactorTile tl = ftiles[f0 + nn + b];
    panel_factor_blk_body(L, tl, dscratch, info_out, Lf_factor, lds, tid, in);
  } else {
    const swc::FrontTile u = utiles[u0 + (b - nw)];
    front_update_body<MODE, false>(L, Lf_update, u, in, dscratch_u, lds, tid);
  }
}

// LDS (doubles) of k_front_factor: the widest panel's working matrix (16-column blocks),
// the one-wave items' buffers, the deferred tiles' entries of A, whichever takes most.  A
// level of panels of at most 32 columns takes half of what 64 columns need, so twice
// the workgroups fit on a CU.
inline size_t front_factor_lds(int nwave_items, int widest, int ndefer) {
  size_t d = 0;
  if (nwave_items) d = 4 * kSmallLds;
  if (widest) d = std::max(d, (size_t)((widest + 15) / 16 * 16 * kWld));
  if (ndefer) d = std::max(d, (size_t)kUpdateLds);
  return d * sizeof(double);
}
