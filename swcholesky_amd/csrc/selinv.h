// Work lists of the selected inverse, built once per symbolic structure.
//
// Z = A^{-1} on the pattern of L, supernode J with L = [L11; L21] (w columns, m rows R
// below), root level first:
//   T = L11^{-1},  U = L21 T               from L alone
//   Z21 = -Z(R,R) U                        Z(R,R) read from the ancestors' Z
//   Z11 = T^T T - U^T Z21
// T and U wait for no other supernode: they are made for a whole chunk of levels in four
// launches (64 x 64 diagonal blocks, those of at most 16 columns, columns of blocks below
// them, U), so that only the last two steps follow the chain of levels, three launches a
// level.  A chunk holds as many
// levels as fit kSelChunk values (its T and U are read again soon, from the caches), and at
// least one.  One thread per entry in four launches a level before, with every entry's own
// serial sum, -> this: 3.9 -> 0.54 ms on a 256^2 GMRF (65,536 unknowns, 13 levels; 0.16 ms
// of it T and U, whose wide root is a chain of six blocks).  Narrow supernodes with few rows (kSelSmallW, kSelSmallM) are one workgroup's
// work in one launch.
#pragma once
#include <cstdint>
#include <vector>

namespace swc {

constexpr int kSelTile = 32;     // output tile of a product
constexpr int kSelBlock = 64;    // block of T = L11^{-1}
constexpr int kSelSmallW = 16;   // a small supernode: w and m at most these; its Z(R,R), U
constexpr int kSelSmallM = 64;   // and Z21 fit the LDS of a workgroup, one lane a row
constexpr int kSelRunCols = 16;  // columns of a gather item
constexpr int kSelRows = 256;    // rows of a gather item, one thread each
constexpr int64_t kSelChunk = 1 << 23;  // 64 MB of T and U

struct SelNode {
  int64_t vbase;  // value offset of (row 0, column 0), ld = nrow
  int64_t moff;   // [T; U], row major, ld = w
  int64_t zoff;   // Z(R,R), m x m; -1 for a small supernode
  int w, nrow;
  int rows_off;   // offset into Ls of its row 0
  int run0;       // its first run
};

// Columns j0 .. j0 + nj - 1 of Z(R,R) that are columns of one ancestor K: entry (i, j) is
// Z[zbase + R(j) ld + rel[i]], R(j) the global column, rel[i] the place of row i of R in
// K's row list (rel = the run's part of the positions, entries below j0 unused).
struct SelRun {
  int64_t zbase;  // K's value offset less its first column's ld
  int64_t rel;
  int j0, nj, ld;
  int rows_off;  // offset into Ls of K's row 0
  int node;
  int pad;
};

struct SelItem {
  int node, a, b, c;
};

struct SelPlan {
  std::vector<SelNode> nodes;  // root level first
  std::vector<SelRun> runs;
  std::vector<int> jrun;  // per row below (rows_off + w + j): its run
  int64_t nrel = 0, msize = 0, zsize = 0;
  std::vector<SelItem> diag, diag16, cols, u;     // by chunk: {node, block} (16: <= 16 rows), {node, block column}, {node, row, column}
  std::vector<SelItem> gather, small, z21, z11;   // by level: {run, j, i}, {node}, {node, row, column}
  std::vector<int> chunk_diag, chunk_diag16, chunk_cols, chunk_u;  // offsets per chunk
  std::vector<int> chunk_lvl;                        // first level of each chunk, one more at the end
  std::vector<int> lvl_gather, lvl_small, lvl_z21, lvl_z11, lvl_m;  // lvl_m: most rows below of a small supernode
};

// ns supernodes: super (first columns, ns + 1), pi (row list offsets), px (value offsets),
// rows Ls.
SelPlan build_selinv(int n, int ns, const int* super, const int64_t* pi, const int64_t* px,
                     const int* Ls);

}  // namespace swc
