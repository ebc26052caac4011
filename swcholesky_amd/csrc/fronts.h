// Multifrontal factorization plan: the device work lists of the default factor
// schedule, built once per symbolic structure.
//
// Every supernode s (w columns, R rows, m = R - w rows below) has, beside its
// block of L, a frontal update matrix U_s (m x m, lower triangle, column-major) in
// an arena, whose offsets count on behind L's (rounded up to 32 values):
//   U_s = (sum over children c of U_c at their landing positions) - L21 L21^T,
// and a supernode's own columns start from A plus the children's U_c.  So every
// product is a dense block of one supernode (rows consecutive, inner dimension the
// supernode's columns), and what a supernode passes up the tree is read once per
// ancestor level by its parent alone.  The left-looking plan (plan.h) instead
// applies every descendant's product to every tile it reaches: its products land
// sparsely in the tiles (about 57% full at the top of a 64^3 grid) and a tile near
// the root runs through a serial list of hundreds of short products.  Factor + solve,
// left-looking -> multifrontal (ms, same solve): 64^3 26.6 -> 21.4, 32^3 mixed 6.01 ->
// 4.94, 2D 100^2 1.04 -> 0.68, a mesh of 20,000 points 2.11 -> 1.41, 256 uneven 2D
// instances 4.69 -> 2.81.  The arena takes about as much memory as L (1.5 GB beside
// 1.6 GB at 64^3) and holds nothing between factorizations, so the handle gives it up first
// when the device has no room.
//
// A supernode is cut into panels of at most 64 columns, its rows into tiles of at
// most 64.  Level l runs two launches: F_l factors the panels of level l (a first
// panel is assembled there, from A and the children), U_l applies them to the later
// panels and to U_s.  Every entry is summed in a fixed order that depends on its own
// supernode and children only.
#pragma once
#include <cstdint>
#include <vector>

namespace swc {

// A child's U landing in one tile: the e-th set bit of rmask is the tile row that
// U row e (counted from src) lands on, the e-th set bit of cmask the tile column
// that U column e lands on.
struct Gather {
  int64_t src;  // value offset of the child's first landing row and column
  int ld;
  int pad;
  uint64_t rmask, cmask;
};

// An entry of A in a tile: value q, tile position row + 64 column.
struct AEntry {
  int q;
  int pos;
};

// One update of one tile (U launch): target -= A B^T over k source columns, both
// operands rows of the tile's own supernode.
struct FrontTile {
  int64_t vbase;  // value offset of the tile's (row 0, column 0)
  int64_t asrc;   // value offset of the first source column at the tile's row 0
  int64_t bsrc;   // ... at the row of the tile's column 0
  int ld, sld;    // leading dimensions of target and source
  int k;
  int nr, nc;
  int diag;       // 1: only rows >= columns exist
  int first;      // 1: the tile is assembled here (gathers, entries of A) and not read
  int upd;        // 1: a tile of U (a descendant update), 0: of the supernode's own columns
  int g0, g1;     // [g0, g1) gathers, first touch only
  int a0, a1;     // [a0, a1) entries of A, first touch only
  int slot;       // >= 0: a copy of the diagonal block for the next factor launch goes here
  int row;        // tile row it is (its column: row - (asrc - bsrc) / 64), for the order of a launch
};

// One tile of a panel being factored (F launch); fields named as in Tile.
struct FactorTile {
  int64_t vbase;  // the panel's value offset of (row 0, column 0)
  int r0, nr, kind, slot, ld, ncol, c0;
  int first;      // 1: assembled here from the lists below
  int g0, g1, a0, a1;      // the tile's
  int dg0, dg1, da0, da1;  // the diagonal tile's
};

// A front of at most 64 rows, 16 columns and 48 rows below them: assembled, factored and
// its U formed by one wave.  Its gathers carry one mask over the front's rows (rmask = cmask).
struct SmallFront {
  int64_t vbase, ubase;
  int R, w, ldu, c0;
  int g0, g1, a0, a1;
};

struct FrontPlan {
  int nlevel = 0;
  int64_t usize = 0;         // doubles of the U arena
  int64_t diag_scratch = 0;  // doubles of diagonal-block copies
  int64_t npanel = 0;
  std::vector<Gather> gathers;
  std::vector<AEntry> aents;
  std::vector<FactorTile> ftiles;   // by level: panels of <= 16 columns, then the others
  std::vector<int> lvl_f, lvl_fn;   // nlevel+1 offsets; nlevel: narrow ones first in their level
  std::vector<int> lvl_widest;      // nlevel: widest panel of the others (0: none)
  std::vector<SmallFront> small;    // by level
  std::vector<int> lvl_small;       // nlevel+1
  std::vector<FrontTile> utiles;    // by level
  std::vector<int> lvl_u;           // nlevel+1
  std::vector<int> lvl_ud;          // nlevel: deferred tiles, last in their level: they run in the
                                    // next level's F launch
  std::vector<int> lvl_kmax;        // nlevel: most source columns of a tile of U_l
  std::vector<double> lvl_flops;    // useful flops of U_l
  double update_flops = 0, factor_flops = 0;
};

// pos[e]: position of A2 entry e's row in its supernode's row list; src: the input
// value of each A2 entry (null: its own index).  Returns false (plan untouched
// beyond use) for a structure whose supernodes do not pass their rows up one tree:
// a supernode's rows below its columns that are not all rows of the supernode owning
// the first of them, or descendant sets that are not those of the row lists; and for one
// whose update matrices are not worth their size.
bool build_fronts(int n, int nsuper, const int* super, const int64_t* pi, const int64_t* px,
                  int64_t xsize, const int* Ls, const int* prunePtr, const int* pruneSet,
                  const int* A2p, const int64_t* src, const int* pos, int rlb, FrontPlan& F);

}  // namespace swc
