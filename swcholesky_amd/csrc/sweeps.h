// Work lists of the triangular solves, built once per symbolic structure.
//
// Each sweep is one persistent launch whose workgroups claim items from a ticket counter
// in list order and pass each other only vector entries: an entry not yet computed holds
// a reserved bit pattern, and whoever needs it reads it again until it does not.  L is
// only read, so no cache is written back or invalidated inside the launch, and there are
// no launches per level.  Bound: the chain of 64-column panels (about 3 us each: an entry's
// way through memory, 64 substitution steps), above that HBM.  Per-level launches -> this
// (ms): 64^3, one right-hand side 4.58 (382 launches) -> 1.55, vector 48^3 with 32 28.4 ->
// 10.4, a 2D 100^2 solve alone 0.35 -> 0.08.
//
// List order is a topological order of the waits: an item waits only for entries that
// items before it produce.  An item in work has every earlier item claimed by a running
// workgroup, and the earliest unfinished one never waits for an unfinished one, so the
// launch cannot deadlock, whatever share of it is resident.
//
// A supernode of w columns and m rows below is cut into blocks of 64: column panels and
// row blocks [64 p, 64 p + 64) of its own rows ("own"), row blocks from row w ("below").
// Narrow supernodes (w <= 16, m <= kSmallRows) are one wave's work from start to finish; with
// more rows below the row blocks' items run side by side.  Limits of 256 / 1024 / 4096 rows
// (ms, one and 8 right-hand sides): 3000 single columns above a border of 600 0.69 / 0.27 / 0.27
// and 4.0 / 0.38 / 0.38, 1500 above a border of 2000 0.66 / 0.66 / 0.32 and 3.7 / 3.7 / 0.66.
#pragma once
#include <cstdint>
#include <vector>

namespace swc {

constexpr int kSmallRows = 4096;

// A narrow supernode.
struct SweepSmall {
  int64_t vbase;  // value offset of (row 0, column 0)
  int64_t voff;   // offset of its contribution vector
  int R, w, c0;   // rows, columns, first global column
  int rows_off;   // offset into Ls of its row 0
};

enum SweepKind {
  kSweepOwn = 0,    // forward: an own row block; backward: a column panel
  kSweepBelow = 1,  // forward: a row block below; backward: part of a panel's rows below
  kSweepSmall = 2   // narrow supernodes [first, first + count) of the small list
};

// Forward: rows [row0, row0 + nr) of the supernode, x of its panels 0 .. nq - 1 applied.
// Backward: columns [col0, col0 + nr) of panel p, over rows [row0, row1) below (by list)
// and, for a panel, own row blocks p + 1 .. np - 1; `parts` earlier-made partial sums.
struct SweepItem {
  int64_t vbase;  // value offset of the supernode's (row 0, column 0)
  int64_t out;    // forward below: V offset of row0; backward below: slot in the partials;
                  // backward own: first slot of its partials
  int ld, w, c0;  // the supernode's rows, width, first global column
  int kind;
  int p;          // own block / panel index
  int nr;
  int row0, row1;
  int nq;         // forward: panels to apply; backward own: number of partials
  int rows_off;   // offset into Ls of the supernode's row 0
  int first, count;  // small ones
};

struct SweepPlan {
  std::vector<SweepSmall> small;   // by level, ascending
  std::vector<int> lvl_small16;    // of those, first in their level: the ones taken 16 lanes each
  std::vector<int> lvl_small;      // small ones of the launches before the persistent one:
                                   // level l holds [lvl_small[l], lvl_small[l + 1])
  std::vector<SweepItem> fwd, bwd;
  int64_t psize = 0;               // doubles of backward partials per right-hand side
  int64_t one_each = 1;            // most right-hand sides that go one to an item
};

// Several right-hand sides go one to an item, or 16 to an item with L read once for them.
// The chain of an item with one is the shorter one, so that is better while the longest chain
// is what takes the time: while the right-hand sides together read no more of L per step of it
// (a 64-column panel, or 64 entries of a column's list of contributions, about 3 us) than comes
// from memory meanwhile, 12 MB, and their chains, where a step is an item of its own, are no
// more than 300, beyond which they wait for each other's places on the device.  One against
// 16 to an item (ms): 24^3 with 16 right-hand sides 0.46 and 0.54, with 33 0.76 and 0.58; 48^3
// with 2 0.92 and 1.35, with 8 2.04 and 1.63; 600 2D instances with 2 0.94 and 0.97, with 3 1.23
// and 1.08; tridiagonal 20,000 in natural order with 300 8.6 and 9.5, with 400 11.5 and 9.6; an
// arrow with a border of 30 with 2 0.93 and 4.8.
constexpr int64_t kStepBytes = 12000000, kChains = 300;
inline bool sweep_by_16(const SweepPlan& W, int nrhs) { return nrhs > 1 && nrhs > W.one_each; }

// Level of every supernode: one above the highest of those whose rows below meet its
// columns.  From the row lists, which say what the sweeps (and the selected inverse) read and
// wait for; a caller's descendant sets may leave out a supernode whose rows hold only zeros.
std::vector<int> supernode_levels(int nsuper, const int* super, const int64_t* pi, const int* Ls);

// voff[s]: offset of the contribution vector of s; gptr: offsets of the columns' lists of
// contributions.  maxpart: most doubles of partials.
void build_sweeps(int nsuper, const int* super, const int64_t* pi, const int64_t* px, const int* Ls,
                  const int64_t* voff, const int64_t* gptr, int64_t maxpart, SweepPlan& W);

}  // namespace swc
