// Builds the multifrontal factorization plan (see fronts.h).
#include "fronts.h"

#include <algorithm>
#include <map>
#include <memory>
#include <tuple>

namespace swc {

namespace {

constexpr int T = 64;  // panel width and tile height

// First-fit arena over levels: blocks live from the level that writes them to the
// level that last reads them.
class Arena {
 public:
  int64_t take(int64_t len) {
    for (auto it = free_.begin(); it != free_.end(); ++it)
      if (it->second >= len) {
        const int64_t at = it->first, left = it->second - len;
        free_.erase(it);
        if (left) free_[at + len] = left;
        return at;
      }
    const int64_t at = end_;
    end_ += len;
    return at;
  }
  void give(int64_t at, int64_t len) {
    auto it = free_.emplace(at, len).first;
    auto nx = std::next(it);
    if (nx != free_.end() && it->first + it->second == nx->first) {
      it->second += nx->second;
      free_.erase(nx);
    }
    if (it != free_.begin()) {
      auto pv = std::prev(it);
      if (pv->first + pv->second == it->first) {
        pv->second += it->second;
        free_.erase(it);
      }
    }
  }
  int64_t size() const { return end_; }

 private:
  std::map<int64_t, int64_t> free_;
  int64_t end_ = 0;
};

}  // namespace

// Orders a launch's tiles (sorted by k) so that workgroups of one XCD, which share an L2
// and get every eighth workgroup, work on square groups of neighbouring tiles: side * side
// tiles read 2 side operand blocks, a run down a column of tiles 1 + side^2.  A group goes
// to the XCD with the least work so far.  Groups of 8 x 8 tiles need 16 blocks of 64 rows,
// up to 4 MB at k = 512, what an L2 holds; a launch of few tiles gets smaller groups, so
// that every XCD has several, and keeps its order below 4 x 64 tiles.
static void order_for_xcds(std::vector<FrontTile>& tiles) {
  constexpr int kXcds = 8;
  const int n = (int)tiles.size();
  int side = 1;
  while (side < 8 && (side + 1) * (side + 1) * 64 <= n) ++side;
  if (side == 1) return;
  struct Group {
    int k;
    std::vector<int> tiles;
  };
  std::vector<Group> groups;
  std::map<std::tuple<int64_t, int, int, int>, int> index;
  for (int i = 0; i < n; ++i) {
    const FrontTile& u = tiles[i];
    const int col = u.row - (int)((u.asrc - u.bsrc) / T);
    // supernode, step and kind have one source offset of tile row 0
    const auto key = std::make_tuple(u.asrc - (int64_t)T * u.row, u.k, u.row / side, col / side);
    const auto it = index.emplace(key, (int)groups.size());
    if (it.second) groups.push_back({u.k, {}});
    groups[it.first->second].tiles.push_back(i);
  }
  std::vector<int> queue[kXcds];
  int64_t load[kXcds] = {};
  for (const Group& g : groups) {  // in order of decreasing k
    const int x = (int)(std::min_element(load, load + kXcds) - load);
    load[x] += (int64_t)g.tiles.size() * (g.k + 32);
    queue[x].insert(queue[x].end(), g.tiles.begin(), g.tiles.end());
  }
  std::vector<FrontTile> out;
  out.reserve(n);
  size_t at[kXcds] = {};
  for (int i = 0; (int)out.size() < n; ++i) {
    int x = i % kXcds;
    if (at[x] == queue[x].size())  // its queue has run out: from the longest
      for (int y = 0; y < kXcds; ++y)
        if (queue[y].size() - at[y] > queue[x].size() - at[x]) x = y;
    out.push_back(tiles[queue[x][at[x]++]]);
  }
  tiles.swap(out);
}

// The update matrices take about as much as L (1.2 times at most on grids, meshes and dense
// matrices), but far more where many small supernodes lie below a wide border: every one of
// them then writes the border's whole triangle and the border reads it (16 bytes an entry at
// 4.3 TB/s), while the left-looking plan runs through the border's descendants one after
// another, about 3 us each, but takes longer over the border itself.  Factorizations, left-
// looking and multifrontal (ms), of single columns below a border: 300 x 600 (arena 199 times
// L) 1.34 and 1.18, 300 x 1000 (230) 1.74 and 2.07, 300 x 2000 (260) 3.2 and 4.0, 1000 x 1000
// (499) 3.6 and 5.8, 1500 x 2000 (30 GB) 5.7 and 13.8, but 30 x 4000 (29) 4.7 and 3.4, and by the
// longer chain 3000 x 600 (443) 8.8 and 7.2.  More than 4 times L takes 32 GiB at most.
static bool arena_pays(int64_t usize, int64_t xsize, int nsuper, const int* prunePtr) {
  if (usize <= 4 * xsize) return true;
  if (usize > (int64_t)1 << 32) return false;
  int most = 0;  // descendants of one supernode
  for (int s = 0; s < nsuper; ++s) most = std::max(most, prunePtr[s + 1] - prunePtr[s]);
  return usize <= 200 * xsize || 16.0 * (double)usize / 4.3e6 <= 3.0 * most;
}

bool build_fronts(int n, int nsuper, const int* super, const int64_t* pi, const int64_t* px,
                  int64_t xsize, const int* Ls, const int* prunePtr, const int* pruneSet,
                  const int* A2p, const int64_t* src, const int* pos, int rlb, FrontPlan& F) {
  std::vector<int> col2sup(n);
  for (int s = 0; s < nsuper; ++s)
    for (int c = super[s]; c < super[s + 1]; ++c) col2sup[c] = s;
  auto width = [&](int s) { return super[s + 1] - super[s]; };
  auto nrows = [&](int s) { return (int)(pi[s + 1] - pi[s]); };

  // ---- the tree, and where each supernode's rows land in its parent's ----
  // rel[roff[s] + j] = position of row w + j of s in the parent's row list
  std::vector<int> parent(nsuper, -1);
  std::vector<int64_t> roff(nsuper + 1, 0);
  for (int s = 0; s < nsuper; ++s) {
    // the kernels' 32-bit tile offsets reach 64 columns of this many rows
    if (nrows(s) > 2000000) return false;
    roff[s + 1] = roff[s] + nrows(s) - width(s);
  }
  std::vector<int> rel((size_t)roff[nsuper]);
  std::vector<int> nchild(nsuper + 1, 0);
  int64_t npairs = 0;  // (descendant, ancestor it updates)
  for (int s = 0; s < nsuper; ++s) {
    const int w = width(s), m = nrows(s) - w;
    if (m == 0) continue;
    const int* rows = Ls + pi[s] + w;
    const int p = col2sup[rows[0]];
    parent[s] = p;
    nchild[p + 1]++;
    const int* prow = Ls + pi[p];
    const int plen = nrows(p);
    int* out = rel.data() + roff[s];
    // the parent's own columns are consecutive: no search below its width
    const int pw = width(p);
    int j = 0;
    for (; j < m && rows[j] < super[p + 1]; ++j) out[j] = rows[j] - super[p];
    for (int i = pw; j < m; ++j) {
      while (i < plen && prow[i] < rows[j]) ++i;
      if (i == plen || prow[i] != rows[j]) return false;
      out[j] = i;
    }
    for (j = 0; j < m; ++npairs) {
      const int q = col2sup[rows[j]];
      while (j < m && rows[j] < super[q + 1]) ++j;
    }
  }
  if ((int64_t)prunePtr[nsuper] != npairs) return false;
  // the same sets, not only as many: every listed descendant once, meeting the supernode
  std::vector<int> seen(nsuper, -1);
  for (int s = 0; s < nsuper; ++s)
    for (int t = prunePtr[s]; t < prunePtr[s + 1]; ++t) {
      const int d = pruneSet[t];
      if (d < 0 || d >= s || seen[d] == s) return false;
      seen[d] = s;
      const int* r0 = Ls + pi[d] + width(d);
      const int* r1 = Ls + pi[d + 1];
      const int* it = std::lower_bound(r0, r1, super[s]);
      if (it == r1 || *it >= super[s + 1]) return false;
    }
  for (int s = 0; s < nsuper; ++s) nchild[s + 1] += nchild[s];
  std::vector<int> child((size_t)nchild[nsuper]);
  {
    std::vector<int> fill(nchild.begin(), nchild.end() - 1);
    for (int s = 0; s < nsuper; ++s)
      if (parent[s] >= 0) child[fill[parent[s]]++] = s;
  }

  // ---- levels: panel p of s at level start + p; a parent after its children ----
  auto npan = [&](int s) { return (width(s) + T - 1) / T; };
  std::vector<int> start(nsuper, 0);
  F.nlevel = 0;
  for (int s = 0; s < nsuper; ++s) {
    const int end = start[s] + npan(s);
    F.nlevel = std::max(F.nlevel, end);
    if (parent[s] >= 0) start[parent[s]] = std::max(start[parent[s]], end);
  }
  std::vector<int> by_start(nsuper), lvl_s(F.nlevel + 1, 0);
  for (int s = 0; s < nsuper; ++s) lvl_s[start[s] + 1]++;
  for (int l = 0; l < F.nlevel; ++l) lvl_s[l + 1] += lvl_s[l];
  {
    std::vector<int> fill(lvl_s.begin(), lvl_s.end() - 1);
    for (int s = 0; s < nsuper; ++s) by_start[fill[start[s]]++] = s;
  }

  // ---- the arena: U_s lives from its first pass (the end of the first block of rlb
  // panels) until the parent's first block has ended (by then every tile of the
  // parent has been assembled), and one level more for deferred tiles.  Supernodes of
  // one lifetime share a block (a batch has millions of supernodes, few lifetimes) ----
  std::vector<int64_t> ux(nsuper, -1);
  auto ldu_of = [&](int s) { return (nrows(s) - width(s) + 7) & ~7; };
  {
    struct Life {
      std::vector<int> sn;
      int64_t len = 0, at = 0;
    };
    std::vector<std::map<int, Life>> born(F.nlevel);  // by level, then by the level it ends
    std::vector<std::vector<const Life*>> dead(F.nlevel + 1);
    for (int s = 0; s < nsuper; ++s) {
      if (parent[s] < 0) continue;
      const int p = parent[s];
      Life& f = born[start[s] + std::min(npan(s), rlb) - 1]
                    [std::min(F.nlevel, start[p] + std::min(npan(p), rlb) + 1)];
      f.sn.push_back(s);
    }
    Arena ar;
    const int64_t ubase = (xsize + 31) & ~(int64_t)31;
    for (int l = 0; l < F.nlevel; ++l) {
      for (const Life* f : dead[l]) ar.give(f->at, f->len);
      for (auto& [end, f] : born[l]) {
        for (int s : f.sn) {
          ux[s] = f.len;
          f.len += (int64_t)ldu_of(s) * (nrows(s) - width(s));
        }
        f.at = ar.take(f.len);
        for (int s : f.sn) ux[s] += ubase + f.at;
        dead[end].push_back(&f);
      }
    }
    F.usize = ar.size() ? ubase - xsize + ar.size() : 0;
    if (!arena_pays(F.usize, xsize, nsuper, prunePtr)) return false;
  }

  // ---- entries of A by tile of L: tile (panel p, row tile t) of s ----
  std::vector<int64_t> tbase(nsuper + 1, 0);
  auto ltiles = [&](int s) {  // tiles of all panels
    const int64_t nt = (nrows(s) + T - 1) / T, np = npan(s);
    return np * nt - np * (np - 1) / 2;
  };
  for (int s = 0; s < nsuper; ++s) tbase[s + 1] = tbase[s] + ltiles(s);
  auto tile_id = [&](int s, int p, int t) {
    const int64_t nt = (nrows(s) + T - 1) / T;
    return tbase[s] + p * nt - (int64_t)p * (p - 1) / 2 + t;
  };
  const int64_t nnz = A2p[n];
  std::vector<int> aptr((size_t)tbase[nsuper] + 1, 0);
  F.aents.resize((size_t)nnz);
  {
    // the first tile of column j's panel, less its row tile
    auto base = [&](int j) {
      const int s = col2sup[j], p = (j - super[s]) / T;
      return tile_id(s, p, 0) - p;
    };
    for (int j = 0; j < n; ++j) {
      int* cnt = aptr.data() + base(j) + 1;
      for (int e = A2p[j]; e < A2p[j + 1]; ++e) cnt[pos[e] / T]++;
    }
    for (size_t i = 1; i < aptr.size(); ++i) aptr[i] += aptr[i - 1];
    std::vector<int> fill(aptr.begin(), aptr.end() - 1);
    for (int j = 0; j < n; ++j) {
      const int col = T * ((j - super[col2sup[j]]) % T);
      int* at = fill.data() + base(j);
      for (int e = A2p[j]; e < A2p[j + 1]; ++e)
        F.aents[at[pos[e] / T]++] = {(int)(src ? src[e] : e), pos[e] % T + col};
    }
  }

  // ---- gathers of one supernode's tiles ----
  struct Cut {
    int lo;
    uint64_t mask;
  };
  // The children's rows by blocks of 64 of the supernode's rows from one row on, and the
  // children with rows in each block: a supernode of thousands of small children, each in
  // few of its blocks, has a tile ask only those (the upload of a tree of 30,000 points whose
  // root has 3434 columns: 15.0 ms with every child asked, 4.7 now).
  struct Cuts {
    std::vector<std::vector<Cut>> of;     // by child
    std::vector<std::vector<int>> child;  // by block, ascending
  };
  Cuts cl, cu;  // from row 0, and from row w
  auto cut = [&](int s, int from, int len, Cuts& out) {
    const int nch = nchild[s + 1] - nchild[s], nb = (len + T - 1) / T;
    if ((int)out.of.size() < nch) out.of.resize(nch);
    if ((int)out.child.size() < nb) out.child.resize(nb);
    for (int b = 0; b < nb; ++b) out.child[b].clear();
    for (int k = 0; k < nch; ++k) {
      const int c = child[nchild[s] + k];
      const int* r = rel.data() + roff[c];
      const int m = (int)(roff[c + 1] - roff[c]);
      std::vector<Cut>& of = out.of[k];
      of.assign(nb, Cut{});
      for (int e = int(std::lower_bound(r, r + m, from) - r); e < m;) {
        const int b = (r[e] - from) / T;
        of[b].lo = e;
        for (; e < m && r[e] < from + T * (b + 1); ++e) of[b].mask |= 1ull << (r[e] - from - T * b);
        out.child[b].push_back(k);
      }
    }
  };
  auto add_gathers = [&](int s, const Cuts& cuts, int I, int J, int nc) {
    const uint64_t keep = nc >= 64 ? ~0ull : (1ull << nc) - 1;
    for (int k : cuts.child[cuts.child[I].size() <= cuts.child[J].size() ? I : J]) {
      const int c = child[nchild[s] + k];
      const Cut &rc = cuts.of[k][I], &cc = cuts.of[k][J];
      const uint64_t rm = rc.mask, cm = cc.mask & keep;
      if (!rm || !cm) continue;
      const int ld = ldu_of(c);
      F.gathers.push_back({ux[c] + rc.lo + (int64_t)cc.lo * ld, ld, 0, rm, cm});
    }
  };

  // ---- tiles, by the level of their launch ----
  struct Lvl {
    std::vector<FactorTile> fn, fw;
    std::vector<FrontTile> uc, ud;  // critical, deferrable
    std::vector<SmallFront> small;
  };
  std::vector<Lvl> lv(F.nlevel);
  for (int l0 = 0; l0 < F.nlevel; ++l0)
    for (int bi = lvl_s[l0]; bi < lvl_s[l0 + 1]; ++bi) {
      const int s = by_start[bi], w = width(s), R = nrows(s), m = R - w, np = npan(s);
      const int nt = (R + T - 1) / T, ntu = (m + T - 1) / T, ldu = ldu_of(s);
      cut(s, 0, R, cl);
      cut(s, w, m, cu);
      F.npanel += np;
      const double dw = w, dm = m;
      F.factor_flops += dw * dw * dw / 3.0 + dm * dw * dw;
      if (R <= T && w <= 16 && m <= 48) {
        SmallFront f{};
        f.vbase = px[s];
        f.ubase = m ? ux[s] : 0;
        f.R = R;
        f.w = w;
        f.ldu = ldu;
        f.c0 = super[s];
        f.g0 = (int)F.gathers.size();
        add_gathers(s, cl, 0, 0, 64);
        f.g1 = (int)F.gathers.size();
        f.a0 = aptr[tbase[s]];
        f.a1 = aptr[tbase[s] + 1];
        lv[l0].small.push_back(f);
        F.update_flops += dw * dm * (dm + 1);
        continue;
      }
      // factor tiles of panel p, at its level
      for (int p = 0; p < np; ++p) {
        const int nc = std::min(T, w - T * p);
        FactorTile d{};
        for (int t = 0; t < nt - p; ++t) {
          FactorTile f{};
          f.vbase = px[s] + (int64_t)T * p * R + T * p;
          f.r0 = T * t;
          f.nr = std::min(T, R - T * p - T * t);
          f.kind = t == 0 ? 0 : 1;
          f.slot = -1;
          f.ld = R;
          f.ncol = nc;
          f.c0 = super[s] + T * p;
          f.first = p == 0;
          if (f.first) {
            f.g0 = (int)F.gathers.size();
            add_gathers(s, cl, t, 0, nc);
            f.g1 = (int)F.gathers.size();
            f.a0 = aptr[tile_id(s, 0, t)];
            f.a1 = aptr[tile_id(s, 0, t) + 1];
            if (t == 0) d = f;
            f.dg0 = d.g0;
            f.dg1 = d.g1;
            f.da0 = d.a0;
            f.da1 = d.a1;
          }
          Lvl& L = lv[l0 + p];
          (nc <= 16 ? L.fn : L.fw).push_back(f);
        }
      }
      // updates: step p, over blocks of rlb panels
      for (int p = 0; p < np; ++p) {
        Lvl& L = lv[l0 + p];
        const int b0 = p - p % rlb, b1 = std::min(b0 + rlb, np);
        const bool last = p + 1 == b1;
        const int q0 = last ? b0 : p;  // source panels q0 .. p
        const int k = std::min(w, T * (p + 1)) - T * q0;
        const int64_t sbase = px[s] + (int64_t)T * q0 * R;
        const bool first = q0 == 0 && p < rlb && (last || p == 0);
        for (int q = p + 1; q < (last ? np : b1); ++q)
          for (int t = 0; t < nt - q; ++t) {
            FrontTile u{};
            u.vbase = px[s] + (int64_t)T * q * R + T * (q + t);
            u.asrc = sbase + T * (q + t);
            u.bsrc = sbase + T * q;
            u.ld = u.sld = R;
            u.k = k;
            u.nr = std::min(T, R - T * (q + t));
            u.nc = std::min(T, w - T * q);
            u.diag = t == 0;
            u.row = q + t;
            u.slot = -1;
            // the panels of the first block are first touched by panel 0, the later
            // ones by the whole first block
            u.first = first && (q < b1 ? p == 0 : true);
            if (u.first) {
              u.g0 = (int)F.gathers.size();
              add_gathers(s, cl, q + t, q, u.nc);
              u.g1 = (int)F.gathers.size();
              u.a0 = aptr[tile_id(s, q, t)];
              u.a1 = aptr[tile_id(s, q, t) + 1];
            }
            if (q == p + 1 && t == 0) u.slot = 0;  // numbered below
            (q == p + 1 ? L.uc : L.ud).push_back(u);
          }
        if (last)
          for (int b = 0; b < ntu; ++b)
            for (int a = b; a < ntu; ++a) {
              FrontTile u{};
              u.vbase = ux[s] + (int64_t)T * b * ldu + T * a;
              u.asrc = sbase + w + T * a;
              u.bsrc = sbase + w + T * b;
              u.ld = ldu;
              u.sld = R;
              u.k = k;
              u.nr = std::min(T, m - T * a);
              u.nc = std::min(T, m - T * b);
              u.diag = a == b;
              u.row = a;
              u.upd = 1;
              u.slot = -1;
              u.first = q0 == 0;
              if (u.first) {
                u.g0 = (int)F.gathers.size();
                add_gathers(s, cu, a, b, u.nc);
                u.g1 = (int)F.gathers.size();
              }
              (p + 1 == np ? L.uc : L.ud).push_back(u);
            }
      }
    }

  // ---- flatten ----
  F.lvl_f.assign(F.nlevel + 1, 0);
  F.lvl_fn.assign(F.nlevel, 0);
  F.lvl_widest.assign(F.nlevel, 0);
  F.lvl_small.assign(F.nlevel + 1, 0);
  F.lvl_u.assign(F.nlevel + 1, 0);
  F.lvl_ud.assign(F.nlevel, 0);
  F.lvl_flops.assign(F.nlevel, 0.0);
  F.lvl_kmax.assign(F.nlevel, 0);
  auto flops = [](const FrontTile& u) {
    const double pairs = u.diag ? u.nc * (u.nc + 1) / 2.0 + (double)(u.nr - u.nc) * u.nc
                                : (double)u.nr * u.nc;
    return 2.0 * pairs * u.k;
  };
  for (int l = 0; l < F.nlevel; ++l) {
    Lvl& L = lv[l];
    // Deferred tiles overlap the next level's panel factorization.  It pays where the
    // critical ones are light; the launch durations are estimated as for the
    // left-looking levels (plan.cpp).
    auto us = [&](const FrontTile& u) { return 3.0 + 1.4 * flops(u) / 1e5; };
    double cm = 0, cs = 0, dm = 0, ds = 0;
    for (const FrontTile& u : L.uc) {
      cm = std::max(cm, us(u));
      cs += us(u);
    }
    for (const FrontTile& u : L.ud) {
      dm = std::max(dm, us(u));
      ds += us(u);
    }
    auto span = [](double mx, double sum) { return std::max(mx, sum / 512 + 0.5 * mx); };
    const bool defer = ds > 0 && l + 1 < F.nlevel &&
                       span(cm, cs) + std::max(20.0, span(dm, ds)) <
                           0.95 * (span(std::max(cm, dm), cs + ds) + 20.0);
    if (!defer) {
      L.uc.insert(L.uc.end(), L.ud.begin(), L.ud.end());
      L.ud.clear();
    }
    auto heavier = [](const FrontTile& a, const FrontTile& b) { return a.k > b.k; };
    std::stable_sort(L.uc.begin(), L.uc.end(), heavier);
    std::stable_sort(L.ud.begin(), L.ud.end(), heavier);
    if (!L.uc.empty()) F.lvl_kmax[l] = L.uc.front().k;
    order_for_xcds(L.uc);
    // diagonal copies: made by U_l, read by F_{l+1}
    int64_t off = 0;
    std::vector<std::pair<int64_t, int>> slots;  // panel's value offset -> slot
    for (FrontTile& u : L.uc)
      if (u.slot >= 0) {
        u.slot = (int)off;
        slots.push_back({u.vbase, (int)off});
        off += (int64_t)u.nc * u.nc;
      }
    F.diag_scratch = std::max(F.diag_scratch, off);
    std::sort(slots.begin(), slots.end());
    if (l + 1 < F.nlevel)
      for (auto* v : {&lv[l + 1].fn, &lv[l + 1].fw})
        for (FactorTile& f : *v)
          if (!f.first) {
            auto it = std::lower_bound(slots.begin(), slots.end(), std::make_pair(f.vbase, -1));
            f.slot = it->second;
          }
    F.lvl_ud[l] = (int)L.ud.size();
    for (auto* v : {&L.uc, &L.ud}) {
      for (const FrontTile& u : *v) F.lvl_flops[l] += flops(u);
      F.utiles.insert(F.utiles.end(), v->begin(), v->end());
    }
    F.update_flops += F.lvl_flops[l];
    F.lvl_u[l + 1] = (int)F.utiles.size();
    F.lvl_fn[l] = (int)L.fn.size();
    for (const FactorTile& f : L.fw) F.lvl_widest[l] = std::max(F.lvl_widest[l], f.ncol);
    F.ftiles.insert(F.ftiles.end(), L.fn.begin(), L.fn.end());
    F.ftiles.insert(F.ftiles.end(), L.fw.begin(), L.fw.end());
    F.lvl_f[l + 1] = (int)F.ftiles.size();
    F.small.insert(F.small.end(), L.small.begin(), L.small.end());
    F.lvl_small[l + 1] = (int)F.small.size();
  }
  return true;
}

}  // namespace swc

// ---- host-only introspection (C ABI) ----
#include <cstring>
#include <exception>
#include <string>

#include "capi_common.h"

struct swc_front_plan {
  swc::FrontPlan F;
};

extern "C" {

int swc_front_plan_build(int n, const int* blockSet, int supNo, const size_t* lC, const int* Ls,
                         const size_t* Li_ptr, const int* prunePtr, const int* pruneSet,
                         const int* A2p, const int* A2i, int rlb, swc_front_plan** out) {
  if (!out || !blockSet || !lC || !Ls || !Li_ptr || !prunePtr || !A2p || !A2i || supNo <= 0 ||
      rlb < 1 || (!pruneSet && prunePtr[supNo] != 0))
    return swc_set_error(SWC_EINVAL, "swc_front_plan_build: bad argument");
  *out = nullptr;
  try {
    std::vector<int64_t> pi(supNo + 1), px(supNo);
    for (int s = 0; s <= supNo; ++s) pi[s] = (int64_t)Li_ptr[blockSet[s]];
    int64_t xsize = 0;
    std::vector<int> pos((size_t)A2p[n]);
    for (int s = 0; s < supNo; ++s) {
      px[s] = (int64_t)lC[blockSet[s]];
      xsize = std::max(xsize, px[s] + (pi[s + 1] - pi[s]) * (blockSet[s + 1] - blockSet[s]));
      for (int j = blockSet[s]; j < blockSet[s + 1]; ++j)
        for (int e = A2p[j]; e < A2p[j + 1]; ++e) {
          const int* it = std::lower_bound(Ls + pi[s], Ls + pi[s + 1], A2i[e]);
          if (it == Ls + pi[s + 1] || *it != A2i[e])
            return swc_set_error(SWC_EINVAL, "swc_front_plan_build: A2 outside the structure");
          pos[e] = (int)(it - (Ls + pi[s]));
        }
    }
    auto h = std::make_unique<swc_front_plan>();
    if (!swc::build_fronts(n, supNo, blockSet, pi.data(), px.data(), xsize, Ls, prunePtr, pruneSet,
                           A2p, nullptr, pos.data(), rlb, h->F))
      return swc_set_error(SWC_EINVAL, "swc_front_plan_build: no front tree");
    *out = h.release();
    return SWC_OK;
  } catch (const std::exception& e) {
    return swc_set_error(SWC_EINVAL, std::string("swc_front_plan_build: ") + e.what());
  }
}

void swc_front_plan_free(swc_front_plan* p) { delete p; }

int swc_front_plan_sizes(const swc_front_plan* p, int64_t* out) {
  if (!p || !out) return swc_set_error(SWC_EINVAL, "swc_front_plan_sizes: null argument");
  const swc::FrontPlan& F = p->F;
  const int64_t v[] = {F.nlevel, F.usize, F.diag_scratch, (int64_t)F.gathers.size(),
                       (int64_t)F.aents.size(), (int64_t)F.ftiles.size(), (int64_t)F.small.size(),
                       (int64_t)F.utiles.size(), sizeof(swc::Gather), sizeof(swc::AEntry),
                       sizeof(swc::FactorTile), sizeof(swc::SmallFront), sizeof(swc::FrontTile)};
  std::memcpy(out, v, sizeof(v));
  return SWC_OK;
}

int swc_front_plan_export(const swc_front_plan* p, int which, void* dst) {
  if (!p || !dst) return swc_set_error(SWC_EINVAL, "swc_front_plan_export: null argument");
  const swc::FrontPlan& F = p->F;
  auto cp = [&](const auto& v) {
    if (!v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
    return SWC_OK;
  };
  switch (which) {
    case 0: return cp(F.gathers);
    case 1: return cp(F.aents);
    case 2: return cp(F.ftiles);
    case 3: return cp(F.lvl_f);
    case 4: return cp(F.lvl_fn);
    case 5: return cp(F.small);
    case 6: return cp(F.lvl_small);
    case 7: return cp(F.utiles);
    case 8: return cp(F.lvl_u);
    case 9: return cp(F.lvl_ud);
    default: return swc_set_error(SWC_EINVAL, "swc_front_plan_export: unknown array id");
  }
}

}  // extern "C"
