// Builds the solves' work lists (see sweeps.h).
#include "sweeps.h"

#include <algorithm>

namespace swc {

std::vector<int> supernode_levels(int nsuper, const int* super, const int64_t* pi, const int* Ls) {
  std::vector<int> lev(nsuper, 0), col2sup(nsuper ? super[nsuper] : 0);
  for (int s = 0; s < nsuper; ++s)
    for (int c = super[s]; c < super[s + 1]; ++c) col2sup[c] = s;
  for (int s = 0; s < nsuper; ++s) {  // rows below belong to later supernodes
    const int* r = Ls + pi[s] + (super[s + 1] - super[s]);
    const int* end = Ls + pi[s + 1];
    while (r < end) {
      const int t = col2sup[*r];
      lev[t] = std::max(lev[t], lev[s] + 1);
      while (r < end && *r < super[t + 1]) ++r;
    }
  }
  return lev;
}

void build_sweeps(int nsuper, const int* super, const int64_t* pi, const int64_t* px, const int* Ls,
                  const int64_t* voff, const int64_t* gptr, int64_t maxpart, SweepPlan& W) {
  W = SweepPlan();
  auto width = [&](int s) { return super[s + 1] - super[s]; };
  auto nrows = [&](int s) { return (int)(pi[s + 1] - pi[s]); };
  auto small = [&](int s) { return width(s) <= 16 && nrows(s) - width(s) <= kSmallRows; };
  const std::vector<int> lev = supernode_levels(nsuper, super, pi, Ls);
  int nlev = 0;
  for (int s = 0; s < nsuper; ++s) nlev = std::max(nlev, lev[s] + 1);
  std::vector<int> lptr(nlev + 1, 0), order(nsuper), nsmall(nlev, 0);
  for (int s = 0; s < nsuper; ++s) {
    lptr[lev[s] + 1]++;
    nsmall[lev[s]] += small(s);
  }
  for (int l = 0; l < nlev; ++l) lptr[l + 1] += lptr[l];
  {
    std::vector<int> fill(lptr.begin(), lptr.end() - 1);
    for (int s = 0; s < nsuper; ++s) order[fill[lev[s]]++] = s;
  }
  // Leading levels of narrow supernodes only get launches of their own while they are
  // large: one wave each without a claim (a claim takes ~12 ns of the one counter, a
  // launch ~8 us; from 512 or 8192 on 64^3, a 500^2 GMRF and 600 2D instances take the same,
  // within 1%).
  int plain = 0;
  while (plain < nlev && nsmall[plain] == lptr[plain + 1] - lptr[plain] && nsmall[plain] >= 2048)
    ++plain;
  std::vector<int> first_small(nlev);
  for (int l = 0; l < nlev; ++l) {
    first_small[l] = (int)W.small.size();
    for (int i = lptr[l]; i < lptr[l + 1]; ++i) {
      const int s = order[i];
      if (!small(s)) continue;
      W.small.push_back({px[s], voff[s], nrows(s), width(s), super[s], (int)pi[s]});
    }
  }
  W.lvl_small.assign(first_small.begin(), first_small.begin() + plain);
  W.lvl_small.push_back(plain < nlev ? first_small[plain] : (int)W.small.size());
  // Of a leading level, the supernodes with at most 16 rows below come first: 16 lanes each
  // in a launch of their own, where they are all or again 2048.
  for (int l = 0; l + 1 < (int)W.lvl_small.size(); ++l) {
    const auto b = W.small.begin() + W.lvl_small[l], e = W.small.begin() + W.lvl_small[l + 1];
    const auto few = [](const SweepSmall& s) { return s.R - s.w <= 16; };
    const int n16 = (int)(std::stable_partition(b, e, few) - b);
    W.lvl_small16.push_back(n16 == e - b || n16 >= 2048 ? n16 : 0);
  }
  // Rows below per backward partial, doubled until the partials fit.  256 / 512 / 1024 / 4096
  // (ms): 64^3 with one right-hand side 1.61 / 1.53 / 1.51 / 1.34, with 8 3.80 / 3.38 / 3.27 / 2.77,
  // vector 40^3 1.87 / 1.85 / 1.79 / 1.59: parts were meant to shorten the chain, which they do not
  // on these, but they keep an item's share of a supernode of very many rows bounded.
  int chunk = 512;
  auto parts = [&](int s) {
    const int m = nrows(s) - width(s);
    return m > chunk ? (m + chunk - 1) / chunk : 0;
  };
  for (;; chunk *= 2) {
    int64_t total = 0;
    for (int s = 0; s < nsuper; ++s)
      if (!small(s)) total += (int64_t)((width(s) + 63) / 64) * 64 * parts(s);
    if (total <= maxpart || chunk >= (1 << 29)) {
      W.psize = total;
      break;
    }
  }
  auto base = [&](int s) {
    SweepItem it{};
    it.vbase = px[s];
    it.ld = nrows(s);
    it.w = width(s);
    it.c0 = super[s];
    it.rows_off = (int)pi[s];
    return it;
  };
  auto add_small = [&](std::vector<SweepItem>& v, int l) {
    const int n = nsmall[l], per = 4 * std::max(1, n / (4 * 2048));
    for (int i = 0; i < n; i += per) {
      SweepItem it{};
      it.kind = kSweepSmall;
      it.first = first_small[l] + i;
      it.count = std::min(per, n - i);
      v.push_back(it);
    }
  };
  // Within a level: panel 0 of every supernode, then panel 1 of those that have one, and so
  // on, narrow ones, and the row blocks below at last, so that no workgroup holds a place
  // only to wait for the panels of its supernode while other supernodes' are not started.
  // A level that fits the device at once lists its row blocks right after their supernode's
  // panels: they then apply each panel when it comes and are done with the last one.  Limits
  // of 0 / 128 / 512 / 2048 items (ms): 64^3 with one right-hand side 1.51 / 1.50 / 1.53 / 1.77, with 8
  // 3.29 / 3.28 / 3.38 / 3.98, vector 40^3 1.83 / 1.82 / 1.85 / 2.14 (runs of one differ by 1%): any level
  // that fits, two workgroups a CU, does; one that does not loses 15%.
  constexpr int kResident = 512;
  auto np_of = [&](int s) { return (width(s) + 63) / 64; };
  auto below_of = [&](int s) { return (nrows(s) - width(s) + 63) / 64; };
  for (int l = plain; l < nlev; ++l) {
    std::vector<int> sn;
    int64_t total = 0;
    int most = 0;
    for (int i = lptr[l]; i < lptr[l + 1]; ++i) {
      if (small(order[i])) continue;
      sn.push_back(order[i]);
      total += np_of(order[i]) + below_of(order[i]);
      most = std::max(most, np_of(order[i]));
    }
    auto own = [&](int s, int p) {
      SweepItem it = base(s);
      it.kind = kSweepOwn;
      it.p = p;
      it.row0 = 64 * p;
      it.nr = std::min(64, width(s) - 64 * p);
      it.nq = p;
      W.fwd.push_back(it);
    };
    auto below = [&](int s) {
      const int w = width(s), m = nrows(s) - w;
      for (int r = 0; r < m; r += 64) {
        SweepItem it = base(s);
        it.kind = kSweepBelow;
        it.row0 = w + r;
        it.nr = std::min(64, m - r);
        it.nq = np_of(s);
        it.out = voff[s] + r;
        W.fwd.push_back(it);
      }
    };
    if (total <= kResident) {
      for (int s : sn) {
        for (int p = 0; p < np_of(s); ++p) own(s, p);
        below(s);
      }
      add_small(W.fwd, l);
    } else {
      for (int p = 0; p < most; ++p)
        for (int s : sn)
          if (p < np_of(s)) own(s, p);
      add_small(W.fwd, l);
      for (int s : sn) below(s);
    }
  }
  // Backward: the parts of every supernode of a level (they wait for levels above only),
  // then the panels, last ones first, then narrow ones.
  int64_t slot = 0;
  for (int l = nlev - 1; l >= plain; --l) {
    std::vector<int> sn;
    std::vector<int64_t> slot0;
    int most = 0;
    for (int i = lptr[l]; i < lptr[l + 1]; ++i) {
      const int s = order[i];
      if (small(s)) continue;
      sn.push_back(s);
      slot0.push_back(slot);
      slot += (int64_t)64 * np_of(s) * parts(s);
      most = std::max(most, np_of(s));
    }
    for (size_t i = 0; i < sn.size(); ++i) {
      const int s = sn[i], w = width(s), m = nrows(s) - w, k = parts(s);
      for (int p = np_of(s) - 1; p >= 0; --p)
        for (int c = k - 1; c >= 0; --c) {
          SweepItem it = base(s);
          it.kind = kSweepBelow;
          it.p = p;
          it.nr = std::min(64, w - 64 * p);
          it.row0 = w + c * chunk;
          it.row1 = w + std::min(m, (c + 1) * chunk);
          it.out = slot0[i] + 64 * ((int64_t)p * k + c);
          W.bwd.push_back(it);
        }
    }
    for (int q = 0; q < most; ++q)
      for (size_t i = 0; i < sn.size(); ++i) {
        const int s = sn[i], w = width(s), k = parts(s), p = np_of(s) - 1 - q;
        if (p < 0) continue;
        SweepItem it = base(s);
        it.kind = kSweepOwn;
        it.p = p;
        it.nr = std::min(64, w - 64 * p);
        it.row0 = w;
        it.row1 = k ? w : nrows(s);
        it.nq = k;
        it.out = slot0[i] + 64 * (int64_t)p * k;
        W.bwd.push_back(it);
      }
    add_small(W.bwd, l);
  }
  // one right-hand side to an item or 16 (sweep_by_16)
  std::vector<int64_t> steps(nsuper, 0);  // of the longest chain up to a supernode
  std::vector<int> col2sup(nsuper ? super[nsuper] : 0);
  int64_t bytes = 1, longest = 1;
  for (int s = 0; s < nsuper; ++s)
    for (int c = super[s]; c < super[s + 1]; ++c) col2sup[c] = s;
  for (int s = 0; s < nsuper; ++s) {
    int64_t list = 0;
    for (int c = super[s]; c < super[s + 1]; ++c) list = std::max(list, gptr[c + 1] - gptr[c]);
    steps[s] += np_of(s) + list / 64;
    longest = std::max(longest, steps[s]);
    bytes += (int64_t)sizeof(double) * width(s) * nrows(s);
    if (nrows(s) > width(s)) {
      int64_t& up = steps[col2sup[Ls[pi[s] + width(s)]]];
      up = std::max(up, steps[s]);
    }
  }
  const int64_t items = std::max<int64_t>(std::min<int64_t>(W.fwd.size(), longest), 1);
  W.one_each = std::min(kStepBytes * longest / bytes, kChains * longest / items);
}

}  // namespace swc
