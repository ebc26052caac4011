#include "selinv.h"

#include <algorithm>

#include "sweeps.h"

namespace swc {

SelPlan build_selinv(int n, int ns, const int* super, const int64_t* pi, const int64_t* px,
                     const int* Ls) {
  SelPlan P;
  const std::vector<int> lev = supernode_levels(ns, super, pi, Ls);
  std::vector<int> col2sup(n);
  int nlev = 0;
  for (int s = 0; s < ns; ++s) {
    nlev = std::max(nlev, lev[s] + 1);
    for (int c = super[s]; c < super[s + 1]; ++c) col2sup[c] = s;
  }
  std::vector<int> first(nlev + 1, 0), order(ns);  // by level, the root's first
  for (int s = 0; s < ns; ++s) ++first[nlev - lev[s]];
  for (int l = 0; l < nlev; ++l) first[l + 1] += first[l];
  {
    std::vector<int> at(first.begin(), first.end() - 1);
    for (int s = 0; s < ns; ++s) order[at[nlev - 1 - lev[s]]++] = s;
  }
  P.jrun.assign(ns ? (size_t)pi[ns] : 0, 0);
  auto close_chunk = [&](int level) {
    P.chunk_lvl.push_back(level);
    P.chunk_diag.push_back((int)P.diag.size());
    P.chunk_diag16.push_back((int)P.diag16.size());
    P.chunk_cols.push_back((int)P.cols.size());
    P.chunk_u.push_back((int)P.u.size());
  };
  close_chunk(0);
  for (auto* v : {&P.lvl_gather, &P.lvl_small, &P.lvl_z21, &P.lvl_z11}) v->push_back(0);
  int64_t mcur = 0;
  for (int l = 0; l < nlev; ++l) {
    int64_t msize = 0, zcur = 0;
    int mmax = 0;
    for (int q = first[l]; q < first[l + 1]; ++q) {
      const int s = order[q];
      msize += (int64_t)(super[s + 1] - super[s]) * (pi[s + 1] - pi[s]);
    }
    if (mcur > 0 && mcur + msize > kSelChunk) {
      close_chunk(l);
      mcur = 0;
    }
    for (int q = first[l]; q < first[l + 1]; ++q) {
      const int s = order[q], id = (int)P.nodes.size();
      SelNode nd;
      nd.vbase = px[s];
      nd.w = super[s + 1] - super[s];
      nd.nrow = (int)(pi[s + 1] - pi[s]);
      nd.rows_off = (int)pi[s];
      nd.run0 = (int)P.runs.size();
      nd.moff = mcur;
      mcur += (int64_t)nd.w * nd.nrow;
      const int w = nd.w, m = nd.nrow - w;
      const bool small = w <= kSelSmallW && m <= kSelSmallM;
      const int* rows = Ls + pi[s] + w;
      for (int j = 0; j < m;) {
        const int K = col2sup[rows[j]];
        SelRun r;
        r.j0 = j;
        while (j < m && col2sup[rows[j]] == K) P.jrun[pi[s] + w + j++] = (int)P.runs.size();
        r.nj = j - r.j0;
        r.ld = (int)(pi[K + 1] - pi[K]);
        r.zbase = px[K] - (int64_t)super[K] * r.ld;
        r.rel = P.nrel - r.j0;  // indexed by i >= j0
        r.rows_off = (int)pi[K];
        r.node = id;
        r.pad = 0;
        P.nrel += m - r.j0;
        if (!small)
          for (int c = 0; c < r.nj; c += kSelRunCols)
            for (int i = r.j0 + c; i < m; i += kSelRows)
              P.gather.push_back({(int)P.runs.size(), r.j0 + c, i, 0});
        P.runs.push_back(r);
      }
      nd.zoff = -1;
      for (int b = 0; b * kSelBlock < w; ++b) {
        (w - b * kSelBlock <= 16 ? P.diag16 : P.diag).push_back({id, b, 0, 0});
        if ((b + 1) * kSelBlock < w) P.cols.push_back({id, b, 0, 0});
      }
      for (int i = 0; i < m; i += kSelTile)
        for (int c = 0; c < w; c += kSelTile) P.u.push_back({id, i, c, 0});
      if (small) {
        P.small.push_back({id, 0, 0, 0});
        mmax = std::max(mmax, m);
      } else {
        nd.zoff = zcur;
        zcur += (int64_t)m * m;
        for (int i = 0; i < m; i += kSelTile)
          for (int c = 0; c < w; c += kSelTile) P.z21.push_back({id, i, c, 0});
        for (int i = 0; i < w; i += kSelTile)
          for (int c = 0; c <= i; c += kSelTile) P.z11.push_back({id, i, c, 0});
      }
      P.nodes.push_back(nd);
    }
    P.msize = std::max(P.msize, mcur);
    P.zsize = std::max(P.zsize, zcur);
    P.lvl_gather.push_back((int)P.gather.size());
    P.lvl_small.push_back((int)P.small.size());
    P.lvl_z21.push_back((int)P.z21.size());
    P.lvl_z11.push_back((int)P.z11.size());
    P.lvl_m.push_back(mmax);
  }
  close_chunk(nlev);
  // block columns with the longest chains first
  for (size_t c = 0; c + 1 < P.chunk_cols.size(); ++c)
    std::stable_sort(P.cols.begin() + P.chunk_cols[c], P.cols.begin() + P.chunk_cols[c + 1],
                     [&](const SelItem& x, const SelItem& y) {
                       return P.nodes[x.node].w - x.a * kSelBlock > P.nodes[y.node].w - y.a * kSelBlock;
                     });
  return P;
}

}  // namespace swc
