// ed_batch.cpp -- host side of the batched solver: builds one work item per
// (instance, target sector) for the ground state and one per (state, spin,
// +-, orbital pair) for the continued fractions, runs the items of a stage
// together, and hands the results to the instances exactly as their own solve
// would (finalize_states; GFRep 'F').
#include "ed_batch.hpp"

#include <algorithm>
#include <cmath>
#include <functional>
#include <future>
#include <map>
#include <tuple>

#include "ed_instance.hpp"
#include "ed_solvers.hpp"

namespace ed {
namespace {

// packed device copy of many FactorizedHost tables
struct TablePack {
  static constexpr size_t kNone = ~size_t(0);
  std::vector<uint32_t> u32;
  std::vector<double> f64;
  struct Off { size_t up_ptr, up_col, dn_ptr, dn_col, up_val, dn_val, diag, diag_t; uint32_t du, dd, nu, nd; };
  std::vector<Off> offs;
  DevBuf<uint32_t> du32;
  DevBuf<double> df64;
  int add(const FactorizedHost &F) {
    Off o;
    auto put32 = [&](const std::vector<uint32_t> &v) {
      const size_t at = u32.size();
      u32.insert(u32.end(), v.begin(), v.end());
      if (v.empty()) u32.push_back(0);
      return at;
    };
    auto put64 = [&](const std::vector<double> &v) {
      const size_t at = f64.size();
      f64.insert(f64.end(), v.begin(), v.end());
      if (v.empty()) f64.push_back(0.0);
      return at;
    };
    o.up_ptr = put32(F.up_ptr);
    o.up_col = put32(F.up_col);
    o.dn_ptr = put32(F.dn_ptr);
    o.dn_col = put32(F.dn_col);
    o.up_val = put64(F.up_val);
    o.dn_val = put64(F.dn_val);
    o.diag = put64(F.diag);
    o.diag_t = kNone;
    o.du = F.du;
    o.dd = F.dd;
    o.nu = (uint32_t)F.up_col.size();
    o.nd = (uint32_t)F.dn_col.size();
    offs.push_back(o);
    return (int)offs.size() - 1;
  }
  void upload() {
    du32.upload(u32);
    df64.upload(f64);
  }
  // LDS bytes of an item of this sector held in LDS
  size_t lds(int k, int nvec, size_t ntri) const {
    const Off &o = offs[k];
    return batch_lds_bytes(nvec, ntri, o.du, o.dd, o.nu, o.nd);
  }
  BatchSector view(int k) const {
    const Off &o = offs[k];
    BatchSector S;
    S.du = o.du;
    S.dd = o.dd;
    S.up_ptr = du32.p + o.up_ptr;
    S.up_col = du32.p + o.up_col;
    S.dn_ptr = du32.p + o.dn_ptr;
    S.dn_col = du32.p + o.dn_col;
    S.up_val = df64.p + o.up_val;
    S.dn_val = df64.p + o.dn_val;
    S.diag = df64.p + o.diag;
    return S;
  }
  // the sector will be used as a wide item: its diagonal in lane order too
  // (before upload)
  void use_wide(int k) {
    Off &o = offs[k];
    if (o.dd <= o.du || o.diag_t != kNone) return;
    o.diag_t = f64.size();
    f64.resize(f64.size() + (size_t)o.du * o.dd);
    for (uint32_t u = 0; u < o.du; ++u)
      for (uint32_t d = 0; d < o.dd; ++d) f64[o.diag_t + (size_t)u * o.dd + d] = f64[o.diag + (size_t)d * o.du + u];
  }
  // entries of the longest row of the smaller half's table (a wide item's rows)
  uint32_t longest_row(int k) const {
    const Off &o = offs[k];
    const uint32_t *p = u32.data() + (o.dd > o.du ? o.up_ptr : o.dn_ptr), n = std::min(o.du, o.dd);
    uint32_t m = 0;
    for (uint32_t r = 0; r < n; ++r) m = std::max(m, p[r + 1] - p[r]);
    return m;
  }
  WideItem wide(int k, int swap) const {
    const Off &o = offs[k];
    WideItem w;
    w.lp = du32.p + (swap ? o.dn_ptr : o.up_ptr);
    w.lc = du32.p + (swap ? o.dn_col : o.up_col);
    w.lv = df64.p + (swap ? o.dn_val : o.up_val);
    w.rp = du32.p + (swap ? o.up_ptr : o.dn_ptr);
    w.rc = du32.p + (swap ? o.up_col : o.dn_col);
    w.rv = df64.p + (swap ? o.up_val : o.dn_val);
    w.dg = df64.p + (swap ? o.diag_t : o.diag);
    return w;
  }
};

// where a wide item's alpha_k and beta_{k-1} go: a continued fraction's own
// arrays, a ground state's tridiagonal arrays tri (M long each)
void wide_coefficients(const BatchCFItem &it, double *, size_t, WideItem &w) {
  w.a = it.a;
  w.b = it.b;
}
void wide_coefficients(const BatchGSItem &, double *tri, size_t M, WideItem &w) {
  w.a = tri;
  w.b = tri + M - 1;
}

// execution class of an item: from LDS with one or four waves, the same with a
// ground state's tridiagonal arrays in memory, with the other items of its shape
// in lockstep, or (fractions) from registers
enum Cls { kLds = 0, kLdsFour = 1, kLdsTri = 2, kLdsTriFour = 3, kWide = 4, kTile = 5 };
constexpr int kLdsClasses = 4;
// Both halves up to two tiles of 16: the register kernel at any size (512
// points of the 2x3 sweep, 225-400 states: 67 ms of LDS kernels -> 31 ms; 2x2
// with 2 bath orbitals 34.3 -> 26.5 ms a whole sweep, with 1 23.6 -> 20.7; 24 -
// 36 states, where neither kernel counts: level).
constexpr uint32_t kTileDim = 32;

// items held in LDS with at least this many states get four waves (the
// steps are latency-bound; more waves per item hide more of it)
constexpr uint32_t kFourWaveDim = 128;

// Vectors of the wide items advanced together: what the 256 MB memory-side
// cache holds beside the tables.  (4 points of 108 900-state fractions: 60 MB
// 217 ms, 192 MB 199, 400 MB 201, all at once 201: the bound also keeps the
// workspace small.)
constexpr size_t kWideBytes = size_t(192) << 20;

// Target sectors of at most this many states: an instance's own continued
// fractions run together too.  One after the other through the single-sector
// recurrence, each step of each fraction pays two dependent launches (8-site
// chain, 72 fractions of 3 920 states: 626 ms against 9.3 together; plaquette +
// 7 bath, 213 444 states: 542 against 101; + 8 bath, 731 808: 260 against 173);
// from there on one product fills the chip and its tuned kernels win (+ 9
// bath, 2.9 M states: 1.24 s against 1.81 together).
constexpr size_t kTogetherDim = size_t(1) << 20;
// The same for a single fraction a part (one orbital): 213 444 states 46 ms alone
// against 35 here, 731 808 states 24.9 against 26.1; three of them 75 and 45.
constexpr size_t kAloneDim = size_t(1) << 19;
// Room for the levels that the fractions of a part may have (each 32 bytes, both
// parts): a level limit meant as none would ask for it at once.
constexpr size_t kTogetherLevels = size_t(1) << 22;

// LDS decides between one workgroup an item and lockstep: a workgroup with
// vectors in memory, the only other way to keep an item by itself, took 1.3 to
// 8 times the lockstep's time over sectors of 2 450 to 108 900 states (64
// points of 3 920-state fractions 21.6 -> 17.7 ms, 4 points of 108 900-state
// ones 1 630 -> 162 ms).
Cls classify(size_t lds, uint32_t dim) {
  if (lds <= kBatchLdsCap) return dim >= kFourWaveDim ? kLdsFour : kLds;
  return kWide;
}

// A ground state: many steps allowed (max_iter_lanczos 5 000: 240 KB of
// tridiagonal arrays) do not send a small sector to the lockstep kernels, whose
// three launches a step are for sectors that fill them (512 points of 2x2, 16 to
// 36 states: 4.4 ms, from LDS 2.4; of 2x3, 300 to 400 states: 23.0 and 9.5).
Cls classify_gs(size_t lds, size_t lds_without_tri, uint32_t dim) {
  const Cls c = classify(lds, dim);
  if (c != kWide || lds_without_tri > kBatchLdsCap) return c;
  return dim >= kFourWaveDim ? kLdsTriFour : kLdsTri;
}

// one launch per LDS class
template <typename Item, typename Launch>
void launch_classes(const std::vector<Item> &items, const std::vector<Cls> &cls, const size_t (&lds_max)[kLdsClasses / 2],
                    Launch launch) {
  std::vector<Item> part[kLdsClasses];
  for (size_t k = 0; k < items.size(); ++k)
    if (cls[k] < kLdsClasses) part[cls[k]].push_back(items[k]);
  DevBuf<Item> d[kLdsClasses];
  for (int c = 0; c < kLdsClasses; ++c) {
    if (part[c].empty()) continue;
    d[c].upload(part[c]);
    launch(d[c].p, (int)part[c].size(), c & 1 ? 256 : 64, lds_max[c / 2], c < kLdsTri);
  }
  sync();
}

// The register-tile fractions, by tile shape.  As many as the SIMDs hold two of (a
// wave each) or fewer go as one launch of the shape that holds them all: what a
// larger tile adds is zero, term by term, and the launches' dependent steps would
// add up (2x1 with 5 bath orbitals, halves of 1 to 21 states, whole solve of 2
// points: 2.14 ms shape by shape, 1.83 so; 12 points of 2x3 5.9 and 4.7).
constexpr size_t kTilesAtOnce = 2048;
using TileParts = std::vector<BatchCFItem>[2][2];
void sort_tiles(const TablePack &tabs, const std::vector<BatchCFItem> &items, const std::vector<Cls> &cls,
                const std::vector<int> &tab, TileParts &part) {
  size_t ntile = 0;
  int rmax = 0, cmax = 0;
  for (size_t k = 0; k < items.size(); ++k)
    if (cls[k] == kTile) {
      ++ntile;
      rmax |= tabs.offs[tab[k]].dd > 16;
      cmax |= tabs.offs[tab[k]].du > 16;
    }
  const bool one = ntile <= kTilesAtOnce;
  for (size_t k = 0; k < items.size(); ++k)
    if (cls[k] == kTile)
      part[one ? rmax : tabs.offs[tab[k]].dd > 16][one ? cmax : tabs.offs[tab[k]].du > 16].push_back(items[k]);
}

// Launch groups that do not depend on each other, with few enough items in all to
// leave part of the chip idle: side by side, each but the first on a host thread
// and stream of its own, since one after the other their dependent steps add up
// (2x2 with 3 bath orbitals, 35 x 21 states from LDS and 21 x 7 in tiles, whole
// solve of 2 points: 4.45 ms one after the other, 3.59 so).  The inputs are complete
// before the threads start and a thread's work before it ends.
constexpr size_t kBesideItems = 8192;
void run_beside(const std::vector<std::function<void()>> &groups, size_t items) {
  if (groups.size() < 2 || items > kBesideItems) {
    for (const auto &g : groups) g();
    return;
  }
  sync();
  std::vector<std::future<void>> rest;  // (a future of async waits for its thread where it is dropped)
  for (size_t k = 1; k < groups.size(); ++k)
    rest.push_back(std::async(std::launch::async, [&groups, k] {
      groups[k]();
      sync();
    }));
  groups[0]();
  for (auto &f : rest) f.get();
}

// The wide items (tab[k]: item k's sector), by shape and then in groups whose
// vectors (nvec each) fit kWideBytes: run(shape, device items, sources, n).
// ntri doubles of tridiagonal arrays per item are handed out when nonzero.
template <typename Item, typename Run>
void launch_wide(const TablePack &tabs, const std::vector<Item> &items, const std::vector<Cls> &cls,
                 const std::vector<int> &tab, int nvec, size_t ntri, Run run) {
  std::map<std::pair<uint32_t, uint32_t>, std::vector<size_t>> shapes;
  for (size_t k = 0; k < items.size(); ++k)
    if (cls[k] == kWide) shapes[{tabs.offs[tab[k]].du, tabs.offs[tab[k]].dd}].push_back(k);
  for (const auto &sh : shapes) {
    const size_t dim = (size_t)sh.first.first * sh.first.second;
    const size_t per = std::max<size_t>(1, kWideBytes / (8 * (size_t)nvec * dim));
    const size_t ngrp = (sh.second.size() + per - 1) / per, len = (sh.second.size() + ngrp - 1) / ngrp;
    for (size_t g0 = 0; g0 < sh.second.size(); g0 += len) {
      const int n = (int)std::min(len, sh.second.size() - g0);
      uint32_t emax = 0;
      for (int k = 0; k < n; ++k) emax = std::max(emax, tabs.longest_row(tab[sh.second[g0 + k]]));
      const WideShape W = wide_shape(sh.first.first, sh.first.second, emax);
      const size_t scal = 2 * (size_t)W.nwg + kWideScalars + ntri;
      DevBuf<double> u((size_t)nvec * dim * n), sc(scal * n);
      std::vector<WideItem> wi(n);
      std::vector<Item> src(n);
      for (int k = 0; k < n; ++k) {
        const size_t i = sh.second[g0 + k];
        src[k] = items[i];
        wi[k] = tabs.wide(tab[i], W.swap);
        wi[k].u = u.p + (size_t)nvec * dim * k;
        wi[k].part = sc.p + scal * k;
        wi[k].sc = wi[k].part + 2 * (size_t)W.nwg;
        wide_coefficients(items[i], ntri ? wi[k].sc + kWideScalars : nullptr, ntri / kTriArrays, wi[k]);
      }
      DevBuf<WideItem> dw;
      DevBuf<Item> ds;
      dw.upload(wi);
      ds.upload(src);
      run(W, dw.p, ds.p, n);
    }
  }
  sync();
}

// The one-body tables and the diagonal are linear in the term values: the
// tables of every operator of a term list at unit value, merged on the union
// of their patterns, give each instance's tables as a weighted sum.
struct UnitTables {
  FactorizedHost pat;                             // union pattern (values unused)
  std::vector<std::vector<double>> up, dn, diag;  // per operator, on pat
};

UnitTables unit_tables(const TermList &T, const Sector &sec) {
  UnitTables U;
  std::vector<FactorizedHost> F;
  for (const auto &tc : T.terms) {
    TermList t1;
    t1.L = T.L;
    t1.terms = {{tc.first, 1.0}};
    F.push_back(factorized_tables(t1, sec));
  }
  U.pat.du = F[0].du;
  U.pat.dd = F[0].dd;
  // union of the rows of one spin, then every operator's values on it
  auto merge = [&](bool up, std::vector<uint32_t> &ptr, std::vector<uint32_t> &col,
                   std::vector<std::vector<double>> &val) {
    const uint32_t nrow = up ? U.pat.du : U.pat.dd;
    ptr.assign(1, 0);
    std::vector<uint32_t> row;
    for (uint32_t r = 0; r < nrow; ++r) {
      row.clear();
      for (const FactorizedHost &f : F) {
        const auto &fp = up ? f.up_ptr : f.dn_ptr;
        const auto &fc = up ? f.up_col : f.dn_col;
        row.insert(row.end(), fc.begin() + fp[r], fc.begin() + fp[r + 1]);
      }
      std::sort(row.begin(), row.end());
      row.erase(std::unique(row.begin(), row.end()), row.end());
      col.insert(col.end(), row.begin(), row.end());
      ptr.push_back((uint32_t)col.size());
    }
    val.assign(F.size(), std::vector<double>(col.size(), 0.0));
    for (size_t k = 0; k < F.size(); ++k) {
      const auto &fp = up ? F[k].up_ptr : F[k].dn_ptr;
      const auto &fc = up ? F[k].up_col : F[k].dn_col;
      const auto &fv = up ? F[k].up_val : F[k].dn_val;
      for (uint32_t r = 0; r < nrow; ++r)
        for (uint32_t e = fp[r]; e < fp[r + 1]; ++e) {
          const auto b = col.begin() + ptr[r], en = col.begin() + ptr[r + 1];
          val[k][std::lower_bound(b, en, fc[e]) - col.begin()] += fv[e];
        }
    }
  };
  merge(true, U.pat.up_ptr, U.pat.up_col, U.up);
  merge(false, U.pat.dn_ptr, U.pat.dn_col, U.dn);
  for (const FactorizedHost &f : F) U.diag.push_back(f.diag);
  return U;
}

// the tables of term list T in sector sec (same operators, in the same
// order, as the list the unit tables were built from)
FactorizedHost combine_tables(const UnitTables &U, const TermList &T) {
  FactorizedHost F = U.pat;
  auto sum = [&](const std::vector<std::vector<double>> &u, std::vector<double> &out) {
    out.assign(u[0].size(), 0.0);
    for (size_t k = 0; k < u.size(); ++k) {
      const double v = T.terms[k].second;
      if (v == 0.0) continue;
      for (size_t i = 0; i < out.size(); ++i) out[i] += v * u[k][i];
    }
  };
  sum(U.up, F.up_val);
  sum(U.dn, F.dn_val);
  sum(U.diag, F.diag);
  return F;
}

// unit tables per (operator list, sector), built once per batched solve
struct TableCache {
  std::map<std::pair<std::vector<const Operator *>, Sector>, UnitTables> m;
  FactorizedHost get(const TermList &T, const Sector &sec) {
    if (T.terms.empty()) return factorized_tables(T, sec);
    std::vector<const Operator *> ops;
    for (const auto &tc : T.terms) ops.push_back(tc.first);
    auto key = std::make_pair(std::move(ops), sec);
    auto it = m.find(key);
    if (it == m.end()) it = m.emplace(key, unit_tables(T, sec)).first;
    return combine_tables(it->second, T);
  }
};

// device maps of c / c^dagger_a on a sector, built once per batched solve
struct MapCache {
  struct Set { DevBuf<int32_t> map; DevBuf<int8_t> sgn, upar; };
  std::map<std::tuple<int, int, int, int, int>, std::unique_ptr<Set>> m;  // (L, Nup, Ndw, pm, a)
  Set &get(int L, const Sector &src, int pm, int a) {
    auto key = std::make_tuple(L, src.Nup(), src.Ndw(), pm, a);
    auto it = m.find(key);
    if (it != m.end()) return *it->second;
    const CdagMaps C = cdag_maps(L, pm, a, src);
    auto M = std::make_unique<Set>();
    M->map.upload(C.map.empty() ? std::vector<int32_t>{-1} : C.map);
    M->sgn.upload(C.sgn.empty() ? std::vector<int8_t>{1} : C.sgn);
    M->upar.upload(C.upar.empty() ? std::vector<int8_t>{1} : C.upar);
    return *(m[key] = std::move(M));
  }
};

// all orbital pairs o1 >= o2, row by row
std::vector<std::pair<int, int>> all_pairs(int ns) {
  std::vector<std::pair<int, int>> p;
  for (int o1 = 0; o1 < ns; ++o1)
    for (int o2 = 0; o2 <= o1; ++o2) p.push_back({o1, o2});
  return p;
}

// one item per orbital pair of c^{pm} on state st, the target sector and the
// result arrays left to the caller
void append_pairs(std::vector<BatchCFItem> &items, MapCache &maps, int L, const std::vector<std::pair<int, int>> &pairs,
                  const State &st, int spin, int pm) {
  const uint32_t du_s = half_basis(L, st.sec.Nup())->dim;
  std::vector<const MapCache::Set *> of(L, nullptr);  // by orbital: one lookup each, not one per pair
  const auto get = [&](int o) -> const MapCache::Set & {
    if (!of[o]) of[o] = &maps.get(L, st.sec, pm, o + spin * L);
    return *of[o];
  };
  for (const auto &p : pairs) {
    const MapCache::Set &m0 = get(p.first);
    BatchCFItem it;
    it.gs = st.psi.p;
    it.du_s = du_s;
    it.spin = spin;
    it.norb = p.second == p.first ? 1 : 2;
    it.map[0] = m0.map.p;
    it.sgn[0] = m0.sgn.p;
    it.upar = m0.upar.p;
    if (p.second != p.first) {
      const MapCache::Set &m1 = get(p.second);
      it.map[1] = m1.map.p;
      it.sgn[1] = m1.sgn.p;
    }
    items.push_back(it);
  }
}

// Runs the fractions of items (tab[k]: item k's sector in tabs, not uploaded
// yet) into av (max_cf per item), bv (max_cf + 1) and out (2).
void run_fractions(TablePack &tabs, std::vector<BatchCFItem> &items, const std::vector<int> &tab, int max_cf,
                   double acc, DevBuf<double> &av, DevBuf<double> &bv, DevBuf<double> &out) {
  std::vector<Cls> cls(items.size());
  size_t lds_max[2] = {0, 0};
  for (size_t k = 0; k < items.size(); ++k) {
    const TablePack::Off &o = tabs.offs[tab[k]];
    if (o.du <= kTileDim && o.dd <= kTileDim) {
      cls[k] = kTile;
      continue;
    }
    const size_t b = tabs.lds(tab[k], kCfVectors, 0);
    cls[k] = classify(b, tabs.offs[tab[k]].du * tabs.offs[tab[k]].dd);
    if (cls[k] == kWide) tabs.use_wide(tab[k]);
    else lds_max[0] = std::max(lds_max[0], b);
  }
  tabs.upload();
  vlog("batch: %zu continued-fraction items, tables and maps built", items.size());
  av.alloc(std::max<size_t>((size_t)max_cf * items.size(), 1));
  bv.alloc(std::max<size_t>((size_t)(max_cf + 1) * items.size(), 1));
  out.alloc(std::max<size_t>(2 * items.size(), 1));
  for (size_t k = 0; k < items.size(); ++k) {
    BatchCFItem &it = items[k];
    it.S = tabs.view(tab[k]);
    it.a = av.p + (size_t)max_cf * k;
    it.b = bv.p + (size_t)(max_cf + 1) * k;
    it.out = out.p + 2 * k;
  }
  TileParts tiles;
  sort_tiles(tabs, items, cls, tab, tiles);
  std::vector<std::function<void()>> groups;
  size_t nlds = 0, ntile = 0;
  for (Cls c : cls) nlds += c < kLdsClasses;
  if (nlds)
    groups.push_back([&] {
      launch_classes(items, cls, lds_max, [&](const BatchCFItem *d, int n, int block, size_t lds, bool) {
        batch_cf(d, n, block, lds, max_cf, acc, stream());
      });
    });
  for (int r = 0; r < 2; ++r)
    for (int c = 0; c < 2; ++c) {
      if (tiles[r][c].empty()) continue;
      ntile += tiles[r][c].size();
      groups.push_back([&, r, c] {
        DevBuf<BatchCFItem> d;
        d.upload(tiles[r][c]);
        tile_cf(d.p, (int)tiles[r][c].size(), r + 1, c + 1, max_cf, acc, stream());
      });
    }
  run_beside(groups, nlds + ntile);
  launch_wide(tabs, items, cls, tab, 2, 0, [&](const WideShape &W, const WideItem *w, const BatchCFItem *q, int n) {
    wide_cf(W, w, q, n, max_cf, acc, stream());
  });
}

bool batchable(const Instance &I) {
  const Params &P = params();
  (void)P;
  if (I.gs_solved) return false;
  if (I.format != 'G' && I.format != 'F') return false;
  if (!terms_factorizable(I.terms())) return false;
  if (params().getc("Ground_state_method") != 'L') return false;
  if (params().geti("n_states") > 1) return false;
  if (params().getb("host_random_start")) return false;
  return true;
}

}  // namespace

void solve_batch(const std::vector<Instance *> &insts, bool want_gf) {
  check_cancel();
  Params &P = params();
  const int max_iter = (int)P.geti("max_iter_lanczos");
  const double accur = P.getd("accur_lanczos");
  const int max_cf = (int)P.geti("max_iter_CF");
  const double acc_cf = P.getd("accur_continued_fraction");
  const uint64_t seed = (uint64_t)P.geti("seed");

  std::vector<Instance *> todo;
  for (Instance *I : insts) {
    if (batchable(*I)) todo.push_back(I);
    else I->ground_state_solve();
  }
  vlog("batch: %zu instances batched, %zu solved one by one", todo.size(), insts.size() - todo.size());

  TableCache cache;
  // ---- ground states: one item per (instance, target sector) ----
  if (!todo.empty()) {
    TablePack tabs;
    struct GSRef { Instance *I; Sector s; int tab; uint32_t dim; };
    std::vector<GSRef> refs;
    size_t gs_len = 0;
    for (Instance *I : todo) {
      const TermList T = I->terms();
      for (const auto &s : I->targets) {
        const size_t dim = sector_dim(I->model->L, s);
        if (dim == 0) continue;
        if (dim > 0xffffffffull) fail(ED_ERR_UNSUPPORTED, "batched sector too large");
        refs.push_back({I, s, tabs.add(cache.get(T, s)), (uint32_t)dim});
        gs_len += dim;
      }
    }
    const size_t ntri = (size_t)kTriArrays * (max_iter + 2);
    std::vector<Cls> cls(refs.size());
    std::vector<int> tab(refs.size());
    size_t lds_max[2] = {0, 0}, ntri_mem = 0;
    for (size_t k = 0; k < refs.size(); ++k) {
      const size_t b = tabs.lds(refs[k].tab, kGsVectors, ntri), b0 = tabs.lds(refs[k].tab, kGsVectors, 0);
      cls[k] = classify_gs(b, b0, refs[k].dim);
      tab[k] = refs[k].tab;
      if (cls[k] == kWide) {
        tabs.use_wide(tab[k]);
      } else if (cls[k] >= kLdsTri) {
        lds_max[1] = std::max(lds_max[1], b0);
        ++ntri_mem;
      } else {
        lds_max[0] = std::max(lds_max[0], b);
      }
    }
    tabs.upload();
    vlog("batch: %zu ground-state tables built and uploaded", refs.size());
    // the ground states stay here; each state's vector is a view kept alive by it
    auto gsv = std::make_shared<DevBuf<double>>(std::max<size_t>(gs_len, 1));
    DevBuf<double> out(std::max<size_t>(3 * refs.size(), 1)), tri(std::max<size_t>(ntri * ntri_mem, 1));
    std::vector<BatchGSItem> items(refs.size());
    size_t go = 0, to = 0;
    for (size_t k = 0; k < refs.size(); ++k) {
      BatchGSItem &it = items[k];
      it.S = tabs.view(refs[k].tab);
      it.seed = seed;
      it.gs = gsv->p + go;
      it.out = out.p + 3 * k;
      go += refs[k].dim;
      if (cls[k] == kLdsTri || cls[k] == kLdsTriFour) it.tri = tri.p + ntri * to++;
    }
    launch_classes(items, cls, lds_max, [&](const BatchGSItem *d, int n, int block, size_t lds, bool tri_lds) {
      batch_gs(d, n, block, lds, tri_lds, max_iter, accur, stream());
    });
    launch_wide(tabs, items, cls, tab, 3, ntri, [&](const WideShape &W, const WideItem *w, const BatchGSItem *q, int n) {
      wide_gs(W, w, q, n, max_iter, accur, stream());
    });
    const std::vector<double> res = out.to_host();
    if (verbose()) {
      double sum = 0.0, mx = 0.0;
      for (size_t k = 0; k < refs.size(); ++k) {
        sum += res[3 * k + 1];
        mx = std::max(mx, res[3 * k + 1]);
      }
      vlog("batch: %zu ground-state items solved (Lanczos steps: mean %.1f, max %.0f)", refs.size(),
           refs.empty() ? 0.0 : sum / refs.size(), mx);
    }
    // states per instance, then the instance's own weighting
    std::map<Instance *, std::vector<std::unique_ptr<State>>> cand;
    for (size_t k = 0; k < refs.size(); ++k) {
      if (res[3 * k + 2] != 0.0)
        fail(ED_ERR_NOT_CONVERGED, "Lanczos procedure exceeded " + std::to_string(max_iter) + " iterations (instance " +
                                       std::to_string(refs[k].I->label) + ", sector " + refs[k].s.name() + ")");
      auto st = std::make_unique<State>();
      st->sec = refs[k].s;
      st->energy = res[3 * k];
      st->psi = DevBuf<double>::view(items[k].gs, refs[k].dim, gsv);
      cand[refs[k].I].push_back(std::move(st));
    }
    sync();
    vlog("batch: ground states copied out");
    for (Instance *I : todo) {
      I->states = std::move(cand[I]);
      I->finalize_states();
    }
    vlog("batch: states finalized");
  }
  if (!want_gf) return;
  check_cancel();

  // ---- Green functions: continued fractions batched, other methods one by one ----
  std::vector<Instance *> cf;
  for (Instance *I : insts) {
    if (I->gf_solved) continue;
    if (I->gf_method == 'F' && std::find(todo.begin(), todo.end(), I) != todo.end()) cf.push_back(I);
    else I->green_function_solve();
  }
  if (cf.empty()) return;
  TablePack tabs;
  std::map<std::pair<Instance *, Sector>, int> tab_of;
  MapCache maps;
  struct CFRef { State *st; int pm; int fid; };
  std::vector<CFRef> refs;
  std::vector<BatchCFItem> items;
  std::vector<int> tab;
  auto store = std::make_shared<CfStore>();
  int nfrac = 0;
  // numbered spin by spin: a Green-function call evaluates one spin's run of fractions
  for (int spin = 0; spin < 2; ++spin) {
    for (Instance *I : cf) {
      if (spin && !(I->mixing & 4)) continue;
      const int L = I->model->L, ns = I->model->n_sites;
      const auto pairs = all_pairs(ns);
      const TermList T = I->terms();
      for (auto &stp : I->states) {
        State &st = *stp;
        GFRep &G = st.gf[spin];
        G = GFRep();
        G.kind = 'F';
        G.n = ns;
        G.store = store;
        G.frac0 = nfrac;
        nfrac += ns * (ns + 1);
        for (int pm = -1; pm <= 1; pm += 2) {
          const Sector tgt = shift_sector(st.sec, pm, spin);
          if (!sector_valid(L, tgt)) continue;
          const size_t dt = sector_dim(L, tgt);
          if (dt == 0) continue;
          if (dt > 0xffffffffull) fail(ED_ERR_UNSUPPORTED, "batched sector too large");
          auto key = std::make_pair(I, tgt);
          auto ti = tab_of.find(key);
          const int t = ti != tab_of.end() ? ti->second : (tab_of[key] = tabs.add(cache.get(T, tgt)));
          append_pairs(items, maps, L, pairs, st, spin, pm);
          tab.resize(items.size(), t);
          for (int idx = 0; (int)refs.size() < (int)items.size(); ++idx)
            refs.push_back({&st, pm, G.frac0 + 2 * idx + (pm == 1 ? 0 : 1)});
        }
      }
    }
  }
  DevBuf<double> av, bv, out;
  run_fractions(tabs, items, tab, max_cf, acc_cf, av, bv, out);
  const std::vector<double> res = out.to_host();
  // the store: fraction f holds n_f coefficients (0 where psi vanished or no
  // target sector exists)
  std::vector<int> len(nfrac + 1, 0), fid(refs.size());
  std::vector<double> e0(refs.size()), wt(refs.size());
  std::vector<int8_t> pmv(refs.size());
  for (size_t k = 0; k < refs.size(); ++k) {
    const CFRef &r = refs[k];
    len[r.fid] = std::max(0, (int)res[2 * k]);
    fid[k] = r.fid;
    e0[k] = r.st->energy;
    wt[k] = r.st->weight;
    pmv[k] = (int8_t)r.pm;
  }
  std::vector<int> off(nfrac + 1, 0);
  size_t total = 0;
  for (int f = 0; f < nfrac; ++f) {
    off[f] = (int)total;
    total += (size_t)len[f];
    if (total > 0x7fffffffull) fail(ED_ERR_UNSUPPORTED, "batched continued fractions: too many coefficients");
  }
  off[nfrac] = (int)total;
  store->nfrac = nfrac;
  store->off.upload(off);
  store->A.alloc(std::max<size_t>(total, 1));
  store->B.alloc(std::max<size_t>(total, 1));
  DevBuf<int> dfid;
  DevBuf<double> de0, dwt;
  DevBuf<int8_t> dpm;
  dfid.upload(fid);
  de0.upload(e0);
  dwt.upload(wt);
  dpm.upload(pmv);
  batch_cf_store((int)refs.size(), max_cf, out.p, av.p, bv.p, dfid.p, store->off.p, de0.p, dwt.p, dpm.p,
                 store->A.p, store->B.p, stream());
  sync();
  vlog("batch: %zu continued fractions built and stored on the device (%zu coefficients)", refs.size(), total);
  for (Instance *I : cf) I->gf_solved = true;
  vlog("batch: continued fractions stored");
}

bool fractions_together(const Instance &I, const TermList &T, const State &st, int spin, size_t npairs, long max_cf) {
  Params &P = params();
  if ((I.format != 'G' && I.format != 'F') || P.geti("lanczos_block") == 0 || P.getb("lanczos_reorth") ||
      max_cf <= 0 || (size_t)max_cf > kTogetherLevels / std::max<size_t>(npairs, 1) || !terms_factorizable(T))
    return false;
  const size_t limit = npairs > 1 ? kTogetherDim : kAloneDim;
  for (int pm = -1; pm <= 1; pm += 2) {
    const Sector tgt = shift_sector(st.sec, pm, spin);
    if (sector_valid(I.model->L, tgt) && sector_dim(I.model->L, tgt) > limit) return false;
  }
  return true;
}

std::vector<Fraction> state_fractions(const Instance &I, const TermList &T, const State &st, int spin,
                                      const std::vector<std::pair<int, int>> &pairs, int max_cf) {
  const int L = I.model->L;
  TablePack tabs;
  MapCache maps;
  std::vector<BatchCFItem> items;
  std::vector<int> tab, at;
  std::vector<Fraction> F(2 * pairs.size());
  for (int pm = -1; pm <= 1; pm += 2) {
    const Sector tgt = shift_sector(st.sec, pm, spin);
    if (!sector_valid(L, tgt) || sector_dim(L, tgt) == 0) continue;
    append_pairs(items, maps, L, pairs, st, spin, pm);
    tab.resize(items.size(), tabs.add(factorized_tables(T, tgt)));
    for (size_t k = 0; k < pairs.size(); ++k) at.push_back(2 * (int)k + (pm < 0));
  }
  if (items.empty()) return F;
  DevBuf<double> av, bv, out;
  run_fractions(tabs, items, tab, max_cf, params().getd("accur_continued_fraction"), av, bv, out);
  const std::vector<double> a = av.to_host(), b = bv.to_host(), res = out.to_host();
  for (size_t k = 0; k < items.size(); ++k) {
    const int n = (int)res[2 * k];
    if (n <= 0) continue;  // psi vanishes
    const double *ak = a.data() + (size_t)max_cf * k, *bk = b.data() + (size_t)(max_cf + 1) * k;
    Fraction &f = F[at[k]];
    f.norm2 = res[2 * k + 1];
    f.a.assign(ak, ak + n);
    f.b.assign(bk, bk + n + 1);
    f.b[0] = 1.0;
  }
  return F;
}

}  // namespace ed
