// ALE ingest and the per-family plan compiler (host C++).
#include "host.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <unordered_map>
#include <numeric>
#include <thread>

#include "../../include/whale_amd.h"

namespace whale {

// ---------------------------------------------------------------------------
// ALE v0.4 text -> CCD.  Follows parse_aleobserve / parse_body /
// addleafclades! / addubiquitous! and CCD(ale, wm, spmap)
// (src/ccd.jl:102-121, 147-248).
// ---------------------------------------------------------------------------
namespace {

struct Line {
  std::vector<std::string> w;  // whitespace-separated fields
};

bool num(const std::string& s, double& v) {
  char* e = nullptr;
  v = std::strtod(s.c_str(), &e);
  return e && *e == 0 && !s.empty();
}
bool inum(const std::string& s, long& v) {
  char* e = nullptr;
  v = std::strtol(s.c_str(), &e, 10);
  return e && *e == 0 && !s.empty();
}

}  // namespace

std::string parse_ale(const char* text, size_t len, const std::unordered_map<std::string, int>& spmap,
                      CCDHost& out) {
  // split(alestring, "#")[2:end-1]
  std::vector<std::pair<size_t, size_t>> pieces;
  size_t st = 0;
  for (size_t i = 0; i <= len; ++i) {
    if (i == len || text[i] == '#') { pieces.push_back({st, i}); st = i + 1; }
  }
  if (pieces.size() != 10) return "Not a valid .ale file (expected 8 sections)";
  std::map<std::string, std::vector<Line>> sec;
  for (size_t k = 1; k + 1 < pieces.size(); ++k) {
    std::string s(text + pieces[k].first, text + pieces[k].second);
    std::string t;
    t.reserve(s.size());
    for (size_t i = 0; i < s.size(); ++i) {
      if (s[i] == ':' && i + 1 < s.size() && s[i + 1] == '\t') { ++i; continue; }  // ":\t" => ""
      t += s[i];
    }
    size_t nl = t.find('\n');
    std::string header = t.substr(0, nl);
    std::vector<Line> lines;
    size_t pos = nl == std::string::npos ? t.size() : nl + 1;
    while (pos < t.size()) {
      size_t e = t.find('\n', pos);
      if (e == std::string::npos) e = t.size();
      if (e > pos) {
        Line L;
        size_t a = pos;
        while (a < e) {
          while (a < e && isspace((unsigned char)t[a])) ++a;
          size_t b = a;
          while (b < e && !isspace((unsigned char)t[b])) ++b;
          if (b > a) L.w.emplace_back(t.substr(a, b - a));
          a = b;
        }
        lines.push_back(std::move(L));
      }
      pos = e + 1;
    }
    sec[header] = std::move(lines);
  }
  for (const char* h : {"observations", "Bip_counts", "Dip_counts", "leaf-id", "set-id"})
    if (!sec.count(h)) return std::string("ALE section missing: ") + h;
  for (const char* h : {"Bip_counts", "Dip_counts", "leaf-id", "set-id"})
    if (sec[h].size() == 1) return std::string("ALE section with a single line is not a table: ") + h;
  double obs;
  if (sec["observations"].size() != 1 || sec["observations"][0].w.empty() || !num(sec["observations"][0].w[0], obs))
    return "bad #observations";
  std::map<long, double> bip;
  for (auto& L : sec["Bip_counts"]) {
    long k; double v;
    if (L.w.size() < 2 || !inum(L.w[0], k) || !num(L.w[1], v)) return "bad #Bip_counts line";
    bip[k] = v;
  }
  struct D { long a, b; double c; };
  std::map<long, std::vector<D>> dip;
  for (auto& L : sec["Dip_counts"]) {
    long k, a, b; double c;
    if (L.w.size() < 4 || !inum(L.w[0], k) || !inum(L.w[1], a) || !inum(L.w[2], b) || !num(L.w[3], c))
      return "bad #Dip_counts line";
    dip[k].push_back({a, b, c});
  }
  std::map<long, std::string> leafname;  // ALE leaf id -> name
  for (auto& L : sec["leaf-id"]) {
    long id;
    if (L.w.size() < 2 || !inum(L.w[1], id)) return "bad #leaf-id line";
    leafname[id] = L.w[0];
  }
  std::map<long, std::vector<long>> sets;  // sorted by set id, as sort!(OrderedDict(...))
  for (auto& L : sec["set-id"]) {
    long k;
    if (L.w.empty() || !inum(L.w[0], k)) return "bad #set-id line";
    std::vector<long> v;
    for (size_t i = 1; i < L.w.size(); ++i) { long x; if (!inum(L.w[i], x)) return "bad #set-id member"; v.push_back(x); }
    sets[k] = std::move(v);
  }
  // addleafclades!: leaf sets get Bip = observations and no splits; leaf ids
  // inside other sets are replaced by the leaf's set id.
  std::map<long, std::string> leafclade;  // leaf set id -> name
  std::map<long, long> leaf2set;
  for (auto& kv : sets) {
    if (kv.second.size() == 1) {
      auto it = leafname.find(kv.second[0]);
      if (it == leafname.end()) return "set-id names an unknown leaf";
      bip[kv.first] = obs;
      dip[kv.first].clear();
      leafclade[kv.first] = it->second;
      leaf2set[kv.second[0]] = kv.first;
    } else {
      for (auto& x : kv.second) {
        auto it = leaf2set.find(x);
        if (it == leaf2set.end()) return "set-id refers to a leaf before its leaf set";
        x = it->second;
      }
    }
  }
  for (auto& kv : leaf2set) sets[kv.second] = {kv.second};
  // addubiquitous!: the root clade's splits are all complementary pairs (i<j)
  // of the set ids 1..nset, each with count Bip_j.
  long n = (long)leafclade.size();
  long nset = (long)sets.size();
  for (long i = 1; i <= nset; ++i) if (!sets.count(i)) return "set ids are not contiguous";
  long G = nset + 1;
  // Complements are found through an additive hash of the members (a random
  // 64-bit key per leaf): the complement of set i hashes to (sum over all
  // leaves) - h(i).  Every candidate is then checked exactly (sizes add up to
  // the leaves, no common member), and pairs come out in the (i, j) order of
  // the reference's double loop.
  auto key = [](long x) {
    uint64_t z = (uint64_t)x * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  std::vector<uint64_t> h(nset + 1, 0);
  for (long i = 1; i <= nset; ++i)
    for (long x : sets[i]) {
      if (x < 1 || x > nset) return "bad set member";
      h[i] += key(x);
    }
  uint64_t all = 0;
  for (auto& kv : leafclade) all += key(kv.first);
  std::unordered_map<uint64_t, std::vector<long>> by_hash;
  by_hash.reserve((size_t)nset * 2);
  for (long i = 1; i <= nset; ++i) by_hash[h[i]].push_back(i);
  std::vector<char> mark(nset + 1, 0);
  std::vector<D> root;
  double N = 0;
  for (long i = 1; i <= nset; ++i) {
    auto it = by_hash.find(all - h[i]);
    if (it == by_hash.end()) continue;
    const long si = (long)sets[i].size();
    bool marked = false;
    for (long j : it->second) {
      if (j <= i || si + (long)sets[j].size() != n) continue;
      if (!marked) {
        for (long x : sets[i]) mark[x] = 1;
        marked = true;
      }
      bool disjoint = true;
      for (long x : sets[j]) if (mark[x]) { disjoint = false; break; }
      if (!disjoint) continue;
      if (!bip.count(i) || !bip.count(j)) return "missing Bip count";
      if (bip[i] != bip[j]) return "complementary clades have different Bip counts";
      N += bip[i];
      root.push_back({i, j, bip[j]});
    }
    if (marked)
      for (long x : sets[i]) mark[x] = 0;
  }
  if (root.empty()) return "no split of the ubiquitous clade";
  bip[G] = N;
  dip[G] = root;
  {
    std::vector<long> u = sets[root.back().a];
    for (long x : sets[root.back().b]) if (std::find(u.begin(), u.end(), x) == u.end()) u.push_back(x);
    sets[G] = u;
  }
  // CCD: order by (size, set id); p = Dip / Bip
  std::vector<std::pair<long, long>> ord;
  for (auto& kv : sets) ord.push_back({(long)kv.second.size(), kv.first});
  std::sort(ord.begin(), ord.end());
  std::unordered_map<long, int> newid;
  for (size_t i = 0; i < ord.size(); ++i) newid[ord[i].second] = (int)i;
  size_t nc = ord.size();
  out.size.assign(nc, 0);
  out.leaf_species.assign(nc, -1);
  out.split_off.assign(nc + 1, 0);
  out.g1.clear(); out.g2.clear(); out.p.clear();
  for (size_t i = 0; i < nc; ++i) {
    long k = ord[i].second;
    out.size[i] = (int32_t)ord[i].first;
    out.split_off[i] = (int32_t)out.g1.size();
    if (ord[i].first == 1) {
      const std::string& nm = leafclade[k];
      std::string pre = nm.substr(0, nm.find('_'));
      auto it = spmap.find(pre);
      if (it == spmap.end()) return "gene " + nm + ": species " + pre + " is not in the species tree";
      out.leaf_species[i] = it->second;
    }
    auto bi = bip.find(k);
    if (bi == bip.end()) return "clade without a Bip count";
    for (auto& d : dip[k]) {
      auto a = newid.find(d.a), b = newid.find(d.b);
      if (a == newid.end() || b == newid.end()) return "split names an unknown clade";
      out.g1.push_back(a->second);
      out.g2.push_back(b->second);
      out.p.push_back(d.c / bi->second);
    }
    if (ord[i].first > 1 && out.g1.size() == (size_t)out.split_off[i]) return "non-leaf clade without splits";
  }
  out.split_off[nc] = (int32_t)out.g1.size();
  return "";
}

// ---------------------------------------------------------------------------
// plan compiler
// ---------------------------------------------------------------------------
namespace {

struct FamPlan {
  std::string err;
  uint32_t n_clades = 0, max_items = 0, max_slots = 0, n_items = 0;
  std::vector<StageDev> stage;      // item0, seg0 and slots relative to the family
  std::vector<SegDev> seg;          // ell/ibar relative to family
  uint32_t root_seg = 0, root_fs = 0, root_bs = 0, root_recs = 0;
  std::vector<uint32_t> it_seg, it_gid;  // it_seg family-relative
  std::vector<uint32_t> fs4, fs2, bs4, bs2, rec_ops, rec_sid, ent_ops, ent_rec;
  std::vector<uint32_t> lvl_f, lvl_b;
  uint64_t ell = 0, ibar = 0;
  int64_t cells = 0, split_terms = 0, sum_compat = 0, row_steps = 0;
  double cost = 0;
};

// lanes of an item with `terms` terms
uint32_t slot_lanes(uint32_t terms) {
  return std::max(1u, std::min(kSlotLanes, (terms + kSlotRecs - 1) / kSlotRecs));
}

// Deals items to slots (plan.hpp): item k of `items` has cnt[k] terms and
// takes one lane, or up to kSlotLanes adjacent lanes of a 16-lane row when it
// has more than kSlotRecs.  Items with the most terms come first, so that the
// 64 lanes of a chunk have similar counts; the lanes a many-lane item leaves
// at the end of a row go to one-lane items.
// Rows are counted from `offset` slots before the first.
// Returns per lane (k, position) or (-1, 0) for an unused lane.
std::vector<std::pair<int, uint32_t>> deal_slots(const std::vector<uint32_t>& cnt, uint32_t offset) {
  const int n = (int)cnt.size();
  std::vector<int> by(n);
  std::iota(by.begin(), by.end(), 0);
  std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return cnt[a] > cnt[b]; });
  std::vector<std::pair<int, uint32_t>> out;
  std::vector<uint32_t> holes;
  size_t next_hole = 0;
  for (int k : by) {
    const uint32_t u = slot_lanes(cnt[k]);
    if (u == 1 && next_hole < holes.size()) {
      out[holes[next_hole++]] = {k, 0};
      continue;
    }
    if ((out.size() + offset) % kSlotLanes + u > kSlotLanes)
      while ((out.size() + offset) % kSlotLanes) {
        holes.push_back((uint32_t)out.size());
        out.push_back({-1, 0});
      }
    for (uint32_t j = 0; j < u; ++j) out.push_back({k, j});
  }
  return out;
}

void plan_family(const ModelHost& m, int32_t nc, const int32_t* csize, const int32_t* leaf_sp,
                 const int64_t* soff, const int32_t* g1, const int32_t* g2, FamPlan& F) {
  const int W = m.words;
  F.n_clades = nc;
  if (nc < 3) { F.err = "family with fewer than two genes"; return; }
  if (nc > 65535) { F.err = "family with more than 65535 clades"; return; }
  // species bitsets of clades
  std::vector<uint64_t> cb((size_t)nc * W, 0);
  for (int c = 0; c < nc; ++c) {
    if (c > 0 && csize[c] < csize[c - 1]) { F.err = "clades are not sorted by size"; return; }
    int64_t a = soff[c], b = soff[c + 1];
    if (csize[c] == 1) {
      int s = leaf_sp[c];
      if (s < 0 || s >= m.n_species) { F.err = "leaf clade with a bad species"; return; }
      if (b != a) { F.err = "leaf clade with splits"; return; }
      cb[(size_t)c * W + (s >> 6)] |= 1ull << (s & 63);
      continue;
    }
    if (b <= a) { F.err = "non-leaf clade without splits"; return; }
    for (int64_t k = a; k < b; ++k) {
      int x = g1[k], y = g2[k];
      if (x < 0 || y < 0 || x >= c || y >= c) { F.err = "split part is not an earlier clade"; return; }
      if (csize[x] + csize[y] != csize[c]) { F.err = "split part sizes do not add up"; return; }
    }
    int x = g1[a], y = g2[a];
    for (int w = 0; w < W; ++w) cb[(size_t)c * W + w] = cb[(size_t)x * W + w] | cb[(size_t)y * W + w];
  }
  if (csize[nc - 1] <= csize[nc - 2]) {  // the last clade must be the unique largest (ubiquitous) one
    F.err = "the last clade is not the ubiquitous clade";
    return;
  }
  // compatible clades per node: species(γ) ⊆ clade(e)  (src/model.jl:39 iscompatible)
  std::vector<std::vector<int32_t>> comp(m.n);
  std::vector<std::vector<int32_t>> idx(m.n);
  for (int e = 0; e < m.n; ++e) {
    const uint64_t* eb = &m.bits[(size_t)e * W];
    auto& C = comp[e];
    for (int c = 0; c < nc; ++c) {
      const uint64_t* x = &cb[(size_t)c * W];
      bool sub = true;
      for (int w = 0; w < W; ++w) if (x[w] & ~eb[w]) { sub = false; break; }
      if (sub) C.push_back(c);
    }
    if (e == m.root && (int)C.size() != nc) { F.err = "a clade is not compatible with the root"; return; }
  }
  // segments: every node with compatible clades, root last
  std::vector<int> segof(m.n, -1);
  std::vector<int> segnodes;
  for (int e : m.order) if (!comp[e].empty() && e != m.root) segnodes.push_back(e);
  // stages by height; segments of one stage must not share clades (MUL trees)
  std::vector<std::vector<int>> stages;
  {
    std::vector<int> stamp(nc, -1);
    for (int h = 0; h <= m.max_height; ++h) {
      std::vector<int> pending;
      for (int e : segnodes) if (m.height[e] == h) pending.push_back(e);
      while (!pending.empty()) {
        int sid = (int)stages.size();
        stages.push_back({});
        std::vector<int> rest;
        for (int e : pending) {
          bool clash = false;
          for (int c : comp[e]) if (stamp[c] == sid) { clash = true; break; }
          if (clash) { rest.push_back(e); continue; }
          for (int c : comp[e]) stamp[c] = sid;
          stages.back().push_back(e);
        }
        pending.swap(rest);
      }
    }
  }
  // A stage runs max R rows for all its segments, so the rows of a family are
  // the sum of its stages' longest branches.  Stages by height put long
  // branches of different lineages in different stages; a segment may run in
  // any stage after its children's and before its parent's.  A local search
  // moves segments (longest first) to the stage that lowers the modelled cost
  // Σ (max R − 1 + 3) · (2 + ⌈items/64⌉ + 2⌈records/64⌉) — rows times the
  // 64-lane chunks of one row, record chunks weighing double (they gather two
  // operands, and scatter twice in the reverse sweep), plus a stage's set-up —
  // without raising the family's largest stage (its LDS need) or putting
  // clades twice in a stage.
  if (stages.size() > 1) {
    // the height stages take every kGap-th slot; the slots between are empty
    // at first, so a segment can also run between two height stages
    constexpr int kGap = 2;
    const int K = kGap * ((int)stages.size() - 1) + 1;
    std::vector<int> stg(m.n, -1);
    std::vector<int64_t> nrec_of(m.n, 0);
    std::vector<std::vector<int>> mem(K);
    std::vector<int64_t> ni(K, 0), nr(K, 0);
    for (int h = 0; h < (int)stages.size(); ++h)
      for (int e : stages[h]) {
        const int k = kGap * h;
        stg[e] = k;
        mem[k].push_back(e);
        for (int32_t c : comp[e]) nrec_of[e] += soff[c + 1] - soff[c];
        ni[k] += (int64_t)comp[e].size();
        nr[k] += nrec_of[e];
      }
    int64_t cap_i = 0, cap_r = 0;
    for (int k = 0; k < K; ++k) cap_i = std::max(cap_i, ni[k]), cap_r = std::max(cap_r, nr[k]);
    auto rmax_of = [&](int k, int skip) {
      int r = 0;
      for (int e : mem[k]) if (e != skip) r = std::max(r, m.nodes[e].R);
      return r;
    };
    auto cost = [](int rmax, int64_t items, int64_t recs) -> int64_t {
      if (items == 0) return 0;
      return (int64_t)(rmax - 1 + 3) * (2 + (items + 63) / 64 + 2 * ((recs + 63) / 64));
    };
    std::vector<int> rmx(K);
    for (int k = 0; k < K; ++k) rmx[k] = rmax_of(k, -1);
    std::vector<int> by_r(segnodes);
    std::stable_sort(by_r.begin(), by_r.end(), [&](int a, int b) { return m.nodes[a].R > m.nodes[b].R; });
    std::vector<int> mark(nc, -1);
    for (int pass = 0; pass < 8; ++pass) {
      bool moved = false;
      for (int e : by_r) {
        const NodeDev& nd = m.nodes[e];
        const int a = stg[e];
        int lo = 0, hi = K - 1;
        for (int ch : {nd.child0, nd.child1})
          if (ch >= 0 && stg[ch] >= 0) lo = std::max(lo, stg[ch] + 1);
        if (nd.parent >= 0 && nd.parent != m.root) hi = stg[nd.parent] - 1;
        const int64_t ce = (int64_t)comp[e].size(), re = nrec_of[e];
        const int ra = rmax_of(a, e);
        const int64_t drop = cost(ra, ni[a] - ce, nr[a] - re) - cost(rmx[a], ni[a], nr[a]);
        int best = a;
        int64_t gain = 0;
        for (int b = lo; b <= hi; ++b) {
          if (b == a || ni[b] + ce > cap_i || nr[b] + re > cap_r) continue;
          const int64_t d = drop + cost(std::max(rmx[b], nd.R), ni[b] + ce, nr[b] + re) - cost(rmx[b], ni[b], nr[b]);
          if (d >= gain) continue;
          // no clade twice in one stage (MUL trees)
          for (int32_t c : comp[e]) mark[c] = e;
          bool clash = false;
          for (int x : mem[b]) {
            for (int32_t c : comp[x]) if (mark[c] == e) { clash = true; break; }
            if (clash) break;
          }
          for (int32_t c : comp[e]) mark[c] = -1;
          if (clash) continue;
          gain = d;
          best = b;
        }
        if (best == a) continue;
        mem[a].erase(std::find(mem[a].begin(), mem[a].end(), e));
        mem[best].push_back(e);
        ni[a] -= ce, nr[a] -= re, ni[best] += ce, nr[best] += re;
        rmx[a] = ra;
        rmx[best] = std::max(rmx[best], nd.R);
        stg[e] = best;
        moved = true;
      }
      if (!moved) break;
    }
    // non-empty stages in order, segments in the species tree's order
    std::vector<std::vector<int>> out(K);
    for (int e : segnodes) out[stg[e]].push_back(e);
    stages.clear();
    for (auto& st : out) if (!st.empty()) stages.push_back(std::move(st));
  }
  // segment records, ℓ and ī offsets
  auto nkids = [&](int e) { const NodeDev& d = m.nodes[e]; return (d.child0 >= 0) + (d.child1 >= 0); };
  uint64_t ell = 0, ibar = 0;
  for (auto& st : stages) {
    for (int e : st) {
      SegDev s{};
      s.node = (uint32_t)e;
      s.nc = (uint32_t)comp[e].size();
      s.R = (uint32_t)m.nodes[e].R;
      s.ell = (uint32_t)ell;
      ell += (uint64_t)s.R * s.nc;
      s.ibar = nkids(e) ? (uint32_t)ibar : kNone;
      ibar += (uint64_t)nkids(e) * s.nc;
      segof[e] = (int)F.seg.size();
      F.seg.push_back(s);
    }
  }
  {
    SegDev s{};
    s.node = (uint32_t)m.root;
    s.nc = (uint32_t)nc;
    s.R = 1;
    s.ell = (uint32_t)ell;
    ell += nc;
    s.ibar = (uint32_t)ibar;
    ibar += 2ull * nc;
    segof[m.root] = (int)F.seg.size();
    F.root_seg = (uint32_t)F.seg.size();
    F.seg.push_back(s);
  }
  if (ell > 0xffffffffull || ibar > 0xffffffffull) { F.err = "family too large"; return; }
  F.ell = ell;
  F.ibar = ibar;
  for (int e = 0; e < m.n; ++e) {
    if (segof[e] < 0) continue;
    idx[e].assign(nc, -1);
    for (size_t j = 0; j < comp[e].size(); ++j) idx[e][comp[e][j]] = (int32_t)j;
  }
  // A stage's items, records and slots.  Records and entries come item by
  // item, so an item's terms are contiguous and a slot is a range of them.
  std::vector<uint32_t> r0, ne, e0, cnt;
  auto emit_items = [&](const std::vector<int>& segs, StageDev& sd) -> bool {
    uint32_t local = 0;
    for (int e : segs) {
      SegDev& s = F.seg[segof[e]];
      s.item0 = local;
      local += s.nc;
      sd.r_max = std::max(sd.r_max, s.R);
    }
    sd.item0 = (uint32_t)F.it_seg.size();
    sd.seg0 = (uint32_t)segof[segs[0]];
    sd.n_segs = (uint32_t)segs.size();
    sd.n_items = local;
    if (local > 0xffff) { F.err = "stage with more than 65535 items"; return false; }
    const uint32_t rb = (uint32_t)F.rec_ops.size();
    r0.assign(local + 1, 0);
    for (int e : segs) {
      const SegDev& s = F.seg[segof[e]];
      for (uint32_t j = 0; j < s.nc; ++j) {
        const int gid = comp[e][j];
        F.it_seg.push_back((uint32_t)segof[e]);
        F.it_gid.push_back((uint32_t)gid);
        r0[s.item0 + j] = (uint32_t)F.rec_ops.size();
        for (int64_t k = soff[gid]; k < soff[gid + 1]; ++k) {
          const uint32_t l1 = s.item0 + (uint32_t)idx[e][g1[k]], l2 = s.item0 + (uint32_t)idx[e][g2[k]];
          F.rec_ops.push_back(l1 | (l2 << 16));
          F.rec_sid.push_back((uint32_t)(k - soff[0]));
        }
      }
    }
    const uint32_t re = (uint32_t)F.rec_ops.size();
    r0[local] = re;
    // the same splits listed by part: (owner, other part, record)
    ne.assign(local + 1, 0);
    for (uint32_t r = rb; r < re; ++r) ++ne[F.rec_ops[r] & 0xffff], ++ne[F.rec_ops[r] >> 16];
    e0.assign(local + 1, 0);
    e0[0] = 2 * rb;
    for (uint32_t i = 0; i < local; ++i) e0[i + 1] = e0[i] + ne[i];
    F.ent_ops.resize(2 * (size_t)re);
    F.ent_rec.resize(2 * (size_t)re);
    std::vector<uint32_t> at(e0.begin(), e0.end() - 1);
    for (uint32_t i = 0; i < local; ++i)
      for (uint32_t r = r0[i]; r < r0[i + 1]; ++r) {
        const uint32_t x = F.rec_ops[r] & 0xffff, y = F.rec_ops[r] >> 16;
        F.ent_ops[at[x]] = i | (y << 16), F.ent_rec[at[x]++] = r;
        F.ent_ops[at[y]] = i | (x << 16), F.ent_rec[at[y]++] = r;
      }
    return true;
  };
  // slots of some of the stage's items, in one direction
  auto emit_slots = [&](const StageDev& sd, const std::vector<uint32_t>& items, bool fwd, uint32_t offset) -> bool {
    const std::vector<uint32_t>& off = fwd ? r0 : e0;
    std::vector<uint32_t>&s4 = fwd ? F.fs4 : F.bs4, &s2 = fwd ? F.fs2 : F.bs2;
    cnt.resize(items.size());
    for (size_t k = 0; k < items.size(); ++k) {
      cnt[k] = off[items[k] + 1] - off[items[k]];
      if (cnt[k] > kSlotLanes * 0xffffu) { F.err = "clade with too many splits"; return false; }
    }
    for (const auto& [k, pos] : deal_slots(cnt, offset)) {
      if (k < 0) {
        s4.insert(s4.end(), {0xffffffffu, 0xffffffffu, 0u, 0u});
        s2.insert(s2.end(), {0u, 0u});
        continue;
      }
      const uint32_t i = items[(size_t)k], terms = cnt[k];
      const uint32_t u = slot_lanes(terms);
      const uint32_t a = (uint32_t)((uint64_t)terms * pos / u), b = (uint32_t)((uint64_t)terms * (pos + 1) / u);
      const uint32_t si = F.it_seg[sd.item0 + i], gid = F.it_gid[sd.item0 + i];
      const int e = (int)F.seg[si].node;
      const NodeDev& nd = m.nodes[e];
      int32_t kc[2] = {-1, -1};
      const int kids[2] = {nd.child0, nd.child1};
      for (int q = 0; q < 2; ++q) {
        const int ch = kids[q];
        if (ch < 0 || segof[ch] < 0 || idx[ch][gid] < 0) continue;
        const SegDev& cs = F.seg[segof[ch]];
        kc[q] = (int32_t)(cs.ell + (uint64_t)(cs.R - 1) * cs.nc + idx[ch][gid]);
      }
      if (nd.kind == WHALE_NODE_WGD) kc[1] = kc[0];
      uint32_t d;
      if (fwd) {
        d = gid | ((si - sd.seg0) << 16);
      } else if (nd.parent < 0) {
        d = 0;
      } else {
        const SegDev& ps = F.seg[segof[nd.parent]];
        const int x = idx[nd.parent][gid];
        if (x < 0) { F.err = "internal error: clade not compatible with the parent"; return false; }
        d = ps.ibar + (m.nodes[nd.parent].child0 == e ? 0u : ps.nc) + (uint32_t)x;
      }
      s4.insert(s4.end(), {(uint32_t)kc[0], (uint32_t)kc[1], i | (pos << 16) | (pos + 1 == u ? kSlotLead : 0u), d});
      s2.insert(s2.end(), {off[i] + a, (b - a) | (fwd ? 0u : (si - sd.seg0) << 16)});
    }
    return true;
  };
  std::vector<uint32_t> all;
  for (auto& st : stages) {
    StageDev sd{};
    if (!emit_items(st, sd)) return;
    if (sd.n_segs > 0xffff) { F.err = "stage with more than 65535 segments"; return; }
    sd.fs0 = (uint32_t)(F.fs4.size() / 4);
    sd.bs0 = (uint32_t)(F.bs4.size() / 4);
    all.resize(sd.n_items);
    std::iota(all.begin(), all.end(), 0u);
    if (!emit_slots(sd, all, true, 0) || !emit_slots(sd, all, false, 0)) return;
    sd.n_fs = (uint32_t)(F.fs4.size() / 4) - sd.fs0;
    sd.n_bs = (uint32_t)(F.bs4.size() / 4) - sd.bs0;
    F.max_items = std::max(F.max_items, sd.n_items);
    F.max_slots = std::max({F.max_slots, sd.n_fs, sd.n_bs});
    F.stage.push_back(sd);
  }
  F.n_items = (uint32_t)F.it_seg.size();
  {
    StageDev sd{};
    const size_t rec_before = F.rec_ops.size();
    if (!emit_items({m.root}, sd)) return;
    F.root_recs = (uint32_t)(F.rec_ops.size() - rec_before);
    // Root levels by depth: a clade's level is one past the highest level of
    // its splits' parts, so a level reads only finished parts and, in the
    // reverse sweep, only finished owners.  (Runs of clades in size order of
    // which none is a part of another: 21 to 26 levels for the families of 25
    // genes at which depth gives 17 to 22, 116 against 44 for 240 genes.)
    std::vector<uint32_t> depth(nc, 0);
    std::vector<std::vector<uint32_t>> lvl(1);
    for (int c = 0; c < nc; ++c) {
      for (int64_t k = soff[c]; k < soff[c + 1]; ++k) depth[c] = std::max({depth[c], depth[g1[k]] + 1, depth[g2[k]] + 1});
      if (depth[c] >= lvl.size()) lvl.resize(depth[c] + 1);
      lvl[depth[c]].push_back((uint32_t)c);
    }
    F.root_fs = (uint32_t)(F.fs4.size() / 4);
    F.root_bs = (uint32_t)(F.bs4.size() / 4);
    for (size_t L = 0; L <= lvl.size(); ++L) {
      F.lvl_f.push_back((uint32_t)(F.fs4.size() / 4) - F.root_fs);
      F.lvl_b.push_back((uint32_t)(F.bs4.size() / 4) - F.root_bs);
      if (L == lvl.size()) break;
      if (!emit_slots(sd, lvl[L], true, F.lvl_f.back()) || !emit_slots(sd, lvl[L], false, F.lvl_b.back())) return;
    }
  }
  // workload counts (the reference's cell and split-term counts)
  for (auto& s : F.seg) {
    F.cells += (int64_t)s.R * s.nc;
    F.sum_compat += s.nc;
  }
  for (auto& st : stages) {
    for (int e : st) {
      const SegDev& s = F.seg[segof[e]];
      F.row_steps += s.R;
      int64_t sp = 0;
      for (int32_t c : comp[e]) sp += soff[c + 1] - soff[c];
      F.split_terms += (int64_t)(s.R - 1) * sp + (m.nodes[e].kind == WHALE_NODE_LEAF ? 0 : sp * (m.nodes[e].kind == WHALE_NODE_WGD ? 1 : 2));
    }
  }
  F.split_terms += 2 * (soff[nc] - soff[0]);
  uint64_t steps = 1 + F.lvl_f.size();
  for (auto& sd : F.stage) steps += sd.r_max;
  F.cost = (double)steps * 64.0 + (double)F.cells + (double)F.split_terms;
}

}  // namespace

std::string build_plan(const ModelHost& m, int n_fam, const int64_t* fam_clade_off, const int32_t* clade_size,
                       const int32_t* leaf_species, const int64_t* split_off, const int32_t* g1,
                       const int32_t* g2, const double* p, PlanHost& P, int nthreads) {
  std::vector<FamPlan> fp(n_fam);
  int nt = std::max(1, std::min(nthreads, n_fam));
  std::vector<std::thread> th;
  for (int w = 0; w < nt; ++w) {
    th.emplace_back([&, w]() {
      for (int f = w; f < n_fam; f += nt) {
        int64_t c0 = fam_clade_off[f], c1 = fam_clade_off[f + 1];
        plan_family(m, (int32_t)(c1 - c0), clade_size + c0, leaf_species + c0, split_off + c0, g1, g2, fp[f]);
        // g1/g2 are absolute arrays indexed by split; plan_family receives soff into them
      }
    });
  }
  for (auto& t : th) t.join();
  for (int f = 0; f < n_fam; ++f)
    if (!fp[f].err.empty()) return "family " + std::to_string(f) + ": " + fp[f].err;
  // concatenate: every family's offsets first, then the copies on the same threads
  P = PlanHost();
  P.cost_order.resize(n_fam);
  std::iota(P.cost_order.begin(), P.cost_order.end(), 0u);
  std::stable_sort(P.cost_order.begin(), P.cost_order.end(),
                   [&](uint32_t a, uint32_t b) { return fp[a].cost > fp[b].cost; });
  P.fam.resize(n_fam);
  P.fam_seg0.resize(n_fam);
  P.fam_nseg.resize(n_fam);
  uint64_t ell = 0, ibar = 0, item = 0, seg = 0, stage = 0, rec = 0, fs = 0, bs = 0, lvl = 0;
  for (int f = 0; f < n_fam; ++f) {
    const FamPlan& F = fp[f];
    FamDev& d = P.fam[f];
    d.n_clades = F.n_clades;
    d.n_stages = (uint32_t)F.stage.size();
    d.stage0 = (uint32_t)stage;
    d.item0 = (uint32_t)item;
    d.n_items = F.n_items;
    d.clade0 = (uint32_t)fam_clade_off[f];
    d.split0 = (uint32_t)split_off[fam_clade_off[f]];
    d.lvl0 = (uint32_t)lvl;
    d.n_lvl = (uint32_t)F.lvl_f.size() - 1;
    d.max_items = F.max_items;
    d.max_slots = F.max_slots;
    d.root_seg = (uint32_t)(seg + F.root_seg);
    d.root_fs = (uint32_t)(fs + F.root_fs);
    d.root_bs = (uint32_t)(bs + F.root_bs);
    d.root_nfs = F.lvl_f.back();
    d.root_nbs = F.lvl_b.back();
    d.root_recs = F.root_recs;
    d.rec0 = (uint32_t)rec;
    d.n_recs = (uint32_t)F.rec_ops.size();
    d.ell0 = ell;
    d.ibar0 = ibar;
    P.fam_seg0[f] = (uint32_t)seg;
    P.fam_nseg[f] = (uint32_t)F.seg.size();
    stage += F.stage.size();
    item += F.it_seg.size();
    seg += F.seg.size();
    rec += F.rec_ops.size();
    fs += F.fs4.size() / 4;
    bs += F.bs4.size() / 4;
    lvl += F.lvl_f.size();
    ell += F.ell;
    ibar += F.ibar;
    P.max_items = std::max(P.max_items, std::max(F.max_items, F.n_clades));
    P.cells += F.cells;
    P.split_terms += F.split_terms;
    P.sum_compat += F.sum_compat;
    P.row_steps += F.row_steps;
    P.n_clades += F.n_clades;
  }
  for (uint64_t x : {item, 2 * rec, fs, bs})
    if (x > 0xffffffffull) return "batch too large";
  P.stage.resize(stage);
  P.seg.resize(seg);
  P.run.resize(seg);
  P.it_seg.resize(item);
  P.it_gid.resize(item);
  P.fs4.resize(4 * fs);
  P.fs2.resize(2 * fs);
  P.bs4.resize(4 * bs);
  P.bs2.resize(2 * bs);
  P.rec_ops.resize(rec);
  P.rec_p.resize(rec);
  P.ent_ops.resize(2 * rec);
  P.ent_p.resize(2 * rec);
  P.lvl_f.resize(lvl);
  P.lvl_b.resize(lvl);
  auto copy_family = [&](int f) {
    FamPlan& F = fp[f];
    const FamDev& d = P.fam[f];
    const uint32_t seg0 = P.fam_seg0[f];
    const uint32_t fs0 = d.root_fs - F.root_fs, bs0 = d.root_bs - F.root_bs;
    for (size_t k = 0; k < F.stage.size(); ++k) {
      StageDev s = F.stage[k];
      s.item0 += d.item0;
      s.seg0 += seg0;
      s.fs0 += fs0;
      s.bs0 += bs0;
      P.stage[d.stage0 + k] = s;
    }
    for (size_t k = 0; k < F.seg.size(); ++k) {
      const SegDev& s = F.seg[k];
      const NodeDev& nd = m.nodes[s.node];
      P.seg[seg0 + k] = s;
      SegRun& t = P.run[seg0 + k];
      t.ell = s.ell - s.item0;
      t.nc = s.nc;
      t.R = s.R;
      t.tab = (uint32_t)nd.tab;
      t.kn = (uint32_t)nd.kind | (s.node << 2);
      t.c0 = nd.kind == WHALE_NODE_LEAF ? s.node : (uint32_t)nd.child0;
      t.c1 = (uint32_t)(nd.kind == WHALE_NODE_WGD ? nd.wgd : nd.child1);
      t.ibar = s.ibar - s.item0;
    }
    for (size_t i = 0; i < F.it_seg.size(); ++i) P.it_seg[d.item0 + i] = F.it_seg[i] + seg0;
    std::copy(F.it_gid.begin(), F.it_gid.end(), P.it_gid.begin() + d.item0);
    std::copy(F.fs4.begin(), F.fs4.end(), P.fs4.begin() + 4 * (size_t)fs0);
    std::copy(F.fs2.begin(), F.fs2.end(), P.fs2.begin() + 2 * (size_t)fs0);
    std::copy(F.bs4.begin(), F.bs4.end(), P.bs4.begin() + 4 * (size_t)bs0);
    std::copy(F.bs2.begin(), F.bs2.end(), P.bs2.begin() + 2 * (size_t)bs0);
    std::copy(F.rec_ops.begin(), F.rec_ops.end(), P.rec_ops.begin() + d.rec0);
    std::copy(F.ent_ops.begin(), F.ent_ops.end(), P.ent_ops.begin() + 2 * (size_t)d.rec0);
    for (size_t r = 0; r < F.rec_sid.size(); ++r) P.rec_p[d.rec0 + r] = p[d.split0 + F.rec_sid[r]];
    for (size_t k = 0; k < F.ent_rec.size(); ++k)
      P.ent_p[2 * (size_t)d.rec0 + k] = p[d.split0 + F.rec_sid[F.ent_rec[k]]];
    std::copy(F.lvl_f.begin(), F.lvl_f.end(), P.lvl_f.begin() + d.lvl0);
    std::copy(F.lvl_b.begin(), F.lvl_b.end(), P.lvl_b.begin() + d.lvl0);
    F = FamPlan();
  };
  th.clear();
  for (int w = 0; w < nt; ++w)
    th.emplace_back([&, w]() {
      for (int f = w; f < n_fam; f += nt) copy_family(f);
    });
  for (auto& t : th) t.join();
  P.ell_cells = ell;
  P.ibar_cells = ibar;
  int64_t nclades = fam_clade_off[n_fam];
  P.clade_size.resize(nclades);
  for (int64_t c = 0; c < nclades; ++c) P.clade_size[c] = (uint16_t)std::min(clade_size[c], 65535);
  int64_t nsplit = split_off[nclades];
  P.n_splits = nsplit;
  P.split_p.assign(p, p + nsplit);
  return "";
}

}  // namespace whale
