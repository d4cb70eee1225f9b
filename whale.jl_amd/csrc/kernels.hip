// gfx950 kernels around the amalgamated-likelihood DP (the DP's own: dp.hpp).
//
//   k_tables       slice tables ε, φ, ψ of every branch (setmodel!/setslices!,
//                  src/model.jl:162-191; getα/_ϵ/_ϕ/_ψ, src/bdputil.jl:6-11)
//                  plus the per-row partial derivatives the reverse sweep needs
//   k_tail         table adjoint (reverse of the ε recursion, chain rule to
//                  λ, μ, q, η), conditioning (src/condition.jl:21-29) and the
//                  batch sum ℓhood(Σℓ − N·c) (src/core.jl:54,63)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "dev.hpp"
#include "../../include/whale_amd.h"

namespace whale {

// ---------------------------------------------------------------------------
// k_tables: one workgroup.  The slice map over Δt is the Möbius map
//   ε ← (a + (1 − a − b) ε) / (1 − b ε)
// (the linear birth-death extinction pgf, src/model.jl:162-191); r slices
// compose to a map of the same kind, which eps_after evaluates in closed
// form.  The tops of the branches go level by level (a node's bottom value is
// a function of its children's tops), one lane per node; then every row of
// every branch is independent: ε(r−1) in closed form, then the last step and
// the row's φ and ψ as the slice recursion writes them.  Last,
// ∂ε_r/∂(α, β, ε_0) for the reverse sweep's tables: with den_r = 1 - β ε_{r-1},
// D_k(r) = -(∂den_r/∂k)/den_r.
// The time is that of its chains: the levels of the tree, and the rows of the
// longest branch.  So a level's step holds a few FP64 operations and divides
// only (the functions and the loads come before), and the derivatives' chain
// one multiply-add a row, its coefficients formed by all lanes at once in LDS.
// Measured, with α, β and the functions within each step before -> now: 9 taxa
// and 140 rows 23 -> 11 us, 58 taxa and slices of 0.01 53 -> 24 us, 50 taxa and
// 1488 rows 60 -> 26 us.
// ---------------------------------------------------------------------------
struct SliceAB {
  double a, b, dal, dam, dbl, dbm;
};

// α, β of one slice of length t (and their derivatives in λ, μ)
__device__ inline SliceAB slice_ab(double l, double u, double t) {
  SliceAB s{0, 0, 0, 0, 0, 0};
  bool close = (l == u) || (isfinite(l) && isfinite(u) && fabs(l - u) <= 1e-6);
  if (close) {
    double x = 1.0 + l * t;
    s.a = l * t / x;
    s.dal = t / (x * x);
    s.dam = 0.0;
  } else {
    double E = exp(t * (l - u));
    double N = u * (E - 1.0), D = l * E - u;
    s.a = N / D;
    double dNl = u * t * E, dNm = (E - 1.0) - u * t * E;
    double dDl = E + l * t * E, dDm = -l * t * E - 1.0;
    s.dal = (dNl * D - N * dDl) / (D * D);
    s.dam = (dNm * D - N * dDm) / (D * D);
  }
  s.b = (l / u) * s.a;
  s.dbl = s.a / u + (l / u) * s.dal;
  s.dbm = -l * s.a / (u * u) + (l / u) * s.dam;
  return s;
}

// ε after k slices from e0.  The map has the fixed points 1 and ρ = a/b
// (= μ/λ), and z = 1/(1 − ε) moves affinely: z ← κz + b/(1 − a) with
// κ = (1 − b)/(1 − a).  With δ = κ − 1, S = (κ^k − 1)/δ:
//   ε_k = (e0 + S(a − b·e0)/(1 − a)) / (κ^k + S·b(1 − e0)/(1 − a)),
// both sums of non-negative terms while e0 ≤ ρ; for e0 > ρ (a leaf whose
// sampling probability p exceeds μ/λ)
//   (ε_k − ρ)/(1 − ε_k) = κ^k (e0 − ρ)/(1 − e0)
// keeps ε_k = ρ + (excess) free of cancellation.  κ^k and S go through
// log1p/expm1 (κ is near 1 for short slices) and are scaled by κ^−k when
// κ > 1.  Accurate to a few ulp, where k dependent steps drift by k ulp.
// What does not depend on e0 comes first, so that the chain from the leaves to
// the root holds none of the functions.
// δ = κ − 1 of the α and β as they are stored.  Not to be fused with the
// product β is formed by: near λ = μ the difference is all rounding, and S
// needs the very δ that log κ was formed from.
__device__ inline double slice_excess(double a, double b) {
#pragma clang fp contract(off)
  return (a - b) / (1.0 - a);
}
struct Powers {
  double L, X, S;  // k·log κ; κ^±k and S (scaled by κ^−k), the sign that of −L
};
__device__ inline Powers slice_powers(double a, double b, double lg, int k) {
  const double d = slice_excess(a, b);
  Powers w{(double)k * lg, 1.0, (double)k};
  if (d == 0.0) return w;
  const double m = w.L <= 0.0 ? w.L : -w.L;
  w.X = exp(m);
  w.S = (w.L <= 0.0 ? expm1(m) : -expm1(m)) / d;
  return w;
}
__device__ inline double eps_after(double a, double b, const Powers& w, int k, double e0) {
  if (k == 0 || e0 == 1.0) return e0;
  const double om = 1.0 - a;
  if (om == 0.0) return 1.0;
  const double d = slice_excess(a, b);
  if (a < b * e0) {
    const double rho = a / b;
    const double W = (w.L <= 0.0 ? w.X : exp(w.L)) * (e0 - rho) / (1.0 - e0);
    return (rho + W) / (1.0 + W);
  }
  const double al = (a - b * e0) / om, be = b * (1.0 - e0) / om;
  if (d == 0.0) return (e0 + (double)k * al) / (1.0 + (double)k * be);
  if (w.L <= 0.0) return (e0 + w.S * al) / (w.X + w.S * be);
  return (e0 * w.X + w.S * al) / (1.0 + w.S * be);
}

// one slice step from ε' = ep (the row's ε, φ, ψ)
__device__ inline void slice_step(double a, double b, double ep, double* en, double* ph, double* ps, double* den_) {
  const double den = 1.0 - b * ep;
  const double num = a + (1.0 - a - b) * ep;
  *en = num / den;
  *ph = (1.0 - a) * (1.0 - b) / (den * den);
  *ps = (1.0 - a) * (1.0 - b) * b / (den * den * den);
  *den_ = den;
}

// The workspace of k_tables: per node α, β, log κ, the powers of its top and
// its top ε; per row ε and the three coefficients of the derivatives' chain,
// which their values replace.  In LDS where it fits.
size_t tables_work_bytes(int n, int rows) { return 8 * (7 * (size_t)n + 4 * (size_t)rows); }

template <bool InLds>
__global__ __launch_bounds__(1024) void k_tables(ModelDev M, double* eps, double* phi, double* psi,
                                                    double* pack64, float* pack32, double* dnode,
                                                    const int32_t* hlevels, const int32_t* hnodes, int n_levels,
                                                    const int32_t* row_node, double* work) {
  extern __shared__ __align__(16) double s_work[];
  const int n = M.n, rows = M.tab_rows, t = threadIdx.x, nt = blockDim.x;
  double* const A = InLds ? s_work : work;
  double *const B = A + n, *const LG = B + n, *const PL = LG + n, *const PX = PL + n, *const PS = PX + n,
                *const TOP = PS + n;
  double *const EN = TOP + n, *const G = EN + rows, *const CA = G + rows, *const CB = CA + rows;
  const double* lam = M.par;
  const double* mu = M.par + n;
  const double* par_p = M.par + 2 * n;
  const double* par_q = M.par + 3 * n;
  // every node's slice map
  for (int e = t; e < n; e += nt) {
    const NodeDev& d = M.node[e];
    SliceAB s{0, 0, 0, 0, 0, 0};
    Powers w{0.0, 1.0, 0.0};
    double lg = 0.0;
    const bool br = d.R > 1;
    if (br) {
      s = slice_ab(lam[e], mu[e], d.delta);
      lg = log1p(slice_excess(s.a, s.b));
      w = slice_powers(s.a, s.b, lg, d.R - 2);
    }
    A[e] = s.a;
    B[e] = s.b;
    LG[e] = lg;
    PL[e] = w.L;
    PX[e] = w.X;
    PS[e] = w.S;
    const double ia = 1.0 / (1.0 - s.a), ib = 1.0 / (1.0 - s.b);
    // at α or β = 1 no lineage crosses the branch: φ = ψ = 0 and the sums these multiply are 0
    const double v[7] = {s.dal, s.dam, s.dbl, s.dbm, br && isfinite(ia) ? ia : 0.0, br && isfinite(ib) ? ib : 0.0,
                         br ? s.b : 0.0};
#pragma unroll
    for (int j = 0; j < 7; ++j) dnode[(size_t)kDnode * e + j] = v[j];
  }
  // tops, children first: a lane keeps the entry of hnodes that is its own
  const int me = t < n ? hnodes[t] : -1;
  const NodeDev mine = M.node[me >= 0 ? me : 0];
  int lv = -1;
  if (me >= 0) {
    int lo = 0, hi = n_levels;  // the level L with hlevels[L] ≤ t < hlevels[L + 1]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (hlevels[mid] <= t) lo = mid;
      else hi = mid;
    }
    lv = lo;
  }
  auto top = [&](int e, const NodeDev& d) {
    double e0;
    if (d.kind == WHALE_NODE_WGD) {
      const double ec = TOP[d.child0], qq = par_q[d.wgd];
      e0 = qq * (ec * ec) + (1.0 - qq) * ec;
    } else if (d.kind == WHALE_NODE_LEAF) {
      e0 = par_p[e];
    } else {
      e0 = TOP[d.child0] * TOP[d.child1];
    }
    EN[d.tab] = e0;
    double en = e0;
    if (d.R > 1) {
      const double a = A[e], b = B[e];
      double ph, ps, den;
      slice_step(a, b, eps_after(a, b, Powers{PL[e], PX[e], PS[e]}, d.R - 2, e0), &en, &ph, &ps, &den);
      EN[d.tab + d.R - 1] = en;
    }
    TOP[e] = en;
  };
  __syncthreads();
  for (int L = 0; L < n_levels; ++L) {
    if (lv == L) top(me, mine);
    for (int k = t + nt; k < n; k += nt)  // trees of more nodes than lanes
      if (k >= hlevels[L] && k < hlevels[L + 1]) top(hnodes[k], M.node[hnodes[k]]);
    __syncthreads();
  }
  // every row: ε(r−1) in closed form, then the last step
  auto put = [&](size_t i, double v) {
    pack64[i] = v;
    pack32[i] = (float)v;
  };
  const size_t n4 = 4 * (size_t)rows, n6 = 6 * (size_t)rows;
  for (int i = t; i < rows; i += nt) {
    const int e = row_node[i];
    const NodeDev& d = M.node[e];
    const int r = i - d.tab;
    double en, ph = 1.0, ps = 1.0, den;
    if (r == 0) {
      en = EN[i];
    } else {
      const double a = A[e], b = B[e];
      slice_step(a, b, eps_after(a, b, slice_powers(a, b, LG[e], r - 1), r - 1, EN[d.tab]), &en, &ph, &ps, &den);
      if (r == d.R - 1) en = EN[i];  // the top, as the levels wrote it for the parent
      else EN[i] = en;
    }
    eps[i] = en;
    phi[i] = ph;
    psi[i] = ps;
    put(4 * (size_t)i, ph);
    put(n4 + 2 * (size_t)i, ph);
    put(n4 + 2 * (size_t)i + 1, ps);
  }
  __syncthreads();
  // ∂ε_r/∂(α, β, ε_0) as a chain of z ← G z + c
  for (int i = t; i < rows; i += nt) {
    const int e = row_node[i];
    if (i == M.node[e].tab) continue;
    const double a = A[e], b = B[e], ep = EN[i - 1], en = EN[i];
    const double id = 1.0 / (1.0 - b * ep);
    G[i] = ((1.0 - a - b) + b * en) * id;
    CA[i] = (1.0 - ep) * id;
    CB[i] = ep * (en - 1.0) * id;
  }
  __syncthreads();
  for (int e = t; e < n; e += nt) {
    const NodeDev& d = M.node[e];
    double za = 0.0, zb = 0.0, z0 = 1.0;
    const int i1 = d.tab + d.R;
    constexpr int U = 8;  // rows read at once, ahead of the chain
    for (int i0 = d.tab + 1; i0 < i1; i0 += U) {
      double g[U], ca[U], cb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + u, i1 - 1);
        g[u] = G[i], ca[u] = CA[i], cb[u] = CB[i];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + u < i1) {
          G[i0 + u] = z0, CA[i0 + u] = za, CB[i0 + u] = zb;
          za = ca[u] + g[u] * za;
          zb = cb[u] + g[u] * zb;
          z0 = g[u] * z0;
        }
    }
    double* dn = dnode + (size_t)kDnode * e;
    const bool br = d.R > 1;
    dn[7] = z0;
    dn[8] = br ? za : 0.0;
    dn[9] = br ? zb : 0.0;
  }
  __syncthreads();
  for (int i = t; i < rows; i += nt) {
    const int e = row_node[i];
    double ch = 0.0, da = 0.0, db = 0.0, d0 = 0.0;  // row 0 has no slice
    if (i != M.node[e].tab) {
      const double a = A[e], b = B[e], ep = EN[i - 1];
      const double den = 1.0 - b * ep, id = 1.0 / den;
      ch = (1.0 - a) * (1.0 - b) / (den * den * den);
      da = b * CA[i] * id;
      db = (ep + b * CB[i]) * id;
      d0 = b * G[i] * id;
    }
    put(4 * (size_t)i + 1, ch);
    put(4 * (size_t)i + 2, da);
    put(4 * (size_t)i + 3, db);
    put(n6 + i, d0);
  }
}

// ---------------------------------------------------------------------------
// The conditioning term c = log P(condition) (src/condition.jl:11-29) of the
// current parameters and its derivatives in the root's ε, its children's ε
// and η: RootCondition P = 1 − g(ε_f) − g(ε_g) + g(ε_ρ), NonExtinct
// P = 1 − g(ε_ρ), g the root's geometric pgf; none: c = 0.
struct CondTerms {
  double c, dc_er, dc_ef, dc_eg, dc_eta;
};
__device__ inline CondTerms cond_terms(const ModelDev& M, int cond) {
  const NodeDev& rn = M.node[M.root];
  const double eta = M.par[3 * M.n + M.n_wgd];
  const double er = eps_top(M, M.root);
  const double ef = eps_top(M, rn.child0), eg = eps_top(M, rn.child1);
  auto gpgf = [&](double x) { return eta * x / (1.0 - (1.0 - eta) * x); };
  auto dg_ds = [&](double x) { double D = 1.0 - (1.0 - eta) * x; return eta / (D * D); };
  auto dg_deta = [&](double x) { double D = 1.0 - (1.0 - eta) * x; return x * (1.0 - x) / (D * D); };
  CondTerms T{0, 0, 0, 0, 0};
  if (cond == WHALE_COND_ROOT) {
    const double P = 1.0 - gpgf(ef) - gpgf(eg) + gpgf(er);
    T.c = P > 0 ? log(P) : -INFINITY;
    T.dc_ef = -dg_ds(ef) / P;
    T.dc_eg = -dg_ds(eg) / P;
    T.dc_er = dg_ds(er) / P;
    T.dc_eta = (-dg_deta(ef) - dg_deta(eg) + dg_deta(er)) / P;
  } else if (cond == WHALE_COND_NONEXTINCT) {
    const double P = 1.0 - gpgf(er);
    T.c = log(P);
    T.dc_er = -dg_ds(er) / P;
    T.dc_eta = -dg_deta(er) / P;
  }
  return T;
}

// k_mix: one workgroup.  The mixture's per-family log-sum-exp over its
// components (src/core.jl:66-76) and the responsibilities that weight each
// component's reverse sweep.
__global__ __launch_bounds__(1024) void k_mix(const MixComp* X, int K, const double* log_prior, uint32_t n_fam,
                                              int cond, double* out, double* resp) {
  __shared__ double red[1024];
  __shared__ double s_c[kMaxMix];
  __shared__ double s_w[kMaxMix][32];
  const int t = threadIdx.x;
  if (t < K) s_c[t] = cond_terms(X[t].M, cond).c;
  for (int i = t; i < kMaxMix * 32; i += blockDim.x) s_w[i / 32][i % 32] = 0.0;
  __syncthreads();
  double tot = 0.0, wsum[kMaxMix];
  for (int j = 0; j < kMaxMix; ++j) wsum[j] = 0.0;
  for (uint32_t i = t; i < n_fam; i += blockDim.x) {
    double l[kMaxMix], mx = -INFINITY;
    for (int j = 0; j < K; ++j) {
      l[j] = X[j].W.fam_ll[i] + log_prior[j] - s_c[j];
      mx = fmax(mx, l[j]);
    }
    double lse = -INFINITY;
    if (isfinite(mx)) {
      double acc = 0.0;
      for (int j = 0; j < K; ++j) acc += exp(l[j] - mx);
      lse = mx + log(acc);
    }
    for (int j = 0; j < K; ++j) {
      const double r = isfinite(lse) ? exp(l[j] - lse) : 0.0;
      X[j].W.seed[i] = r;
      wsum[j] += r;
      if (resp) resp[(size_t)i * K + j] = r;
    }
    tot += lse;
  }
  red[t] = tot;
  for (int j = 0; j < K; ++j) atomicAdd(&s_w[j][t % 32], wsum[j]);
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (t < w) red[t] += red[t + w];
    __syncthreads();
  }
  if (t < K) {
    double sw = 0.0;
    for (int q = 0; q < 32; ++q) sw += s_w[t][q];
    X[t].W.seed[n_fam] = sw;
  }
  if (t == 0) out[0] = isfinite(red[0]) ? red[0] : -INFINITY;
}

constexpr int kTailThreads = 1024;

// Sum over the workgroup, in every lane of it: lanes of a wave, then waves.
__device__ inline double group_sum(double v, double* part) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < kTailThreads / 64; ++w) s += part[w];
  return s;
}

// The workspace of k_tail, per node: ε̄ of its top and what the chain from the
// root needs of it; the levels of the tree.  In LDS where it fits.
constexpr size_t kTailLds = 48 * 1024;
size_t tail_work_bytes(int n) { return 8 * 4 * (size_t)n; }

// k_tail.  The first workgroup forms Σℓ over the families, the conditioning
// term, and the chain rule from the nodes' sums to ∂λ, ∂μ, ∂q, ∂η.  The
// adjoints of a branch's ε of row 0, α and β are its own sums plus the adjoint
// of its top ε times ∂ε_top/∂(ε_0, α, β) (k_tables); depth by depth, parents
// first, a node's top adjoint takes its parent's row-0 one.  Only that chain
// goes by depth, one multiply-add and two products a level on values loaded
// before it; all else follows for every node at once.
// Results may go to pinned host memory: `out`, and with `host_fam` every
// family's ℓ and the count *fb of families recomputed in FP64.  The other
// workgroups share the families' copy.
// Measured, with the chain on global memory and a tree reduction of Σℓ before
// -> now: 12 families of 9 taxa 13.5 -> 6.4 us, one of 58 taxa 16.7 -> 6.1 us,
// 10,000 of 50 taxa 30 -> 13 us, the three copies to the host (14 us) included
// in the latter figures.
template <bool InLds>
__global__ __launch_bounds__(kTailThreads) void k_tail(ModelDev M, const double* fam_ll, uint32_t n_fam,
                                                       const double* acc_in, double* work, const int32_t* dlevels,
                                                       const int32_t* dnodes, int n_dlevels, int cond, int with_grad,
                                                       double* out, const double* n_eff, double* host_fam,
                                                       const uint32_t* fb, uint32_t* host_fb) {
  extern __shared__ __align__(16) double s_work[];
  __shared__ double part[kTailThreads / 64];
  __shared__ CondTerms s_ct;
  const int t = threadIdx.x, n = M.n;
  if (host_fam)
    for (uint32_t i = blockIdx.x * blockDim.x + t; i < n_fam; i += gridDim.x * blockDim.x) host_fam[i] = fam_ll[i];
  if (blockIdx.x > 0) return;
  const AccLayout AL(n, M.n_wgd);
  double *const EB = InLds ? s_work : work, *const SL = EB + n, *const E0 = SL + n, *const TOP = E0 + n;
  // the last wave forms the conditioning term while the others load
  if (t == kTailThreads - 1) s_ct = cond_terms(M, cond);
  NodeDev mine{};
  int me = -1, lv = -1;
  if (with_grad) {
    for (int e = t; e < n; e += blockDim.x) {
      const double* dn = M.dnode + (size_t)kDnode * e;
      EB[e] = acc_in[AL.eps + e];
      SL[e] = dn[7];
      E0[e] = acc_in[AL.e0 + e];
      TOP[e] = eps_top(M, e);
    }
    if (t < n) {  // a lane's own entry of dnodes, in level lv
      me = dnodes[t];
      mine = M.node[me];
      int lo = 0, hi = n_dlevels;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (dlevels[mid] <= t) lo = mid;
        else hi = mid;
      }
      lv = lo;
    }
  }
  if (t == 0 && host_fb) *host_fb = fb ? *fb : 0u;
  // Σ ℓ_i
  double s = 0;
#pragma unroll 4
  for (uint32_t i = t; i < n_fam; i += blockDim.x) s += fam_ll[i];
  s = group_sum(s, part);  // its barrier also shows s_ct and the arrays
  const CondTerms CT = s_ct;
  if (t == 0) {
    const double tot = s - (double)n_fam * CT.c;
    out[0] = isfinite(tot) ? tot : -INFINITY;
  }
  if (!with_grad) return;
  if (t == 0) {
    // ε̄ of the top rows: conditioning and root A/B terms beside the DP's
    const NodeDev& rn = M.node[M.root];
    const double eta = M.par[3 * n + M.n_wgd];
    const double er = TOP[M.root];
    const double A_ = acc_in[AL.rootA], B_ = acc_in[AL.rootB];
    const double xi = 1.0 - (1.0 - eta) * er;
    const double dA_deta = (-xi + (1.0 - eta) * er) / eta - (1.0 - eta) * xi / (eta * eta);
    const double dA_der = -(1.0 - eta) * (1.0 - eta) / eta;
    const double dB_deta = (1.0 - er) / (xi * xi) - 2.0 * eta * (1.0 - er) * er / (xi * xi * xi);
    const double dB_der = -eta / (xi * xi) + 2.0 * eta * (1.0 - er) * (1.0 - eta) / (xi * xi * xi);
    const double Ng = n_eff ? *n_eff : (double)n_fam;  // the families' weight in the gradient
    EB[M.root] += A_ * dA_der + B_ * dB_der - Ng * CT.dc_er;
    EB[rn.child0] += -Ng * CT.dc_ef;
    EB[rn.child1] += -Ng * CT.dc_eg;
    out[1 + 2 * n + M.n_wgd] = A_ * dA_deta + B_ * dB_deta - Ng * CT.dc_eta;
  }
  __syncthreads();
  // parents before children: ε̄ of a node's row 0 into its children's tops
  // (row 0 of ε: the product of the children's tops, or the WGD retention map)
  auto down = [&](int e, const NodeDev& d) {
    const double g = SL[e] * EB[e] + E0[e];
    if (d.kind == WHALE_NODE_WGD) {
      const double qq = M.par[3 * n + d.wgd];
      EB[d.child0] += g * (2.0 * qq * TOP[d.child0] + (1.0 - qq));
    } else if (d.kind == WHALE_NODE_SPECIATION || d.kind == WHALE_NODE_ROOT) {
      EB[d.child0] += g * TOP[d.child1];
      EB[d.child1] += g * TOP[d.child0];
    }
  };
  for (int L = 0; L < n_dlevels; ++L) {
    if (lv == L) down(me, mine);
    for (int k = t + (int)blockDim.x; k < n; k += blockDim.x)  // trees of more nodes than lanes
      if (k >= dlevels[L] && k < dlevels[L + 1]) down(dnodes[k], M.node[dnodes[k]]);
    __syncthreads();
  }
  double* dl = out + 1;
  double* dm = out + 1 + n;
  double* dq = out + 1 + 2 * n;
  for (int e = t; e < n; e += blockDim.x) {
    const NodeDev& d = M.node[e];
    const double* dn = M.dnode + (size_t)kDnode * e;
    const double gt = EB[e];
    const double ga = dn[8] * gt + acc_in[AL.da + e], gb = dn[9] * gt + acc_in[AL.db + e];
    dl[e] = d.R > 1 ? ga * dn[0] + gb * dn[2] : 0.0;
    dm[e] = d.R > 1 ? ga * dn[1] + gb * dn[3] : 0.0;
    if (d.kind == WHALE_NODE_WGD) {
      const double ec = TOP[d.child0];
      dq[d.wgd] = acc_in[AL.q + d.wgd] + (SL[e] * gt + E0[e]) * (ec * ec - ec);
    }
  }
}

// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, uint32_t v, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}
// k_reset: what an evaluation starts from, in one launch: its tickets, the
// gradient's accumulators (n_acc 0: none) and the FP32 form's flags and count
// of flagged families (n_flag 0: none).
__global__ void k_reset(uint32_t* ticket, int n_ticket, double* acc, int n_acc, uint32_t* flag, int n_flag,
                        uint32_t* fb) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
  for (int i = i0; i < n_ticket; i += step) ticket[i] = 0u;
  for (int i = i0; i < n_acc; i += step) acc[i] = 0.0;
  for (int i = i0; i < n_flag; i += step) flag[i] = 0u;
  if (i0 == 0 && n_flag > 0) fb[0] = 0u;
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
static size_t real_size(int mode) { return mode == WHALE_FP32_SCALED ? sizeof(float) : sizeof(double); }

// node constants: ε at the top, leafℙ, q; for the reverse sweep also 1/(1-α), 1/(1-β), β
static size_t nodec_bytes(size_t real, bool bwd, int n, int nwgd) {
  return align16(((bwd ? 5 : 2) * (size_t)n + (size_t)(nwgd > 0 ? nwgd : 1)) * real);
}

size_t fwd_shared_bytes(int mode, int n, int nwgd) {
  const size_t s = real_size(mode);
  return kCtlBytes + nodec_bytes(s, false, n, nwgd);
}

size_t bwd_shared_bytes(int mode, int n, int nwgd) {
  const size_t s = real_size(mode);
  return kCtlBytes + acc_lds_bytes(AccLayout(n, nwgd).n) +
         nodec_bytes(s, true, n, nwgd);
}

hipError_t launch_forward(int mode, bool store_all, const LaunchCfg& C, hipStream_t st, const BatchDev& B,
                          const ModelDev& M, const WorkRaw& W, int32_t fam_single, uint32_t fam_begin,
                          uint32_t fam_end, const uint32_t* fam_count, const MixComp* X, int K) {
  if (mode == WHALE_FP64_PLAIN)
    return fwd_variant<double, false>(store_all, C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
  if (mode == WHALE_FP32_SCALED)
    return fwd_variant<float, true>(store_all, C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
  return fwd_variant<double, true>(store_all, C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
}

hipError_t launch_backward(int mode, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                           const WorkRaw& W, int32_t fam_single, uint32_t fam_begin, uint32_t fam_end,
                           const uint32_t* fam_count, const MixComp* X, int K) {
  if (mode == WHALE_FP64_PLAIN)
    return bwd_variant<double, false>(C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
  if (mode == WHALE_FP32_SCALED)
    return bwd_variant<float, true>(C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
  return bwd_variant<double, true>(C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
}

hipError_t launch_fused(int mode, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                        const WorkRaw& W, uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count, int grad,
                        const FusedSlots& SL) {
  if (mode == WHALE_FP64_PLAIN)
    return fused_variant<double, false>(C, st, B, M, W, fam_begin, fam_end, fam_count, grad, SL);
  if (mode == WHALE_FP32_SCALED)
    return fused_variant<float, true>(C, st, B, M, W, fam_begin, fam_end, fam_count, grad, SL);
  return fused_variant<double, true>(C, st, B, M, W, fam_begin, fam_end, fam_count, grad, SL);
}

hipError_t launch_mix(hipStream_t st, const MixComp* X, int K, const double* log_prior, uint32_t n_fam, int cond,
                      double* out, double* resp) {
  if (K < 1 || K > kMaxMix) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mix, dim3(1), dim3(1024), 0, st, X, K, log_prior, n_fam, cond, out, resp);
  return hipGetLastError();
}

hipError_t launch_tables(hipStream_t st, const ModelDev& M, double* eps, double* phi, double* psi, double* pack64,
                         float* pack32, double* dnode, const int32_t* hlevels, const int32_t* hnodes, int n_levels,
                         const int32_t* row_node, double* work) {
  const size_t lds = tables_work_bytes(M.n, M.tab_rows);
  if (work) {
    hipLaunchKernelGGL(k_tables<false>, dim3(1), dim3(1024), 0, st, M, eps, phi, psi, pack64, pack32, dnode, hlevels,
                       hnodes, n_levels, row_node, work);
    return hipGetLastError();
  }
  if (lds > kTabLds) return hipErrorInvalidValue;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tables<true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_tables<true>, dim3(1), dim3(1024), lds, st, M, eps, phi, psi, pack64, pack32, dnode, hlevels,
                     hnodes, n_levels, row_node, work);
  return hipGetLastError();
}

hipError_t launch_tail(hipStream_t st, const ModelDev& M, const double* fam_ll, uint32_t n_fam, const double* acc,
                       double* work, const int32_t* dlevels, const int32_t* dnodes, int n_dlevels, int cond,
                       int with_grad, double* out, const double* n_eff, double* host_fam, const uint32_t* fb,
                       uint32_t* host_fb) {
  // a workgroup for every 2048 families that go to the host
  const int grid = host_fam ? (int)std::min<uint32_t>(64, 1 + (n_fam - 1) / 2048) : 1;
  const size_t lds = tail_work_bytes(M.n);
  if (!with_grad || lds <= kTailLds)
    hipLaunchKernelGGL(k_tail<true>, dim3(grid), dim3(kTailThreads), with_grad ? lds : 0, st, M, fam_ll, n_fam, acc,
                       work, dlevels, dnodes, n_dlevels, cond, with_grad, out, n_eff, host_fam, fb, host_fb);
  else
    hipLaunchKernelGGL(k_tail<false>, dim3(grid), dim3(kTailThreads), 0, st, M, fam_ll, n_fam, acc, work, dlevels,
                       dnodes, n_dlevels, cond, with_grad, out, n_eff, host_fam, fb, host_fb);
  return hipGetLastError();
}
hipError_t launch_reset(hipStream_t st, uint32_t* ticket, int n_ticket, double* acc, int n_acc, uint32_t* flag,
                        int n_flag, uint32_t* fb) {
  const int most = std::max(std::max(n_ticket, n_acc), n_flag);
  hipLaunchKernelGGL(k_reset, dim3(std::min(64, (most + 255) / 256)), dim3(256), 0, st, ticket, n_ticket, acc, n_acc,
                     flag, n_flag, fb);
  return hipGetLastError();
}
hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t v, int n) {
  hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, p, v, n);
  return hipGetLastError();
}


// ---------------------------------------------------------------------------
// k_backtrack: stochastic backtracking of reconciled trees from the stored ℓ
// (backtrack!, src/track.jl:188-414).  One wave per (family, sample): a depth
// first walk over slice states (species node e, clade γ,
// slice row t) that picks each event with probability term / ℓ_e(γ, t), the
// terms taken in the reference's order: inside a branch "no event"
// (φ_t ℓ(γ, t-1)) then each duplication (p ψ_t ℓ(γ1, t-1) ℓ(γ2, t-1)); at a
// speciation node the two losses then both speciations of every split; at a
// WGD node non-retention ((1 - q + 2qε_f) ℓ_f(γ)) then each retained split; at
// the root each split's root duplication (ξ(1-η)/η) and both speciations
// (η(1-ε)/ξ²), then the two losses.  Uniform draws come from a counter-based
// generator of (seed, family, sample), one per inter- or intra-branch step in
// depth-first order.  Scaled forms: every term is formed relative to 2^E(γ) of
// the state's clade.
//
// A walk is a chain of dependent loads (the clade's column in a segment, ℓ),
// so the lanes take what does not depend on each other: the rows of a branch
// that the walk may pass without an event (a lane a row, each with its own
// draw of the counter), and the splits of a state (a lane a split).  The terms
// are subtracted from the draw one by one in order.  What the walk needs of
// every branch is gathered in LDS first.  Measured (100 families of 8 to 120
// genes on 13 taxa, 4 trees each): one lane a walk 11.9 ms, this 0.75 ms; with
// the call's copies 13.5 ms, and by groups of 4, 16 and 64 lanes 4.1, 2.9 and
// 2.0 ms.  64,000 walks of 1000 families: 87 ms, now 31 (groups of 4: 42).
// ---------------------------------------------------------------------------
constexpr uint64_t kBtStep = 0x9E3779B97F4A7C15ull;
__device__ __forceinline__ double bt_uniform(uint64_t st) {  // the draw of counter st
  uint64_t z = st;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * 0x1.0p-53;
}

struct BtCell {
  double v;  // stored value (0 when the clade is not compatible with the branch)
  int E;     // its clade's exponent (0 in the plain form)
};
// a branch of the family: its node and its segment's clades and ℓ block (nc =
// 0: none)
struct BtBranch {
  uint64_t ell;
  uint32_t nc, R, item0;
  int32_t kind, fc, gc, tab, wgd;
  double eps;   // ε at the top
};

struct BtCtx {
  const BtDev& D;
  const ModelDev& M;
  FamDev F;
  uint32_t f;
  bool f64;  // this family's ℓ is in the FP64 region
  const BtBranch* lds;  // all branches in LDS, or null
  __device__ __forceinline__ BtBranch gather(int e) const {
    const NodeDev& nd = M.node[e];
    BtBranch b{0, 0u, (uint32_t)nd.R, 0u, nd.kind, nd.child0, nd.child1, nd.tab, nd.wgd, eps_top(M, e)};
    const int32_t s = D.node_seg[(size_t)f * M.n + e];
    if (s < 0) return b;
    const SegDev sg = D.seg[s];
    b.item0 = D.seg_item[s];
    b.ell = F.ell0 + sg.ell;
    b.nc = sg.nc;
    return b;
  }
  __device__ __forceinline__ BtBranch branch(int e) const { return lds ? lds[e] : gather(e); }
  const uint16_t* ids;  // the family's items' clades in LDS, or null
  // columns of N clades in branch b (~0: not compatible): the segment's clades
  // are in increasing id, the root's are all clades in order
  template <int N>
  __device__ __forceinline__ void columns(const BtBranch& b, const int (&g)[N], uint32_t (&col)[N]) const {
    if (b.nc == 0 || b.kind == WHALE_NODE_ROOT) {
#pragma unroll
      for (int i = 0; i < N; ++i) col[i] = b.nc ? (uint32_t)g[i] : ~0u;
    } else if (ids) {
      search(ids + (b.item0 - F.item0), b.nc, g, col);
    } else {
      search(D.it_gid + b.item0, b.nc, g, col);
    }
  }
  template <int N, typename Id>
  __device__ __forceinline__ static void search(const Id* id, uint32_t nc, const int (&g)[N], uint32_t (&col)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) col[i] = 0u;  // clades of the segment below g
    for (uint32_t step = 1u << (31 - __clz((int)nc)); step; step >>= 1) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const uint32_t x = col[i] + step;
        if (x <= nc && id[x - 1] < (uint32_t)g[i]) col[i] = x;
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (col[i] == nc || id[col[i]] != (uint32_t)g[i]) col[i] = ~0u;
  }
  // ℓ of column col of branch b at row t
  __device__ __forceinline__ BtCell cell(const BtBranch& b, uint32_t col, int g, int t) const {
    BtCell c{0.0, 0};
    if (col == ~0u || t < 1 || (uint32_t)t > b.R) return c;
    const uint64_t idx = b.ell + (uint64_t)(t - 1) * b.nc + col;
    c.v = f64 ? D.ell64[idx] : (D.ell_float ? (double)((const float*)D.ell)[idx] : ((const double*)D.ell)[idx]);
    if (D.E && c.v != 0.0) c.E = D.E[F.clade0 + g];
    return c;
  }
};

// term x·a·b relative to 2^Eg, a, b two cells
__device__ __forceinline__ double bt_rel2(double x, const BtCell& a, const BtCell& b, int Eg) {
  if (a.v == 0.0 || b.v == 0.0 || x == 0.0) return 0.0;
  return ldexp(x * a.v * b.v, a.E + b.E - Eg);
}
__device__ __forceinline__ double bt_rel1(double x, const BtCell& a, int Eg) {
  if (a.v == 0.0 || x == 0.0) return 0.0;
  return ldexp(x * a.v, a.E - Eg);
}

struct BtState {
  int e, g, t;
};
// events; a split's are kept as event | split << 3
enum BtEvent { kBtRootDup, kBtSpec, kBtSpecSwap, kBtLossG, kBtLossF, kBtNoWgd, kBtWgd, kBtDup, kBtNone = -1 };

// states a walk keeps on its stack in LDS; one that needs more keeps
// the others in global memory
constexpr uint32_t kBtStack = 64;

__global__ __launch_bounds__(64) void k_backtrack(BtDev D, ModelDev M, uint32_t fam_begin, uint32_t n_fams,
                                                  uint32_t n_samples, uint64_t seed, uint32_t cap, int32_t* counts,
                                                  int32_t* nodes, int32_t* stack, int staged, uint32_t staged_ids) {
  // BtBranch[n] when staged; then the clades of the family's items, if there
  // are no more than staged_ids
  extern __shared__ __align__(16) unsigned char s_branch[];
  __shared__ int4 s_stack[kBtStack];
  const uint32_t lane = threadIdx.x;
  const uint64_t id = blockIdx.x + (uint64_t)blockIdx.y * gridDim.x;
  if (id >= (uint64_t)n_fams * n_samples) return;
  const uint32_t fi = (uint32_t)(id / n_samples), smp = (uint32_t)(id % n_samples);
  const uint32_t f = fam_begin + fi;
  BtCtx X{D, M, D.fam[f], f, D.fam64 ? D.fam64[f] != 0 : false, nullptr, nullptr};
  if (staged) {
    BtBranch* const all = (BtBranch*)s_branch;
    uint16_t* const ids = (uint16_t*)(all + M.n);
    const bool fit = X.F.n_items <= staged_ids;
    for (int e = (int)lane; e < M.n; e += 64) all[e] = X.gather(e);
    if (fit)
      for (uint32_t i = lane; i < X.F.n_items; i += 64) ids[i] = (uint16_t)D.it_gid[X.F.item0 + i];
    __syncthreads();
    X.lds = all;
    if (fit) X.ids = ids;
  }
  uint64_t st = seed ^ (kBtStep * (uint64_t)(f + 1)) ^ (0xD1B54A32D192ED03ull * (uint64_t)(smp + 1));
  int4* const out = (int4*)nodes + id * (uint64_t)cap;
  int4* const deep = (int4*)stack + id * (uint64_t)cap;
  const double eta = M.par[3 * M.n + M.n_wgd];
  uint32_t n = 0, sp = 0;
  bool over = false;

  auto lane_of = [](double x, int l) -> double {
    const long long y = __builtin_bit_cast(long long, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)y, l), hi = (uint32_t)__builtin_amdgcn_readlane((int)(y >> 32), l);
    return __builtin_bit_cast(double, (long long)(((uint64_t)hi << 32) | lo));
  };
  auto add = [&](const BtState& s, int par) -> int {
    if (n >= cap) {
      over = true;
      return -1;
    }
    if (lane == 0) out[n] = make_int4(s.g, s.e, s.t, par);
    return (int)n++;
  };

  BtState s{M.root, (int)X.F.n_clades - 1, 1};
  int cur = add(s, -1);
  int ce = s.e, cg = s.g;  // the branch and clade of node cur
  while (!over) {
    // The state s at node `cur`; a branch of the walk ends at a leaf or a loss.
    // r is what is left of the draw, `hit` the event at which it fell below 0,
    // `last` the last one with weight.
    double r = 0.0;
    int hit = kBtNone, last = kBtNone;
    auto take = [&](double x, int event) {
      if (hit != kBtNone || !(x > 0.0)) return;
      last = event;
      r -= x;
      if (r < 0.0) hit = event;
    };
    // the N terms of each split k0..k1, in order: fill(k, x) forms split k's
    auto splits = [&](auto n_, uint32_t k0, uint32_t k1, const int (&event)[3], auto&& fill) {
      constexpr int N = decltype(n_)::value;
      for (uint32_t kb = k0; kb < k1 && hit == kBtNone; kb += 64) {
        double x[N];
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = 0.0;
        if (kb + lane < k1) fill(kb + lane, x);
        bool any = false;
#pragma unroll
        for (int i = 0; i < N; ++i) any |= x[i] > 0.0;
        for (uint64_t m = __ballot(any); m && hit == kBtNone; m &= m - 1) {
          const int l = __builtin_ctzll(m);
#pragma unroll
          for (int i = 0; i < N; ++i) take(lane_of(x[i], l), event[i] | (int)((kb + (uint32_t)l - k0) << 3));
        }
      }
    };
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, 3> I3;
    uint32_t k0 = 0;
    if (s.g >= 0) {
      const BtBranch b = X.branch(s.e);
      const uint32_t ca = X.F.clade0 + (uint32_t)s.g;
      k0 = D.spl_off[ca];
      const uint32_t k1 = D.spl_off[ca + 1];
      const int gs[1] = {s.g};
      uint32_t col[1];
      X.columns(b, gs, col);
      if (s.t > 1 && D.clade_size[ca] == 1) s.t = 1;  // a one-gene clade does not duplicate along the branch
      while (s.t > 1) {
        // lane j: the step from row t - j, had the steps before it no event
        const int row = s.t - (int)lane;
        const BtCell me = X.cell(b, col[0], s.g, row), lo = X.cell(b, col[0], s.g, row - 1);
        double left = bt_uniform(st + (uint64_t)(lane + 1) * kBtStep) * me.v;
        if (row > 1) left -= bt_rel1(M.phi[b.tab + row - 1], lo, me.E);
        const uint64_t m = __ballot(row > 1 && !(left < 0.0));
        if (m == 0) {
          const int steps = min(64, s.t - 1);
          st += (uint64_t)steps * kBtStep;
          s.t -= steps;
          continue;
        }
        const int l = __builtin_ctzll(m);
        st += (uint64_t)(l + 1) * kBtStep;
        s.t -= l;
        r = lane_of(left, l);
        const int Eg = __builtin_amdgcn_readlane(me.E, l);
        const double ps = M.psi[b.tab + s.t - 1];
        const int ev[3] = {kBtDup, 0, 0};
        splits(I1{}, k0, k1, ev, [&](uint32_t k, double (&x)[1]) {
          const int g[2] = {(int)(D.spl_g[k] & 0xffff), (int)(D.spl_g[k] >> 16)};
          uint32_t c[2];
          X.columns(b, g, c);
          x[0] = bt_rel2(D.split_p[k] * ps, X.cell(b, c[0], g[0], s.t - 1), X.cell(b, c[1], g[1], s.t - 1), Eg);
        });
        s.t -= 1;
        if (last != kBtNone) break;  // the split where r fell below 0, or (rounding) the last one with weight
      }                              // otherwise only "no event" has weight
      if (last == kBtNone && b.kind != WHALE_NODE_LEAF) {
        const BtCell me = X.cell(b, col[0], s.g, 1);
        const int Eg = me.E;
        st += kBtStep;
        r = bt_uniform(st) * me.v;
        const int fc = b.fc, gc = b.gc;
        const BtBranch bf = X.branch(fc);
        const int tf = (int)bf.R;
        if (b.kind == WHALE_NODE_WGD) {
          const double q = M.par[3 * M.n + b.wgd];
          uint32_t c1[1];
          X.columns(bf, gs, c1);
          take(bt_rel1(1.0 - q + 2.0 * q * bf.eps, X.cell(bf, c1[0], s.g, tf), Eg), kBtNoWgd);
          const int ev[3] = {kBtWgd, 0, 0};
          splits(I1{}, k0, k1, ev, [&](uint32_t k, double (&x)[1]) {
            const int g[2] = {(int)(D.spl_g[k] & 0xffff), (int)(D.spl_g[k] >> 16)};
            uint32_t c[2];
            X.columns(bf, g, c);
            x[0] = bt_rel2(q * D.split_p[k], X.cell(bf, c[0], g[0], tf), X.cell(bf, c[1], g[1], tf), Eg);
          });
        } else {
          const BtBranch bg = X.branch(gc);
          const int tg = (int)bg.R;
          double cA = 0.0, cB = 1.0;
          if (b.kind == WHALE_NODE_ROOT) {
            const double eps = b.eps, xi = 1.0 - (1.0 - eta) * eps;
            cA = xi * (1.0 - eta) / eta;
            cB = eta * (1.0 - eps) / (xi * xi);
          }
          uint32_t cf[1], cg_[1];
          X.columns(bf, gs, cf);
          X.columns(bg, gs, cg_);
          const double lossg = bt_rel1(bg.eps * cB, X.cell(bf, cf[0], s.g, tf), Eg);
          const double lossf = bt_rel1(bf.eps * cB, X.cell(bg, cg_[0], s.g, tg), Eg);
          auto spec = [&](uint32_t k, double p, double* x) {
            const int g[2] = {(int)(D.spl_g[k] & 0xffff), (int)(D.spl_g[k] >> 16)};
            uint32_t c[2], d[2];
            X.columns(bf, g, c);
            X.columns(bg, g, d);
            x[0] = bt_rel2(p, X.cell(bf, c[0], g[0], tf), X.cell(bg, d[1], g[1], tg), Eg);
            x[1] = bt_rel2(p, X.cell(bg, d[0], g[0], tg), X.cell(bf, c[1], g[1], tf), Eg);
          };
          if (b.kind == WHALE_NODE_ROOT) {
            const int ev[3] = {kBtRootDup, kBtSpec, kBtSpecSwap};
            splits(I3{}, k0, k1, ev, [&](uint32_t k, double (&x)[3]) {
              const int g1 = (int)(D.spl_g[k] & 0xffff), g2 = (int)(D.spl_g[k] >> 16);
              const double p = D.split_p[k];
              x[0] = bt_rel2(p * cA, X.cell(b, (uint32_t)g1, g1, 1), X.cell(b, (uint32_t)g2, g2, 1), Eg);
              spec(k, p * cB, x + 1);
            });
          }
          take(lossg, kBtLossG);
          take(lossf, kBtLossF);
          if (b.kind != WHALE_NODE_ROOT) {
            const int ev[3] = {kBtSpec, kBtSpecSwap, 0};
            splits(I2{}, k0, k1, ev, [&](uint32_t k, double (&x)[2]) { spec(k, D.split_p[k], x); });
          }
        }
      }
    }
    const int event = hit != kBtNone ? hit : last;  // rounding may leave r >= 0: the last one with weight
    if (event != kBtNone) {
      // next states in the reference's order: the first is walked first
      const BtBranch b = X.branch(s.e);
      const int fc = b.fc, gc = b.gc, kind = event & 7;
      const uint32_t g12 = kind < kBtLossG || kind > kBtNoWgd ? D.spl_g[k0 + (uint32_t)(event >> 3)] : 0u;
      const int g1 = (int)(g12 & 0xffff), g2 = (int)(g12 >> 16);
      auto top = [&](int e) -> int { return (int)X.branch(e).R; };
      BtState a, z{0, 0, 0};
      switch (kind) {
        case kBtRootDup: a = {s.e, g1, 1}, z = {s.e, g2, 1}; break;
        case kBtSpec: a = {fc, g1, top(fc)}, z = {gc, g2, top(gc)}; break;
        case kBtSpecSwap: a = {gc, g1, top(gc)}, z = {fc, g2, top(fc)}; break;
        case kBtLossG: a = {fc, s.g, top(fc)}, z = {gc, -1, 0}; break;
        case kBtLossF: a = {gc, s.g, top(gc)}, z = {fc, -1, 0}; break;
        case kBtNoWgd: a = {fc, s.g, top(fc)}; break;
        case kBtWgd: a = {fc, g1, top(fc)}, z = {fc, g2, top(fc)}; break;
        default: a = {s.e, g1, s.t}, z = {s.e, g2, s.t}; break;
      }
      const uint32_t nn = kind == kBtNoWgd ? 1u : 2u;
      if (sp + nn > cap) {
        over = true;
        break;
      }
      // a new node when its (clade, branch) differs from the node it came from
      // ((b::BackTracker)(newstate), src/track.jl:172-180): known already here
      if (nn == 2) {
        const bool same = z.g == cg && z.e == ce;
        const int4 q = make_int4(z.e, z.g, z.t | (same ? INT32_MIN : 0), cur);
        if (lane == 0) {
          if (sp < kBtStack) s_stack[sp] = q;
          else deep[sp] = q;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        ++sp;
      }
      s = a;
      if (a.g != cg || a.e != ce) {
        cur = add(a, cur);
        ce = a.e, cg = a.g;
      }
    } else {
      if (sp == 0) break;
      --sp;
      int4 q = make_int4(0, 0, 0, 0);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (sp < kBtStack) {
        q = s_stack[sp];
      } else {
        if (lane == 0) q = deep[sp];  // by the lane that wrote it
        q.x = __builtin_amdgcn_readfirstlane(q.x);
        q.y = __builtin_amdgcn_readfirstlane(q.y);
        q.z = __builtin_amdgcn_readfirstlane(q.z);
        q.w = __builtin_amdgcn_readfirstlane(q.w);
      }
      s = {q.x, q.y, q.z & INT32_MAX};
      ce = s.e, cg = s.g;
      cur = q.w;
      if (q.z >= 0) cur = add(s, cur);
    }
  }
  if (lane == 0) counts[id] = over ? -1 : (int32_t)n;
}

// one workgroup per walk
static dim3 bt_grid(uint64_t walks) {
  const uint64_t x = std::min<uint64_t>(walks, 1u << 30);
  return dim3((uint32_t)x, (uint32_t)((walks + x - 1) / x));
}

hipError_t launch_backtrack(hipStream_t st, const BtDev& D, const ModelDev& M, uint32_t fam_begin, uint32_t n_fams,
                            uint32_t n_samples, uint64_t seed, uint32_t cap, int32_t* counts, int32_t* nodes,
                            int32_t* stack, uint32_t max_items) {
  const uint64_t walks = (uint64_t)n_fams * n_samples;
  if (walks == 0) return hipSuccess;
  // In LDS: the branches of trees of up to 512 nodes, then the items' clades
  // of families of up to 8000 or so; larger ones read them from global
  // memory at each step.  24 KB a walk leave six walks to a compute unit.
  const size_t lim = 24 * 1024, lds = sizeof(BtBranch) * (size_t)M.n;
  const int staged = lds <= lim;
  const uint32_t ids = staged ? std::min<uint32_t>(max_items, (uint32_t)((lim - lds) / 2)) : 0u;
  hipLaunchKernelGGL(k_backtrack, bt_grid(walks), dim3(64), staged ? lds + 2 * (size_t)ids : 0, st, D, M,
                     fam_begin, n_fams, n_samples, seed, cap, counts, nodes, stack, staged, ids);
  return hipGetLastError();
}

// k_bt_pack: the walks' nodes one after the other, so that only what they hold
// is copied to the host: walk i's start at first[i], at its turn at `cursor`.
__global__ __launch_bounds__(64) void k_bt_pack(const int32_t* counts, const int4* nodes, uint64_t walks,
                                                uint32_t cap, unsigned long long* first, unsigned long long* cursor,
                                                int4* packed) {
  const uint64_t id = blockIdx.x + (uint64_t)blockIdx.y * gridDim.x;
  if (id >= walks) return;
  const int n = counts[id];
  if (n <= 0) return;
  __shared__ unsigned long long s_at;
  if (threadIdx.x == 0) first[id] = s_at = atomicAdd(cursor, (unsigned long long)n);
  __syncthreads();
  const uint64_t at = s_at;
  for (int i = (int)threadIdx.x; i < n; i += 64) packed[at + i] = nodes[id * cap + i];
}

hipError_t launch_bt_pack(hipStream_t st, uint64_t walks, const int32_t* counts, const int32_t* nodes, uint32_t cap,
                          uint64_t* first, uint64_t* cursor, int32_t* packed) {
  hipLaunchKernelGGL(k_bt_pack, bt_grid(walks), dim3(64), 0, st, counts, (const int4*)nodes, walks, cap,
                     (unsigned long long*)first, (unsigned long long*)cursor, (int4*)packed);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// k_det_sum: the batch's gradient accumulators as the sum of the per-family
// slots in an order that depends on the number of families alone, so that the
// result does not depend on which workgroup evaluated which family, or when.
// A workgroup sums 16 accumulators (a 128-byte line of every slot), 64 lanes
// each; lane r takes families r, r + 64, …, and the lanes' sums are added
// pairwise.  One lane an accumulator is a chain of n_fam loads: 190 us for 777
// families of 50 taxa.
// ---------------------------------------------------------------------------
constexpr int kDetCols = 16, kDetLanes = 64;
__global__ __launch_bounds__(kDetCols * kDetLanes) void k_det_sum(const double* slots, uint32_t n_fam, int ncol,
                                                                  double* out) {
  __shared__ double s[kDetLanes][kDetCols];
  const int c = threadIdx.x % kDetCols, r = threadIdx.x / kDetCols;
  const int j = blockIdx.x * kDetCols + c;
  double t = 0.0;
  if (j < ncol) {
#pragma unroll 8
    for (uint32_t f = (uint32_t)r; f < n_fam; f += kDetLanes) t += slots[(size_t)f * ncol + j];
  }
  s[r][c] = t;
  for (int w = kDetLanes / 2; w > 0; w >>= 1) {
    __syncthreads();
    if (r < w) s[r][c] += s[r + w][c];
  }
  if (r == 0 && j < ncol) out[j] = s[0][c];
}

hipError_t launch_det_sum(hipStream_t st, const double* slots, uint32_t n_fam, int ncol, double* out) {
  hipLaunchKernelGGL(k_det_sum, dim3((ncol + kDetCols - 1) / kDetCols), dim3(kDetCols * kDetLanes), 0, st, slots, n_fam,
                     ncol, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// fixed workspace of the evaluation that allocates nothing
// ---------------------------------------------------------------------------
// Every GPU the library runs on holds one copy of this array until the
// process ends.  Host code never passes its name to a kernel (on the host it
// is a stand-in, not a device address): the device address of each GPU's copy
// comes from hipGetSymbolAddress, once per device, and only that is used.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

hipError_t scratch_address(int device, void** out) {
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device) return hipErrorInvalidDevice;  // the caller makes `device` current
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[device] = p;
  }
  *out = addr[device];
  return hipSuccess;
}

}  // namespace whale
