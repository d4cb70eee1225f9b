// Device code of the amalgamated-likelihood DP: the forward recursion and the
// reverse sweep of one family, and the kernels that run them over a batch.
// Each arithmetic has its own translation unit (dp_fp64.hip, dp_fp32.hip,
// dp_fp64s.hip), which instantiates the launch templates at the end.
//
//   k_forward      the DP of every family (whale!/whalewgd!/within_branch!/
//                  whaleroot!, src/core.jl:83-158), one family per wavefront
//                  (several families per workgroup) or per team of up to
//                  kMaxTeam wavefronts, stage by stage, the items of a stage in
//                  lockstep row by row, row buffers in LDS
//   k_backward     reverse sweep of the same DAG: d logL / d ℓ, accumulated
//                  into d logL / d(α, β, ε of row 0, ε, q, A, B) per node
//   k_fused        both for one family after the other, under a memory budget
//
// Precision: Real = double (plain: exactly the reference's recursion) or
// float/double with per-clade power-of-two exponents (Scaled).  In the scaled
// forms the value of clade γ is stored as v = ℓ·2^-E(γ) with one exponent per
// (family, clade), fixed the first time γ gets a non-zero value.  Because
// every term of the recursion multiplies ℓ(γ1)·ℓ(γ2) into ℓ(γ) or carries
// ℓ(γ) itself, all scaling folds into one coefficient per split,
// p·2^(E(γ1)+E(γ2)-E(γ)); rows then run on plain Real arithmetic.
//
// What bounds these kernels is the chain of dependent rows of a family (a
// stage's row r needs all of row r-1): some hundred rows, each a trip through
// LDS.  The layout (plan.hpp) makes that trip as short as it can be: an item's
// lane gathers its splits' parts, adds them, applies φ_r and ψ_r to the value
// it holds in a register and writes the new value to the other row buffer, one
// LDS round trip per row with no atomics; the reverse sweep does the same over
// the splits an item is a part of.  Everything constant over the rows sits in
// registers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "dev.hpp"
#include "../../include/whale_amd.h"

// a lambda that is part of its function's body: kept out of line, the lanes'
// state it takes by reference would live in scratch memory
#define WHALE_INLINE __attribute__((always_inline))

namespace whale {

constexpr int kUndef = -0x40000000;  // exponent not yet fixed
constexpr int kWG = 64;              // lanes of a wave
// A clade's exponent is fixed at its first non-zero value, which can be far
// smaller than its later values (e.g. a large in-paralog clade grows by ~2^120
// along one branch as more slices become available for its duplications).
// New non-leaf clades therefore start at 2^-kBirth, leaving 2^(128+kBirth) of
// growth and 2^-(126-kBirth) of decay before FP32 runs out of range; a family
// that still leaves the range is recomputed in FP64 (see k_forward's flag).
constexpr int kBirth = 40;
// A clade that had no value before the current stage ("young") may still grow
// by many powers of two within this stage's branch (a large in-paralog clade
// gains a factor per slice as more slices hold its duplications).  Because it
// has no stored values elsewhere, its exponent can be raised in place: when
// its FP32 value passes 2^kBump the clade is renormalised and the rows it
// already wrote on this branch are rescaled.  The window [2^-kBirth, 2^kBump]
// is kept narrow because a split's coefficient p·2^(E1+E2-E) spans the ratio
// of the parent's value to the product of its parts' values (two windows and
// one 1/ψ): 2^(kBump + 2·kBirth + log2(1/ψ)) must stay inside FP32.  A narrow
// window also ends the stage low, with room to grow in the stages above.
constexpr int kBump = 16;
template <typename Real>
struct WorkDev {
  Real* ell;
  int32_t* E;         // per clade (scaled forms)
  int32_t* Eit;       // per item: its clade's exponent at the end of its stage (scaled forms, stored rows)
  Real* ibar;
  double* fam_ll;
  double* acc;        // gradient accumulators
  uint32_t* ticket;
  uint32_t* flag;
  uint32_t* fb;
  unsigned char* gws;
  double* acc_fam;    // deterministic gradients: per-family accumulator slots (null otherwise)
  double* seed;       // per-family weights of the reverse sweep (null: 1)
  __host__ __device__ explicit WorkDev(const WorkRaw& w)
      : ell((Real*)w.ell), E(w.E), Eit(w.Eit), ibar((Real*)w.ibar), fam_ll(w.fam_ll), acc(w.acc), ticket(w.ticket),
        flag(w.flag), fb(w.fb), gws(w.gws), acc_fam(w.acc_fam), seed(w.seed) {}
};

template <typename Real>
__device__ __forceinline__ Real frexp_r(Real x, int* e);
template <>
__device__ __forceinline__ float frexp_r<float>(float x, int* e) { return frexpf(x, e); }
template <>
__device__ __forceinline__ double frexp_r<double>(double x, int* e) { return frexp(x, e); }
template <typename Real>
__device__ __forceinline__ Real ldexp_r(Real x, int e);
template <>
__device__ __forceinline__ float ldexp_r<float>(float x, int e) { return ldexpf(x, e); }
template <>
__device__ __forceinline__ double ldexp_r<double>(double x, int e) { return ldexp(x, e); }

// the mantissa in [1/2, 1) and the exponent of x
__device__ __forceinline__ float mant(float x) { return __builtin_amdgcn_frexp_mantf(x); }
__device__ __forceinline__ double mant(double x) { return __builtin_amdgcn_frexp_mant(x); }
__device__ __forceinline__ int expo(float x) { return __builtin_amdgcn_frexp_expf(x); }
__device__ __forceinline__ int expo(double x) { return __builtin_amdgcn_frexp_exp(x); }

// A sum s·2^k of terms m·2^e of unknown spread (k = kUndef: none yet).  Terms
// have normalised mantissas, so the largest exponent is the largest term's to
// a few binary digits and the others are shifted down to it.  Free of
// branches: a zero is the term 0·2^kUndef.
template <typename Real>
struct XSum {
  Real s;
  int k;
  __device__ __forceinline__ XSum() : s(0), k(kUndef) {}
  template <int N>
  __device__ __forceinline__ void add(const Real (&m)[N], const int (&e)[N]) {
    int K = k;
#pragma unroll
    for (int j = 0; j < N; ++j) K = max(K, e[j]);
    s = ldexp_r(s, k - K);
#pragma unroll
    for (int j = 0; j < N; ++j) s += ldexp_r(m[j], e[j] - K);
    k = K;
  }
  __device__ __forceinline__ void add(Real m, int e) {
    const Real a[1] = {m};
    const int b[1] = {e};
    add(a, b);
  }
  // the sum at exponent e
  __device__ __forceinline__ Real at(int e) const { return ldexp_r(s, k - e); }
  // the sum as a mantissa and its exponent (0, kUndef for 0)
  __device__ __forceinline__ Real split(int* e) const {
    *e = s != Real(0) ? k + expo(s) : kUndef;
    return mant(s);
  }
};
// x·2^e0 as a term
template <typename Real, typename X>
__device__ __forceinline__ void xterm(X x, int e0, Real* m, int* e) {
  *m = (Real)mant(x);
  *e = x != X(0) ? e0 + expo(x) : kUndef;
}
// p·v1·v2·2^e0 as a term: FP32 products are formed in FP64, which holds any of
// them; FP64 ones from the mantissas
template <typename Real>
__device__ __forceinline__ void xprod(Real p, Real v1, Real v2, int e0, Real* m, int* e) {
  if constexpr (sizeof(Real) == sizeof(float)) xterm((double)p * ((double)v1 * v2), e0, m, e);
  else xterm(p * (mant(v1) * mant(v2)), e0 + expo(v1) + expo(v2), m, e);
}
// N records' terms p (F(a) G(b) + G(a) F(b)) 2^(e(a) + e(b)) added to x
template <typename Real, int N>
__device__ __forceinline__ void xpairs(XSum<Real>& x, const Real (&p)[N], const Real (&fa)[N], const Real (&fb)[N],
                                       const Real (&ga)[N], const Real (&gb)[N], const int (&ea)[N],
                                       const int (&eb)[N]) {
  Real m[N];
  int e[N];
  if constexpr (sizeof(Real) == sizeof(float)) {
#pragma unroll
    for (int j = 0; j < N; ++j)
      xterm((double)p[j] * ((double)fa[j] * gb[j] + (double)ga[j] * fb[j]), ea[j] + eb[j], &m[j], &e[j]);
    x.add(m, e);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) xprod(p[j], fa[j], gb[j], ea[j] + eb[j], &m[j], &e[j]);
    x.add(m, e);
#pragma unroll
    for (int j = 0; j < N; ++j) xprod(p[j], ga[j], fb[j], ea[j] + eb[j], &m[j], &e[j]);
    x.add(m, e);
  }
}

// ---------------------------------------------------------------------------
// wave-level reductions
// ---------------------------------------------------------------------------
template <typename Real>
__device__ __forceinline__ Real wave_sum(Real v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWG);
  return v;
}

// The lane `OFF` lower in the wave's 16-lane row (0 where there is none), by DPP.
template <int OFF>
__device__ __forceinline__ int dpp_shr(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x110 + OFF, 0xf, 0xf, false);
}
template <int OFF>
__device__ __forceinline__ float dpp_shr(float v) {
  return __builtin_bit_cast(float, dpp_shr<OFF>(__builtin_bit_cast(int, v)));
}
template <int OFF>
__device__ __forceinline__ double dpp_shr(double v) {
  const long long x = __builtin_bit_cast(long long, v);
  const int lo = dpp_shr<OFF>((int)(x & 0xffffffffll)), hi = dpp_shr<OFF>((int)(x >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}

// Sum of v over the lanes of an item, complete in its last lane: lane `pos`
// of the item adds the lanes below it, 1, 2, 4 and 8 at a time.  `steps` (the
// same in all lanes) is what the wave's widest item needs, 0 when every item
// has one lane, as most chunks do.
template <typename Real>
__device__ __forceinline__ Real slot_sum(Real v, uint32_t pos, int steps) {
  if (steps > 0) {
    Real u = dpp_shr<1>(v);
    v += pos >= 1 ? u : Real(0);
    if (steps > 1) {
      u = dpp_shr<2>(v);
      v += pos >= 2 ? u : Real(0);
      if (steps > 2) {
        u = dpp_shr<4>(v);
        v += pos >= 4 ? u : Real(0);
        if (steps > 3) {
          u = dpp_shr<8>(v);
          v += pos >= 8 ? u : Real(0);
        }
      }
    }
  }
  return v;
}
// the same for sums with exponents
template <int OFF, typename Real>
__device__ __forceinline__ void slot_xstep(XSum<Real>& x, uint32_t pos) {
  const Real s = dpp_shr<OFF>(x.s);
  const int k = dpp_shr<OFF>(x.k);
  const bool in = pos >= (uint32_t)OFF;
  x.add(in ? s : Real(0), in ? k : kUndef);
}
template <typename Real>
__device__ __forceinline__ void slot_xsum(XSum<Real>& x, uint32_t pos, int steps) {
  if (steps > 0) slot_xstep<1>(x, pos);
  if (steps > 1) slot_xstep<2>(x, pos);
  if (steps > 2) slot_xstep<4>(x, pos);
  if (steps > 3) slot_xstep<8>(x, pos);
}
// lane shifts the widest item of the wave needs
__device__ __forceinline__ int slot_steps(uint32_t pos) {
  return __any(pos >= 8) ? 4 : __any(pos >= 4) ? 3 : __any(pos >= 2) ? 2 : __any(pos >= 1) ? 1 : 0;
}

// atomic adds without return: LDS (ds_add) or global (FP64 atomics in L2)
template <typename Real>
__device__ __forceinline__ void lds_add(Real* p, Real v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// a gradient accumulator: the workgroup's copy in LDS, or (trees whose
// accumulators do not fit) the batch's in global memory
struct Acc {
  __attribute__((address_space(3))) double* lds;
  double* glb;
  bool in_lds;
  __device__ __forceinline__ void add(int i, double v) const {
    if (v == 0.0) return;
    if (in_lds) lds_add((double*)(lds + i), v);
    else unsafeAtomicAdd(glb + i, v);
  }
};

// coefficient of a record in the scaled forms: p·2^(E1+E2-E), 0 while any exponent is open
template <typename Real>
__device__ __forceinline__ Real coef_of(Real p, int e1, int e2, int Eg) {
  if (Eg == kUndef || e1 == kUndef || e2 == kUndef) return Real(0);
  return ldexp_r(p, e1 + e2 - Eg);
}

// One wavefront, or a team of wavefronts that fill a workgroup, evaluates one
// family.  The LDS executes a wave's instructions in order, so between the
// rows of a one-wave family it is enough to keep the compiler from moving LDS
// accesses across the boundary: no s_barrier and no wait on outstanding global
// stores.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Where a wave reads back global memory its lanes wrote (ℓ and ī of earlier
// stages, exponents) the stores must have completed: once per stage.
__device__ __forceinline__ void wave_sync_mem() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
// Between two passes over a family's stage buffers.  A team's waves meet at a
// barrier that orders LDS only; with the buffers in global memory (Gws:
// families whose stages do not fit one compute unit's LDS) every pass also
// waits for the previous pass's global stores.
template <bool Team, bool Gws>
__device__ __forceinline__ void tsync() {
  if (Gws) {
    if (Team) __syncthreads();
    else wave_sync_mem();
  } else if (Team) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  } else {
    wave_sync();
  }
}
// where the family's waves read back global memory that one of them wrote
template <bool Team>
__device__ __forceinline__ void tsync_mem() {
  if (Team) __syncthreads();
  else wave_sync_mem();
}

// Pointers with their address space.  A generic pointer to global memory is
// accessed with flat instructions, which count against both the vector-memory
// and the LDS counters, so a later wait for LDS also waits for them; a generic
// pointer into LDS likewise makes every row wait for the last row's stores to
// reach memory.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> glob(T* p) {
  return (gptr<T>)p;
}
template <typename T>
using lptr = __attribute__((address_space(3))) T*;
// a family's stage buffers: LDS or (Gws) global memory
template <bool Gws, typename T>
using bptr = std::conditional_t<Gws, gptr<T>, lptr<T>>;

// A record every lane of the wave loaded from the same address, moved to
// scalar registers.  The kernels write global memory, so the compiler loads
// such records with vector loads and treats their fields as varying across
// lanes; tests on them (item and record counts, row counts) would then be
// exec-mask branches instead of scalar ones.
template <typename T>
__device__ __forceinline__ T uniform(const T& x) {
  static_assert(sizeof(T) % 4 == 0, "a record of whole dwords");
  uint32_t w[sizeof(T) / 4];
  __builtin_memcpy(w, &x, sizeof(T));
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 4); ++k) w[k] = (uint32_t)__builtin_amdgcn_readfirstlane((int)w[k]);
  T y;
  __builtin_memcpy(&y, w, sizeof(T));
  return y;
}

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

// Row `row` of the slice tables (ModelDev::pack64 / pack32): φ_r, ψ_r, and for
// the reverse sweep φ_r, χ_r = ψ_r/β, D_α, D_β, D_ε0.  The rows of a stage are
// read from global memory ahead of their use: a copy in LDS takes a third to
// two thirds of a family's share of it (a 100-taxon tree of 1346 rows: 27 KB in
// the FP32 reverse sweep), and so of the families a compute unit can hold.
template <typename Real>
struct SliceRow {
  Real ph, ps;
};
template <typename Real>
struct SliceRowB {
  Real ph, ch, D[3];
};
template <typename Real>
__device__ __forceinline__ gptr<const Real> slice_pack(const ModelDev& M) {
  if constexpr (sizeof(Real) == sizeof(float)) return glob(M.pack32);
  else return glob(M.pack64);
}
template <typename Real>
__device__ __forceinline__ SliceRow<Real> slice(gptr<const Real> pack, uint32_t rows, uint32_t row) {
  typedef Real Real2 __attribute__((ext_vector_type(2)));
  const Real2 t = ((gptr<const Real2>)(pack + 4 * (size_t)rows))[row];
  return {t.x, t.y};
}
template <typename Real>
__device__ __forceinline__ SliceRowB<Real> slice_b(gptr<const Real> pack, uint32_t rows, uint32_t row) {
  typedef Real Real4 __attribute__((ext_vector_type(4)));
  const Real4 t = ((gptr<const Real4>)pack)[row];
  return {t.x, t.y, {t.z, t.w, pack[6 * (size_t)rows + row]}};
}

// per-node constants of the current parameters in LDS: ε at the top of each
// branch, leafℙ, q per WGD; for the reverse sweep also 1/(1-α), 1/(1-β), β
template <typename Real>
struct NodeC {
  lptr<Real> etop, leafP, q, ia, ib, be;
  __device__ NodeC(lptr<unsigned char> base, int n, int nwgd) {
    etop = (lptr<Real>)base;
    leafP = etop + n;
    q = leafP + n;
    ia = q + (nwgd > 0 ? nwgd : 1);
    ib = ia + n;
    be = ib + n;
  }
  __device__ void fill(const ModelDev& M, bool bwd, int tid, int nthreads) {
    for (int e = tid; e < M.n; e += nthreads) {
      etop[e] = (Real)eps_top(M, e);
      leafP[e] = (Real)M.node[e].leafP;
      if (bwd) {
        const double* d = M.dnode + (size_t)kDnode * e;
        ia[e] = (Real)d[4];
        ib[e] = (Real)d[5];
        be[e] = (Real)d[6];
      }
    }
    for (int w = tid; w < M.n_wgd; w += nthreads) q[w] = (Real)M.par[3 * M.n + w];
  }
};

// clade-size level boundaries of a family's root stage: the first 128 held
// in two registers across the wave and read with readlane (uniform level)
struct LevelBounds {
  uint32_t lo, hi;
  const uint32_t* p;
  __device__ LevelBounds(const uint32_t* lvl, const FamDev& F, uint32_t lane) : p(lvl + F.lvl0) {
    lo = lane <= F.n_lvl ? p[lane] : 0u;
    hi = lane + kWG <= F.n_lvl ? p[kWG + lane] : 0u;
  }
  __device__ __forceinline__ uint32_t at(uint32_t L) const {
    if (L < (uint32_t)kWG) return (uint32_t)__builtin_amdgcn_readlane((int)lo, (int)L);
    if (L < 2u * kWG) return (uint32_t)__builtin_amdgcn_readlane((int)hi, (int)(L - kWG));
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)p[L]);
  }
};

// ---------------------------------------------------------------------------
// LDS of one family, laid out afresh for every stage of n items
// (fwd_stage_bytes, fwd_root_bytes, bwd_stage_bytes, bwd_root_bytes)
// ---------------------------------------------------------------------------
template <typename Real, bool Gws>
struct FwdBuf {  // stage and root alike; the root uses no flags
  bptr<Gws, Real> A, F, G;
  bptr<Gws, int32_t> E;
  bptr<Gws, uint8_t> fl;
  __device__ FwdBuf(bptr<Gws, unsigned char> p, uint32_t n) {
    A = (bptr<Gws, Real>)p;
    F = A + n;
    G = F + n;
    p += align16(3 * (size_t)n * sizeof(Real));
    E = (bptr<Gws, int32_t>)p;
    p += align16(4 * (size_t)n);
    fl = (bptr<Gws, uint8_t>)p;
  }
};
template <typename Real, bool Gws>
struct BwdRootBuf {
  bptr<Gws, Real> A, V, F, G;
  bptr<Gws, int32_t> E;
  __device__ BwdRootBuf(bptr<Gws, unsigned char> p, uint32_t n) {
    A = (bptr<Gws, Real>)p;
    V = A + n;
    F = V + n;
    G = F + n;
    E = (bptr<Gws, int32_t>)(p + align16(4 * (size_t)n * sizeof(Real)));
  }
};
// The root's slots and terms staged behind its arrays when they fit the
// family's region (root_stage_bytes): terms' operands and coefficients, then
// per slot {item, position, lead; first term | count << 16}.
template <typename Real, bool Gws>
struct RootStage {
  bptr<Gws, uint32_t> ops;
  bptr<Gws, Real> c;
  bptr<Gws, u2> slot;
  bool on;
  __device__ RootStage(bptr<Gws, unsigned char> p, size_t used, uint32_t nt, uint32_t ns, uint32_t region) {
    on = !Gws && nt <= 0xffffu && used + root_stage_bytes(sizeof(Real), nt, ns) <= region;
    p += used;
    ops = (bptr<Gws, uint32_t>)p;
    p += align16(4 * (size_t)nt);
    c = (bptr<Gws, Real>)p;
    p += align16(sizeof(Real) * (size_t)nt);
    slot = (bptr<Gws, u2>)p;
  }
};

// terms a lane holds in registers
constexpr int kRecs = (int)kSlotRecs;

constexpr uint8_t kYoung = 1;    // the exponent was open when the stage began
constexpr uint8_t kShifted = 2;  // renormalised in the last row; exponent update pending

// A lane's slot of one chunk in the forward sweep.
template <typename Real, bool Scaled>
struct FwdLane {
  uint32_t ops[kRecs];            // its first terms: the two parts' items
  Real c[kRecs];                  // their coefficients
  Real p[Scaled ? kRecs : 1];     // scaled forms: their probabilities
  uint32_t item, pos, start, cnt, gid;
  uint32_t cell, nc, tab, R;
  u4 k;                           // the segment's second half: kind and node, children
  Real v;                         // the item's value in the current row (lead lane)
  bool lead, young, open;         // open: no value yet, but splits that may bring one
};

// The family index of a workgroup's control words (LDS).
enum { kCtlFam = 0, kCtlDirty = 1 /* two words */, kCtlSum = 4 /* 4 doubles per wave, from this word */ };

// The forward DP of family f by one wave or by the workgroup's team: its
// stages (row buffers in the family's region wb), then its root.  ℓ is
// written through `ell` (the family's cells, relative indices) and the items'
// exponents through `Eit` (absolute items less it_base).
template <typename Real, bool Scaled, bool StoreAll, bool Gws, bool Team>
__device__ __forceinline__ void fwd_family(const BatchDev& B, const ModelDev& M, const WorkDev<Real>& W, uint32_t f,
                                           bptr<Gws, unsigned char> const wb, uint32_t region,
                                           const NodeC<Real>& NC, lptr<uint32_t> ctl, uint32_t lane, Real* ell_arg,
                                           int32_t* Eit_arg, uint32_t it_base) {
  const gptr<const Real> pack = slice_pack<Real>(M);
  const gptr<Real> ell = glob(ell_arg);
  const gptr<int32_t> Eit = glob(Eit_arg);
  constexpr bool kF32 = sizeof(Real) == sizeof(float);
  typedef FwdLane<Real, Scaled> Lane;
  const uint32_t wv = Team ? (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWG) : 0u;
  const uint32_t nw = Team ? blockDim.x / kWG : 1u;
  const uint32_t tid = Team ? threadIdx.x : lane, nt = Team ? blockDim.x : (uint32_t)kWG;
  const FamDev F = uniform(B.fam[f]);
  const gptr<int32_t> E = glob(W.E + F.clade0);
  const gptr<const u4> fs4 = glob(reinterpret_cast<const u4*>(B.fs4));
  const gptr<const u2> fs2 = glob(reinterpret_cast<const u2*>(B.fs2));
  const gptr<const u4> run = glob(reinterpret_cast<const u4*>(B.run));
  const gptr<const uint32_t> rec_ops = glob(B.rec_ops);
  const gptr<const double> rec_p = glob(B.rec_p);
  if (Scaled)
    for (uint32_t c = tid; c < F.n_clades; c += nt) E[c] = kUndef;
  StageDev ahead = B.stage[F.stage0];
  // ---------------- non-root stages
  for (uint32_t s = 0; s < F.n_stages; ++s) {
    const StageDev S = uniform(ahead);
    if (s + 1 < F.n_stages) ahead = B.stage[F.stage0 + s + 1];  // in flight during this stage's rows
    const uint32_t n = S.n_items;
    const FwdBuf<Real, Gws> T(wb, n);  // fits the family's region (size class)
    const auto sE = T.E;
    const uint32_t nch = (S.n_fs + kChunk - 1) / kChunk;
    const uint32_t mych = wv < nch ? min((uint32_t)kRegChunks, (nch - wv + nw - 1) / nw) : 0u;
    const uint32_t over = wv + kRegChunks * nw;  // this wave's first chunk past its registers
    tsync_mem<Team>();  // ℓ and exponents of the stages below; the last readers of the buffers
    auto slot_at = [&](uint32_t ch, u4& a, u2& b) WHALE_INLINE {
      const uint32_t k = ch * kChunk + lane;
      const bool in = k < S.n_fs;
      a = fs4[S.fs0 + (in ? k : 0u)];
      b = fs2[S.fs0 + (in ? k : 0u)];
      if (!in) {
        a = u4{~0u, ~0u, 0u, 0u};
        b = u2{0u, 0u};
      }
    };
    // the slot's words, its segment and its terms (registers)
    auto take_slot = [&](Lane& q, const u4& a, const u2& b) WHALE_INLINE {
      q.item = a.z & 0xffffu;
      q.pos = (a.z >> 16) & 0xfu;
      q.lead = (a.z & kSlotLead) != 0u;
      q.gid = a.w & 0xffffu;
      q.start = b.x;
      q.cnt = b.y;
    };
    auto take_seg = [&](Lane& q, const u4& r) WHALE_INLINE {
      q.cell = r.x + q.item;
      q.nc = r.y;
      q.R = r.z;
      q.tab = r.w;
    };
    auto load_terms = [&](Lane& q) WHALE_INLINE {
      const int most = __any(q.cnt > 2) ? kRecs : __any(q.cnt > 0) ? 2 : 0;  // uniform
#pragma unroll
      for (int j = 0; j < kRecs; ++j) {
        uint32_t o = q.item * 0x10001u;  // past its terms a lane adds 0 times its own value squared
        Real p = 0;
        if (j < most) {
          const bool in = (uint32_t)j < q.cnt;
          const uint32_t k = F.rec0 + (in ? q.start + j : 0u);
          const uint32_t ro = rec_ops[k];
          const Real rp = (Real)rec_p[k];
          o = in ? ro : o;
          p = in ? rp : p;
        }
        q.ops[j] = o;
        if (Scaled) q.p[j] = p;
        else q.c[j] = p;
      }
    };
    Lane q[kRegChunks];
    u4 s4[kRegChunks], r0[kRegChunks], r1[kRegChunks];
    u2 s2[kRegChunks];
#pragma unroll
    for (int c = 0; c < kRegChunks; ++c)
      if ((uint32_t)c < mych) slot_at(wv + c * nw, s4[c], s2[c]);
    {
      Real vf[kRegChunks], vg[kRegChunks];
      int ev[kRegChunks];
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) {
          const uint32_t sg = S.seg0 + (s4[c].w >> 16);
          r0[c] = run[2 * (size_t)sg];
          r1[c] = run[2 * (size_t)sg + 1];
          const int32_t cf = (int32_t)s4[c].x, cg = (int32_t)s4[c].y;
          vf[c] = ell[cf >= 0 ? cf : 0];
          vg[c] = ell[cg >= 0 ? cg : 0];
          ev[c] = Scaled ? E[s4[c].w & 0xffffu] : 0;
          take_slot(q[c], s4[c], s2[c]);
          load_terms(q[c]);
        }
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) {
          take_seg(q[c], r0[c]);
          q[c].k = r1[c];
          q[c].young = Scaled && ev[c] == kUndef;
          q[c].open = false;
          q[c].v = 0;
          if (q[c].lead) {
            T.F[q[c].item] = (int32_t)s4[c].x >= 0 ? vf[c] : Real(0);
            T.G[q[c].item] = (int32_t)s4[c].y >= 0 ? vg[c] : Real(0);
            if (Scaled) {
              sE[q[c].item] = ev[c];
              T.fl[q[c].item] = ev[c] == kUndef ? kYoung : 0;
            }
          }
        }
    }
#pragma unroll 1
    for (uint32_t ch = over; ch < nch; ch += nw) {
      u4 a;
      u2 b;
      slot_at(ch, a, b);
      if (a.z & kSlotLead) {
        const uint32_t i = a.z & 0xffffu;
        const int32_t cf = (int32_t)a.x, cg = (int32_t)a.y;
        const Real vf = ell[cf >= 0 ? cf : 0], vg = ell[cg >= 0 ? cg : 0];
        T.F[i] = cf >= 0 ? vf : Real(0);
        T.G[i] = cg >= 0 ? vg : Real(0);
        if (Scaled) {
          const int e = E[a.w & 0xffffu];
          sE[i] = e;
          T.fl[i] = e == kUndef ? kYoung : 0;
        }
      }
    }
    tsync<Team, Gws>();
    auto cur = T.A;
    auto nxt = T.F;
    // scaled forms: coefficients for the exponents now fixed.  A record of a
    // clade that is still open keeps 0 (the open clade sums explicit exponents).
    auto coefs = [&](Lane& x) WHALE_INLINE {
      const int Eo = sE[x.item];
      x.open = Eo == kUndef && x.cnt > 0;
#pragma unroll
      for (int j = 0; j < kRecs; ++j)
        x.c[j] = coef_of(x.p[Scaled ? j : 0], sE[x.ops[j] & 0xffffu], sE[x.ops[j] >> 16], Eo);
    };
    // a pass over the wave's chunks: those in registers, then the others
    auto load_lane = [&](uint32_t ch, Lane& x) WHALE_INLINE {
      u4 a;
      u2 b;
      slot_at(ch, a, b);
      take_slot(x, a, b);
      const uint32_t sg = S.seg0 + (a.w >> 16);
      const u4 r0 = run[2 * (size_t)sg];
      x.k = run[2 * (size_t)sg + 1];
      take_seg(x, r0);
      load_terms(x);
      x.young = Scaled && (T.fl[x.item] & kYoung) != 0;
      x.open = false;
      x.v = cur[x.item];
    };
    auto each = [&](auto&& fn) WHALE_INLINE {
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) fn(q[c], true);
#pragma unroll 1
      for (uint32_t ch = over; ch < nch; ch += nw) {
        Lane x;
        load_lane(ch, x);
        fn(x, false);
      }
    };
    // the lane's terms j0 .. j0 + kRecs past its registers (0 past its last)
    auto more_terms = [&](const Lane& x, uint32_t j0, uint32_t (&o)[kRecs], Real (&p)[kRecs]) WHALE_INLINE {
#pragma unroll
      for (int j = 0; j < kRecs; ++j) {
        const bool in = j0 + j < x.cnt;
        const uint32_t k = F.rec0 + (in ? x.start + j0 + j : 0u);
        o[j] = in ? rec_ops[k] : x.item * 0x10001u;
        p[j] = in ? (Real)rec_p[k] : Real(0);
      }
    };
    // Row 0: terms from the child branches (whale!/whalewgd!, src/core.jl:95-128).
    // A WGD node's one child stands in both child slots, so both kinds sum
    // p(F(γ1)G(γ2) + G(γ1)F(γ2)).  The scaled forms sum them with exponents; a
    // clade still without one takes it from the sum.  Lanes that read the
    // exponent of a clade that gets one in this pass see either value; its
    // operands are zero, so the term is zero both ways.
    each([&](Lane& x, bool) WHALE_INLINE {
      const uint32_t kind = x.k.x & 3u;
      const int Eo = Scaled ? sE[x.item] : 0;
      const bool open = Scaled && Eo == kUndef;
      Real t = 0;
      XSum<Real> xs;
      // kRecs terms: all operands are read before any is used
      auto terms = [&](const uint32_t (&o)[kRecs], const Real (&p)[kRecs]) WHALE_INLINE {
        Real fa[kRecs], fb[kRecs], ga[kRecs], gb[kRecs];
        int ea[kRecs], eb[kRecs];
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          const uint32_t a = o[j] & 0xffffu, b = o[j] >> 16;
          fa[j] = T.F[a];
          fb[j] = T.F[b];
          ga[j] = T.G[a];
          gb[j] = T.G[b];
          if (Scaled) {
            ea[j] = sE[a];
            eb[j] = sE[b];
          }
        }
        if constexpr (Scaled) {
          xpairs(xs, p, fa, fb, ga, gb, ea, eb);
        } else {
#pragma unroll
          for (int j = 0; j < kRecs; ++j) t += p[j] * (fa[j] * gb[j] + ga[j] * fb[j]);
        }
      };
      if (__any(kind != WHALE_NODE_LEAF && x.cnt > 0)) {
        if constexpr (Scaled) terms(x.ops, x.p);
        else terms(x.ops, x.c);
#pragma unroll 1
        for (uint32_t j0 = kRecs; __any(j0 < x.cnt); j0 += kRecs) {
          uint32_t o[kRecs];
          Real p[kRecs];
          more_terms(x, j0, o, p);
          terms(o, p);
        }
      }
      const int st = slot_steps(x.pos);
      if constexpr (Scaled) slot_xsum(xs, x.pos, st);
      else t = slot_sum(t, x.pos, st);
      if (!x.lead) return;
      if (Scaled && !open) t = xs.at(Eo);
      Real v = 0;
      if (kind == WHALE_NODE_LEAF) {
        if (x.cnt == 0 && x.pos == 0) {  // a clade of one gene (every larger clade has a split)
          const Real lp = NC.leafP[x.k.y];
          if (!Scaled) {
            v = lp;
          } else if (open) {
            int ex;
            v = frexp_r(lp, &ex);
            sE[x.item] = ex;
          } else {
            v = ldexp_r(lp, -Eo);
          }
        }
      } else {
        const Real f0 = T.F[x.item], g0 = T.G[x.item], ef = NC.etop[x.k.y];
        Real base, fac = 1;
        if (kind == WHALE_NODE_WGD) {
          const Real qq = NC.q[x.k.z];
          base = (Real(1) - qq) * f0 + (Real(2) * qq) * ef * f0;
          fac = Real(0.5) * qq;
        } else {
          base = f0 * NC.etop[x.k.z] + g0 * ef;
        }
        if (!open) {
          v = base + fac * t;
        } else if (fac * xs.s != Real(0)) {
          v = ldexp_r(mant(fac * xs.s), -kBirth);
          sE[x.item] = xs.k + expo(fac * xs.s) + kBirth;
        }
      }
      T.A[x.item] = v;
      x.v = v;
      if (StoreAll || x.R == 1) ell[x.cell] = v;
    });
    tsync<Team, Gws>();
    bool any_open = false, any_young = false, dirty = false;
    auto all_coefs = [&]() WHALE_INLINE {
      any_open = false;
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) {
          coefs(q[c]);
          any_open |= q[c].open;
        }
      any_open = __any(any_open);
    };
    int steps = 0;
    uint32_t most = over < nch ? 5u : 0u;  // chunks past the registers may hold any count
    if (Scaled) all_coefs();
#pragma unroll
    for (int c = 0; c < kRegChunks; ++c)
      if ((uint32_t)c < mych) {
        any_young |= q[c].young;
        steps = max(steps, slot_steps(q[c].pos));
        most = max(most, __any(q[c].cnt > kSlotRecs) ? 5u : __any(q[c].cnt > 2) ? 4u : 2u);
      }
    any_young = Scaled && __any(any_young);
    // the new value of an item from the sum over its splits
    auto finish = [&](Lane& x, uint32_t r, Real acc, Real ph, Real ps, bool check, bool& changed) WHALE_INLINE {
      const bool in = r < x.R;
      if (in && !x.open) x.v = fma(ph, x.v, ps * acc);
      if (Scaled && kF32 && check) {
        // A young clade past 2^kBump is renormalised in place (its only values
        // are this branch's rows); its exponent is raised after the row, as
        // other items of this row still read the clade's last row at the old
        // scale.
        const float av = fabsf((float)x.v);
        if (__any(x.young && x.lead && in && av > (float)(1ull << kBump) && av < INFINITY)) {
          if (x.young && x.lead && in && av > (float)(1ull << kBump) && av < INFINITY) {
            int ex;
            (void)frexp_r(x.v, &ex);
            const int sh = ex + kBirth;
            x.v = ldexp_r(x.v, -sh);
            if (StoreAll)
#pragma unroll 1
              for (uint32_t k = 0; k < r; ++k) {
                const gptr<Real> z = ell + (x.cell + k * x.nc);
                *z = ldexp_r(*z, -sh);
              }
            T.G[x.item] = (Real)sh;  // G is free after row 0
            T.fl[x.item] |= kShifted;
            changed = true;
          }
        }
      }
      if (x.lead) {
        nxt[x.item] = x.v;
        if (in && (StoreAll || r + 1 == x.R)) ell[x.cell + r * x.nc] = x.v;
      }
    };
    // Rows 1..R-1: within_branch! (src/core.jl:83-92).  A row in which
    // exponents are open or have changed, or whose terms are not all in
    // registers, takes the general form; the others run in loops for two or
    // all terms a lane, which leave at a row that needs
    // the general form.
    uint32_t r = 1;
    auto flagged = [&]() WHALE_INLINE -> bool {  // the last row changed exponents
      if (!Scaled) return false;
      return Team ? __builtin_amdgcn_readfirstlane((int)ctl[kCtlDirty + (r & 1u)]) != 0 : dirty;
    };
    auto end_row = [&](bool changed) WHALE_INLINE {
      if (Scaled && __any(changed)) {
        dirty = true;
        if (Team && lane == 0) ctl[kCtlDirty + ((r + 1) & 1u)] = 1u;
      }
      tsync<Team, Gws>();
      const auto t = cur;
      cur = nxt;
      nxt = t;
      ++r;
    };
    // After a row that fixed an exponent or renormalised a clade: the new
    // exponents, then every coefficient.  The rows already hold the values at
    // the new scales.  A team learns of it through ctl (two words in turn).
    auto settle = [&]() WHALE_INLINE {
      auto shift = [&](bool lead, uint32_t i) WHALE_INLINE {
        if (lead && (T.fl[i] & kShifted)) {
          sE[i] += (int)T.G[i];
          T.fl[i] &= (uint8_t)~kShifted;
        }
      };
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) shift(q[c].lead, q[c].item);
#pragma unroll 1
      for (uint32_t ch = over; ch < nch; ch += nw) {
        const uint32_t k = ch * kChunk + lane;
        const uint32_t z = k < S.n_fs ? fs4[S.fs0 + k].z : 0u;
        shift((z & kSlotLead) != 0u, z & 0xffffu);
      }
      tsync<Team, Gws>();
      if (Team && threadIdx.x == 0) ctl[kCtlDirty + (r & 1u)] = 0u;
      dirty = false;
      all_coefs();
    };
    const bool all_general = over < nch || most > kSlotRecs || (Team && mych == 0);
    auto general_row = [&]() WHALE_INLINE {
      if (Scaled && flagged()) settle();
      bool changed = false;
      each([&](Lane& x, bool held) WHALE_INLINE {
        if (Scaled && !held) coefs(x);
        Real t = 0;
        const SliceRow<Real> w = slice<Real>(pack, M.tab_rows, x.tab + min(r, x.R - 1));
        XSum<Real> xs;
        // the first value of an open clade sums its terms as (mantissa, exponent) pairs
        auto open_terms = [&](const uint32_t (&o)[kRecs], const Real (&p)[kRecs], const Real (&va)[kRecs],
                              const Real (&vb)[kRecs]) WHALE_INLINE {
          Real m[kRecs];
          int e[kRecs];
#pragma unroll
          for (int j = 0; j < kRecs; ++j) xprod(p[j], va[j], vb[j], sE[o[j] & 0xffffu] + sE[o[j] >> 16], &m[j], &e[j]);
          xs.add(m, e);
        };
        const bool some_open = Scaled && __any(x.open);
        Real va[kRecs], vb[kRecs];
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          va[j] = cur[x.ops[j] & 0xffffu];
          vb[j] = cur[x.ops[j] >> 16];
        }
#pragma unroll
        for (int j = 0; j < kRecs; ++j) t = fma(x.c[j] * va[j], vb[j], t);
        if constexpr (Scaled) {
          if (some_open) open_terms(x.ops, x.p, va, vb);
        }
        if (most > kSlotRecs) {
          const int Eo = Scaled ? sE[x.item] : 0;
#pragma unroll 1
          for (uint32_t j0 = kRecs; __any(j0 < x.cnt); j0 += kRecs) {  // the terms past the lane's registers
            uint32_t o[kRecs];
            Real p[kRecs];
            more_terms(x, j0, o, p);
#pragma unroll
            for (int j = 0; j < kRecs; ++j) {
              va[j] = cur[o[j] & 0xffffu];
              vb[j] = cur[o[j] >> 16];
              const Real c = Scaled ? coef_of(p[j], sE[o[j] & 0xffffu], sE[o[j] >> 16], Eo) : p[j];
              t = fma(c * va[j], vb[j], t);
            }
            if (some_open) open_terms(o, p, va, vb);
          }
        }
        const int st = slot_steps(x.pos);
        t = slot_sum(t, x.pos, st);
        if (some_open) {
          slot_xsum(xs, x.pos, st);
          const Real v = w.ps * xs.s;
          if (x.open && x.lead && r < x.R && v != Real(0)) {
            x.v = ldexp_r(mant(v), -kBirth);
            sE[x.item] = xs.k + expo(v) + kBirth;  // readers of row r-1 see 0 here and skip it
            changed = true;
          }
        }
        finish(x, r, t, w.ph, w.ps, Scaled, changed);
      });
      end_row(changed);
    };
    auto plain_rows = [&](auto km_) WHALE_INLINE {
      constexpr int NC_ = kRegChunks, KM = decltype(km_)::value;
      // φ, ψ of this row and the next: a row's are loaded two rows ahead, so that
      // the wait for them waits for no younger store of a row
      SliceRow<Real> w0[NC_], w1[NC_];
#pragma unroll
      for (int c = 0; c < NC_; ++c) {
        w0[c] = slice<Real>(pack, M.tab_rows, q[c].tab + min(r, q[c].R - 1));
        w1[c] = slice<Real>(pack, M.tab_rows, q[c].tab + min(r + 1, q[c].R - 1));
      }
#pragma unroll 1
      while (r < S.r_max) {
        Real va[NC_][KM], vb[NC_][KM];
        SliceRow<Real> w2[NC_];
#pragma unroll
        for (int c = 0; c < NC_; ++c) {
#pragma unroll
          for (int j = 0; j < KM; ++j) {
            va[c][j] = cur[q[c].ops[j] & 0xffffu];
            vb[c][j] = cur[q[c].ops[j] >> 16];
          }
          w2[c] = slice<Real>(pack, M.tab_rows, q[c].tab + min(r + 2, q[c].R - 1));
        }
        if (flagged()) break;
        Real acc[NC_];
#pragma unroll
        for (int c = 0; c < NC_; ++c) {
          acc[c] = 0;
#pragma unroll
          for (int j = 0; j < KM; ++j) acc[c] = fma(q[c].c[j] * va[c][j], vb[c][j], acc[c]);
        }
        if (steps > 0) {
#pragma unroll
          for (int c = 0; c < NC_; ++c) acc[c] = slot_sum(acc[c], q[c].pos, steps);
        }
        bool changed = false;
#pragma unroll
        for (int c = 0; c < NC_; ++c) {
          finish(q[c], r, acc[c], w0[c].ph, w0[c].ps, any_young, changed);
          w0[c] = w1[c];
          w1[c] = w2[c];
        }
        end_row(changed);
      }
    };
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, kRecs> IK;
    static_assert(kRegChunks == 1, "the row loops hold every chunk of the wave");
#pragma unroll 1
    while (r < S.r_max) {
      if (all_general || any_open || flagged()) {
        general_row();
      } else if (most > 2) {
        plain_rows(IK{});
      } else {
        plain_rows(I2{});
      }
    }
    if (Scaled) {
      if (flagged()) settle();
      // exponents of this stage's clades, for the stages above, ℓ download and the reverse sweep
      auto out = [&](bool lead, uint32_t i, uint32_t gid) WHALE_INLINE {
        if (!lead) return;
        const int e = sE[i];
        E[gid] = e;
        if (StoreAll) Eit[S.item0 - it_base + i] = e;
      };
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) out(q[c].lead, q[c].item, q[c].gid);
#pragma unroll 1
      for (uint32_t ch = over; ch < nch; ch += nw) {
        const uint32_t k = ch * kChunk + lane;
        if (k < S.n_fs) {
          const u4 a = fs4[S.fs0 + k];
          out((a.z & kSlotLead) != 0u, a.z & 0xffffu, a.w & 0xffffu);
        }
      }
    }
  }
  // ---------------- root: all clades, by size level (whaleroot!, src/core.jl:139-158)
  {
    const uint32_t n = F.n_clades;
    const SegDev sg = uniform(B.seg[F.root_seg]);
    const NodeDev& nd = M.node[M.root];
    const double eta = M.par[3 * M.n + M.n_wgd];
    const double er = eps_top(M, M.root);
    const double xi = 1.0 - (1.0 - eta) * er;
    const Real cA = (Real)((1.0 - eta) * xi / eta);
    const Real cB = (Real)(eta * (1.0 - er) / (xi * xi));
    const Real ef = NC.etop[nd.child0], eg = NC.etop[nd.child1];
    const LevelBounds LB(B.lvl_f, F, lane);
    const uint32_t ns = F.root_nfs, rec0 = F.rec0, first = F.n_recs - F.root_recs;
    const FwdBuf<Real, Gws> T(wb, n);
    const RootStage<Real, Gws> RS(wb, fwd_bytes(sizeof(Real), Scaled, n), F.root_recs, ns, region);
    const auto sE = T.E;
    tsync_mem<Team>();
    // tops of the root's two branches
    constexpr int U = 4;
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < ns; k0 += U * nt) {
      u4 a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t k = k0 + u * nt + tid;
        a[u] = fs4[F.root_fs + (k < ns ? k : 0u)];
        if (k >= ns) a[u].z = 0u;
      }
      Real vf[U], vg[U];
      int ev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t cf = (int32_t)a[u].x, cg = (int32_t)a[u].y;
        vf[u] = ell[cf >= 0 ? cf : 0];
        vg[u] = ell[cg >= 0 ? cg : 0];
        ev[u] = Scaled ? E[a[u].z & 0xffffu] : 0;  // root items are the clades
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (a[u].z & kSlotLead) {
          const uint32_t i = a[u].z & 0xffffu;
          T.F[i] = (int32_t)a[u].x >= 0 ? vf[u] : Real(0);
          T.G[i] = (int32_t)a[u].y >= 0 ? vg[u] : Real(0);
          if (Scaled) sE[i] = ev[u];
        }
    }
    tsync<Team, Gws>();
    // Everything that does not depend on other root values, all slots at
    // once: A(γ) = cB·(F(γ)ε_g + G(γ)ε_f + Σ p (F(γ1)G(γ2) + G(γ1)F(γ2))).  A
    // clade without a value below the root ("open") keeps this part as a
    // mantissa in A and its exponent, above kOpen, in E.  The terms are staged
    // for the levels.
    constexpr int kOpen = 1 << 28;
    u4 a0;
    u2 b0;
    auto fetch = [&](uint32_t k) WHALE_INLINE {
      const bool in = k < ns;
      a0 = fs4[F.root_fs + (in ? k : 0u)];
      b0 = fs2[F.root_fs + (in ? k : 0u)];
      if (!in) {
        a0.z = 0u;
        b0 = u2{0u, 0u};
      }
    };
    fetch(wv * kChunk + lane);
#pragma unroll 1
    for (uint32_t k0 = wv * kChunk; k0 < ns; k0 += nt) {
      const u4 a = a0;
      const u2 b = b0;
      const uint32_t i = a.z & 0xffffu, pos = (a.z >> 16) & 0xfu;
      uint32_t o[kRecs];
      Real p[kRecs];
      auto load = [&](uint32_t j0) WHALE_INLINE {
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          const bool in = j0 + j < b.y;
          const uint32_t k = rec0 + (in ? b.x + j0 + j : 0u);
          o[j] = rec_ops[k];
          p[j] = in ? (Real)rec_p[k] : Real(0);
        }
      };
      load(0);
      fetch(k0 + nt + lane);
      if (RS.on && k0 + lane < ns) RS.slot[k0 + lane] = u2{a.z, b.y ? (b.x - first) | (b.y << 16) : 0u};
      const int Eo = Scaled ? sE[i] : 0;
      const bool open = Scaled && (Eo == kUndef || Eo >= kOpen / 2);
      Real t = 0;
      XSum<Real> xs;
#pragma unroll 1
      for (uint32_t j0 = 0; __any(j0 < b.y); j0 += kRecs) {
        if (j0 > 0) load(j0);
        Real fa[kRecs], fb[kRecs], ga[kRecs], gb[kRecs];
        int ea[kRecs], eb[kRecs];
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          const uint32_t x = o[j] & 0xffffu, y = o[j] >> 16;
          fa[j] = T.F[x];
          fb[j] = T.F[y];
          ga[j] = T.G[x];
          gb[j] = T.G[y];
          if (Scaled) {
            ea[j] = sE[x];
            eb[j] = sE[y];
          }
        }
#pragma unroll
        for (int j = 0; j < kRecs; ++j) {
          if (RS.on && j0 + j < b.y) {
            RS.ops[b.x - first + j0 + j] = o[j];
            RS.c[b.x - first + j0 + j] = p[j];
          }
          if (!Scaled) t += p[j] * (fa[j] * gb[j] + ga[j] * fb[j]);
        }
        if constexpr (Scaled) xpairs(xs, p, fa, fb, ga, gb, ea, eb);
      }
      const int st = slot_steps(pos);
      if constexpr (Scaled) slot_xsum(xs, pos, st);
      else t = slot_sum(t, pos, st);
      if (a.z & kSlotLead) {
        Real v;
        if (Scaled && open) {
          int ex;
          xs.s *= cB;
          v = xs.split(&ex);
          if (ex != kUndef) sE[i] = ex + kOpen;
        } else {
          if (Scaled) t = xs.at(Eo);
          v = cB * (T.F[i] * eg + T.G[i] * ef + t);
        }
        T.A[i] = v;
      }
    }
    tsync<Team, Gws>();
    // Levels: the terms cA·p·A(γ1)·A(γ2) of parts in lower levels.  A level's
    // lanes stand at its slots' places modulo 16, as the slots were dealt.
    // Nothing is stored to global memory in here: a load's wait would also
    // wait for the stores before it.
    auto levels = [&](auto staged_) WHALE_INLINE {
      constexpr bool staged = decltype(staged_)::value;
#pragma unroll 1
      for (uint32_t L = 0; L < F.n_lvl; ++L) {
        const uint32_t s0 = LB.at(L), s1 = LB.at(L + 1);
#pragma unroll 1
        for (uint32_t k0 = (s0 & ~15u) + wv * kChunk; k0 < s1; k0 += nt) {
          const uint32_t k = k0 + lane;
          const bool in = k >= s0 && k < s1;
          uint32_t z, r0, cnt;
          if constexpr (staged) {
            const u2 d = RS.slot[in ? k : s0];
            z = d.x;
            r0 = d.y & 0xffffu;
            cnt = d.y >> 16;
          } else {
            const u2 d = fs2[F.root_fs + (in ? k : s0)];
            z = fs4[F.root_fs + (in ? k : s0)].z;
            r0 = d.x;
            cnt = d.y;
          }
          if (!in) z = cnt = 0;
          const uint32_t i = z & 0xffffu, pos = (z >> 16) & 0xfu;
          const int Eo = Scaled ? sE[i] : 0;
          const bool open = Scaled && (Eo == kUndef || Eo >= kOpen / 2);
          Real t = 0;
          XSum<Real> xs;
#pragma unroll 1
          for (uint32_t j0 = 0; __any(j0 < cnt); j0 += kRecs) {
            uint32_t o[kRecs];
            Real p[kRecs], va[kRecs], vb[kRecs];
            int ea[kRecs], eb[kRecs];
#pragma unroll
            for (int j = 0; j < kRecs; ++j) {
              const bool ok = j0 + j < cnt;
              if constexpr (staged) {
                const uint32_t x = ok ? r0 + j0 + j : 0u;
                o[j] = RS.ops[x];
                p[j] = RS.c[x];
              } else {
                const uint32_t x = rec0 + (ok ? r0 + j0 + j : 0u);
                o[j] = rec_ops[x];
                p[j] = (Real)rec_p[x];
              }
              if (!ok) p[j] = 0;
            }
#pragma unroll
            for (int j = 0; j < kRecs; ++j) {
              va[j] = T.A[o[j] & 0xffffu];
              vb[j] = T.A[o[j] >> 16];
              if (Scaled) {
                ea[j] = sE[o[j] & 0xffffu];
                eb[j] = sE[o[j] >> 16];
              }
            }
            if constexpr (Scaled) {
              Real m[kRecs];
              int e[kRecs];
#pragma unroll
              for (int j = 0; j < kRecs; ++j) xprod(p[j], va[j], vb[j], ea[j] + eb[j], &m[j], &e[j]);
              xs.add(m, e);
            } else {
#pragma unroll
              for (int j = 0; j < kRecs; ++j) t = fma(p[j] * va[j], vb[j], t);
            }
          }
          const int st = slot_steps(pos);
          if constexpr (Scaled) slot_xsum(xs, pos, st);
          else t = slot_sum(t, pos, st);
          if (z & kSlotLead) {
            Real v = T.A[i];
            if (!Scaled) {
              v = fma(cA, t, v);
            } else if (!open) {
              v = fma(cA, xs.at(Eo), v);
            } else {
              xs.s *= cA;
              if (Eo != kUndef) xs.add(v, Eo - kOpen);
              int ex;
              v = ldexp_r(xs.split(&ex), -kBirth);
              sE[i] = ex != kUndef ? ex + kBirth : kUndef;
            }
            T.A[i] = v;
          }
        }
        tsync<Team, Gws>();
      }
    };
    if (RS.on) levels(std::true_type{});
    else levels(std::false_type{});
    for (uint32_t i = tid; i < n; i += nt) {
      ell[sg.ell + i] = T.A[i];
      if (Scaled) E[i] = sE[i];
    }
    if (tid == 0) {
      const Real v = T.A[n - 1];
      double ll;
      if (v > Real(0) && isfinite((double)v)) {
        ll = log((double)v);
        if (Scaled) ll += (double)sE[n - 1] * 0.69314718055994530942;
      } else {
        ll = -INFINITY;
        if (Scaled && kF32) {
          // overflow, or everything underflowed: redo this family in FP64 (a true zero stays -Inf there)
          W.flag[f] = 1u;
          W.fb[1 + atomicAdd(W.fb, 1u)] = f;
        }
      }
      W.fam_ll[f] = ll;
    }
  }
}

// ---------------------------------------------------------------------------
// backward (reverse sweep); requires a forward with stored rows
// ---------------------------------------------------------------------------
// A lane's slot of one chunk in the reverse sweep.
template <typename Real>
struct BwdLane {
  uint32_t ops[kRecs];   // its first entries: owner's item, other part's item
  Real c[kRecs];
  uint32_t item, pos, start, cnt;
  uint32_t cell, nc, tab, R;
  u4 k;                  // the segment's second half: kind and node, children, ī
  Real a, v;             // ā(r) and ℓ(r-1) of the item (lead lane)
  Real pf[4];            // ℓ of the next rows down
  Real f, g;             // tops of the child branches (row 0)
  Real be;               // β of the branch
  Real t[3], q1, q2;     // the row sums of d/d(α, β, ε of row 0), see bwd_family
  double d[sizeof(Real) == 4 ? 5 : 1];  // FP32: what was moved out of them every 32 rows
  bool lead;
};

// The reverse sweep of family f by one wave or by the workgroup's team, from
// its stored ℓ (`ell`, relative cells) and its items' exponents (`Eit`,
// absolute items less it_base), writing ī through `ibar` (relative cells).
//
// Down a branch, with S(γ) = Σ c·ā(r)[owner]·ℓ(r-1)[other] over the splits γ
// is a part of: ā(r-1) = φ_r ā(r) + ψ_r S.  Each split is seen by both its
// parts, so d/dψ_r = ½ Σ_γ ℓ(r-1)[γ] S(γ); d/dφ_r = Σ_γ ā(r)[γ] ℓ(r-1)[γ].
// φ_r and ψ_r are functions of the branch's α, β and ε of row 0 alone
// (src/model.jl:182-191): with den_r = 1 - β ε_{r-1}, φ_r = (1-α)(1-β)/den_r²
// and ψ_r = φ_r β/den_r.  So instead of one sum per row and segment (a
// reduction over the segment's lanes every row), every lane folds its item's
// two products into five sums over the rows,
//   q1 = Σ φ_r x_r,  q2 = Σ χ_r y_r (χ = ψ/β),  t_k = Σ (2 φ_r x_r + 3 ψ_r y_r) D_k(r)
// with x = ā(r) ℓ(r-1), y = ½ ℓ(r-1) S, D_k(r) = -(∂den_r/∂k)/den_r for
// k = α, β, ε0, and the segment's lanes are reduced once per stage.
template <typename Real, bool Scaled, bool Gws, bool Team>
__device__ __forceinline__ void bwd_family(const BatchDev& B, const ModelDev& M, const WorkDev<Real>& W, uint32_t f,
                                           bptr<Gws, unsigned char> const wb, uint32_t region,
                                           const Acc& acc, const NodeC<Real>& NC, lptr<uint32_t> ctl, uint32_t lane,
                                           const Real* ell_arg, Real* ibar_arg, const int32_t* Eit_arg,
                                           uint32_t it_base) {
  const gptr<const Real> pack = slice_pack<Real>(M);
  const gptr<const Real> ell = glob(ell_arg);
  const gptr<Real> ibar = glob(ibar_arg);
  const gptr<const int32_t> Eit = glob(Eit_arg);
  constexpr bool kF32 = sizeof(Real) == sizeof(float);
  typedef BwdLane<Real> Lane;
  constexpr int kSpill = kF32 ? 5 : 1;
  const AccLayout AL(M.n, M.n_wgd);
  const uint32_t wv = Team ? (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWG) : 0u;
  const uint32_t nw = Team ? blockDim.x / kWG : 1u;
  const uint32_t tid = Team ? threadIdx.x : lane, nt = Team ? blockDim.x : (uint32_t)kWG;
  // Deterministic gradients: every node's sums of this family go to its own
  // slot with plain stores (each is formed once, in a fixed order); a
  // fixed-order sum over the families follows.  Otherwise they are added to
  // the workgroup's accumulators.
  double* const accF = W.acc_fam ? W.acc_fam + (size_t)f * AL.n : nullptr;
  if (accF) {
    for (int j = (int)tid; j < AL.n; j += (int)nt) accF[j] = 0.0;
    tsync_mem<Team>();
  }
  auto put = [&](int i, double v) WHALE_INLINE {
    if (accF) accF[i] = v;
    else acc.add(i, v);
  };
  const FamDev F = uniform(B.fam[f]);
  const gptr<const u4> bs4 = glob(reinterpret_cast<const u4*>(B.bs4));
  const gptr<const u2> bs2 = glob(reinterpret_cast<const u2*>(B.bs2));
  const gptr<const u4> run = glob(reinterpret_cast<const u4*>(B.run));
  const gptr<const uint32_t> ent_ops = glob(B.ent_ops);
  const gptr<const double> ent_p = glob(B.ent_p);
  const uint32_t ent0 = 2 * F.rec0;
  // ---------------- root
  {
    const uint32_t n = F.n_clades;
    const SegDev sg = uniform(B.seg[F.root_seg]);
    const NodeDev& nd = M.node[M.root];
    const double eta = M.par[3 * M.n + M.n_wgd];
    const double er = eps_top(M, M.root);
    const double xi = 1.0 - (1.0 - eta) * er;
    const Real cA = (Real)((1.0 - eta) * xi / eta);
    const Real cB = (Real)(eta * (1.0 - er) / (xi * xi));
    const Real ef = NC.etop[nd.child0], eg = NC.etop[nd.child1];
    const BwdRootBuf<Real, Gws> T(wb, n);
    const uint32_t ns = F.root_nbs, first = 2 * (F.n_recs - F.root_recs);
    const RootStage<Real, Gws> RS(wb, bwd_root_bytes(sizeof(Real), Scaled, n), 2 * F.root_recs, ns, region);
    const gptr<const int32_t> E = glob(static_cast<const int32_t*>(W.E + F.clade0));
    tsync_mem<Team>();
    const LevelBounds LB(B.lvl_b, F, lane);
    const Real Lr = ell[sg.ell + n - 1];
    if (!(Lr > Real(0) && isfinite((double)Lr))) return;  // likelihood 0: no gradient
    const Real seed = (W.seed ? (Real)W.seed[f] : Real(1)) / Lr;
    constexpr int U = 4;
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < ns; k0 += U * nt) {
      u4 a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t k = k0 + u * nt + tid;
        a[u] = bs4[F.root_bs + (k < ns ? k : 0u)];
        if (k >= ns) a[u].z = 0u;
      }
      Real vv[U], vf[U], vg[U];
      int ev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t cf = (int32_t)a[u].x, cg = (int32_t)a[u].y;
        const uint32_t i = a[u].z & 0xffffu;
        vv[u] = ell[sg.ell + i];
        vf[u] = ell[cf >= 0 ? cf : 0];
        vg[u] = ell[cg >= 0 ? cg : 0];
        ev[u] = Scaled ? E[i] : 0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (a[u].z & kSlotLead) {
          const uint32_t i = a[u].z & 0xffffu;
          T.V[i] = vv[u];
          T.F[i] = (int32_t)a[u].x >= 0 ? vf[u] : Real(0);
          T.G[i] = (int32_t)a[u].y >= 0 ? vg[u] : Real(0);
          if (Scaled) T.E[i] = ev[u];
        }
    }
    tsync<Team, Gws>();
    // kRecs entries of a slot from its j0-th: owner, other part, coefficient
    // p·2^(E(γ) + E(other) - E(owner)) (0 past its last)
    auto scale = [&](uint32_t i, const uint32_t (&o)[kRecs], Real (&c)[kRecs]) WHALE_INLINE {
      const int Ei = T.E[i];
#pragma unroll
      for (int j = 0; j < kRecs; ++j)
        c[j] = c[j] != Real(0) ? coef_of(c[j], Ei, T.E[o[j] >> 16], T.E[o[j] & 0xffffu]) : Real(0);
    };
    auto entries = [&](uint32_t x0, uint32_t j0, uint32_t cnt, uint32_t i, uint32_t (&o)[kRecs],
                       Real (&c)[kRecs]) WHALE_INLINE {
#pragma unroll
      for (int j = 0; j < kRecs; ++j) {
        const bool ok = j0 + j < cnt;
        const uint32_t x = ent0 + (ok ? x0 + j0 + j : first);
        o[j] = ent_ops[x];
        c[j] = ok ? (Real)ent_p[x] : Real(0);
      }
      if (Scaled) scale(i, o, c);
    };
    // the entries staged for the levels and the pass after them
    if (RS.on) {
#pragma unroll 1
      for (uint32_t k0 = wv * kChunk; k0 < ns; k0 += nt) {
        const uint32_t k = k0 + lane;
        const u2 b = bs2[F.root_bs + (k < ns ? k : 0u)];
        const uint32_t z = bs4[F.root_bs + (k < ns ? k : 0u)].z;
        const uint32_t cnt = k < ns ? b.y & 0xffffu : 0u;
        if (k < ns) RS.slot[k] = u2{z, cnt ? (b.x - first) | (cnt << 16) : 0u};
#pragma unroll 1
        for (uint32_t j0 = 0; __any(j0 < cnt); j0 += kRecs) {
          uint32_t o[kRecs];
          Real c[kRecs];
          entries(b.x, j0, cnt, z & 0xffffu, o, c);
#pragma unroll
          for (int j = 0; j < kRecs; ++j)
            if (j0 + j < cnt) {
              RS.ops[b.x - first + j0 + j] = o[j];
              RS.c[b.x - first + j0 + j] = c[j];
            }
        }
      }
      tsync<Team, Gws>();
    }
    double sA = 0, sB = 0, sF = 0, sG = 0;
    auto sweep = [&](auto staged_) WHALE_INLINE {
      constexpr bool staged = decltype(staged_)::value;
      auto slot_of = [&](uint32_t k, bool in, uint32_t& z, uint32_t& r0, uint32_t& cnt) WHALE_INLINE {
        if constexpr (staged) {
          const u2 d = RS.slot[k];
          z = d.x;
          r0 = d.y & 0xffffu;
          cnt = d.y >> 16;
        } else {
          const u2 d = bs2[F.root_bs + k];
          z = bs4[F.root_bs + k].z;
          r0 = d.x;
          cnt = d.y & 0xffffu;
        }
        if (!in) z = cnt = 0;
      };
      auto terms_of = [&](uint32_t r0, uint32_t j0, uint32_t cnt, uint32_t i, uint32_t (&o)[kRecs],
                          Real (&c)[kRecs]) WHALE_INLINE {
        if constexpr (staged) {
#pragma unroll
          for (int j = 0; j < kRecs; ++j) {
            const bool ok = j0 + j < cnt;
            o[j] = RS.ops[ok ? r0 + j0 + j : 0u];
            c[j] = RS.c[ok ? r0 + j0 + j : 0u];
            if (!ok) c[j] = 0;
          }
        } else {
          entries(r0, j0, cnt, i, o, c);
        }
      };
      // d logL / d ℓ of the root's clades, levels from the last (the ubiquitous
      // clade) down: cA Σ c·ā(owner)·ℓ(other) over the splits a clade is a part
      // of, whose owners are in higher levels.  FP32 terms that are not in LDS
      // are read ahead of the chain: a level's first terms during the level
      // before it, by slot words read another level before.  Reads in the level
      // itself are three dependent trips to memory, 4400 to 5800 clocks a level
      // (5000 families 2918 -> 2831 us, 10,000 8666 -> 8572).  FP64 lanes lack
      // the registers: one family of 240 genes 1372 -> 1427 us.
      if constexpr (staged || !kF32) {
#pragma unroll 1
        for (int L = (int)F.n_lvl - 1; L >= 0; --L) {
          const uint32_t s0 = LB.at((uint32_t)L), s1 = LB.at((uint32_t)L + 1);
#pragma unroll 1
          for (uint32_t k0 = (s0 & ~15u) + wv * kChunk; k0 < s1; k0 += nt) {
            const uint32_t k = k0 + lane;
            const bool in = k >= s0 && k < s1;
            uint32_t z, r0, cnt;
            slot_of(in ? k : s0, in, z, r0, cnt);
            const uint32_t i = z & 0xffffu, pos = (z >> 16) & 0xfu;
            Real t = 0;
#pragma unroll 1
            for (uint32_t j0 = 0; __any(j0 < cnt); j0 += kRecs) {
              uint32_t o[kRecs];
              Real c[kRecs], a[kRecs], v[kRecs];
              terms_of(r0, j0, cnt, i, o, c);
#pragma unroll
              for (int j = 0; j < kRecs; ++j) {
                a[j] = T.A[o[j] & 0xffffu];
                v[j] = T.V[o[j] >> 16];
              }
#pragma unroll
              for (int j = 0; j < kRecs; ++j) t = j0 + j < cnt ? fma(cA * a[j] * c[j], v[j], t) : t;
            }
            t = slot_sum(t, pos, slot_steps(pos));
            if (z & kSlotLead) T.A[i] = i == n - 1 ? seed : t;
          }
          tsync<Team, Gws>();
        }
      } else {
        auto level = [&](uint32_t s0, uint32_t s1, auto&& first) WHALE_INLINE {
#pragma unroll 1
          for (uint32_t k0 = (s0 & ~15u) + wv * kChunk; k0 < s1; k0 += nt) {
            const uint32_t k = k0 + lane;
            const bool in = k >= s0 && k < s1, lead_chunk = k0 < (s0 & ~15u) + nt;
            uint32_t z, r0, cnt;
            uint32_t o[kRecs];
            Real c[kRecs];
            if (lead_chunk) {
              first(z, r0, cnt, o, c);
              if (!in) z = cnt = 0;
            } else {
              slot_of(in ? k : s0, in, z, r0, cnt);
            }
            const uint32_t i = z & 0xffffu, pos = (z >> 16) & 0xfu;
            Real t = 0;
#pragma unroll 1
            for (uint32_t j0 = 0; __any(j0 < cnt); j0 += kRecs) {
              Real a[kRecs], v[kRecs];
              if (!lead_chunk || j0 > 0) terms_of(r0, j0, cnt, i, o, c);
              else if (Scaled) scale(i, o, c);
#pragma unroll
              for (int j = 0; j < kRecs; ++j) {
                a[j] = T.A[o[j] & 0xffffu];
                v[j] = T.V[o[j] >> 16];
              }
#pragma unroll
              for (int j = 0; j < kRecs; ++j) t = j0 + j < cnt ? fma(cA * a[j] * c[j], v[j], t) : t;
            }
            t = slot_sum(t, pos, slot_steps(pos));
            if (z & kSlotLead) T.A[i] = i == n - 1 ? seed : t;
          }
          tsync<Team, Gws>();
        };
        struct Words {
          uint32_t z;
          u2 d;
        };
        struct Terms {
          uint32_t z, r0, cnt, o[kRecs];
          double p[kRecs];
        };
        // of level L (0 below the first): this lane's first slot, its terms
        auto words = [&](Words& w, int L) WHALE_INLINE {
          const uint32_t s0 = LB.at((uint32_t)max(L, 0));
          const uint32_t k = min((s0 & ~15u) + wv * kChunk + lane, ns - 1);
          w.d = bs2[F.root_bs + k];
          w.z = bs4[F.root_bs + k].z;
        };
        auto terms = [&](Terms& x, const Words& w) WHALE_INLINE {
          x.z = w.z;
          x.r0 = w.d.x;
          x.cnt = w.d.y & 0xffffu;
#pragma unroll
          for (int j = 0; j < kRecs; ++j) {
            const uint32_t y = ent0 + ((uint32_t)j < x.cnt ? x.r0 + j : first);
            x.o[j] = ent_ops[y];
            x.p[j] = ent_p[y];
          }
        };
        // level L from x; y takes the terms of the next level from its words,
        // whose place takes the words of the level after
        auto step = [&](int L, Terms& x, Terms& y, Words& wy, Words& wx) WHALE_INLINE {
          terms(y, wy);
          words(wx, L - 2);
          level(LB.at((uint32_t)L), LB.at((uint32_t)L + 1),
                [&](uint32_t& z, uint32_t& r0, uint32_t& cnt, uint32_t(&o)[kRecs], Real(&c)[kRecs]) WHALE_INLINE {
                  z = x.z, r0 = x.r0, cnt = x.cnt;
#pragma unroll
                  for (int j = 0; j < kRecs; ++j) {
                    o[j] = x.o[j];
                    c[j] = (uint32_t)j < cnt ? (Real)x.p[j] : Real(0);
                  }
                });
        };
        Words w0, w1;
        Terms t0, t1;
        words(w0, (int)F.n_lvl - 1);
        words(w1, (int)F.n_lvl - 2);
        terms(t0, w0);
#pragma unroll 1
        for (int L = (int)F.n_lvl - 1; L >= 0; L -= 2) {
          step(L, t0, t1, w1, w0);
          if (L > 0) step(L - 1, t1, t0, w0, w1);
        }
      }
      // With every ā known, all slots at once: with SF = Σ c·ā(owner)·G(other)
      // and SG likewise with F, ī of the tops is cB(ā ε_g + SF), cB(ā ε_f + SG);
      // and the sums of d/dA, d/dB and the root children's ε.  The sums take
      // the coefficient with the other part's value first: c·ā passes FP32's
      // range where c·ā·ℓ does not.
#pragma unroll 1
      for (uint32_t k0 = wv * kChunk; k0 < ns; k0 += nt) {
        const uint32_t k = k0 + lane;
        uint32_t z, r0, cnt;
        slot_of(k < ns ? k : 0u, k < ns, z, r0, cnt);
        const uint32_t i = z & 0xffffu, pos = (z >> 16) & 0xfu;
        Real tv = 0, tf = 0, tg = 0, tb = 0;
#pragma unroll 1
        for (uint32_t j0 = 0; __any(j0 < cnt); j0 += kRecs) {
          uint32_t o[kRecs];
          Real c[kRecs];
          terms_of(r0, j0, cnt, i, o, c);
#pragma unroll
          for (int j = 0; j < kRecs; ++j) {
            const uint32_t y = o[j] >> 16;
            const Real a = T.A[o[j] & 0xffffu], g = T.G[y], x = a * c[j];
            tv = fma(c[j] * T.V[y], a, tv);
            tb = fma(c[j] * g, a, tb);
            tf = fma(x, T.F[y], tf);
            tg = fma(x, g, tg);
          }
        }
        const int st = slot_steps(pos);
        tv = slot_sum(tv, pos, st);
        tf = slot_sum(tf, pos, st);
        tg = slot_sum(tg, pos, st);
        tb = slot_sum(tb, pos, st);
        if (z & kSlotLead) {
          const Real a = T.A[i], v = T.V[i], vf = T.F[i], vg = T.G[i];
          ibar[sg.ibar + i] = cB * (a * eg + tg);
          ibar[sg.ibar + n + i] = cB * (a * ef + tf);
          sA += 0.5 * ((double)v * tv);
          sB += (double)vf * tb + (double)a * ((double)vf * eg + (double)vg * ef);
          sF += (double)a * vf;
          sG += (double)a * vg;
        }
      }
    };
    if (RS.on) sweep(std::true_type{});
    else sweep(std::false_type{});
    sA = wave_sum(sA);
    sB = wave_sum(sB);
    sF = wave_sum(sF);
    sG = wave_sum(sG);
    if (Team) {  // the waves' parts in order
      const lptr<double> part = (lptr<double>)(ctl + kCtlSum);
      if (lane == 0) {
        part[4 * wv] = sA;
        part[4 * wv + 1] = sB;
        part[4 * wv + 2] = sF;
        part[4 * wv + 3] = sG;
      }
      tsync<Team, false>();
      if (threadIdx.x == 0)
        for (uint32_t k = 1; k < nw; ++k) {
          sA += part[4 * k];
          sB += part[4 * k + 1];
          sF += part[4 * k + 2];
          sG += part[4 * k + 3];
        }
    }
    if (tid == 0) {
      put(AL.rootA, sA);
      put(AL.rootB, sB);
      put(AL.eps + nd.child1, (double)cB * sF);
      put(AL.eps + nd.child0, (double)cB * sG);
    }
  }
  // ---------------- non-root stages, top down
  StageDev ahead = B.stage[F.stage0 + F.n_stages - 1];
  for (int s = (int)F.n_stages - 1; s >= 0; --s) {
    const StageDev S = uniform(ahead);
    if (s > 0) ahead = B.stage[F.stage0 + s - 1];
    const uint32_t n = S.n_items;
    typedef bptr<Gws, Real> Buf;
    const Buf buf = (Buf)wb;  // five arrays of n
    const auto sE = (bptr<Gws, int32_t>)(buf + n);  // until the rows begin
    const uint32_t nch = (S.n_bs + kChunk - 1) / kChunk;
    const uint32_t mych = wv < nch ? min((uint32_t)kRegChunks, (nch - wv + nw - 1) / nw) : 0u;
    const uint32_t over = wv + kRegChunks * nw;
    const int rtop = (int)S.r_max - 1;
    tsync_mem<Team>();  // ī written by the stage above
    auto slot_at = [&](uint32_t ch, u4& a, u2& b) WHALE_INLINE {
      const uint32_t k = ch * kChunk + lane;
      const bool in = k < S.n_bs;
      a = bs4[S.bs0 + (in ? k : 0u)];
      b = bs2[S.bs0 + (in ? k : 0u)];
      if (!in) {
        a = u4{~0u, ~0u, 0u, 0u};
        b = u2{0u, 0u};
      }
    };
    auto take = [&](Lane& q, const u4& a, const u2& b, const u4& r0, const u4& r1) WHALE_INLINE {
      q.item = a.z & 0xffffu;
      q.pos = (a.z >> 16) & 0xfu;
      q.lead = (a.z & kSlotLead) != 0u;
      q.start = b.x;
      q.cnt = b.y & 0xffffu;
      q.cell = r0.x + q.item;
      q.nc = r0.y;
      q.R = r0.z;
      q.tab = r0.w;
      q.k = r1;
      q.be = NC.be[r1.x >> 2];
#pragma unroll
      for (int k = 0; k < 3; ++k) q.t[k] = 0;
      q.q1 = q.q2 = 0;
#pragma unroll
      for (int k = 0; k < kSpill; ++k) q.d[k] = 0.0;
    };
    auto load_terms = [&](Lane& q) WHALE_INLINE {
      const int most = __any(q.cnt > 2) ? kRecs : __any(q.cnt > 0) ? 2 : 0;  // uniform
#pragma unroll
      for (int j = 0; j < kRecs; ++j) {
        uint32_t o = q.item * 0x10001u;
        Real p = 0;
        if (j < most) {
          const bool in = (uint32_t)j < q.cnt;
          const uint32_t k = ent0 + (in ? q.start + j : 0u);
          const uint32_t eo = ent_ops[k];
          const Real ep = (Real)ent_p[k];
          o = in ? eo : o;
          p = in ? ep : p;
        }
        q.ops[j] = o;
        q.c[j] = p;
      }
    };
    // ℓ of row x of the lane's item (of the nearest row below its top or above its bottom)
    auto row_at = [&](const Lane& q, int x) WHALE_INLINE -> Real {
      const int y = max(min(x, (int)q.R - 2), 0);
      return ell[q.cell + (uint32_t)y * q.nc];
    };
    auto eit_at = [&](uint32_t i) WHALE_INLINE -> int { return Eit[S.item0 - it_base + i]; };
    Lane q[kRegChunks];
    {
      u4 s4[kRegChunks];
      u2 s2[kRegChunks];
      int ev[kRegChunks];
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) slot_at(wv + c * nw, s4[c], s2[c]);
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) {
          const uint32_t sg = S.seg0 + (s2[c].y >> 16);
          const u4 r0 = run[2 * (size_t)sg], r1 = run[2 * (size_t)sg + 1];
          const int32_t cf = (int32_t)s4[c].x, cg = (int32_t)s4[c].y;
          q[c].a = ibar[s4[c].w];
          const Real vf = ell[cf >= 0 ? cf : 0], vg = ell[cg >= 0 ? cg : 0];
          ev[c] = Scaled ? eit_at(s4[c].z & 0xffffu) : 0;
          take(q[c], s4[c], s2[c], r0, r1);
          q[c].f = cf >= 0 ? vf : Real(0);
          q[c].g = cg >= 0 ? vg : Real(0);
          load_terms(q[c]);
        }
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) {
          q[c].v = row_at(q[c], rtop - 1);
#pragma unroll
          for (int u = 0; u < 4; ++u) q[c].pf[u] = row_at(q[c], rtop - 2 - u);
        }
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych && q[c].lead) {
          buf[q[c].item] = q[c].a;
          buf[2 * n + q[c].item] = q[c].v;
          if (Scaled) sE[q[c].item] = ev[c];
        }
    }
    // Chunks past the registers keep their items' sums behind the row buffers.
    const auto oS = (bptr<Gws, double>)(wb + align16(5 * (size_t)n * sizeof(Real)));
#pragma unroll 1
    for (uint32_t ch = over; ch < nch; ch += nw) {
      u4 a;
      u2 b;
      slot_at(ch, a, b);
      const u4 r0 = run[2 * (size_t)(S.seg0 + (b.y >> 16))];
      if (a.z & kSlotLead) {
        const uint32_t i = a.z & 0xffffu;
        const int y = max(min(rtop - 1, (int)r0.z - 2), 0);
        buf[i] = ibar[a.w];
        buf[2 * n + i] = ell[r0.x + i + (uint32_t)y * r0.y];
        if (Scaled) sE[i] = eit_at(i);
        for (int j = 0; j < 5; ++j) oS[(size_t)j * n + i] = 0.0;
      }
    }
    tsync<Team, Gws>();
    int steps = 0;
    uint32_t most = 0;
#pragma unroll
    for (int c = 0; c < kRegChunks; ++c)
      if ((uint32_t)c < mych) {
        if (Scaled) {
          const int Ei = sE[q[c].item];
#pragma unroll
          for (int j = 0; j < kRecs; ++j)
            q[c].c[j] = coef_of(q[c].c[j], Ei, sE[q[c].ops[j] >> 16], sE[q[c].ops[j] & 0xffffu]);
        }
        steps = max(steps, slot_steps(q[c].pos));
        most = max(most, __any(q[c].cnt > kSlotRecs) ? 5u : __any(q[c].cnt > 2) ? 4u : 2u);
      }
    if (Scaled) tsync<Team, Gws>();  // sE's array is the next row's ā
    Buf curA = buf, nxtA = buf + n, curV = buf + 2 * n, nxtV = buf + 3 * n;
    // a pass over the wave's chunks: those in registers, then the others
    auto each = [&](auto&& fn) WHALE_INLINE {
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c)
        if ((uint32_t)c < mych) fn(q[c], true);
#pragma unroll 1
      for (uint32_t ch = over; ch < nch; ch += nw) {
        Lane x;
        u4 a;
        u2 b;
        slot_at(ch, a, b);
        const uint32_t sg = S.seg0 + (b.y >> 16);
        const u4 r0 = run[2 * (size_t)sg], r1 = run[2 * (size_t)sg + 1];
        take(x, a, b, r0, r1);
        load_terms(x);
        if (Scaled) {
          const int Ei = eit_at(x.item);
#pragma unroll
          for (int j = 0; j < kRecs; ++j)
            x.c[j] = coef_of(x.c[j], Ei, eit_at(x.ops[j] >> 16), eit_at(x.ops[j] & 0xffffu));
        }
        x.a = curA[x.item];
        x.v = curV[x.item];
        const int32_t cf = (int32_t)a.x, cg = (int32_t)a.y;
        const Real vf = ell[cf >= 0 ? cf : 0], vg = ell[cg >= 0 ? cg : 0];
        x.f = cf >= 0 ? vf : Real(0);
        x.g = cg >= 0 ? vg : Real(0);
        fn(x, false);
      }
    };
    // the entries past a lane's registers
    auto rest = [&](const Lane& x, auto&& fn) WHALE_INLINE {
      const int Ei = Scaled ? eit_at(x.item) : 0;
#pragma unroll 1
      for (uint32_t j = kRecs; j < x.cnt; ++j) {
        const uint32_t k = ent0 + x.start + j;
        const uint32_t own = ent_ops[k] & 0xffffu, y = ent_ops[k] >> 16;
        Real c = (Real)ent_p[k];
        if (Scaled) c = coef_of(c, Ei, eit_at(y), eit_at(own));
        fn(c * curA[own], y);
      }
    };
    // one row of an item: its share of the sums, then ā(r-1); vn = ℓ(r-2)
    auto finish = [&](Lane& x, int r, Real S_, const SliceRowB<Real>& w_, Real vn) WHALE_INLINE {
      const bool in = r < (int)x.R;
      const Real X = in ? w_.ph * (x.a * x.v) : Real(0);
      const Real Y = in ? w_.ch * (Real(0.5) * x.v * S_) : Real(0);
      const Real w = fma(Real(3) * x.be, Y, Real(2) * X);
      x.q1 += X;
      x.q2 += Y;
#pragma unroll
      for (int k = 0; k < 3; ++k) x.t[k] = fma(w, w_.D[k], x.t[k]);
      x.a = in ? fma(w_.ph, x.a, x.be * w_.ch * S_) : x.a;
      x.v = vn;
      if (x.lead) {
        nxtA[x.item] = x.a;
        nxtV[x.item] = x.v;
      }
    };
    auto spill32 = [&](Lane& x) WHALE_INLINE {  // the FP32 row sums go to FP64
      if constexpr (kF32) {
        x.d[0] += (double)x.t[0];
        x.d[1] += (double)x.t[1];
        x.d[2] += (double)x.t[2];
        x.d[3] += (double)x.q1;
        x.d[4] += (double)x.q2;
        x.t[0] = x.t[1] = x.t[2] = x.q1 = x.q2 = 0;
      }
    };
    // d/dα, d/dβ, d/dε0 of the item's rows
    auto row_sums = [&](const Lane& x, double (&o)[3]) WHALE_INLINE {
      double t0 = (double)x.t[0], t1 = (double)x.t[1], t2 = (double)x.t[2], q1 = (double)x.q1, q2 = (double)x.q2;
      if constexpr (kF32) t0 += x.d[0], t1 += x.d[1], t2 += x.d[2], q1 += x.d[3], q2 += x.d[4];
      const uint32_t node = x.k.x >> 2;
      const double S1 = q1 + (double)x.be * q2;
      o[0] = t0 - S1 * (double)NC.ia[node];
      o[1] = t1 - S1 * (double)NC.ib[node] + q2;
      o[2] = t2;
    };
    auto step_sync = [&]() WHALE_INLINE {
      tsync<Team, Gws>();
      Buf t = curA;
      curA = nxtA;
      nxtA = t;
      t = curV;
      curV = nxtV;
      nxtV = t;
    };
    // Rows: loops for two or all entries a lane; waves
    // whose terms are not all in registers take the general form.
    auto rows = [&](auto km_) WHALE_INLINE {
      constexpr int NC_ = kRegChunks, KM = decltype(km_)::value;
      SliceRowB<Real> wn[NC_];  // the next row's
#pragma unroll
      for (int c = 0; c < NC_; ++c)
        wn[c] = slice_b<Real>(pack, M.tab_rows, q[c].tab + (uint32_t)min(rtop, (int)q[c].R - 1));
#pragma unroll 1
      for (int rb = rtop; rb >= 1; rb -= 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // ℓ is loaded four rows ahead of its use
          const int r = rb - u;
          if (r >= 1) {
            Real a_[NC_][KM], v_[NC_][KM], S_[NC_], vn[NC_];
            SliceRowB<Real> w[NC_];
#pragma unroll
            for (int c = 0; c < NC_; ++c) {
#pragma unroll
              for (int j = 0; j < KM; ++j) {
                a_[c][j] = curA[q[c].ops[j] & 0xffffu];
                v_[c][j] = curV[q[c].ops[j] >> 16];
              }
              w[c] = wn[c];
              wn[c] = slice_b<Real>(pack, M.tab_rows, q[c].tab + (uint32_t)max(min(r, (int)q[c].R) - 1, 0));
            }
#pragma unroll
            for (int c = 0; c < NC_; ++c) {
              vn[c] = q[c].pf[u];
              q[c].pf[u] = row_at(q[c], r - 6);
            }
#pragma unroll
            for (int c = 0; c < NC_; ++c) {
              S_[c] = 0;
#pragma unroll
              for (int j = 0; j < KM; ++j) S_[c] = fma(q[c].c[j] * a_[c][j], v_[c][j], S_[c]);
            }
            if (steps > 0) {
#pragma unroll
              for (int c = 0; c < NC_; ++c) S_[c] = slot_sum(S_[c], q[c].pos, steps);
            }
#pragma unroll
            for (int c = 0; c < NC_; ++c) finish(q[c], r, S_[c], w[c], vn[c]);
            step_sync();
          }
        }
        if (kF32 && ((rb - rtop) & 31) == 0 && rb != rtop) {
#pragma unroll
          for (int c = 0; c < NC_; ++c) spill32(q[c]);
        }
      }
    };
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, kRecs> IK;
    if (over < nch || most > kSlotRecs || (Team && mych == 0)) {
#pragma unroll 1
      for (int r = rtop; r >= 1; --r) {
        each([&](Lane& x, bool held) WHALE_INLINE {
          Real t = 0;
          const SliceRowB<Real> w = slice_b<Real>(pack, M.tab_rows, x.tab + (uint32_t)min(r, (int)x.R - 1));
#pragma unroll
          for (int j = 0; j < kRecs; ++j) t = fma(x.c[j] * curA[x.ops[j] & 0xffffu], curV[x.ops[j] >> 16], t);
          rest(x, [&](Real c, uint32_t y) WHALE_INLINE { t = fma(c, curV[y], t); });
          t = slot_sum(t, x.pos, slot_steps(x.pos));
          finish(x, r, t, w, row_at(x, r - 2));
          if (!held) {
            double o[3];
            row_sums(x, o);
            if (x.lead)
              for (int j = 0; j < 3; ++j) oS[(size_t)j * n + x.item] += o[j];
          } else if (kF32 && ((rtop - r) & 31) == 31) {
            spill32(x);
          }
        });
        step_sync();
      }
    } else if (most > 2) {
      rows(IK{});
    } else {
      rows(I2{});
    }
    // ---- row 0: adjoints of the child tops, ε and q.  With SF(γ) = Σ
    // c·ā[owner]·G[other] and SG(γ) likewise with F over the splits γ is a part
    // of (a WGD node's one child stands in both slots):
    //   speciation  ī0 = ε_g ā + SF, ī1 = ε_f ā + SG, ε̄_f += ā G, ε̄_g += ā F
    //   WGD         ī0 = q SF + (1 - q + 2 q ε_f) ā, ε̄_f += 2 q ā F,
    //               q̄ += ½ F SF - ā F + 2 ε_f ā F
    const Buf bF = curV, bG = nxtV;
    each([&](Lane& x, bool) WHALE_INLINE {
      if (x.lead) {
        bF[x.item] = x.f;
        bG[x.item] = x.g;
      }
    });
    tsync<Team, Gws>();
    each([&](Lane& x, bool held) WHALE_INLINE {
      const uint32_t kind = x.k.x & 3u;
      Real SF = 0, SG = 0;
#pragma unroll
      for (int j = 0; j < kRecs; ++j) {
        const Real c = x.c[j] * curA[x.ops[j] & 0xffffu];
        SF = fma(c, bG[x.ops[j] >> 16], SF);
        SG = fma(c, bF[x.ops[j] >> 16], SG);
      }
      rest(x, [&](Real c, uint32_t y) WHALE_INLINE {
        SF = fma(c, bG[y], SF);
        SG = fma(c, bF[y], SG);
      });
      const int st = slot_steps(x.pos);
      SF = slot_sum(SF, x.pos, st);
      SG = slot_sum(SG, x.pos, st);
      Real e0 = 0, e1 = 0;
      if (x.lead && kind != WHALE_NODE_LEAF) {
        const Real ef = NC.etop[x.k.y];
        const uint32_t ib = x.k.w + x.item;
        if (kind == WHALE_NODE_WGD) {
          const Real qq = NC.q[x.k.z];
          ibar[ib] = fma(qq, SF, ((Real(1) - qq) + Real(2) * qq * ef) * x.a);
          e0 = Real(2) * qq * (x.a * x.f);
          e1 = x.f * (Real(0.5) * SF - x.a + Real(2) * ef * x.a);
        } else {
          ibar[ib] = fma(x.a, NC.etop[x.k.z], SF);
          ibar[ib + x.nc] = fma(x.a, ef, SG);
          e0 = x.a * x.g;
          e1 = x.a * x.f;
        }
      }
      x.pf[0] = e0;
      x.pf[1] = e1;
      if (!held && x.lead) {
        oS[3 * (size_t)n + x.item] = (double)e0;
        oS[4 * (size_t)n + x.item] = (double)e1;
      }
    });
    tsync<Team, Gws>();
    // ---- the items' sums by segment: 8 lanes a segment, then once into the
    // node's accumulators
    each([&](Lane& x, bool held) WHALE_INLINE {
      if (!x.lead) return;
      double o[5];
      if (held) {
        double w[3];
        row_sums(x, w);
        o[0] = w[0], o[1] = w[1], o[2] = w[2], o[3] = (double)x.pf[0], o[4] = (double)x.pf[1];
      } else {
        for (int j = 0; j < 5; ++j) o[j] = oS[(size_t)j * n + x.item];
      }
#pragma unroll
      for (int j = 0; j < 5; ++j) buf[(size_t)j * n + x.item] = (Real)o[j];
    });
    tsync<Team, Gws>();
#pragma unroll 1
    for (uint32_t g0 = 8 * wv; g0 < S.n_segs; g0 += 8 * nw) {
      const uint32_t g = g0 + lane / 8;
      const uint32_t sg = S.seg0 + (g < S.n_segs ? g : 0u);
      const u4 r0 = run[2 * (size_t)sg], r1 = run[2 * (size_t)sg + 1];
      const uint32_t i0 = glob(B.seg)[sg].item0, i1 = g < S.n_segs ? i0 + r0.y : i0;
      double z[5] = {0, 0, 0, 0, 0};
      for (uint32_t i = i0 + (lane & 7u); i < i1; i += 8)
#pragma unroll
        for (int j = 0; j < 5; ++j) z[j] += (double)buf[(size_t)j * n + i];
#pragma unroll
      for (int j = 0; j < 5; ++j) z[j] = slot_sum(z[j], lane & 7u, 3);
      if ((lane & 7u) == 7u && g < S.n_segs) {
        const int node = (int)(r1.x >> 2);
        const uint32_t kind = r1.x & 3u;
        put(AL.da + node, z[0]);
        put(AL.db + node, z[1]);
        put(AL.e0 + node, z[2]);
        if (kind != WHALE_NODE_LEAF) {
          put(AL.eps + (int)r1.y, z[3]);
          put((kind == WHALE_NODE_WGD ? AL.q : AL.eps) + (int)r1.z, z[4]);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
constexpr int kMaxFPW = 8;   // families (one wave each) per workgroup, at most
constexpr int kMaxWaves = 12; // waves per workgroup, at most (kMaxTeam of one family, or kMaxFPW)
static_assert(kMaxTeam <= kMaxWaves && kMaxFPW <= kMaxWaves, "launch bounds");
// Resident waves per SIMD the kernels are compiled for; a wave has 512 over it
// registers.  The rows are chains of LDS round trips, so a large batch runs at
// the rate that the waves of a SIMD cover each other's waits.  Measured
// (10,000 families of 50 taxa, FP32 gradient, two evaluations): one chunk a
// wave and four waves a SIMD 9.4 ms, two waves 11.3 ms; two chunks a wave and
// two waves a SIMD 10.1 ms.  FP64 lanes hold twice the registers: with four
// waves a SIMD they spill (6,000 families, scaled FP64 gradient: 3.8 ms, three
// waves 3.4 ms).
template <typename Real>
constexpr int kWavesPerEU = sizeof(Real) == 4 ? 4 : 3;

// A mixture launch's workgroup takes its component's model, workspace and,
// when given, family order and count.  The component is read into scalar
// registers: as vector loads its pointers would be kept in vector registers,
// about 50 of them, throughout the kernel.
template <typename Real>
__device__ __forceinline__ void mix_select(const MixComp* X, int K, BatchDev& B, ModelDev& M, WorkDev<Real>& W,
                                           const uint32_t*& fam_count) {
  if (K <= 0) return;
  const MixComp x = uniform(X[blockIdx.x % (uint32_t)K]);
  M = x.M;
  W = WorkDev<Real>(x.W);
  if (x.order) B.order = x.order;
  if (x.count) fam_count = x.count;
}

// The workgroup's shared LDS: control words, the gradient's accumulators when they fit, node constants; then the families'
// regions (fwd_shared_bytes, bwd_shared_bytes).
template <typename Real>
struct Shared {
  lptr<uint32_t> ctl;
  Acc acc;
  NodeC<Real> NC;
  __device__ __forceinline__ Shared(lptr<unsigned char> p, const ModelDev& M, const WorkDev<Real>& W, bool bwd)
      : ctl((lptr<uint32_t>)p),
        acc{(lptr<double>)(p + kCtlBytes), W.acc,
            bwd && acc_lds_bytes(AccLayout(M.n, M.n_wgd).n) != 0},
        NC(p + kCtlBytes + (bwd ? acc_lds_bytes(AccLayout(M.n, M.n_wgd).n) : 0),
           M.n, M.n_wgd) {
    if (threadIdx.x < kCtlBytes / 4) ctl[threadIdx.x] = 0u;
    if (acc.in_lds) {
      const int na = AccLayout(M.n, M.n_wgd).n;
      for (int j = threadIdx.x; j < na; j += (int)blockDim.x) acc.lds[j] = 0.0;
    }
    NC.fill(M, bwd, threadIdx.x, (int)blockDim.x);
    __syncthreads();
  }
  // the workgroup's sums into the batch's
  __device__ void flush(const ModelDev& M) const {
    if (!acc.in_lds) return;
    __syncthreads();
    const int na = AccLayout(M.n, M.n_wgd).n;
    for (int j = threadIdx.x; j < na; j += (int)blockDim.x) {
      const double v = acc.lds[j];
      if (v != 0.0) unsafeAtomicAdd(acc.glb + j, v);
    }
  }
};

// the family's stage buffers: its share of the dynamic LDS, or (Gws) its
// region of the global workspace
template <bool Gws>
__device__ __forceinline__ bptr<Gws, unsigned char> region_of(unsigned char* smem, unsigned char* gws, const LdsCfg& L,
                                                              size_t slot, uint32_t in_group) {
  if constexpr (Gws) return glob(gws) + slot * L.wave_bytes;
  else return (lptr<unsigned char>)smem + L.shared_bytes + in_group * L.wave_bytes;
}

// The next family of a launch: the wave's, or (Team) the workgroup's; kNone
// when there are none left.
template <bool Team>
__device__ __forceinline__ uint32_t next_family(const BatchDev& B, uint32_t* ticket, lptr<uint32_t> ctl, int32_t fam_single,
                                                uint32_t fam_begin, uint32_t fam_end, bool first) {
  if (fam_single >= 0) return first && (Team || threadIdx.x < kWG) ? (uint32_t)fam_single : kNone;
  uint32_t k = 0;
  if (Team) {
    __syncthreads();  // the last family's readers of the word are done
    if (threadIdx.x == 0) ctl[kCtlFam] = atomicAdd(ticket, 1u);
    __syncthreads();
    k = ctl[kCtlFam];
  } else if (threadIdx.x % kWG == 0) {
    k = atomicAdd(ticket, 1u);
  }
  k = fam_begin + (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
  if (k >= fam_end) return kNone;
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)B.order[k]);  // wave-uniform: family data in scalar registers
}

template <typename Real, bool Scaled, bool StoreAll, bool Gws, bool Team>
__global__ __launch_bounds__(kWG* kMaxWaves, kWavesPerEU<Real>) void k_forward(BatchDev B, ModelDev M, WorkDev<Real> W,
                                                                       LdsCfg L, int32_t fam_single,
                                                                       uint32_t fam_begin, uint32_t fam_end,
                                                                       const uint32_t* fam_count, const MixComp* X,
                                                                       int K) {
  mix_select(X, K, B, M, W, fam_count);
  if (fam_count) fam_end = fam_begin + *fam_count;
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t lane = threadIdx.x % kWG;
  const uint32_t wv = Team ? 0u : threadIdx.x / kWG;
  const Shared<Real> sh((lptr<unsigned char>)smem, M, W, false);
  const auto wb = region_of<Gws>(smem, W.gws, L, blockIdx.x, wv);
  for (bool first = true;; first = false) {
    const uint32_t f = next_family<Team>(B, W.ticket, sh.ctl, fam_single, fam_begin, fam_end, first);
    if (f == kNone) break;
    fwd_family<Real, Scaled, StoreAll, Gws, Team>(B, M, W, f, wb, L.wave_bytes, sh.NC, sh.ctl, lane,
                                                        W.ell + B.fam[f].ell0, W.Eit, 0u);
  }
}

template <typename Real, bool Scaled, bool Gws, bool Team>
__global__ __launch_bounds__(kWG* kMaxWaves, kWavesPerEU<Real>) void k_backward(BatchDev B, ModelDev M, WorkDev<Real> W,
                                                                        LdsCfg L, int32_t fam_single,
                                                                        uint32_t fam_begin, uint32_t fam_end,
                                                                        const uint32_t* fam_count, const MixComp* X,
                                                                        int K) {
  mix_select(X, K, B, M, W, fam_count);
  if (fam_count) fam_end = fam_begin + *fam_count;
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t lane = threadIdx.x % kWG;
  const uint32_t wv = Team ? 0u : threadIdx.x / kWG;
  const Shared<Real> sh((lptr<unsigned char>)smem, M, W, true);
  const auto wb = region_of<Gws>(smem, W.gws, L, blockIdx.x, wv);
  for (bool first = true;; first = false) {
    const uint32_t f = next_family<Team>(B, W.ticket, sh.ctl, fam_single, fam_begin, fam_end, first);
    if (f == kNone) break;
    if (Scaled && sizeof(Real) == sizeof(float) && W.flag[f]) continue;  // done by the FP64 pass
    bwd_family<Real, Scaled, Gws, Team>(B, M, W, f, wb, L.wave_bytes, sh.acc, sh.NC, sh.ctl, lane,
                                              W.ell + B.fam[f].ell0, W.ibar + B.fam[f].ibar0, W.Eit, 0u);
  }
  if (!W.acc_fam) sh.flush(M);
}

// k_fused: the forward DP and (grad) the reverse sweep of each family by one
// wave or team, with the family's stored rows, ī and exponents in its own slot
// of a scratch buffer.  A family's rows live only while it is worked on, so ℓ
// takes (resident families) x (the launch's largest family) instead of every
// cell of the batch: the evaluation under a memory budget for ℓ.  Shared LDS
// as in the reverse sweep; a family's region fits both directions.
template <typename Real, bool Scaled, bool Gws, bool Team>
__global__ __launch_bounds__(kWG* kMaxWaves, kWavesPerEU<Real>) void k_fused(BatchDev B, ModelDev M, WorkDev<Real> W,
                                                                     LdsCfg L, uint32_t fam_begin, uint32_t fam_end,
                                                                     const uint32_t* fam_count, int grad,
                                                                     FusedSlots SL) {
  if (fam_count) fam_end = fam_begin + *fam_count;
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t lane = threadIdx.x % kWG;
  const uint32_t wv = Team ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWG);
  const Shared<Real> sh((lptr<unsigned char>)smem, M, W, true);
  const size_t slot = (size_t)blockIdx.x * (Team ? 1 : blockDim.x / kWG) + wv;
  const auto wb = region_of<Gws>(smem, W.gws, L, slot, wv);
  unsigned char* const sp = SL.base + slot * SL.slot_bytes;
  Real* const ell = reinterpret_cast<Real*>(sp);
  Real* const ibar = reinterpret_cast<Real*>(sp + SL.ibar_off);
  int32_t* const Eit = reinterpret_cast<int32_t*>(sp + SL.eit_off);
  for (bool first = true;; first = false) {
    const uint32_t f = next_family<Team>(B, W.ticket, sh.ctl, -1, fam_begin, fam_end, first);
    if (f == kNone) break;
    const uint32_t item0 = B.fam[f].item0;
    tsync_mem<Team>();  // the slot's previous family is done with it
    fwd_family<Real, Scaled, true, Gws, Team>(B, M, W, f, wb, L.wave_bytes, sh.NC, sh.ctl, lane, ell, Eit, item0);
    if (!grad) continue;
    tsync_mem<Team>();  // the forward's rows, exponents and flag are visible to the family's waves
    if (Scaled && sizeof(Real) == sizeof(float) &&
        __hip_atomic_load(&W.flag[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)
      continue;  // done by the FP64 pass
    bwd_family<Real, Scaled, Gws, Team>(B, M, W, f, wb, L.wave_bytes, sh.acc, sh.NC, sh.ctl, lane, ell, ibar, Eit,
                                               item0);
  }
  if (grad && !W.acc_fam) sh.flush(M);
}

// ---------------------------------------------------------------------------
// launch wrappers (instantiated once per arithmetic)
// ---------------------------------------------------------------------------
template <typename K, typename... Args>
static hipError_t go(K kern, int grid, int waves, size_t lds, hipStream_t st, Args... args) {
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kWG * waves), lds, st, args...);
  return hipGetLastError();
}

// a launch's shape is one the kernels accept
static inline bool shape_ok(const LaunchCfg& C) {
  if (C.fpw < 1 || C.team < 1 || C.grid < 1 || C.fpw * C.team > kMaxWaves) return false;
  return C.team == 1 ? C.fpw <= kMaxFPW && !C.gws : C.fpw == 1 && C.team <= kMaxTeam;
}

template <typename R, bool S, bool A>
static hipError_t fwd_go(const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M, const WorkRaw& W,
                         int32_t fam_single, uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count,
                         const MixComp* X, int K) {
  const size_t lds = C.lds();
  const WorkDev<R> w(W);
  if (!shape_ok(C) || K < 0 || K > kMaxMix || (K > 0 && (!X || fam_single >= 0))) return hipErrorInvalidValue;
  const int grid = C.grid * (K > 0 ? K : 1);
#define WHALE_FWD(GWS, TEAM)                                                                                  \
  return go(k_forward<R, S, A, GWS, TEAM>, grid, C.fpw * C.team, lds, st, B, M, w, C.L, fam_single, fam_begin, \
            fam_end, fam_count, X, K)
  if (C.gws) {  // stage buffers in the global workspace
    if (!W.gws || K > 0) return hipErrorInvalidValue;
    WHALE_FWD(true, true);
  }
  if (C.team > 1) WHALE_FWD(false, true);
  WHALE_FWD(false, false);
#undef WHALE_FWD
}

template <typename R, bool S>
hipError_t fwd_variant(bool store_all, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                       const WorkRaw& W, int32_t fam_single, uint32_t fam_begin, uint32_t fam_end,
                       const uint32_t* fam_count, const MixComp* X, int K) {
  return store_all ? fwd_go<R, S, true>(C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K)
                   : fwd_go<R, S, false>(C, st, B, M, W, fam_single, fam_begin, fam_end, fam_count, X, K);
}

template <typename R, bool S>
hipError_t bwd_variant(const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M, const WorkRaw& W,
                       int32_t fam_single, uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count,
                       const MixComp* X, int K) {
  const size_t lds = C.lds();
  const WorkDev<R> w(W);
  if (!shape_ok(C) || K < 0 || K > kMaxMix || (K > 0 && (!X || fam_single >= 0))) return hipErrorInvalidValue;
  const int grid = C.grid * (K > 0 ? K : 1);
#define WHALE_BWD(GWS, TEAM)                                                                               \
  return go(k_backward<R, S, GWS, TEAM>, grid, C.fpw * C.team, lds, st, B, M, w, C.L, fam_single, fam_begin, \
            fam_end, fam_count, X, K)
  if (C.gws) {
    if (!W.gws || K > 0) return hipErrorInvalidValue;
    WHALE_BWD(true, true);
  }
  if (C.team > 1) WHALE_BWD(false, true);
  WHALE_BWD(false, false);
#undef WHALE_BWD
}

template <typename R, bool S>
hipError_t fused_variant(const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M, const WorkRaw& W,
                         uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count, int grad,
                         const FusedSlots& SL) {
  const size_t lds = C.lds();
  const WorkDev<R> w(W);
  if (!shape_ok(C) || !SL.base || (C.gws && !W.gws)) return hipErrorInvalidValue;
#define WHALE_FUSED(GWS, TEAM)                                                                                 \
  return go(k_fused<R, S, GWS, TEAM>, C.grid, C.fpw * C.team, lds, st, B, M, w, C.L, fam_begin, fam_end, fam_count, \
            grad, SL)
  if (C.gws) WHALE_FUSED(true, true);
  if (C.team > 1) WHALE_FUSED(false, true);
  WHALE_FUSED(false, false);
#undef WHALE_FUSED
}

}  // namespace whale

// the three launch templates of one arithmetic
#define WHALE_DP_INSTANTIATE(R, S)                                                                                   \
  namespace whale {                                                                                                  \
  template hipError_t fwd_variant<R, S>(bool, const LaunchCfg&, hipStream_t, const BatchDev&, const ModelDev&,        \
                                        const WorkRaw&, int32_t, uint32_t, uint32_t, const uint32_t*, const MixComp*, \
                                        int);                                                                        \
  template hipError_t bwd_variant<R, S>(const LaunchCfg&, hipStream_t, const BatchDev&, const ModelDev&,              \
                                        const WorkRaw&, int32_t, uint32_t, uint32_t, const uint32_t*, const MixComp*, \
                                        int);                                                                        \
  template hipError_t fused_variant<R, S>(const LaunchCfg&, hipStream_t, const BatchDev&, const ModelDev&,            \
                                          const WorkRaw&, uint32_t, uint32_t, const uint32_t*, int,                  \
                                          const FusedSlots&);                                                        \
  }
