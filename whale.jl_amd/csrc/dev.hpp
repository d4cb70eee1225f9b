// Device-side views of the model, the batch plan and the per-call workspace,
// and the launch wrappers the C ABI calls.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "plan.hpp"

namespace whale {

struct BatchDev {
  const FamDev* fam;
  const StageDev* stage;
  const SegDev* seg;
  const SegRun* run;
  const uint32_t* fs4;   // slots: 4 and 2 words each (plan.hpp)
  const uint32_t* fs2;
  const uint32_t* bs4;
  const uint32_t* bs2;
  const uint32_t* rec_ops;
  const double* rec_p;
  const uint32_t* ent_ops;
  const double* ent_p;
  const uint32_t* it_gid;
  const uint16_t* clade_size;
  const double* split_p;
  const uint32_t* lvl_f;
  const uint32_t* lvl_b;
  const uint32_t* order;   // families in processing order
  uint32_t n_fam;
};

struct ModelDev {
  const NodeDev* node;
  const double* eps;
  const double* phi;
  const double* psi;
  const double* par;       // [λ(n), μ(n), p(n), q(n_wgd), η]
  // the slice tables as the DP reads them, in FP64 and FP32: per row φ, χ = ψ/β,
  // D_α, D_β; then per row φ, ψ; then per row D_ε0 (k_tables)
  const double* pack64;
  const float* pack32;
  const double* dnode;     // per node kDnode values (k_tables)
  int n;
  int n_wgd;
  int root;
  int tab_rows;
};

// per node: ∂α/∂λ, ∂α/∂μ, ∂β/∂λ, ∂β/∂μ; 1/(1-α), 1/(1-β), β; ∂ε_top/∂(ε of
// row 0), ∂ε_top/∂α, ∂ε_top/∂β (all 0 for a node of one row)
constexpr int kDnode = 10;

__device__ __forceinline__ double eps_top(const ModelDev& M, int node) {
  const NodeDev& d = M.node[node];
  return M.eps[d.tab + d.R - 1];
}

// type-erased workspace (ell, ibar hold float or double)
struct WorkRaw {
  void* ell;
  int32_t* E;         // per clade
  int32_t* Eit;       // per item
  void* ibar;
  double* fam_ll;
  double* acc;
  uint32_t* ticket;
  uint32_t* flag;     // per family: 1 if the FP32 form left its range (recomputed in FP64)
  uint32_t* fb;       // fb[0] = number of such families, fb[1..] = their indices
  unsigned char* gws; // stage buffers of launches whose families do not fit LDS (LaunchCfg::gws)
  double* acc_fam = nullptr;  // deterministic gradients: per-family accumulator slots
  // per-family weights of the reverse sweep (null: 1): family f's adjoint is
  // seeded with seed[f] / L_f, and seed[n_fam] = Σ seed scales the
  // conditioning term's derivative (mixture responsibilities)
  double* seed = nullptr;
};

// gradient accumulator layout (doubles): per node the derivatives of logL in
// the branch's α, β and ε of row 0 through its φ_r, ψ_r, and in ε at its top;
// then q per WGD and the root's constants
struct AccLayout {
  int da, db, e0, eps, q, rootA, rootB, n;
  __host__ __device__ AccLayout(int nodes, int nwgd) {
    da = 0;
    db = nodes;
    e0 = 2 * nodes;
    eps = 3 * nodes;
    q = 4 * nodes;
    rootA = q + nwgd;
    rootB = rootA + 1;
    n = rootB + 1;
  }
};

__host__ __device__ constexpr size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

// Chunks of slots a wave holds in registers; a stage with more than its team
// holds streams the rest from memory every row.
constexpr int kRegChunks = 1;
constexpr int kMaxTeam = 12;  // most waves of one family (three a SIMD)

// LDS of one family, laid out afresh for every stage from its item count n
// (s = bytes per Real).  The same functions size the launches on the host and
// carve the buffers on the device.
//   forward stage, root:  A F G [n] | E [n], flags [n] (scaled forms)
//   reverse stage:        five arrays [n] | row sums, 5 doubles an item, when the
//                         stage has more slots than the largest team's registers
//   reverse root:         A V F G [n] | E [n] (scaled forms)
__host__ __device__ inline size_t fwd_bytes(size_t s, bool scaled, size_t n) {
  return align16(3 * n * s) + (scaled ? align16(4 * n) + align16(n) : 0);
}
__host__ __device__ inline size_t bwd_stage_bytes(size_t s, size_t n, size_t slots) {
  return align16(5 * n * s) + (slots > kRegChunks * (size_t)kChunk ? 40 * n : 0);
}
__host__ __device__ inline size_t bwd_root_bytes(size_t s, bool scaled, size_t n) {
  return align16(4 * n * s) + (scaled ? align16(4 * n) : 0);
}

//   the root's terms and slots, staged behind its arrays when they fit:
//                         operands, coefficients [nt] | slots, 8 bytes each [ns]
__host__ __device__ inline size_t root_stage_bytes(size_t s, size_t nt, size_t ns) {
  return align16(4 * nt) + align16(s * nt) + 8 * ns;
}

// LDS family d needs (s bytes per value): its largest non-root stage and its
// root, with the root's terms staged or not
__host__ __device__ inline size_t fam_lds_bytes(const FamDev& d, size_t s, bool scaled, bool fwd, int team,
                                                bool staged) {
  const size_t a = fwd ? fwd_bytes(s, scaled, d.max_items) : bwd_stage_bytes(s, d.max_items, (d.max_slots + team - 1) / team);
  size_t b = fwd ? fwd_bytes(s, scaled, d.n_clades) : bwd_root_bytes(s, scaled, d.n_clades);
  if (staged) b += root_stage_bytes(s, (fwd ? 1 : 2) * (size_t)d.root_recs, fwd ? d.root_nfs : d.root_nbs);
  return a > b ? a : b;
}

// A launch of k_forward / k_backward: every family of a workgroup has
// `wave_bytes` of LDS (laid out per stage); `shared_bytes` (control words,
// reverse-sweep accumulators, node constants) come first and are
// shared by the workgroup.
struct LdsCfg {
  uint32_t wave_bytes;
  uint32_t shared_bytes;
};

// a launch: `fpw` families of one wave each per workgroup, or one family of
// `team` waves.  With `gws` the families' stage
// buffers (wave_bytes each) live in a global workspace instead of LDS, one
// family per workgroup: the path of families whose largest stage does not fit
// one compute unit's LDS.
struct LaunchCfg {
  int grid = 1;
  int fpw = 1;
  int team = 1;
  int waves_per_cu = 0;  // families per compute unit the LDS allows
  bool gws = false;
  LdsCfg L{};
  size_t lds() const { return (size_t)L.shared_bytes + (gws ? 0 : (size_t)fpw * L.wave_bytes); }
  size_t gws_bytes() const { return gws ? (size_t)grid * fpw * L.wave_bytes : 0; }
};

constexpr size_t kCtlBytes = 16 + 32 * kMaxTeam;  // control words and the waves' partial sums of a workgroup
// the gradient's accumulators in LDS (0: too many, they are added to global memory)
__host__ __device__ inline size_t acc_lds_bytes(int n) { return n <= 4096 ? align16(8 * (size_t)n) : 0; }
size_t fwd_shared_bytes(int mode, int n, int nwgd);
size_t bwd_shared_bytes(int mode, int n, int nwgd);

// forward/backward launch: `mode` is WHALE_FP64_PLAIN / WHALE_FP32_SCALED /
// WHALE_FP64_SCALED; fam_single >= 0 runs that one family (first family of a
// 1-block grid), otherwise waves or teams take families order[fam_begin .. fam_end)
// from the ticket.  fam_count, if not null, replaces fam_end with a count read
// on the device (the FP64 pass over families listed by the FP32 pass).
// One component of a mixture launch: with K components the grid is K times
// the launch's, and workgroup w works for component w % K with that
// component's model (tables), workspace (tickets included), and, when not
// null, its own family order and count (the FP64 pass over families its
// FP32 pass flagged).
struct MixComp {
  ModelDev M;
  WorkRaw W;
  const uint32_t* order = nullptr;
  const uint32_t* count = nullptr;
};
constexpr int kMaxMix = 8;

// the launches of one arithmetic (dp.hpp; instantiated in dp_*.hip)
template <typename R, bool S>
hipError_t fwd_variant(bool store_all, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                       const WorkRaw& W, int32_t fam_single, uint32_t fam_begin, uint32_t fam_end,
                       const uint32_t* fam_count, const MixComp* X, int K);
template <typename R, bool S>
hipError_t bwd_variant(const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M, const WorkRaw& W,
                       int32_t fam_single, uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count,
                       const MixComp* X, int K);
struct FusedSlots;
template <typename R, bool S>
hipError_t fused_variant(const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M, const WorkRaw& W,
                         uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count, int grad,
                         const FusedSlots& SL);
hipError_t launch_forward(int mode, bool store_all, const LaunchCfg& C, hipStream_t st, const BatchDev& B,
                          const ModelDev& M, const WorkRaw& W, int32_t fam_single, uint32_t fam_begin,
                          uint32_t fam_end, const uint32_t* fam_count = nullptr, const MixComp* X = nullptr,
                          int K = 0);
hipError_t launch_backward(int mode, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                           const WorkRaw& W, int32_t fam_single, uint32_t fam_begin, uint32_t fam_end,
                           const uint32_t* fam_count = nullptr, const MixComp* X = nullptr, int K = 0);
// per family i: ℓ_ij = fam_ll_j[i] + log prior_j − c_j over the K components
// (c_j the component's conditioning term), r_ij = exp(ℓ_ij − logsumexp_j ℓ_ij)
// into seed_j[i] and Σ_i r_ij into seed_j[n_fam]; out[0] = Σ_i logsumexp_j ℓ_ij
// (−inf if not finite); resp (n_fam × K, may be null) = r
hipError_t launch_mix(hipStream_t st, const MixComp* X, int K, const double* log_prior, uint32_t n_fam, int cond,
                      double* out, double* resp);
// per-family slots of the fused forward + reverse launch: each holds one
// family's stored rows (from byte 0), ī (from ibar_off) and its items'
// exponents (from eit_off)
struct FusedSlots {
  unsigned char* base = nullptr;
  uint64_t slot_bytes = 0;
  uint64_t ibar_off = 0;
  uint64_t eit_off = 0;
};
hipError_t launch_fused(int mode, const LaunchCfg& C, hipStream_t st, const BatchDev& B, const ModelDev& M,
                        const WorkRaw& W, uint32_t fam_begin, uint32_t fam_end, const uint32_t* fam_count, int grad,
                        const FusedSlots& SL);
hipError_t launch_tables(hipStream_t st, const ModelDev& M, double* eps, double* phi, double* psi, double* pack64,
                         float* pack32, double* dnode, const int32_t* hlevels, const int32_t* hnodes, int n_levels,
                         const int32_t* row_node, double* work);
// the workspace of launch_tables: in LDS up to kTabLds (`work` null), else `work`
constexpr size_t kTabLds = 128 * 1024;
size_t tables_work_bytes(int n, int rows);
// n_eff (null: n_fam) holds the family count the conditioning term's
// derivative is scaled by (Σ of the reverse sweep's family weights)
hipError_t launch_tail(hipStream_t st, const ModelDev& M, const double* fam_ll, uint32_t n_fam, const double* acc,
                       double* work, const int32_t* dlevels, const int32_t* dnodes, int n_dlevels, int cond,
                       int with_grad, double* out, const double* n_eff = nullptr, double* host_fam = nullptr,
                       const uint32_t* fb = nullptr, uint32_t* host_fb = nullptr);
size_t tail_work_bytes(int n);  // `work` of launch_tail
hipError_t launch_reset(hipStream_t st, uint32_t* ticket, int n_ticket, double* acc, int n_acc, uint32_t* flag,
                        int n_flag, uint32_t* fb);
hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t v, int n);
hipError_t launch_det_sum(hipStream_t st, const double* slots, uint32_t n_fam, int ncol, double* out);

// What the backtracking sampler reads: the stored ℓ (FP32 or FP64 values,
// plus the FP64 region of families an FP32 call evaluated in FP64), the
// clades' exponents, each (family, node)'s segment, each segment's first
// item (its clades in increasing id), and every clade's split list.
struct BtDev {
  const FamDev* fam;
  const SegDev* seg;
  const uint32_t* it_gid;
  const uint32_t* seg_item;   // absolute first item of each segment
  const int32_t* node_seg;    // [family][node]: segment, or -1 (no compatible clade)
  const uint32_t* spl_off;    // per absolute clade: its splits [spl_off[c], spl_off[c + 1])
  const uint32_t* spl_g;      // per split: g1 | g2 << 16 (family-local clade ids)
  const double* split_p;
  const uint16_t* clade_size;
  const void* ell;
  const double* ell64;
  const int32_t* E;           // null in the plain form
  const uint8_t* fam64;       // per family: 1 if its ℓ is in ell64 (null: none)
  int ell_float;              // the main region holds FP32 values
};
hipError_t launch_backtrack(hipStream_t st, const BtDev& D, const ModelDev& M, uint32_t fam_begin, uint32_t n_fams,
                            uint32_t n_samples, uint64_t seed, uint32_t cap, int32_t* counts, int32_t* nodes,
                            int32_t* stack, uint32_t max_items);
hipError_t launch_bt_pack(hipStream_t st, uint64_t walks, const int32_t* counts, const int32_t* nodes, uint32_t cap,
                          uint64_t* first, uint64_t* cursor, int32_t* packed);

// The fixed per-GPU workspace of whale_logpdf_noalloc (a file-scope device
// array in kernels.hip) and its device address on `device`, which must be the
// current device; found once per device and kept.
constexpr size_t kScratchBytes = 64ull << 20;
constexpr int kMaxDevices = 64;
hipError_t scratch_address(int device, void** out);

}  // namespace whale
