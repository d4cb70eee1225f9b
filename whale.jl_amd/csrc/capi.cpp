// C ABI (include/whale_amd.h): contexts, models, CCD ingest, device batches
// and the evaluation entry points.  Host code; kernels live in kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>
#include <memory>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/whale_amd.h"
#include "dev.hpp"
#include "host.hpp"

using namespace whale;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) return fail(WHALE_EHIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// device buffer owned by a handle
struct DBuf {
  void* p = nullptr;
  size_t n = 0;
  ~DBuf() { if (p) (void)hipFree(p); }
  hipError_t alloc(size_t bytes) {
    if (bytes <= n && p) return hipSuccess;
    if (p) { (void)hipFree(p); p = nullptr; n = 0; }
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipSuccess) n = bytes;
    return e;
  }
  void free() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  template <typename T> T* as() const { return static_cast<T*>(p); }
};

template <typename V>
hipError_t upload(DBuf& b, const V& v, hipStream_t st, bool wait = true) {
  const size_t n = v.size() * sizeof(v[0]);
  hipError_t e = b.alloc(n);
  if (e != hipSuccess || v.empty()) return e;
  e = hipMemcpyAsync(b.p, v.data(), n, hipMemcpyHostToDevice, st);
  if (e != hipSuccess || !wait) return e;
  return hipStreamSynchronize(st);
}

// waits for a stream at the end of a scope
struct StreamWait {
  hipStream_t st;
  ~StreamWait() { (void)hipStreamSynchronize(st); }
};

}  // namespace

struct whale_batch;
namespace {
constexpr int kLayouts = 6;
// The searchable launch shape of a batch.
struct Tuning {
  uint32_t bounds[5] = {10 * 1024, 14 * 1024, 20 * 1024, 28 * 1024, 48 * 1024};  // class bounds (bytes of row state, fam_size)
  int layout = 0;      // index into kLayoutOrder / kLayoutLane
  int waves_cap = 8;   // resident families per compute unit a launch aims for
};
// Class launch orders (largest first within a stream) and the stream of each
// class, for the candidate layouts.  Layout 0 was chosen by hand among a
// dozen on the 10,000-family workload; the others are what the search tries.
constexpr int kLayoutOrder[kLayouts][6] = {
    {5, 4, 1, 3, 2, 0}, {5, 4, 3, 2, 1, 0}, {5, 4, 3, 2, 1, 0},
    {5, 4, 3, 2, 1, 0}, {5, 4, 3, 2, 1, 0}, {5, 4, 3, 2, 1, 0}};
constexpr int kLayoutLane[kLayouts][6] = {  // stream of class 0..5
    {2, 2, 1, 0, 1, 0},   // 5 then 3 | 4 then 2 | 1 then 0
    {0, 1, 2, 0, 1, 2},   // 5, 2 | 4, 1 | 3, 0
    {0, 0, 1, 1, 2, 2},   // 5, 4 | 3, 2 | 1, 0
    {1, 2, 0, 2, 1, 0},   // 5, 2 | 4, 0 | 3, 1
    {2, 1, 0, 0, 1, 2},   // 5, 0 | 4, 1 | 3, 2
    {1, 1, 2, 1, 2, 0}};  // 5 alone | 4, 2 | 3, 1, 0

// family tickets: one per class and direction, two for the FP64 pass after an
// FP32 pass, two for the families routed to FP64 from the start, two for the
// families whose stages do not fit LDS
constexpr int kTickets = 18;
constexpr int kTicketHbm = 16;
int assign_classes(whale_batch* b);
int plan_batch_launches(whale_batch* b);
int ensure_gws(whale_batch* b, bool* moved);
void drop_graphs(whale_batch* b);
uint64_t full_bytes(const whale_batch* b);
int replan(whale_batch* b);

// LDS family d needs in `mode` when `team` waves evaluate it (fam_lds_bytes)
size_t fam_lds(const whale::FamDev& d, int mode, bool fwd, int team, bool staged) {
  return whale::fam_lds_bytes(d, mode == WHALE_FP32_SCALED ? 4 : 8, mode != WHALE_FP64_PLAIN, fwd, team, staged);
}
// The size a family is classed by: the registers its largest stage takes, at
// 80 bytes of row state a slot (an FP32 lane's).
size_t fam_size(const whale::FamDev& d) { return 80 * (size_t)d.max_slots; }
// the fewest waves that hold every stage of a family in registers (kRegChunks
// chunks a wave), at most kMaxTeam
int fam_team(uint32_t max_slots) {
  constexpr uint32_t held = whale::kRegChunks * whale::kChunk;
  return std::max(1, std::min(whale::kMaxTeam, (int)((max_slots + held - 1) / held)));
}
}  // namespace

struct whale_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipStream_t side = nullptr;   // size classes run here and on side3 beside the context's stream
  hipStream_t side3 = nullptr;
  hipStream_t side2 = nullptr;  // families routed to FP64 run here
  hipEvent_t fork[8] = {};
  int n_cu = 256;
  size_t lds_wg = 64 * 1024;   // LDS one workgroup may allocate
  size_t lds_cu = 64 * 1024;   // LDS of one compute unit
  bool timing = false;
  hipEvent_t ev[6] = {};
  hipEvent_t user[16] = {};
  double last_ms[5] = {0, 0, 0, 0, 0};
  unsigned char* scratch = nullptr;  // this device's copy of the fixed workspace (whale_logpdf_noalloc)
};

struct whale_model {
  whale_ctx* ctx = nullptr;
  ModelHost h;
  DBuf nodes, eps, phi, psi, pack64, pack32, dnode, par, hlv, hnd, dlv, dnd, rown, twork, ebar;
  int n_hlevels = 0, n_dlevels = 0;
  bool has_params = false;
  std::vector<double> host_par;
  ModelDev dev() const {
    ModelDev M;
    M.node = nodes.as<NodeDev>();
    M.eps = eps.as<double>();
    M.phi = phi.as<double>();
    M.psi = psi.as<double>();
    M.par = par.as<double>();
    M.pack64 = pack64.as<double>();
    M.pack32 = pack32.as<float>();
    M.dnode = dnode.as<double>();
    M.n = h.n;
    M.n_wgd = h.n_wgd;
    M.root = h.root;
    M.tab_rows = h.tab_rows;
    return M;
  }
};

struct whale_ccd {
  CCDHost c;
};

struct whale_batch {
  whale_model* model = nullptr;
  int device = 0;
  PlanHost plan;
  DBuf fam, stage, seg, run, it_gid, fs4, fs2, bs4, bs2, rec_ops, rec_p, ent_ops, ent_p, clade_size, split_p, lvl_f,
      lvl_b, order;
  // workspace.  ell/ibar hold the main pass (FP32 or FP64 values) in
  // their first 8 bytes per element and, for FP32 runs, the FP64 recomputation
  // of families that left the FP32 range after the first align8(4 * n) bytes.
  DBuf ell, E, Eit, ibar, fam_ll, acc, ticket, flag, fb;
  // the families' split lists (per absolute clade: first split; per split:
  // g1 | g2 << 16) and, built on the first backtracking call, each
  // (family, node)'s segment and each segment's first item; the sampler's
  // output and stack buffers
  DBuf spl_off, spl_g, node_seg, seg_item, fam64, bt_counts, bt_nodes, bt_stack;
  // stage buffers of the launches that run them in global memory
  // (LaunchCfg::gws): the launches on the context's stream use the first
  // gws_main bytes, the FP64 evaluation of routed families (on its own
  // stream, concurrently) the rest
  DBuf gws;
  size_t gws_main = 0;
  uint64_t n_rec = 0;
  uint32_t n_fam = 0;
  // size classes by the LDS one family needs: families order[cls_lo[c] .. cls_hi[c])
  static constexpr int kClasses = 6;
  uint32_t cls_lo[kClasses] = {}, cls_hi[kClasses] = {};
  // Families whose largest stage, in the FP64-scaled form, does not fit the
  // LDS of one compute unit (or `lds_limit`, when set): order[hbm_lo ..
  // hbm_hi), first in `order`; they run one per workgroup with their stage
  // buffers in the global workspace `gws`.
  uint32_t hbm_lo = 0, hbm_hi = 0;
  size_t lds_limit = 0;  // 0: the device's LDS per workgroup
  LaunchCfg cfg_hbm[3][2];
  // Launch-shape parameters (whale_batch_autotune searches them): the LDS
  // bounds of the size classes, how the classes are spread over the three
  // streams, and the most waves per compute unit a launch plans for.
  Tuning tune;
  // Memory budget for the stored rows of ℓ (0: none).  When the whole
  // batch's ℓ, ī and exponents exceed it, evaluations without stored ℓ
  // for the caller run the fused forward + reverse launches, whose per-wave
  // slots hold one family at a time (k_fused); their launch shapes and slots,
  // per mode, are planned on first use.
  size_t ell_budget = 0;
  bool fused_ok[3] = {};
  LaunchCfg fcfg[3][kClasses], fcfg_hbm[3], fcfg_route[3], fcfg_fb;
  FusedSlots fslot[3][kClasses], fslot_hbm[3], fslot_route[3], fslot_fb[3];
  size_t fused_bytes[3] = {};
  DBuf fslots;
  bool full_ok = false;  // ell, Eit and ibar allocated for every family
  // Deterministic gradients: each family's accumulators land in its own slot
  // of acc_fam, and a fixed-order sum over families follows, so that repeated
  // evaluations give bit-identical gradients.
  bool det = false;
  DBuf acc_fam;
  // Per-family weights of the reverse sweep (whale_batch_set_seeds): n_fam
  // seeds, then their sum; used by gradient calls while `seeded`.
  bool seeded = false;
  DBuf seed;
  // Mixture evaluations (whale_mixture_eval): one workspace per component,
  // the per-launch component tables, the log priors, the result and the
  // responsibilities.
  struct MixWork {
    DBuf ell, E, Eit, ibar, fam_ll, acc, ticket, flag, fb, seed, out;
  };
  std::vector<std::unique_ptr<MixWork>> mixw;
  DBuf mixsel, mixprior, mixout, mixresp;
  LaunchCfg cfg[3][2][kClasses];   // [mode][forward, backward][class]
  // the launches of one evaluation: a class, or adjacent classes as one launch
  // (plan_groups); a group's largest class names its entry of cfg and ticket
  struct Group {
    int cls, lane;
    uint32_t lo, hi;   // order_host[lo, hi)
    LaunchCfg cfg[2];  // forward, backward
  };
  std::vector<Group> groups[3];
  // the same for a mixture of mix_k components (0: not planned since the classes were)
  std::vector<Group> mix_groups[3];
  int mix_k[3] = {0, 0, 0};
  LaunchCfg cfg_fb[2];             // FP64 pass over families the FP32 form could not represent
  int last_mode = -1;
  int last_launch = WHALE_LAUNCH_BATCHED;
  bool last_store_all = false;
  uint32_t last_fallback = 0;  // families of the last FP32 call computed in FP64
  // Families whose FP32 values left the range in an earlier call: FP32 calls
  // evaluate them in FP64 with per-clade exponents from the start, beside the
  // FP32 classes (other modes treat them like any family).  They sit last in
  // `order`, at [route_lo, n_fam).
  std::vector<uint8_t> routed;
  std::vector<uint32_t> flagged_once;  // recomputed in FP64 by the last call, routed from the next
  uint32_t route_lo = 0;
  LaunchCfg cfg_route[3][2];
  std::vector<uint32_t> order_host;
  // captured evaluations, keyed by (mode, gradient, keep ℓ), and pinned result staging
  hipGraphExec_t graph[3][2][2][2] = {};  // [mode][gradient][keep ℓ][fused]
  double* pin_out = nullptr;
  double* pin_fam = nullptr;
  ~whale_batch() {
    for (auto& a : graph) for (auto& b2 : a) for (auto& c2 : b2) for (auto& g : c2) if (g) (void)hipGraphExecDestroy(g);
    if (pin_out) (void)hipHostFree(pin_out);
    if (pin_fam) (void)hipHostFree(pin_fam);
  }
  BatchDev dev() const {
    BatchDev B;
    B.fam = fam.as<FamDev>();
    B.stage = stage.as<StageDev>();
    B.seg = seg.as<SegDev>();
    B.run = run.as<SegRun>();
    B.fs4 = fs4.as<uint32_t>();
    B.fs2 = fs2.as<uint32_t>();
    B.bs4 = bs4.as<uint32_t>();
    B.bs2 = bs2.as<uint32_t>();
    B.rec_ops = rec_ops.as<uint32_t>();
    B.rec_p = rec_p.as<double>();
    B.ent_ops = ent_ops.as<uint32_t>();
    B.ent_p = ent_p.as<double>();
    B.it_gid = it_gid.as<uint32_t>();
    B.clade_size = clade_size.as<uint16_t>();
    B.split_p = split_p.as<double>();
    B.lvl_f = lvl_f.as<uint32_t>();
    B.lvl_b = lvl_b.as<uint32_t>();
    B.order = order.as<uint32_t>();
    B.n_fam = n_fam;
    return B;
  }
  WorkRaw work() const {
    WorkRaw W;
    W.ell = ell.p;
    W.E = E.as<int32_t>();
    W.Eit = Eit.as<int32_t>();
    W.ibar = ibar.p;
    W.fam_ll = fam_ll.as<double>();
    W.acc = acc.as<double>();
    W.ticket = ticket.as<uint32_t>();
    W.flag = flag.as<uint32_t>();
    W.fb = fb.as<uint32_t>();
    W.gws = gws.as<unsigned char>();
    return W;
  }
  // the FP64 region used for families recomputed after an FP32 pass
  WorkRaw work_fallback() const { return fallback_of(work()); }
  WorkRaw fallback_of(WorkRaw W) const {
    W.ell = (char*)W.ell + fp32_bytes(plan.ell_cells);
    W.ibar = (char*)W.ibar + fp32_bytes(plan.ibar_cells);
    return W;
  }
  static uint64_t fp32_bytes(uint64_t n) { return ((4 * n + 7) / 8) * 8; }
};

extern "C" {

const char* whale_last_error(void) { return g_err.c_str(); }

int whale_ctx_create(int device, whale_ctx** out) {
  if (!out) return fail(WHALE_EINVAL, "out is NULL");
  int n = 0;
  HIPCHK(hipGetDeviceCount(&n));
  if (device < 0 || device >= n) return fail(WHALE_EINVAL, "no such HIP device");
  HIPCHK(hipSetDevice(device));
  auto c = std::make_unique<whale_ctx>();
  c->device = device;
  HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  HIPCHK(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
  HIPCHK(hipStreamCreateWithFlags(&c->side2, hipStreamNonBlocking));
  HIPCHK(hipStreamCreateWithFlags(&c->side3, hipStreamNonBlocking));
  for (auto& e : c->fork) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  hipDeviceProp_t prop;
  HIPCHK(hipGetDeviceProperties(&prop, device));
  c->n_cu = prop.multiProcessorCount;
  {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device) == hipSuccess && v > 0)
      c->lds_wg = (size_t)v;
    c->lds_cu = c->lds_wg;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device) == hipSuccess && v > 0)
      c->lds_cu = std::max(c->lds_wg, (size_t)v);
  }
  for (auto& e : c->ev) HIPCHK(hipEventCreate(&e));
  for (auto& e : c->user) HIPCHK(hipEventCreate(&e));
  {  // the device address of this GPU's fixed workspace, with the device current
    void* p = nullptr;
    HIPCHK(scratch_address(device, &p));
    c->scratch = static_cast<unsigned char*>(p);
  }
  *out = c.release();
  return WHALE_OK;
}

int whale_ctx_destroy(whale_ctx* c) {
  if (!c) return WHALE_OK;
  (void)hipSetDevice(c->device);
  for (auto& e : c->ev) if (e) (void)hipEventDestroy(e);
  for (auto& e : c->user) if (e) (void)hipEventDestroy(e);
  for (auto& e : c->fork) if (e) (void)hipEventDestroy(e);
  if (c->side) (void)hipStreamDestroy(c->side);
  if (c->side2) (void)hipStreamDestroy(c->side2);
  if (c->side3) (void)hipStreamDestroy(c->side3);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return WHALE_OK;
}

void* whale_ctx_stream(whale_ctx* c) { return c ? (void*)c->stream : nullptr; }

int whale_ctx_record(whale_ctx* c, int32_t slot) {
  if (!c || slot < 0 || slot >= 16) return fail(WHALE_EINVAL, "bad context or event slot");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipEventRecord(c->user[slot], c->stream));
  return WHALE_OK;
}

int whale_ctx_elapsed(whale_ctx* c, int32_t a, int32_t b, double* ms) {
  if (!c || !ms || a < 0 || a >= 16 || b < 0 || b >= 16) return fail(WHALE_EINVAL, "bad context or event slot");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipEventSynchronize(c->user[b]));
  float f = 0;
  HIPCHK(hipEventElapsedTime(&f, c->user[a], c->user[b]));
  *ms = f;
  return WHALE_OK;
}

int whale_ctx_set_timing(whale_ctx* c, int32_t en) {
  if (!c) return fail(WHALE_EINVAL, "ctx is NULL");
  c->timing = en != 0;
  return WHALE_OK;
}

int whale_last_timings(whale_ctx* c, double* ms5) {
  if (!c || !ms5) return fail(WHALE_EINVAL, "NULL argument");
  for (int i = 0; i < 5; ++i) ms5[i] = c->last_ms[i];
  return WHALE_OK;
}

int whale_model_create(whale_ctx* ctx, int32_t n, const int32_t* parent, const int32_t* kind, const int32_t* child0,
                       const int32_t* child1, const int32_t* n_slices, const double* slice_len,
                       const double* leaf_prob, const int32_t* wgd_index, const int32_t* leaf_species,
                       int32_t n_species, const int32_t* order, int32_t condition, whale_model** out) {
  if (!ctx || !out || n <= 0 || !parent || !kind || !child0 || !child1 || !n_slices || !slice_len || !leaf_prob ||
      !wgd_index || !leaf_species || !order)
    return fail(WHALE_EINVAL, "whale_model_create: NULL or empty argument");
  if (condition < 0 || condition > 2) return fail(WHALE_EINVAL, "unknown condition");
  if (n_species <= 0) return fail(WHALE_EINVAL, "n_species must be positive");
  auto m = std::make_unique<whale_model>();
  m->ctx = ctx;
  ModelHost& h = m->h;
  h.n = n;
  h.n_species = n_species;
  h.cond = condition;
  h.words = (n_species + 63) / 64;
  h.nodes.resize(n);
  int nwgd = 0, roots = 0;
  for (int i = 0; i < n; ++i) {
    NodeDev& d = h.nodes[i];
    d.kind = kind[i];
    d.child0 = child0[i];
    d.child1 = child1[i];
    d.parent = parent[i];
    d.R = n_slices[i] + 1;
    d.wgd = wgd_index[i];
    d.leafP = leaf_prob[i];
    d.delta = slice_len[i];
    d.pad = 0;
    if (n_slices[i] < 0) return fail(WHALE_EINVAL, "negative slice count");
    auto okc = [&](int c) { return c >= 0 && c < n && parent[c] == i; };
    switch (d.kind) {
      case WHALE_NODE_LEAF:
        if (d.child0 != -1 || d.child1 != -1) return fail(WHALE_EINVAL, "leaf with children");
        if (leaf_species[i] < 0 || leaf_species[i] >= n_species) return fail(WHALE_EINVAL, "leaf species out of range");
        break;
      case WHALE_NODE_WGD:
        if (!okc(d.child0) || d.child1 != -1) return fail(WHALE_EINVAL, "WGD node needs exactly one child");
        if (d.wgd < 0) return fail(WHALE_EINVAL, "WGD node without a q index");
        nwgd = std::max(nwgd, d.wgd + 1);
        break;
      case WHALE_NODE_SPECIATION:
      case WHALE_NODE_ROOT:
        if (!okc(d.child0) || !okc(d.child1)) return fail(WHALE_EINVAL, "speciation/root node needs two children");
        break;
      default:
        return fail(WHALE_EINVAL, "unknown node kind");
    }
    if (d.kind == WHALE_NODE_ROOT) { ++roots; h.root = i; if (parent[i] != -1) return fail(WHALE_EINVAL, "root with a parent"); }
    else if (parent[i] < 0 || parent[i] >= n) return fail(WHALE_EINVAL, "non-root node without a parent");
  }
  if (roots != 1) return fail(WHALE_EINVAL, "the tree needs exactly one root");
  h.n_wgd = nwgd;
  // order must list every node once, children before parents
  std::vector<int> pos(n, -1);
  for (int k = 0; k < n; ++k) {
    if (order[k] < 0 || order[k] >= n || pos[order[k]] >= 0) return fail(WHALE_EINVAL, "order is not a permutation");
    pos[order[k]] = k;
  }
  for (int i = 0; i < n; ++i)
    if (parent[i] >= 0 && pos[parent[i]] < pos[i]) return fail(WHALE_EINVAL, "order lists a parent before a child");
  if (order[n - 1] != h.root) return fail(WHALE_EINVAL, "order must end with the root");
  h.order.assign(order, order + n);
  // species bitsets, heights, table offsets
  h.bits.assign((size_t)n * h.words, 0);
  h.height.assign(n, 0);
  for (int e : h.order) {
    const NodeDev& d = h.nodes[e];
    uint64_t* b = &h.bits[(size_t)e * h.words];
    if (d.kind == WHALE_NODE_LEAF) {
      b[leaf_species[e] >> 6] |= 1ull << (leaf_species[e] & 63);
    } else {
      for (int c : {d.child0, d.child1}) {
        if (c < 0) continue;
        for (int w = 0; w < h.words; ++w) b[w] |= h.bits[(size_t)c * h.words + w];
        h.height[e] = std::max(h.height[e], h.height[c] + 1);
      }
    }
  }
  h.max_height = h.height[h.root];
  h.tab_off.assign(n + 1, 0);
  for (int i = 0; i < n; ++i) {
    h.nodes[i].tab = h.tab_off[i];
    h.tab_off[i + 1] = h.tab_off[i] + h.nodes[i].R;
  }
  h.tab_rows = h.tab_off[n];
  // height levels (children first) and depth levels (parents first)
  std::vector<int32_t> hlv, hnd, dlv, dnd;
  for (int L = 0; L <= h.max_height; ++L) {
    hlv.push_back((int32_t)hnd.size());
    for (int e : h.order) if (h.height[e] == L) hnd.push_back(e);
  }
  hlv.push_back((int32_t)hnd.size());
  std::vector<int> depth(n, 0);
  int maxd = 0;
  for (int k = n - 1; k >= 0; --k) {
    int e = h.order[k];
    if (parent[e] >= 0) depth[e] = depth[parent[e]] + 1;
    maxd = std::max(maxd, depth[e]);
  }
  for (int L = 0; L <= maxd; ++L) {
    dlv.push_back((int32_t)dnd.size());
    for (int e = 0; e < n; ++e) if (depth[e] == L) dnd.push_back(e);
  }
  dlv.push_back((int32_t)dnd.size());
  m->n_hlevels = (int)hlv.size() - 1;
  m->n_dlevels = (int)dlv.size() - 1;
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  HIPCHK(upload(m->nodes, h.nodes, st));
  HIPCHK(upload(m->hlv, hlv, st));
  HIPCHK(upload(m->hnd, hnd, st));
  HIPCHK(upload(m->dlv, dlv, st));
  HIPCHK(upload(m->dnd, dnd, st));
  std::vector<int32_t> rown;  // every table row's node
  for (int e = 0; e < n; ++e) rown.insert(rown.end(), (size_t)h.nodes[e].R, e);
  HIPCHK(upload(m->rown, rown, st));
  if (const size_t tw = tables_work_bytes(n, h.tab_rows); tw > kTabLds || tw > ctx->lds_wg) HIPCHK(m->twork.alloc(tw));
  HIPCHK(m->eps.alloc(sizeof(double) * h.tab_rows));
  HIPCHK(m->phi.alloc(sizeof(double) * h.tab_rows));
  HIPCHK(m->psi.alloc(sizeof(double) * h.tab_rows));
  HIPCHK(m->pack64.alloc(sizeof(double) * 7 * h.tab_rows));
  HIPCHK(m->pack32.alloc(sizeof(float) * 7 * h.tab_rows));
  HIPCHK(m->dnode.alloc(sizeof(double) * kDnode * n));
  HIPCHK(m->par.alloc(sizeof(double) * (3 * n + nwgd + 1)));
  HIPCHK(m->ebar.alloc(tail_work_bytes(n)));
  *out = m.release();
  return WHALE_OK;
}

int whale_model_destroy(whale_model* m) {
  if (!m) return WHALE_OK;
  (void)hipSetDevice(m->ctx->device);
  delete m;
  return WHALE_OK;
}

int whale_model_set_params(whale_model* m, const double* lambda, const double* mu, const double* q, int32_t n_q,
                           double eta, const double* p) {
  if (!m || !lambda || !mu) return fail(WHALE_EINVAL, "whale_model_set_params: NULL argument");
  const int n = m->h.n;
  if (n_q < m->h.n_wgd || (m->h.n_wgd > 0 && !q)) return fail(WHALE_EINVAL, "too few q values for the WGD nodes");
  std::vector<double>& hp = m->host_par;
  hp.assign(3 * n + m->h.n_wgd + 1, 0.0);
  for (int i = 0; i < n; ++i) {
    hp[i] = lambda[i];
    hp[n + i] = mu[i];
    hp[2 * n + i] = p ? p[i] : 0.0;
  }
  for (int w = 0; w < m->h.n_wgd; ++w) hp[3 * n + w] = q[w];
  hp[3 * n + m->h.n_wgd] = eta;
  whale_ctx* c = m->ctx;
  HIPCHK(hipSetDevice(c->device));
  if (c->timing) HIPCHK(hipEventRecord(c->ev[0], c->stream));
  HIPCHK(hipMemcpyAsync(m->par.p, hp.data(), hp.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
  HIPCHK(launch_tables(c->stream, m->dev(), m->eps.as<double>(), m->phi.as<double>(), m->psi.as<double>(),
                       m->pack64.as<double>(), m->pack32.as<float>(), m->dnode.as<double>(), m->hlv.as<int32_t>(), m->hnd.as<int32_t>(),
                       m->n_hlevels, m->rown.as<int32_t>(), m->twork.as<double>()));
  if (c->timing) HIPCHK(hipEventRecord(c->ev[1], c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (c->timing) {
    float ms;
    HIPCHK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    c->last_ms[0] = ms;
  }
  m->has_params = true;
  return WHALE_OK;
}

int whale_model_table_offsets(const whale_model* m, int32_t* off) {
  if (!m || !off) return fail(WHALE_EINVAL, "NULL argument");
  for (int i = 0; i <= m->h.n; ++i) off[i] = m->h.tab_off[i];
  return WHALE_OK;
}

int whale_model_tables(whale_model* m, double* eps, double* phi, double* psi) {
  if (!m) return fail(WHALE_EINVAL, "NULL model");
  if (!m->has_params) return fail(WHALE_ESTATE, "parameters not set");
  HIPCHK(hipSetDevice(m->ctx->device));
  size_t b = sizeof(double) * m->h.tab_rows;
  if (eps) HIPCHK(hipMemcpy(eps, m->eps.p, b, hipMemcpyDeviceToHost));
  if (phi) HIPCHK(hipMemcpy(phi, m->phi.p, b, hipMemcpyDeviceToHost));
  if (psi) HIPCHK(hipMemcpy(psi, m->psi.p, b, hipMemcpyDeviceToHost));
  return WHALE_OK;
}

int whale_ccd_parse(const char* text, size_t len, const char* const* names, const int32_t* ids, int32_t n_names,
                    whale_ccd** out) {
  if (!text || !out || (n_names > 0 && (!names || !ids))) return fail(WHALE_EINVAL, "whale_ccd_parse: NULL argument");
  std::unordered_map<std::string, int> sp;
  for (int k = 0; k < n_names; ++k) sp[names[k]] = ids[k];
  auto c = std::make_unique<whale_ccd>();
  std::string err = parse_ale(text, len, sp, c->c);
  if (!err.empty()) return fail(WHALE_EPARSE, err);
  *out = c.release();
  return WHALE_OK;
}

int whale_ccd_parse_many(const char* const* texts, const size_t* lens, int32_t n, const char* const* names,
                         const int32_t* ids, int32_t n_names, int32_t n_threads, whale_ccd** out, int32_t* bad) {
  if (bad) *bad = -1;
  if (n < 0 || (n > 0 && (!texts || !lens || !out)) || (n_names > 0 && (!names || !ids)))
    return fail(WHALE_EINVAL, "whale_ccd_parse_many: NULL argument");
  std::unordered_map<std::string, int> sp;
  for (int k = 0; k < n_names; ++k) sp[names[k]] = ids[k];
  std::vector<std::unique_ptr<whale_ccd>> res(n);
  std::vector<std::string> err(n);
  const unsigned hw = std::min(std::max(1u, std::thread::hardware_concurrency()), 16u);
  const int nt = std::max(1, std::min(n_threads > 0 ? (int)n_threads : (int)hw, (int)n));
  auto work = [&](int w) {
    for (int i = w; i < n; i += nt) {
      if (!texts[i]) {
        err[i] = "NULL text";
        continue;
      }
      auto c = std::make_unique<whale_ccd>();
      err[i] = parse_ale(texts[i], lens[i], sp, c->c);
      if (err[i].empty()) res[i] = std::move(c);
    }
  };
  std::vector<std::thread> th;
  for (int w = 1; w < nt; ++w) th.emplace_back(work, w);
  work(0);
  for (auto& t : th) t.join();
  for (int i = 0; i < n; ++i)
    if (!res[i]) {
      if (bad) *bad = i;
      return fail(WHALE_EPARSE, "family " + std::to_string(i) + ": " + err[i]);
    }
  for (int i = 0; i < n; ++i) out[i] = res[i].release();
  return WHALE_OK;
}

int whale_ccd_shape(const whale_ccd* c, int32_t* nc, int32_t* ns) {
  if (!c || !nc || !ns) return fail(WHALE_EINVAL, "NULL argument");
  *nc = (int32_t)c->c.size.size();
  *ns = (int32_t)c->c.g1.size();
  return WHALE_OK;
}

int whale_ccd_export(const whale_ccd* c, int32_t* size, int32_t* leaf_species, int32_t* split_off, int32_t* g1,
                     int32_t* g2, double* p) {
  if (!c) return fail(WHALE_EINVAL, "NULL ccd");
  const CCDHost& h = c->c;
  if (size) std::copy(h.size.begin(), h.size.end(), size);
  if (leaf_species) std::copy(h.leaf_species.begin(), h.leaf_species.end(), leaf_species);
  if (split_off) std::copy(h.split_off.begin(), h.split_off.end(), split_off);
  if (g1) std::copy(h.g1.begin(), h.g1.end(), g1);
  if (g2) std::copy(h.g2.begin(), h.g2.end(), g2);
  if (p) std::copy(h.p.begin(), h.p.end(), p);
  return WHALE_OK;
}

int whale_ccd_destroy(whale_ccd* c) {
  delete c;
  return WHALE_OK;
}

int whale_batch_create(whale_model* m, int32_t n_fam, const int64_t* fam_clade_off, const int32_t* clade_size,
                       const int32_t* leaf_species, const int64_t* split_off, const int32_t* g1, const int32_t* g2,
                       const double* p, whale_batch** out) {
  if (!m || !out || n_fam <= 0 || !fam_clade_off || !clade_size || !leaf_species || !split_off || !g1 || !g2 || !p)
    return fail(WHALE_EINVAL, "whale_batch_create: NULL or empty argument");
  if (fam_clade_off[0] != 0) return fail(WHALE_EINVAL, "fam_clade_off[0] must be 0");
  for (int f = 0; f < n_fam; ++f)
    if (fam_clade_off[f + 1] < fam_clade_off[f]) return fail(WHALE_EINVAL, "fam_clade_off is not increasing");
  int64_t nc = fam_clade_off[n_fam];
  for (int64_t c = 0; c < nc; ++c) {
    if (split_off[c + 1] < split_off[c]) return fail(WHALE_EINVAL, "split_off is not increasing");
    if (clade_size[c] < 1) return fail(WHALE_EINVAL, "clade size must be positive");
  }
  if (nc > 0xffffffffLL || split_off[nc] > 0xffffffffLL) return fail(WHALE_EINVAL, "batch too large");
  auto b = std::make_unique<whale_batch>();
  b->model = m;
  b->device = m->ctx->device;
  unsigned hw = std::max(1u, std::thread::hardware_concurrency());
  std::string err = build_plan(m->h, n_fam, fam_clade_off, clade_size, leaf_species, split_off, g1, g2, p, b->plan,
                               (int)std::min(hw, 16u));
  if (!err.empty()) return fail(WHALE_EINVAL, err);
  PlanHost& P = b->plan;
  b->n_fam = (uint32_t)n_fam;
  b->routed.assign(n_fam, 0);
  {
    const int rc = assign_classes(b.get());
    if (rc != WHALE_OK) return rc;
  }
  whale_ctx* c = m->ctx;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = c->stream;
  {
    const int rc = ensure_gws(b.get(), nullptr);
    if (rc != WHALE_OK) return rc;
  }
  // copies queued together: every source lives until the wait below
  std::vector<uint32_t> so(nc + 1), sg((size_t)split_off[nc]);
  const StreamWait wait_copies{st};  // also where a copy fails
  HIPCHK(upload(b->fam, P.fam, st, false));
  HIPCHK(upload(b->stage, P.stage, st, false));
  HIPCHK(upload(b->seg, P.seg, st, false));
  HIPCHK(upload(b->run, P.run, st, false));
  HIPCHK(upload(b->it_gid, P.it_gid, st, false));
  HIPCHK(upload(b->fs4, P.fs4, st, false));
  HIPCHK(upload(b->fs2, P.fs2, st, false));
  HIPCHK(upload(b->bs4, P.bs4, st, false));
  HIPCHK(upload(b->bs2, P.bs2, st, false));
  HIPCHK(upload(b->rec_ops, P.rec_ops, st, false));
  HIPCHK(upload(b->rec_p, P.rec_p, st, false));
  HIPCHK(upload(b->ent_ops, P.ent_ops, st, false));
  HIPCHK(upload(b->ent_p, P.ent_p, st, false));
  HIPCHK(upload(b->clade_size, P.clade_size, st, false));
  HIPCHK(upload(b->split_p, P.split_p, st, false));
  HIPCHK(upload(b->lvl_f, P.lvl_f, st, false));
  HIPCHK(upload(b->lvl_b, P.lvl_b, st, false));
  HIPCHK(upload(b->order, b->order_host, st, false));
  {
    for (int64_t c = 0; c <= nc; ++c) so[c] = (uint32_t)split_off[c];
    for (size_t k = 0; k < sg.size(); ++k) sg[k] = (uint32_t)g1[k] | ((uint32_t)g2[k] << 16);
    HIPCHK(upload(b->spl_off, so, st, false));
    HIPCHK(upload(b->spl_g, sg, st, false));
  }
  b->n_rec = P.rec_ops.size();

  HIPCHK(b->E.alloc(sizeof(int32_t) * std::max<int64_t>(1, nc)));

  HIPCHK(b->flag.alloc(sizeof(uint32_t) * n_fam));
  HIPCHK(b->fb.alloc(sizeof(uint32_t) * (n_fam + 1)));
  HIPCHK(b->fam_ll.alloc(sizeof(double) * n_fam));
  AccLayout AL(m->h.n, m->h.n_wgd);
  HIPCHK(b->acc.alloc(sizeof(double) * AL.n));
  HIPCHK(b->ticket.alloc(sizeof(uint32_t) * kTickets));
  HIPCHK(hipHostMalloc((void**)&b->pin_out, sizeof(double) * (3 + 2 * m->h.n + m->h.n_wgd), hipHostMallocDefault));
  HIPCHK(hipHostMalloc((void**)&b->pin_fam, sizeof(double) * n_fam, hipHostMallocDefault));
  HIPCHK(hipStreamSynchronize(st));
  // release host copies the device now owns (keep what ℓ download needs)
  for (auto* v : {&P.fs4, &P.fs2, &P.bs4, &P.bs2, &P.rec_ops, &P.ent_ops}) RawVec<uint32_t>().swap(*v);
  RawVec<double>().swap(P.rec_p);
  RawVec<double>().swap(P.ent_p);
  *out = b.release();
  return WHALE_OK;
}

int whale_batch_destroy(whale_batch* b) {
  if (!b) return WHALE_OK;
  (void)hipSetDevice(b->device);  // the model may already be gone
  delete b;
  return WHALE_OK;
}

int whale_batch_fallbacks(const whale_batch* b, int32_t* n) {
  if (!b || !n) return fail(WHALE_EINVAL, "NULL argument");
  *n = (int32_t)b->last_fallback;
  return WHALE_OK;
}

int whale_batch_launches(const whale_batch* b, int32_t mode, int64_t* o) {
  static_assert(whale_batch::kClasses == WHALE_SIZE_CLASSES, "size classes of the C ABI");
  if (!b || !o) return fail(WHALE_EINVAL, "NULL argument");
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  for (int dir = 0; dir < 2; ++dir)
    for (int k = 0; k < whale_batch::kClasses; ++k) {
      const LaunchCfg& C = b->cfg[mode][dir][k];
      int64_t* r = o + 8 * (whale_batch::kClasses * dir + k);
      r[0] = b->cls_hi[k] - b->cls_lo[k];
      r[1] = C.fpw;
      r[2] = 0;  // the slice tables are read from global memory
      r[3] = C.grid;
      r[4] = (int64_t)C.lds();
      r[5] = C.L.shared_bytes;
      r[6] = 0;
      r[7] = C.L.wave_bytes;
    }
  return WHALE_OK;
}

int whale_batch_hbm_families(const whale_batch* b, int32_t* n) {
  if (!b || !n) return fail(WHALE_EINVAL, "NULL argument");
  *n = (int32_t)(b->hbm_hi - b->hbm_lo);
  return WHALE_OK;
}

int whale_batch_set_lds_limit(whale_batch* b, int64_t bytes) {
  if (!b) return fail(WHALE_EINVAL, "NULL argument");
  if (bytes < 0) return fail(WHALE_EINVAL, "negative LDS limit");
  HIPCHK(hipSetDevice(b->device));
  b->lds_limit = (size_t)bytes;
  int rc = assign_classes(b);
  if (rc != WHALE_OK) return rc;
  if ((rc = ensure_gws(b, nullptr)) != WHALE_OK) return rc;
  HIPCHK(hipMemcpy(b->order.p, b->order_host.data(), sizeof(uint32_t) * b->n_fam, hipMemcpyHostToDevice));
  drop_graphs(b);
  return WHALE_OK;
}

int whale_batch_set_ell_budget(whale_batch* b, int64_t bytes) {
  if (!b) return fail(WHALE_EINVAL, "NULL argument");
  if (bytes < 0) return fail(WHALE_EINVAL, "negative budget");
  HIPCHK(hipSetDevice(b->device));
  b->ell_budget = (size_t)bytes;
  for (bool& x : b->fused_ok) x = false;
  drop_graphs(b);
  if (b->ell_budget && full_bytes(b) > b->ell_budget && b->full_ok) {
    // the stored form's buffers are given back; a call that keeps ℓ allocates them again
    b->ell.free();
    b->Eit.free();
    b->ibar.free();
    b->full_ok = false;
    if (b->last_store_all) b->last_mode = -1;  // nothing stored any more
  }
  return WHALE_OK;
}

int whale_batch_set_deterministic(whale_batch* b, int32_t on) {
  if (!b) return fail(WHALE_EINVAL, "NULL argument");
  HIPCHK(hipSetDevice(b->device));
  const bool was = b->det;
  b->det = on != 0;
  const int rc = replan(b);
  if (rc != WHALE_OK) {
    b->det = was;
    (void)replan(b);
    return rc;
  }
  return WHALE_OK;
}

int whale_batch_ell_bytes(const whale_batch* b, int64_t* out3) {
  if (!b || !out3) return fail(WHALE_EINVAL, "NULL argument");
  out3[0] = (int64_t)full_bytes(b);
  size_t fz = 0;
  for (int m = 0; m < 3; ++m)
    if (b->fused_ok[m]) fz = std::max(fz, b->fused_bytes[m]);
  out3[1] = (int64_t)fz;
  out3[2] = (int64_t)((b->full_ok ? b->ell.n + b->Eit.n + b->ibar.n : 0) + b->fslots.n);
  return WHALE_OK;
}

int whale_batch_stats(const whale_batch* b, int64_t* o) {
  if (!b || !o) return fail(WHALE_EINVAL, "NULL argument");
  const PlanHost& P = b->plan;
  o[0] = b->n_fam;
  o[1] = P.n_clades;
  o[2] = P.n_splits;
  o[3] = P.cells;
  o[4] = P.split_terms;
  o[5] = P.sum_compat;
  o[6] = (int64_t)P.it_seg.size();
  o[7] = (int64_t)b->rec_ops.n / sizeof(uint32_t);
  o[8] = (int64_t)P.stage.size();
  o[9] = P.row_steps;
  o[10] = P.max_items;
  o[11] = (int64_t)P.ell_cells;
  return WHALE_OK;
}

namespace {

// Launch shape of one forward or backward launch over families that need
// `wave` bytes of LDS each and `team` waves: the shape with the most resident
// families per compute unit (LDS-limited, at most `cap`), then the fewest
// families per workgroup.
constexpr int kMaxFPW = 8;

bool plan_launch(const whale_model* m, bool fwd, int mode, size_t wave, uint64_t nfam, bool multi, int team,
                 LaunchCfg* out, int cap) {
  wave = align16(std::max<size_t>(wave, 16));
  const size_t shared = fwd ? fwd_shared_bytes(mode, m->h.n, m->h.n_wgd) : bwd_shared_bytes(mode, m->h.n, m->h.n_wgd);
  int best_fpw = 0, best_fams = 0, best_wg = 0;
  for (int fpw = 1; fpw <= (multi && team == 1 ? kMaxFPW : 1); ++fpw) {
    const size_t lds = shared + (size_t)fpw * wave;
    if (lds > m->ctx->lds_wg) break;
    const int wg = (int)std::min<size_t>(m->ctx->lds_cu / lds, (size_t)std::max(1, cap / fpw));
    if (wg * fpw > best_fams) {
      best_fpw = fpw;
      best_fams = wg * fpw;
      best_wg = wg;
    }
  }
  if (best_fpw == 0) return false;
  LaunchCfg C;
  C.fpw = best_fpw;
  C.team = team;
  C.waves_per_cu = best_fams;
  C.L.wave_bytes = (uint32_t)wave;
  C.L.shared_bytes = (uint32_t)shared;
  const uint64_t need = (nfam + C.fpw - 1) / C.fpw;
  C.grid = (int)std::max<uint64_t>(1, std::min<uint64_t>((uint64_t)m->ctx->n_cu * best_wg, need));
  *out = C;
  return true;
}

// A launch over the families `fams` (both directions when `fused`): a
// family's region fits the largest of them, its team the widest stage.
bool plan_families(const whale_batch* b, bool fwd, int mode, const uint32_t* fams, size_t nf, uint64_t grid_fams,
                   bool multi, LaunchCfg* out, bool force_gws = false, bool fused = false) {
  uint32_t slots = 0;
  for (size_t j = 0; j < nf; ++j) slots = std::max(slots, b->plan.fam[fams[j]].max_slots);
  auto need_of = [&](int team, bool staged) {
    size_t need = 16;
    for (size_t j = 0; j < nf; ++j) {
      const FamDev& d = b->plan.fam[fams[j]];
      need = std::max(need, fam_lds(d, mode, fwd, team, staged));
      if (fused) need = std::max(need, fam_lds(d, mode, !fwd, team, staged));
    }
    return need;
  };
  const int team = fam_team(slots);
  // the root's terms are staged in LDS unless reading them from global memory
  // lets more than a third more families share a compute unit
  LaunchCfg x, y;
  const int cap = b->tune.waves_cap;
  const bool ox = !force_gws && plan_launch(b->model, fwd, mode, need_of(team, true), grid_fams, multi, team, &x, cap);
  const bool oy = !force_gws && plan_launch(b->model, fwd, mode, need_of(team, false), grid_fams, multi, team, &y, cap);
  if (ox || oy) {
    *out = ox && (!oy || 4 * x.waves_per_cu >= 3 * y.waves_per_cu) ? x : y;
    return true;
  }
  // the stage buffers in global memory: one family per workgroup by the
  // largest team, only the node constants (and accumulators) in LDS
  const whale_model* m = b->model;
  const size_t need = need_of(kMaxTeam, false);
  LaunchCfg g;
  g.gws = true;
  g.fpw = 1;
  g.team = kMaxTeam;
  g.waves_per_cu = 1;
  g.L.wave_bytes = (uint32_t)align16(need);
  g.L.shared_bytes = (uint32_t)(fwd ? fwd_shared_bytes(mode, m->h.n, m->h.n_wgd)
                                    : bwd_shared_bytes(mode, m->h.n, m->h.n_wgd));
  if (g.L.shared_bytes > m->ctx->lds_wg || need > 0xffffffffull) return false;
  g.grid = (int)std::max<uint64_t>(1, std::min<uint64_t>((uint64_t)m->ctx->n_cu, grid_fams));
  *out = g;
  return true;
}

// whether family d runs with its stage buffers in LDS: its FP64-scaled
// stages (the largest form) fit the LDS limit in both directions
bool fits_lds(const whale_batch* b, const FamDev& d) {
  const whale_model* m = b->model;
  size_t lim = m->ctx->lds_wg;
  if (b->lds_limit) lim = std::min(lim, b->lds_limit);
  const int md = WHALE_FP64_SCALED, team = fam_team(d.max_slots);
  const size_t f = fwd_shared_bytes(md, m->h.n, m->h.n_wgd) + align16(fam_lds(d, md, true, team, false));
  const size_t r =
      bwd_shared_bytes(md, m->h.n, m->h.n_wgd) + align16(fam_lds(d, md, false, team, false));
  return f <= lim && r <= lim;
}

// The launches of one evaluation.  Launches on one stream run one after the
// other, and a family takes as long alone as beside others, so a batch that
// the GPU holds at once runs as few launches as leave it resident: adjacent
// classes share a launch (by the largest's team; a smaller family's idle waves
// wait at barriers) while the waves and the LDS of all families stay within
// kFill times what the compute units hold.  Larger batches keep their classes,
// each of which fills the GPU.  Measured, classes apart -> together, per pass:
// 100 families, FP64 gradient, 818 -> 500 us; 1000 families, FP32 gradient,
// 1990 -> 1310 us (1.6 times what the GPU holds; by kFill 1 in four launches
// 1760); 777 families of 50 taxa, scaled FP64, 3350 -> 2200 us (kFill 1: 3140).
// Past kFill the idle waves cost more than the launches: 5000 families, 2.5
// times what the GPU holds, 3160 us apart, 3690 in two launches.
// `comps`: that many components of a mixture run in every launch.
void plan_groups(const whale_batch* b, int mode, int comps, std::vector<whale_batch::Group>& out) {
  const whale_model* m = b->model;
  out.clear();
  const uint32_t* ord = b->order_host.data();
  for (int j = 0; j < whale_batch::kClasses; ++j) {
    const int k = kLayoutOrder[b->tune.layout][j];
    if (b->cls_hi[k] > b->cls_lo[k])
      out.push_back({k, kLayoutLane[b->tune.layout][k], b->cls_lo[k], b->cls_hi[k], {b->cfg[mode][0][k], b->cfg[mode][1][k]}});
  }
  std::vector<whale_batch::Group> cls = out;  // largest class first, as in order_host
  std::sort(cls.begin(), cls.end(), [](const auto& x, const auto& y) { return x.cls > y.cls; });
  const int nc = (int)cls.size();
  constexpr double kFill = 2.0;
  const double waves = kFill * m->ctx->n_cu * (mode == WHALE_FP32_SCALED ? 16 : 12);
  const double lds = kFill * (double)m->ctx->n_cu * (double)m->ctx->lds_cu;
  // waves and LDS of a launch's families
  auto load = [&](const whale_batch::Group& g, double* w, double* l) {
    for (int d = 0; d < 2; ++d) {
      const double n = (double)comps * (g.hi - g.lo);
      w[d] += n * g.cfg[d].team;
      l[d] += n * (double)g.cfg[d].lds() / g.cfg[d].fpw;
    }
  };
  auto fits = [&](const std::vector<whale_batch::Group>& gs, double* total) {
    double w[2] = {0, 0}, l[2] = {0, 0};
    for (const auto& g : gs) load(g, w, l);
    *total = w[0];
    return std::max(w[0], w[1]) <= waves && std::max(l[0], l[1]) <= lds;
  };
  double total;
  if (nc < 2 || !fits(cls, &total)) return;
  // launches of classes i..j (largest first), planned when first asked for
  std::vector<whale_batch::Group> range((size_t)nc * nc);
  std::vector<char> known((size_t)nc * nc, 0);
  std::vector<whale_batch::Group> best;
  double best_total = 0;
  for (uint32_t cut = 0; cut < 1u << (nc - 1); ++cut) {  // bit i: a launch ends after class i
    const size_t n = (size_t)__builtin_popcount(cut) + 1;
    if (!best.empty() && n > best.size()) continue;
    std::vector<whale_batch::Group> gs;
    bool ok = true;
    for (int i = 0, j; i < nc && ok; i = j + 1) {
      for (j = i; j < nc - 1 && !(cut >> j & 1); ++j) {}
      whale_batch::Group& g = range[(size_t)i * nc + j];
      char& state = known[(size_t)i * nc + j];
      if (!state) {
        g = cls[i];
        g.hi = cls[j].hi;
        state = 1;
        if (j > i)
          for (int d = 0; d < 2; ++d)
            if (!plan_families(b, d == 0, mode, ord + g.lo, g.hi - g.lo, g.hi - g.lo, true, &g.cfg[d]) || g.cfg[d].gws) state = 2;
      }
      ok = state == 1;
      gs.push_back(g);
    }
    if (!ok || !fits(gs, &total)) continue;
    if (best.empty() || n < best.size() || total < best_total) {
      best = gs;
      best_total = total;
    }
  }
  if (best.empty() || (int)best.size() == nc) return;
  out = best;
  for (size_t g = 0; g < out.size(); ++g) out[g].lane = (int)g % 3;
}

// launch shapes of every class, mode and direction, and of the FP64 pass over
// families the FP32 form could not represent
int plan_batch_launches(whale_batch* b) {
  const whale_model* m = b->model;
  for (int mode = 0; mode < 3; ++mode)
    for (int dir = 0; dir < 2; ++dir)
      if (b->hbm_hi > b->hbm_lo &&
          !plan_families(b, dir == 0, mode, b->order_host.data() + b->hbm_lo, b->hbm_hi - b->hbm_lo,
                         b->hbm_hi - b->hbm_lo, false, &b->cfg_hbm[mode][dir], true))
        return fail(WHALE_EINVAL, "the node constants do not fit the LDS of one compute unit");
  for (int mode = 0; mode < 3; ++mode)
    for (int dir = 0; dir < 2; ++dir)
      for (int k = 0; k < whale_batch::kClasses; ++k) {
        const uint32_t lo = b->cls_lo[k], hi = b->cls_hi[k];
        if (!plan_families(b, dir == 0, mode, b->order_host.data() + lo, hi - lo, hi - lo, true, &b->cfg[mode][dir][k]))
          return fail(WHALE_EINVAL, "a family's largest stage does not fit the LDS of one compute unit");
      }
  for (int mode = 0; mode < 3; ++mode) {
    plan_groups(b, mode, 1, b->groups[mode]);
    b->mix_k[mode] = 0;
  }
  for (int dir = 0; dir < 2; ++dir)
    if (!plan_families(b, dir == 0, WHALE_FP64_SCALED, b->order_host.data(), b->order_host.size(),
                       (uint64_t)m->ctx->n_cu, false, &b->cfg_fb[dir]))
      return fail(WHALE_EINVAL, "a family's largest stage does not fit the LDS of one compute unit");
  return WHALE_OK;
}

// Size classes by the widest stage of a family (fam_size), so that the
// families of a launch want the same number of waves.
// Order: largest class first, costliest families first in a class, families
// routed to FP64 last.  Then the launch shapes.
int assign_classes(whale_batch* b) {
  const PlanHost& P = b->plan;
  const uint32_t* bounds = b->tune.bounds;
  std::vector<uint32_t> cls[whale_batch::kClasses], rt, hbm;
  for (uint32_t f : P.cost_order) {
    if (b->routed[f]) {
      rt.push_back(f);
      continue;
    }
    if (!fits_lds(b, P.fam[f])) {
      hbm.push_back(f);
      continue;
    }
    const size_t need = fam_size(P.fam[f]);
    int k = whale_batch::kClasses - 1;
    while (k > 0 && need <= bounds[k - 1]) --k;
    cls[k].push_back(f);
  }
  b->order_host.clear();
  b->hbm_lo = 0;
  b->order_host.insert(b->order_host.end(), hbm.begin(), hbm.end());
  b->hbm_hi = (uint32_t)b->order_host.size();
  for (int k = whale_batch::kClasses - 1; k >= 0; --k) {
    b->cls_lo[k] = (uint32_t)b->order_host.size();
    b->order_host.insert(b->order_host.end(), cls[k].begin(), cls[k].end());
    b->cls_hi[k] = (uint32_t)b->order_host.size();
  }
  b->route_lo = (uint32_t)b->order_host.size();
  b->order_host.insert(b->order_host.end(), rt.begin(), rt.end());
  for (bool& x : b->fused_ok) x = false;  // fused shapes follow the classes
  int rc = plan_batch_launches(b);
  if (rc != WHALE_OK) return rc;
  for (int mode = 0; mode < 3; ++mode)
    for (int dir = 0; dir < 2; ++dir)
      if (!rt.empty() &&
          !plan_families(b, dir == 0, mode == WHALE_FP32_SCALED ? WHALE_FP64_SCALED : mode, rt.data(), rt.size(),
                         rt.size(), true, &b->cfg_route[mode][dir]))
        return fail(WHALE_EINVAL, "a family's largest stage does not fit the LDS of one compute unit");
  return WHALE_OK;
}

// The global workspace for the stage buffers of every launch planned with
// them in global memory (the class of families that do not fit LDS, the FP64
// passes over flagged or routed families, and per-family launches of the
// former).  Grows only; captured evaluations must be dropped when it moves.
int ensure_gws(whale_batch* b, bool* moved) {
  size_t main = 0, route = 0;
  for (int mode = 0; mode < 3; ++mode)
    for (int dir = 0; dir < 2; ++dir) {
      if (b->hbm_hi > b->hbm_lo) main = std::max(main, b->cfg_hbm[mode][dir].gws_bytes());
      if (b->route_lo < b->n_fam) route = std::max(route, b->cfg_route[mode][dir].gws_bytes());
    }
  for (int dir = 0; dir < 2; ++dir) main = std::max(main, b->cfg_fb[dir].gws_bytes());
  for (int mode = 0; mode < 3; ++mode)
    if (b->fused_ok[mode]) {
      main = std::max(main, std::max(b->fcfg_hbm[mode].gws_bytes(), b->fcfg_fb.gws_bytes()));
      if (b->route_lo < b->n_fam) route = std::max(route, b->fcfg_route[mode].gws_bytes());
    }
  for (uint32_t k = b->hbm_lo; k < b->hbm_hi; ++k)
    for (int dir = 0; dir < 2; ++dir)
      main = std::max(main, align16(fam_lds(b->plan.fam[b->order_host[k]], WHALE_FP64_SCALED, dir == 0, kMaxTeam, false)));
  main = (main + 255) & ~(size_t)255;
  const size_t need = main + route;
  if (moved) *moved = main != b->gws_main || need > b->gws.n;
  b->gws_main = main;
  if (need == 0 || need <= b->gws.n) return WHALE_OK;
  HIPCHK(b->gws.alloc(need));
  return WHALE_OK;
}

void drop_graphs(whale_batch* b) {
  for (auto& a : b->graph)
    for (auto& b2 : a)
      for (auto& c2 : b2)
        for (auto& g : c2)
          if (g) {
            (void)hipGraphExecDestroy(g);
            g = nullptr;
          }
}

// ℓ and ī of every family (8 bytes per value, or 4 with the FP64 region of
// recomputed families after it in the FP32 form) and the items' exponents
uint64_t full_bytes(const whale_batch* b) {
  const PlanHost& P = b->plan;
  return (16 + 12 * std::max<uint64_t>(1, P.ell_cells)) + 4 * std::max<uint64_t>(1, P.it_seg.size()) +
         (16 + 12 * std::max<uint64_t>(1, P.ibar_cells));
}

int ensure_full(whale_batch* b) {
  if (b->full_ok) return WHALE_OK;
  const PlanHost& P = b->plan;
  HIPCHK(b->ell.alloc(16 + 12 * std::max<uint64_t>(1, P.ell_cells)));
  HIPCHK(b->Eit.alloc(4 * std::max<uint64_t>(1, P.it_seg.size())));
  HIPCHK(b->ibar.alloc(16 + 12 * std::max<uint64_t>(1, P.ibar_cells)));
  b->full_ok = true;
  return WHALE_OK;
}

// a slot of a fused launch over `fams`: the largest family's rows, ī and exponents
void fused_slot(const whale_batch* b, int mode, const uint32_t* fams, size_t nf, FusedSlots* out) {
  const PlanHost& P = b->plan;
  const uint64_t s = mode == WHALE_FP32_SCALED ? 4 : 8;
  uint64_t cells = 1, ibar = 1, items = 1;
  for (size_t j = 0; j < nf; ++j) {
    const uint32_t f = fams[j];
    const FamDev& d = P.fam[f];
    const bool last = f + 1 == b->n_fam;
    cells = std::max(cells, (last ? P.ell_cells : P.fam[f + 1].ell0) - d.ell0);
    ibar = std::max(ibar, (last ? P.ibar_cells : P.fam[f + 1].ibar0) - d.ibar0);
    items = std::max<uint64_t>(items, d.n_items);
  }
  auto al = [](uint64_t x) { return (x + 255) & ~(uint64_t)255; };
  FusedSlots S;
  S.ibar_off = al(cells * s);
  S.eit_off = S.ibar_off + al(ibar * s);
  S.slot_bytes = S.eit_off + al(items * 4);
  *out = S;
}

// Shapes and slots of every fused launch of `mode` (classes, families in
// global memory, routed families, the FP64 pass over flagged ones), their
// grids shrunk so that all slots fit the budget (at least one workgroup per
// launch), and the slot buffer.
int plan_fused(whale_batch* b, int mode) {
  const whale_model* m = b->model;
  const uint32_t* ord = b->order_host.data();
  const int smode = mode == WHALE_FP32_SCALED ? WHALE_FP64_SCALED : mode;  // routed and flagged families
  struct Item { LaunchCfg* c; FusedSlots* s; };
  std::vector<Item> items;
  for (int k = 0; k < whale_batch::kClasses; ++k) {
    const uint32_t lo = b->cls_lo[k], hi = b->cls_hi[k];
    if (hi == lo) continue;
    if (!plan_families(b, false, mode, ord + lo, hi - lo, hi - lo, true, &b->fcfg[mode][k], false, true))
      return fail(WHALE_EINVAL, "no fused launch shape");
    fused_slot(b, mode, ord + lo, hi - lo, &b->fslot[mode][k]);
    items.push_back({&b->fcfg[mode][k], &b->fslot[mode][k]});
  }
  if (b->hbm_hi > b->hbm_lo) {
    const uint32_t nh = b->hbm_hi - b->hbm_lo;
    if (!plan_families(b, false, mode, ord + b->hbm_lo, nh, nh, false, &b->fcfg_hbm[mode], true, true))
      return fail(WHALE_EINVAL, "no fused launch shape");
    fused_slot(b, mode, ord + b->hbm_lo, nh, &b->fslot_hbm[mode]);
    items.push_back({&b->fcfg_hbm[mode], &b->fslot_hbm[mode]});
  }
  if (b->route_lo < b->n_fam) {
    const uint32_t nr = b->n_fam - b->route_lo;
    if (!plan_families(b, false, smode, ord + b->route_lo, nr, nr, true, &b->fcfg_route[mode], false, true))
      return fail(WHALE_EINVAL, "no fused launch shape");
    fused_slot(b, smode, ord + b->route_lo, nr, &b->fslot_route[mode]);
    items.push_back({&b->fcfg_route[mode], &b->fslot_route[mode]});
  }
  if (mode == WHALE_FP32_SCALED) {
    if (!plan_families(b, false, WHALE_FP64_SCALED, ord, b->n_fam, (uint64_t)m->ctx->n_cu, false, &b->fcfg_fb, false, true))
      return fail(WHALE_EINVAL, "no fused launch shape");
    fused_slot(b, WHALE_FP64_SCALED, ord, b->n_fam, &b->fslot_fb[mode]);
    items.push_back({&b->fcfg_fb, &b->fslot_fb[mode]});
  }
  auto total = [&]() {
    uint64_t t = 0;
    for (auto& it : items) t += (uint64_t)it.c->grid * it.c->fpw * it.s->slot_bytes;
    return t;
  };
  if (b->ell_budget && total() > b->ell_budget) {
    const double f = (double)b->ell_budget / (double)total();
    for (auto& it : items) it.c->grid = std::max(1, (int)((double)it.c->grid * f));
  }
  uint64_t off = 0;
  for (auto& it : items) off += (uint64_t)it.c->grid * it.c->fpw * it.s->slot_bytes;
  const void* before = b->fslots.p;
  HIPCHK(b->fslots.alloc(std::max<uint64_t>(off, 256)));
  if (b->fslots.p != before)
    for (bool& x : b->fused_ok) x = false;  // every mode's slots start at the buffer; one mode runs at a time
  off = 0;
  for (auto& it : items) {
    it.s->base = b->fslots.as<unsigned char>() + off;
    off += (uint64_t)it.c->grid * it.c->fpw * it.s->slot_bytes;
  }
  b->fused_bytes[mode] = off;
  b->fused_ok[mode] = true;
  bool moved = false;
  const int rc = ensure_gws(b, &moved);
  if (rc != WHALE_OK) return rc;
  drop_graphs(b);  // captured evaluations hold the previous slots
  return WHALE_OK;
}

bool use_fused(const whale_batch* b, int32_t launch, bool keep) {
  return b->ell_budget && launch == WHALE_LAUNCH_BATCHED && !keep && full_bytes(b) > b->ell_budget;
}

// All device work of one evaluation on the context's stream (capturable: no
// memset nodes, no host synchronisation).  Timing events only when `timed`.
// `ws`, when given, replaces the batch's workspace (and `ws_out` the model's
// result buffer); the results then stay on the device.
int enqueue(whale_batch* b, int mode, int32_t launch, bool grad, bool store_all, bool timed,
            const WorkRaw* ws = nullptr, double* ws_out = nullptr, bool fused = false) {
  whale_model* m = b->model;
  whale_ctx* c = m->ctx;
  hipStream_t st = c->stream;
  const BatchDev B = b->dev();
  const ModelDev M = m->dev();
  WorkRaw W = ws ? *ws : b->work();
  W.acc_fam = b->det && grad ? b->acc_fam.as<double>() : nullptr;
  W.seed = b->seeded && grad ? b->seed.as<double>() : nullptr;
  const AccLayout AL(m->h.n, m->h.n_wgd);
  if (timed) HIPCHK(hipEventRecord(c->ev[1], st));
  const uint32_t nf = b->n_fam;
  const bool fp32 = mode == WHALE_FP32_SCALED;
  HIPCHK(launch_reset(st, W.ticket, kTickets, W.acc, grad ? AL.n : 0, W.flag, fp32 ? (int)nf : 0, W.fb));
  // families the FP32 pass could not represent, recomputed in FP64 with per-clade exponents
  BatchDev Bfb = B;
  Bfb.order = W.fb + 1;
  WorkRaw Wfb = b->fallback_of(W);
  // The size classes run on three streams at once (the context's stream and
  // two side streams), each taking classes largest first: a class's launch
  // holds a compute unit's LDS until its slowest family ends, and the classes
  // beside it fill what the others leave free.
  auto batched = [&](int dir) -> int {
    constexpr int kLanes = 3;
    hipStream_t lanes[kLanes] = {st, c->side, c->side3};
    const std::vector<whale_batch::Group>& groups = b->groups[mode];
    bool used[kLanes] = {};
    for (const auto& g : groups) used[g.lane] = true;
    HIPCHK(hipEventRecord(c->fork[3 * dir], st));
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) HIPCHK(hipStreamWaitEvent(lanes[l], c->fork[3 * dir], 0));
    if (b->hbm_hi > b->hbm_lo) {  // families with their stage buffers in global memory
      WorkRaw Wh = W;
      Wh.ticket = W.ticket + kTicketHbm + dir;
      const LaunchCfg& C = b->cfg_hbm[mode][dir];
      if (dir == 0) HIPCHK(launch_forward(mode, store_all, C, st, B, M, Wh, -1, b->hbm_lo, b->hbm_hi));
      else HIPCHK(launch_backward(mode, C, st, B, M, Wh, -1, b->hbm_lo, b->hbm_hi));
    }
    for (const auto& g : groups) {
      WorkRaw Wk = W;
      Wk.ticket = W.ticket + whale_batch::kClasses * dir + g.cls;
      if (dir == 0) HIPCHK(launch_forward(mode, store_all, g.cfg[0], lanes[g.lane], B, M, Wk, -1, g.lo, g.hi));
      else HIPCHK(launch_backward(mode, g.cfg[1], lanes[g.lane], B, M, Wk, -1, g.lo, g.hi));
    }
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) {
        HIPCHK(hipEventRecord(c->fork[3 * dir + l], lanes[l]));
        HIPCHK(hipStreamWaitEvent(st, c->fork[3 * dir + l], 0));
      }
    return WHALE_OK;
  };
  // logL and gradient: each stream runs its classes' forwards, then their
  // reverse sweeps, with no join between (a family's reverse sweep needs only
  // its own forward), so the reverse sweeps of one stream overlap the last
  // forwards of the others instead of waiting for the slowest forward of the
  // batch.
  auto interleaved = [&]() -> int {
    constexpr int kLanes = 3;
    hipStream_t lanes[kLanes] = {st, c->side, c->side3};
    const std::vector<whale_batch::Group>& groups = b->groups[mode];
    bool used[kLanes] = {};
    for (const auto& g : groups) used[g.lane] = true;
    HIPCHK(hipEventRecord(c->fork[0], st));
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) HIPCHK(hipStreamWaitEvent(lanes[l], c->fork[0], 0));
    const bool hbm = b->hbm_hi > b->hbm_lo;
    WorkRaw Wh = W;
    if (hbm) {
      Wh.ticket = W.ticket + kTicketHbm;
      HIPCHK(launch_forward(mode, store_all, b->cfg_hbm[mode][0], st, B, M, Wh, -1, b->hbm_lo, b->hbm_hi));
    }
    for (const auto& g : groups) {
      WorkRaw Wk = W;
      Wk.ticket = W.ticket + g.cls;
      HIPCHK(launch_forward(mode, store_all, g.cfg[0], lanes[g.lane], B, M, Wk, -1, g.lo, g.hi));
    }
    if (hbm) {
      Wh.ticket = W.ticket + kTicketHbm + 1;
      HIPCHK(launch_backward(mode, b->cfg_hbm[mode][1], st, B, M, Wh, -1, b->hbm_lo, b->hbm_hi));
    }
    for (const auto& g : groups) {
      WorkRaw Wk = W;
      Wk.ticket = W.ticket + whale_batch::kClasses + g.cls;
      HIPCHK(launch_backward(mode, g.cfg[1], lanes[g.lane], B, M, Wk, -1, g.lo, g.hi));
    }
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) {
        HIPCHK(hipEventRecord(c->fork[3 + l], lanes[l]));
        HIPCHK(hipStreamWaitEvent(st, c->fork[3 + l], 0));
      }
    return WHALE_OK;
  };
  auto single = [&](int dir, uint32_t f, const WorkRaw& Wf) -> int {
    LaunchCfg C;
    if (!plan_families(b, dir == 0, mode, &f, 1, 1, false, &C))
      return fail(WHALE_EINVAL, "a family's largest stage does not fit the LDS of one compute unit");
    C.grid = 1;
    if (dir == 0) HIPCHK(launch_forward(mode, store_all, C, st, B, M, Wf, (int32_t)f, 0, 0));
    else HIPCHK(launch_backward(mode, C, st, B, M, Wf, (int32_t)f, 0, 0));
    return WHALE_OK;
  };
  int rc;
  if (fused) {
    // every family's forward and reverse sweep by one wave, its rows in the
    // wave's slot (k_fused); the same streams and classes as the stored form
    const int rmode = fp32 ? WHALE_FP64_SCALED : mode;
    const bool routed = b->route_lo < nf;
    if (routed) {
      HIPCHK(hipEventRecord(c->fork[6], st));
      HIPCHK(hipStreamWaitEvent(c->side2, c->fork[6], 0));
      WorkRaw Wr = W;
      if (Wr.gws) Wr.gws += b->gws_main;
      Wr.ticket = W.ticket + 2 * whale_batch::kClasses + 2;
      HIPCHK(launch_fused(rmode, b->fcfg_route[mode], c->side2, B, M, Wr, b->route_lo, nf, nullptr, grad ? 1 : 0,
                          b->fslot_route[mode]));
      HIPCHK(hipEventRecord(c->fork[7], c->side2));
    }
    constexpr int kLanes = 3;
    hipStream_t lanes[kLanes] = {st, c->side, c->side3};
    const int* kOrder = kLayoutOrder[b->tune.layout];
    const int* kLane = kLayoutLane[b->tune.layout];
    bool used[kLanes] = {};
    for (int k = 0; k < whale_batch::kClasses; ++k)
      if (b->cls_hi[k] > b->cls_lo[k]) used[kLane[k]] = true;
    HIPCHK(hipEventRecord(c->fork[0], st));
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) HIPCHK(hipStreamWaitEvent(lanes[l], c->fork[0], 0));
    if (b->hbm_hi > b->hbm_lo) {
      WorkRaw Wh = W;
      Wh.ticket = W.ticket + kTicketHbm;
      HIPCHK(launch_fused(mode, b->fcfg_hbm[mode], st, B, M, Wh, b->hbm_lo, b->hbm_hi, nullptr, grad ? 1 : 0,
                          b->fslot_hbm[mode]));
    }
    for (int j = 0; j < whale_batch::kClasses; ++j) {
      const int k = kOrder[j];
      if (b->cls_hi[k] == b->cls_lo[k]) continue;
      WorkRaw Wk = W;
      Wk.ticket = W.ticket + k;
      HIPCHK(launch_fused(mode, b->fcfg[mode][k], lanes[kLane[k]], B, M, Wk, b->cls_lo[k], b->cls_hi[k], nullptr,
                          grad ? 1 : 0, b->fslot[mode][k]));
    }
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) {
        HIPCHK(hipEventRecord(c->fork[3 + l], lanes[l]));
        HIPCHK(hipStreamWaitEvent(st, c->fork[3 + l], 0));
      }
    if (fp32) {
      Wfb.ticket = W.ticket + 2 * whale_batch::kClasses;
      HIPCHK(launch_fused(WHALE_FP64_SCALED, b->fcfg_fb, st, Bfb, M, Wfb, 0, 0, W.fb, grad ? 1 : 0,
                          b->fslot_fb[mode]));
    }
    if (timed) HIPCHK(hipEventRecord(c->ev[2], st));
    if (routed) HIPCHK(hipStreamWaitEvent(st, c->fork[7], 0));
    if (timed) HIPCHK(hipEventRecord(c->ev[3], st));
  } else {
  // families routed to FP64: their whole evaluation on the second side stream
  const bool routed = launch == WHALE_LAUNCH_BATCHED && b->route_lo < nf;
  if (routed) {
    HIPCHK(hipEventRecord(c->fork[6], st));
    HIPCHK(hipStreamWaitEvent(c->side2, c->fork[6], 0));
    const int rmode = fp32 ? WHALE_FP64_SCALED : mode;
    WorkRaw Wr = fp32 ? b->fallback_of(W) : W;
    if (Wr.gws) Wr.gws += b->gws_main;  // its own stage-buffer region: it runs beside the other launches
    Wr.ticket = W.ticket + 2 * whale_batch::kClasses + 2;
    HIPCHK(launch_forward(rmode, store_all, b->cfg_route[mode][0], c->side2, B, M, Wr, -1, b->route_lo, nf));
    if (grad) {
      Wr.ticket = W.ticket + 2 * whale_batch::kClasses + 3;
      HIPCHK(launch_backward(rmode, b->cfg_route[mode][1], c->side2, B, M, Wr, -1, b->route_lo, nf));
    }
    HIPCHK(hipEventRecord(c->fork[7], c->side2));
  }
  // per-kernel timing keeps the forward and reverse phases apart
  const bool inter = launch == WHALE_LAUNCH_BATCHED && grad && !timed;
  if (inter) {
    if ((rc = interleaved()) != WHALE_OK) return rc;
  } else if (launch == WHALE_LAUNCH_BATCHED) {
    if ((rc = batched(0)) != WHALE_OK) return rc;
  } else {
    for (uint32_t k = 0; k < nf; ++k)
      if ((rc = single(0, b->order_host[k], W)) != WHALE_OK) return rc;
  }
  if (fp32) {
    Wfb.ticket = W.ticket + 2 * whale_batch::kClasses;
    HIPCHK(launch_forward(WHALE_FP64_SCALED, store_all, b->cfg_fb[0], st, Bfb, M, Wfb, -1, 0, 0, W.fb));
  }
  if (timed) HIPCHK(hipEventRecord(c->ev[2], st));
  if (grad) {
    if (inter) {
      // the reverse sweeps ran above
    } else if (launch == WHALE_LAUNCH_BATCHED) {
      if ((rc = batched(1)) != WHALE_OK) return rc;
    } else {
      for (uint32_t k = 0; k < nf; ++k)
        if ((rc = single(1, b->order_host[k], W)) != WHALE_OK) return rc;
    }
    if (fp32) {
      WorkRaw Wfb2 = Wfb;
      Wfb2.ticket = W.ticket + 2 * whale_batch::kClasses + 1;
      HIPCHK(launch_backward(WHALE_FP64_SCALED, b->cfg_fb[1], st, Bfb, M, Wfb2, -1, 0, 0, W.fb));
    }
  }
  if (routed) HIPCHK(hipStreamWaitEvent(st, c->fork[7], 0));
  if (timed) HIPCHK(hipEventRecord(c->ev[3], st));
  }
  if (W.acc_fam) HIPCHK(launch_det_sum(st, W.acc_fam, nf, AL.n, W.acc));
  // the results go to the caller's device buffer, or from the kernel straight
  // to the batch's pinned ones (three copies took 14 us of a small evaluation)
  const int n = m->h.n, nw = m->h.n_wgd;
  HIPCHK(launch_tail(st, M, W.fam_ll, nf, W.acc, m->ebar.as<double>(), m->dlv.as<int32_t>(), m->dnd.as<int32_t>(),
                     m->n_dlevels, m->h.cond, grad ? 1 : 0, ws ? ws_out : b->pin_out, W.seed ? W.seed + nf : nullptr,
                     ws ? nullptr : b->pin_fam, fp32 ? W.fb : nullptr,
                     ws ? nullptr : reinterpret_cast<uint32_t*>(&b->pin_out[2 + 2 * n + nw])));
  if (timed) HIPCHK(hipEventRecord(c->ev[4], st));
  return WHALE_OK;
}

int run(whale_batch* b, int32_t mode_in, int32_t launch, bool grad, double* out_family, double* out_total,
        double* d_lambda, double* d_mu, double* d_q, double* d_eta) {
  if (!b || !out_total) return fail(WHALE_EINVAL, "NULL argument");
  whale_model* m = b->model;
  whale_ctx* c = m->ctx;
  if (!m->has_params) return fail(WHALE_ESTATE, "parameters not set (whale_model_set_params)");
  const int mode = mode_in & 0xff;
  const bool keep = (mode_in & 0x100) != 0;
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  if (launch != WHALE_LAUNCH_BATCHED && launch != WHALE_LAUNCH_PER_FAMILY) return fail(WHALE_EINVAL, "unknown launch");
  const bool store_all = grad || keep;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = c->stream;
  if (!b->flagged_once.empty()) {
    for (uint32_t f : b->flagged_once) b->routed[f] = 1;
    b->flagged_once.clear();
    int rc = assign_classes(b);
    if (rc != WHALE_OK) return rc;
    if ((rc = ensure_gws(b, nullptr)) != WHALE_OK) return rc;
    HIPCHK(hipMemcpy(b->order.p, b->order_host.data(), sizeof(uint32_t) * b->n_fam, hipMemcpyHostToDevice));
    drop_graphs(b);
  }
  const bool fused = use_fused(b, launch, keep);
  if (b->det && grad) {
    const AccLayout AL(m->h.n, m->h.n_wgd);
    HIPCHK(b->acc_fam.alloc(sizeof(double) * (size_t)b->n_fam * AL.n));
  }
  if (fused) {
    if (!b->fused_ok[mode]) {
      const int rc = plan_fused(b, mode);
      if (rc != WHALE_OK) return rc;
    }
  } else {
    const int rc = ensure_full(b);
    if (rc != WHALE_OK) return rc;
  }
  if (launch == WHALE_LAUNCH_BATCHED && !c->timing) {
    // replay the captured evaluation (captured on first use)
    hipGraphExec_t& ge = b->graph[mode][grad ? 1 : 0][keep ? 1 : 0][fused ? 1 : 0];
    if (!ge) {
      HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
      int rc = enqueue(b, mode, launch, grad, store_all, false, nullptr, nullptr, fused);
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(st, &g);
      if (rc != WHALE_OK) { if (g) (void)hipGraphDestroy(g); return rc; }
      HIPCHK(e);
      e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      HIPCHK(e);
    }
    HIPCHK(hipGraphLaunch(ge, st));
  } else {
    int rc = enqueue(b, mode, launch, grad, store_all, c->timing, nullptr, nullptr, fused);
    if (rc != WHALE_OK) return rc;
  }
  HIPCHK(hipStreamSynchronize(st));
  if (c->timing) {
    float a, bb, cc, dd;
    HIPCHK(hipEventElapsedTime(&a, c->ev[1], c->ev[2]));
    HIPCHK(hipEventElapsedTime(&bb, c->ev[2], c->ev[3]));
    HIPCHK(hipEventElapsedTime(&cc, c->ev[3], c->ev[4]));
    HIPCHK(hipEventElapsedTime(&dd, c->ev[1], c->ev[4]));
    c->last_ms[1] = a;
    c->last_ms[2] = bb;
    c->last_ms[3] = cc;
    c->last_ms[4] = dd;
  }
  const int n = m->h.n, nw = m->h.n_wgd;
  const double* o = b->pin_out;
  *out_total = o[0];
  if (out_family) std::copy(b->pin_fam, b->pin_fam + b->n_fam, out_family);
  if (grad) {
    if (d_lambda) std::copy(o + 1, o + 1 + n, d_lambda);
    if (d_mu) std::copy(o + 1 + n, o + 1 + 2 * n, d_mu);
    if (d_q) std::copy(o + 1 + 2 * n, o + 1 + 2 * n + nw, d_q);
    if (d_eta) *d_eta = o[1 + 2 * n + nw];
  }
  b->last_mode = mode;
  b->last_store_all = store_all && !fused;
  b->last_launch = launch;
  b->last_fallback = 0;
  if (mode == WHALE_FP32_SCALED) {
    const uint32_t fresh = *reinterpret_cast<const uint32_t*>(&o[2 + 2 * n + nw]);
    b->last_fallback = fresh + (launch == WHALE_LAUNCH_BATCHED ? b->n_fam - b->route_lo : 0);
    if (fresh && launch == WHALE_LAUNCH_BATCHED) {
      // these families will be evaluated in FP64 from the start by later FP32 calls
      std::vector<uint32_t> list(fresh);
      HIPCHK(hipMemcpy(list.data(), b->fb.as<uint32_t>() + 1, sizeof(uint32_t) * fresh, hipMemcpyDeviceToHost));
      for (uint32_t f : list) b->flagged_once.push_back(f);
    }
  }
  return WHALE_OK;
}

}  // namespace

namespace {

// Re-plans the batch for its current tuning and drops captured evaluations.
int replan(whale_batch* b) {
  int rc = assign_classes(b);
  if (rc != WHALE_OK) return rc;
  if ((rc = ensure_gws(b, nullptr)) != WHALE_OK) return rc;
  HIPCHK(hipMemcpy(b->order.p, b->order_host.data(), sizeof(uint32_t) * b->n_fam, hipMemcpyHostToDevice));
  drop_graphs(b);
  return WHALE_OK;
}

// Median wall time (ms) of `reps` captured evaluations after one untimed one
// (which captures the graph), as a caller sees them: launch to results on the host.
int time_evals(whale_batch* b, int mode, bool grad, int reps, double* ms) {
  const whale_model* m = b->model;
  std::vector<double> fam(b->n_fam), dl(m->h.n), dm(m->h.n), dq(std::max(1, m->h.n_wgd));
  double tot = 0, de = 0;
  std::vector<double> t;
  for (int i = 0; i <= reps; ++i) {
    const auto t0 = std::chrono::steady_clock::now();
    const int rc = run(b, mode, WHALE_LAUNCH_BATCHED, grad, fam.data(), &tot, dl.data(), dm.data(), dq.data(), &de);
    if (rc != WHALE_OK) return rc;
    const auto t1 = std::chrono::steady_clock::now();
    if (i > 0) t.push_back(std::chrono::duration<double, std::milli>(t1 - t0).count());
  }
  std::sort(t.begin(), t.end());
  *ms = t[t.size() / 2];
  return WHALE_OK;
}

// The workload a tuning applies to: device, arithmetic, gradient or not, and
// every family's shape as the planner sees it.
void tune_key(const whale_batch* b, int mode, bool grad, std::string* key) {
  const whale_model* m = b->model;
  uint64_t h = 1469598103934665603ull;
  auto mix = [&](uint64_t v) {
    for (int i = 0; i < 8; ++i) {
      h ^= (v >> (8 * i)) & 0xff;
      h *= 1099511628211ull;
    }
  };
  mix(b->n_fam);
  mix((uint64_t)m->h.tab_rows);
  mix((uint64_t)m->h.n);
  for (const FamDev& d : b->plan.fam) {
    mix(d.n_clades);
    mix(d.max_items);
    mix(d.max_slots);
    mix(d.n_recs);
    mix(d.n_stages);
  }
  hipDeviceProp_t prop;
  std::string arch = "gpu";
  if (hipGetDeviceProperties(&prop, m->ctx->device) == hipSuccess) arch = prop.gcnArchName;
  for (char& ch : arch)
    if (ch == ' ' || ch == ':') ch = '_';
  char buf[256];
  snprintf(buf, sizeof buf, "%s/cu%d/lds%zu/mode%d/grad%d/%016llx", arch.c_str(), m->ctx->n_cu, m->ctx->lds_wg, mode,
           grad ? 1 : 0, (unsigned long long)h);
  *key = buf;
}

bool valid_tuning(const Tuning& t) {
  if (t.layout < 0 || t.layout >= kLayouts || t.waves_cap < 1 || t.waves_cap > 32) return false;
  for (int i = 0; i < 5; ++i) {
    if (t.bounds[i] < 1024) return false;
    if (i > 0 && t.bounds[i] <= t.bounds[i - 1]) return false;
  }
  return true;
}

bool cache_lookup(const char* path, const std::string& key, Tuning* t) {
  if (!path || !*path) return false;
  std::ifstream f(path);
  std::string line;
  bool found = false;
  while (std::getline(f, line)) {  // the last line for a key wins
    std::istringstream is(line);
    std::string k;
    Tuning u;
    double ms = 0;
    if (!(is >> k) || k != key) continue;
    for (auto& x : u.bounds) is >> x;
    is >> u.layout >> u.waves_cap >> ms;
    if (is && valid_tuning(u)) {
      *t = u;
      found = true;
    }
  }
  return found;
}

void cache_store(const char* path, const std::string& key, const Tuning& t, double ms) {
  if (!path || !*path) return;
  std::ofstream f(path, std::ios::app);
  if (!f) return;  // a cache that cannot be written only costs a search next time
  f << key;
  for (auto x : t.bounds) f << ' ' << x;
  f << ' ' << t.layout << ' ' << t.waves_cap << ' ' << ms << '\n';
}

}  // namespace

int whale_batch_autotune(whale_batch* b, int32_t mode, int32_t gradient, int32_t reps, const char* cache_path,
                         int64_t* out8, double* out_ms2) {
  if (!b) return fail(WHALE_EINVAL, "NULL argument");
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  if (!b->model->has_params) return fail(WHALE_ESTATE, "parameters not set (whale_model_set_params)");
  if (b->model->ctx->timing) return fail(WHALE_ESTATE, "per-kernel timing is on; the search times graph replays");
  reps = std::max(1, std::min(reps, 50));
  const bool grad = gradient != 0;
  HIPCHK(hipSetDevice(b->device));
  std::string key;
  tune_key(b, mode, grad, &key);
  const Tuning start = b->tune;
  int rc;
  double t_start = 0, t_best = 0;
  int evals = 0;
  Tuning best;
  if (cache_lookup(cache_path, key, &best)) {
    b->tune = best;
    if ((rc = replan(b)) != WHALE_OK) return rc;
    if ((rc = time_evals(b, mode, grad, reps, &t_best)) != WHALE_OK) return rc;
    t_start = t_best;
  } else {
    // coordinate search from the current shape, accepting a change only when
    // it is at least 1 % faster (run-to-run noise is below that)
    auto timed = [&](const Tuning& t, double* ms) -> int {
      b->tune = t;
      int r = replan(b);
      if (r == WHALE_OK) r = time_evals(b, mode, grad, reps, ms);
      ++evals;
      return r;
    };
    best = start;
    if ((rc = timed(best, &t_start)) != WHALE_OK) return rc;
    t_best = t_start;
    auto consider = [&](const Tuning& t) -> int {
      if (!valid_tuning(t)) return WHALE_OK;
      double ms = 0;
      const int r = timed(t, &ms);
      if (r != WHALE_OK) return r;
      if (ms < 0.99 * t_best) {
        best = t;
        t_best = ms;
      }
      return WHALE_OK;
    };
    // the layouts at the starting bounds, then a descent from each of the two
    // fastest: their basins differ, and at the starting bounds the two are
    // often within the timing noise of each other
    std::vector<std::pair<double, int>> lay{{t_start, start.layout}};
    for (int l = 0; l < kLayouts; ++l) {
      if (l == start.layout) continue;
      Tuning t = start;
      t.layout = l;
      if (!valid_tuning(t)) continue;
      double ms = 0;
      if ((rc = timed(t, &ms)) != WHALE_OK) return rc;
      lay.push_back({ms, l});
    }
    std::sort(lay.begin(), lay.end());
    Tuning overall = start;
    double overall_ms = t_start;
    for (size_t d = 0; d < std::min<size_t>(2, lay.size()); ++d) {
      best = start;
      best.layout = lay[d].second;
      t_best = lay[d].first;
      // two rounds: the best layout depends on the class bounds and the
      // other way round, so the layouts are tried again once the bounds
      // have moved
      for (int round = 0; round < 2; ++round) {
        const Tuning before = best;
        if (round > 0)
          for (int l = 0; l < kLayouts; ++l) {
            if (l == best.layout) continue;
            Tuning t = best;
            t.layout = l;
            if ((rc = consider(t)) != WHALE_OK) return rc;
          }
        for (int cap : {4, 6, 8, 12, 16}) {
          if (cap == best.waves_cap) continue;
          Tuning t = best;
          t.waves_cap = cap;
          if ((rc = consider(t)) != WHALE_OK) return rc;
        }
        for (int pass = 0; pass < 2; ++pass)
          for (int i = 0; i < 5; ++i)
            for (double f : {0.75, 0.9, 1.12, 1.33}) {
              Tuning t = best;
              t.bounds[i] = (uint32_t)((double)best.bounds[i] * f) & ~255u;
              if ((rc = consider(t)) != WHALE_OK) return rc;
            }
        if (round == 0 && std::memcmp(&before, &best, sizeof(Tuning)) == 0) break;  // nothing moved
      }
      if (t_best < overall_ms) {
        overall = best;
        overall_ms = t_best;
      }
    }
    best = overall;
    t_best = overall_ms;
    b->tune = best;
    if ((rc = replan(b)) != WHALE_OK) return rc;
    cache_store(cache_path, key, best, t_best);
  }
  if (out8) {
    for (int i = 0; i < 5; ++i) out8[i] = best.bounds[i];
    out8[5] = best.layout;
    out8[6] = best.waves_cap;
    out8[7] = evals;
  }
  if (out_ms2) {
    out_ms2[0] = t_start;
    out_ms2[1] = t_best;
  }
  return WHALE_OK;
}

int whale_mixture_eval(whale_batch* b, whale_model* const* comps, int32_t K, const double* prior, int32_t mode,
                       int32_t gradient, double* out_total, double* out_fam, double* out_resp, double* out_grad,
                       double* out_dprior) {
  if (!b || !comps || !prior || !out_total) return fail(WHALE_EINVAL, "NULL argument");
  if (K < 1 || K > kMaxMix) return fail(WHALE_EINVAL, "1 to 8 mixture components");
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  if (gradient && !out_grad) return fail(WHALE_EINVAL, "out_grad is NULL");
  if (b->det || use_fused(b, WHALE_LAUNCH_BATCHED, false))
    return fail(WHALE_ESTATE, "mixtures need the stored form without deterministic gradients");
  if (b->hbm_hi > b->hbm_lo) return fail(WHALE_ESTATE, "mixtures need every family's stages in LDS");
  whale_model* m0 = b->model;
  const ModelHost& H = m0->h;
  for (int j = 0; j < K; ++j) {
    const whale_model* m = comps[j];
    if (!m) return fail(WHALE_EINVAL, "NULL component");
    if (!(prior[j] > 0) || !std::isfinite(prior[j])) return fail(WHALE_EINVAL, "prior weights must be positive");
    if (!m->has_params) return fail(WHALE_ESTATE, "component parameters not set (whale_model_set_params)");
    bool same = m->ctx == m0->ctx && m->h.n == H.n && m->h.n_wgd == H.n_wgd && m->h.root == H.root &&
                m->h.tab_rows == H.tab_rows && m->h.cond == H.cond;
    for (int e = 0; same && e < H.n; ++e) {
      const NodeDev &x = m->h.nodes[e], &y = H.nodes[e];
      same = x.kind == y.kind && x.child0 == y.child0 && x.child1 == y.child1 && x.tab == y.tab && x.R == y.R &&
             x.wgd == y.wgd && x.parent == y.parent && x.leafP == y.leafP && x.delta == y.delta;
    }
    if (!same) return fail(WHALE_EINVAL, "mixture components must share the batch's species-tree structure");
  }
  whale_ctx* c = m0->ctx;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = c->stream;
  {
    const int rc = ensure_full(b);
    if (rc != WHALE_OK) return rc;
  }
  const uint32_t nf = b->n_fam;
  const bool fp32 = mode == WHALE_FP32_SCALED;
  const bool grad = gradient != 0;
  const AccLayout AL(H.n, H.n_wgd);
  const int ng = 2 + 2 * H.n + H.n_wgd;  // a tail's output
  // workspaces, sized as the batch's own
  while ((int)b->mixw.size() < K) b->mixw.emplace_back(new whale_batch::MixWork());
  std::vector<WorkRaw> Wj(K);
  for (int j = 0; j < K; ++j) {
    whale_batch::MixWork& x = *b->mixw[j];
    HIPCHK(x.ell.alloc(b->ell.n));
    HIPCHK(x.Eit.alloc(b->Eit.n));
    HIPCHK(x.E.alloc(b->E.n));
    HIPCHK(x.ibar.alloc(b->ibar.n));
    HIPCHK(x.fam_ll.alloc(b->fam_ll.n));
    HIPCHK(x.acc.alloc(b->acc.n));
    HIPCHK(x.ticket.alloc(sizeof(uint32_t) * kTickets));
    HIPCHK(x.flag.alloc(b->flag.n));
    HIPCHK(x.fb.alloc(b->fb.n));
    HIPCHK(x.seed.alloc(sizeof(double) * (nf + 1)));
    HIPCHK(x.out.alloc(sizeof(double) * ng));
    WorkRaw W;
    W.ell = x.ell.p;
    W.Eit = x.Eit.as<int32_t>();
    W.E = x.E.as<int32_t>();
    W.ibar = x.ibar.p;
    W.fam_ll = x.fam_ll.as<double>();
    W.acc = x.acc.as<double>();
    W.ticket = x.ticket.as<uint32_t>();
    W.flag = x.flag.as<uint32_t>();
    W.fb = x.fb.as<uint32_t>();
    W.gws = nullptr;
    W.seed = x.seed.as<double>();  // written by the mixture kernel, read by the reverse sweep
    Wj[j] = W;
  }
  // the component tables of every launch: [launch][component]
  enum { kF = 0, kB = whale_batch::kClasses, kFbF = 2 * whale_batch::kClasses, kFbB, kRtF, kRtB, kSlots };
  std::vector<MixComp> sel((size_t)kSlots * K);
  for (int j = 0; j < K; ++j) {
    const ModelDev M = comps[j]->dev();
    const WorkRaw Wfb = b->fallback_of(Wj[j]);
    for (int k = 0; k < whale_batch::kClasses; ++k) {
      MixComp& f = sel[(size_t)(kF + k) * K + j];
      f.M = M;
      f.W = Wj[j];
      f.W.ticket = Wj[j].ticket + k;
      MixComp& r = sel[(size_t)(kB + k) * K + j];
      r = f;
      r.W.ticket = Wj[j].ticket + whale_batch::kClasses + k;
    }
    MixComp& a = sel[(size_t)kFbF * K + j];
    a.M = M;
    a.W = Wfb;
    a.W.ticket = Wj[j].ticket + 2 * whale_batch::kClasses;
    a.order = Wj[j].fb + 1;
    a.count = Wj[j].fb;
    MixComp& d = sel[(size_t)kFbB * K + j];
    d = a;
    d.W.ticket = Wj[j].ticket + 2 * whale_batch::kClasses + 1;
    MixComp& e = sel[(size_t)kRtF * K + j];
    e.M = M;
    e.W = fp32 ? Wfb : Wj[j];
    e.W.ticket = Wj[j].ticket + 2 * whale_batch::kClasses + 2;
    MixComp& g = sel[(size_t)kRtB * K + j];
    g = e;
    g.W.ticket = Wj[j].ticket + 2 * whale_batch::kClasses + 3;
  }
  HIPCHK(b->mixsel.alloc(sizeof(MixComp) * sel.size()));
  HIPCHK(hipMemcpy(b->mixsel.p, sel.data(), sizeof(MixComp) * sel.size(), hipMemcpyHostToDevice));
  std::vector<double> lp(K);
  for (int j = 0; j < K; ++j) lp[j] = std::log(prior[j]);
  HIPCHK(b->mixprior.alloc(sizeof(double) * K));
  HIPCHK(hipMemcpy(b->mixprior.p, lp.data(), sizeof(double) * K, hipMemcpyHostToDevice));
  HIPCHK(b->mixout.alloc(sizeof(double)));
  HIPCHK(b->mixresp.alloc(sizeof(double) * (size_t)nf * K));
  const MixComp* X = b->mixsel.as<MixComp>();
  auto at = [&](int slot) { return X + (size_t)slot * K; };
  const BatchDev B = b->dev();
  const ModelDev M0 = m0->dev();
  const bool store_all = grad;
  for (int j = 0; j < K; ++j) {
    HIPCHK(launch_reset(st, Wj[j].ticket, kTickets, Wj[j].acc, grad ? AL.n : 0, Wj[j].flag, fp32 ? (int)nf : 0,
                        Wj[j].fb));
  }
  // one direction: every size class as one launch over all components on the
  // three streams, the families routed to FP64 as one launch beside them, and
  // the FP64 pass over the families each component's FP32 pass flagged
  if (b->mix_k[mode] != K) {
    plan_groups(b, mode, K, b->mix_groups[mode]);
    b->mix_k[mode] = K;
  }
  const std::vector<whale_batch::Group>& groups = b->mix_groups[mode];
  auto direction = [&](int dir) -> int {
    constexpr int kLanes = 3;
    hipStream_t lanes[kLanes] = {st, c->side, c->side3};
    bool used[kLanes] = {};
    for (const auto& g : groups) used[g.lane] = true;
    const bool routed = b->route_lo < nf;
    HIPCHK(hipEventRecord(c->fork[3 * dir], st));
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) HIPCHK(hipStreamWaitEvent(lanes[l], c->fork[3 * dir], 0));
    if (routed) HIPCHK(hipStreamWaitEvent(c->side2, c->fork[3 * dir], 0));
    for (const auto& g : groups) {
      if (dir == 0)
        HIPCHK(launch_forward(mode, store_all, g.cfg[0], lanes[g.lane], B, M0, Wj[0], -1, g.lo, g.hi, nullptr,
                              at(kF + g.cls), K));
      else
        HIPCHK(launch_backward(mode, g.cfg[1], lanes[g.lane], B, M0, Wj[0], -1, g.lo, g.hi, nullptr, at(kB + g.cls), K));
    }
    if (routed) {
      const int rmode = fp32 ? WHALE_FP64_SCALED : mode;
      if (dir == 0)
        HIPCHK(launch_forward(rmode, store_all, b->cfg_route[mode][0], c->side2, B, M0, Wj[0], -1, b->route_lo, nf,
                              nullptr, at(kRtF), K));
      else
        HIPCHK(launch_backward(rmode, b->cfg_route[mode][1], c->side2, B, M0, Wj[0], -1, b->route_lo, nf, nullptr,
                               at(kRtB), K));
      HIPCHK(hipEventRecord(c->fork[7], c->side2));
      HIPCHK(hipStreamWaitEvent(st, c->fork[7], 0));
    }
    for (int l = 1; l < kLanes; ++l)
      if (used[l]) {
        HIPCHK(hipEventRecord(c->fork[3 * dir + l], lanes[l]));
        HIPCHK(hipStreamWaitEvent(st, c->fork[3 * dir + l], 0));
      }
    if (fp32) {
      BatchDev Bfb = B;
      if (dir == 0)
        HIPCHK(launch_forward(WHALE_FP64_SCALED, store_all, b->cfg_fb[0], st, Bfb, M0, Wj[0], -1, 0, 0, nullptr,
                              at(kFbF), K));
      else
        HIPCHK(launch_backward(WHALE_FP64_SCALED, b->cfg_fb[1], st, Bfb, M0, Wj[0], -1, 0, 0, nullptr, at(kFbB), K));
    }
    return WHALE_OK;
  };
  int rc = direction(0);
  if (rc != WHALE_OK) return rc;
  // logsumexp over the components, the responsibilities as the reverse sweep's weights
  HIPCHK(launch_mix(st, at(kF), K, b->mixprior.as<double>(), nf, H.cond, b->mixout.as<double>(),
                    b->mixresp.as<double>()));
  if (grad) {
    if ((rc = direction(1)) != WHALE_OK) return rc;
    for (int j = 0; j < K; ++j) {
      const whale_model* m = comps[j];
      HIPCHK(launch_tail(st, m->dev(), Wj[j].fam_ll, nf, Wj[j].acc, m->ebar.as<double>(), m->dlv.as<int32_t>(), m->dnd.as<int32_t>(), m->n_dlevels, H.cond, 1,
                         b->mixw[j]->out.as<double>(), Wj[j].seed + nf));
    }
  }
  HIPCHK(hipStreamSynchronize(st));
  HIPCHK(hipMemcpy(out_total, b->mixout.p, sizeof(double), hipMemcpyDeviceToHost));
  std::vector<double> col(nf + 1);
  for (int j = 0; j < K; ++j) {
    if (out_fam) {
      HIPCHK(hipMemcpy(col.data(), Wj[j].fam_ll, sizeof(double) * nf, hipMemcpyDeviceToHost));
      for (uint32_t i = 0; i < nf; ++i) out_fam[(size_t)i * K + j] = col[i];
    }
    if (grad) {
      std::vector<double> o(ng);
      HIPCHK(hipMemcpy(o.data(), b->mixw[j]->out.p, sizeof(double) * ng, hipMemcpyDeviceToHost));
      std::copy(o.begin() + 1, o.begin() + 1 + (ng - 1), out_grad + (size_t)j * (ng - 1));
    }
    if (out_dprior && grad) {
      double sw = 0;
      HIPCHK(hipMemcpy(&sw, Wj[j].seed + nf, sizeof(double), hipMemcpyDeviceToHost));
      out_dprior[j] = sw / prior[j];
    }
  }
  if (out_resp) HIPCHK(hipMemcpy(out_resp, b->mixresp.p, sizeof(double) * (size_t)nf * K, hipMemcpyDeviceToHost));
  if (out_dprior && !grad) {
    std::vector<double> r((size_t)nf * K);
    HIPCHK(hipMemcpy(r.data(), b->mixresp.p, sizeof(double) * r.size(), hipMemcpyDeviceToHost));
    for (int j = 0; j < K; ++j) {
      double sw = 0;
      for (uint32_t i = 0; i < nf; ++i) sw += r[(size_t)i * K + j];
      out_dprior[j] = sw / prior[j];
    }
  }
  return WHALE_OK;
}

int whale_batch_set_seeds(whale_batch* b, const double* seeds) {
  if (!b) return fail(WHALE_EINVAL, "NULL batch");
  HIPCHK(hipSetDevice(b->model->ctx->device));
  if (!seeds) {
    if (b->seeded) drop_graphs(b);  // captured evaluations hold the seed pointer
    b->seeded = false;
    return WHALE_OK;
  }
  std::vector<double> h(seeds, seeds + b->n_fam);
  double sum = 0;
  for (double x : h) {
    if (!std::isfinite(x) || x < 0) return fail(WHALE_EINVAL, "seeds must be finite and non-negative");
    sum += x;
  }
  h.push_back(sum);
  const void* before = b->seed.p;
  HIPCHK(b->seed.alloc(sizeof(double) * h.size()));
  HIPCHK(hipMemcpy(b->seed.p, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
  if (!b->seeded || b->seed.p != before) drop_graphs(b);
  b->seeded = true;
  return WHALE_OK;
}

int whale_batch_pooled(whale_batch* b, int32_t mode, int32_t* out) {
  if (!b || !out) return fail(WHALE_EINVAL, "NULL argument");
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  *out = 0;
  return WHALE_OK;
}

int whale_batch_set_tuning(whale_batch* b, const int64_t* in7) {
  if (!b || !in7) return fail(WHALE_EINVAL, "NULL argument");
  Tuning t;
  for (int i = 0; i < 5; ++i) t.bounds[i] = (uint32_t)in7[i];
  t.layout = (int)in7[5];
  t.waves_cap = (int)in7[6];
  if (!valid_tuning(t)) return fail(WHALE_EINVAL, "invalid tuning: increasing class bounds >= 1024, layout 0..5, 1..32 waves");
  HIPCHK(hipSetDevice(b->device));
  b->tune = t;
  return replan(b);
}

int whale_batch_get_tuning(const whale_batch* b, int64_t* out7) {
  if (!b || !out7) return fail(WHALE_EINVAL, "NULL argument");
  for (int i = 0; i < 5; ++i) out7[i] = b->tune.bounds[i];
  out7[5] = b->tune.layout;
  out7[6] = b->tune.waves_cap;
  return WHALE_OK;
}

int whale_logpdf(whale_batch* b, int32_t mode, int32_t launch, double* out_family, double* out_total) {
  return run(b, mode, launch, false, out_family, out_total, nullptr, nullptr, nullptr, nullptr);
}

static_assert(kScratchBytes == WHALE_NOALLOC_SCRATCH_BYTES, "fixed workspace size of the C ABI");

int whale_logpdf_noalloc(whale_batch* b, int32_t mode, double* d_family, double* d_total) {
  if (!b || !d_family || !d_total) return fail(WHALE_EINVAL, "whale_logpdf_noalloc: NULL argument");
  if (mode < 0 || mode > 2) return fail(WHALE_EINVAL, "unknown mode");
  whale_model* m = b->model;
  whale_ctx* c = m->ctx;
  if (!m->has_params) return fail(WHALE_ESTATE, "parameters not set (whale_model_set_params)");
  if (!c->scratch) return fail(WHALE_ESTATE, "no fixed workspace on this device");
  // The workspace of a logL evaluation without stored rows, carved from the
  // fixed array: ℓ (FP32 values followed by the FP64 region of families an
  // FP32 pass recomputes, or FP64 values), per-clade exponents, tickets,
  // flags, the list of recomputed families and the stage buffers of
  // global-memory launches.  Per-record coefficients, ī and gradient
  // accumulators are not touched without stored rows or a gradient.
  const PlanHost& P = b->plan;
  auto al = [](uint64_t x) { return (x + 255) & ~(uint64_t)255; };
  const uint64_t cells = P.ell_cells;
  const uint64_t ell_b = mode == WHALE_FP32_SCALED ? whale_batch::fp32_bytes(cells) + 8 * cells : 8 * cells;
  uint64_t off = 0;
  const uint64_t o_ell = off;
  off += al(std::max<uint64_t>(16, ell_b));
  const uint64_t o_E = off;
  off += al(4 * std::max<uint64_t>(1, (uint64_t)P.n_clades));
  const uint64_t o_ticket = off;
  off += al(4 * kTickets);
  const uint64_t o_flag = off;
  off += al(4 * (uint64_t)b->n_fam);
  const uint64_t o_fb = off;
  off += al(4 * ((uint64_t)b->n_fam + 1));
  const uint64_t o_gws = off;
  off += al(b->gws.n);
  if (off > kScratchBytes)
    return fail(WHALE_EINVAL, "whale_logpdf_noalloc: the batch needs " + std::to_string(off) +
                                  " bytes of workspace, more than the fixed " + std::to_string(kScratchBytes) +
                                  " bytes; evaluate it with whale_logpdf");
  unsigned char* base = c->scratch;
  WorkRaw W{};
  W.ell = base + o_ell;
  W.Eit = nullptr;         // not read or written without stored rows
  W.ibar = base + o_ell;   // not read or written without a gradient
  W.acc = nullptr;         // not read or written without a gradient
  W.E = reinterpret_cast<int32_t*>(base + o_E);
  W.ticket = reinterpret_cast<uint32_t*>(base + o_ticket);
  W.flag = reinterpret_cast<uint32_t*>(base + o_flag);
  W.fb = reinterpret_cast<uint32_t*>(base + o_fb);
  W.gws = b->gws.n ? base + o_gws : nullptr;
  W.fam_ll = d_family;
  HIPCHK(hipSetDevice(c->device));
  return enqueue(b, mode, WHALE_LAUNCH_BATCHED, false, false, false, &W, d_total);
}

int whale_logpdf_grad(whale_batch* b, int32_t mode, int32_t launch, double* out_family, double* out_total,
                      double* d_lambda, double* d_mu, double* d_q, double* d_eta) {
  return run(b, mode, launch, true, out_family, out_total, d_lambda, d_mu, d_q, d_eta);
}

int whale_backtrack(whale_batch* b, int32_t family, int32_t n_families, int32_t n_samples, uint64_t seed,
                    int32_t cap, int32_t* counts, int32_t* nodes) {
  if (!b || !counts || !nodes) return fail(WHALE_EINVAL, "NULL argument");
  if (family < 0 || n_families < 1 || (uint64_t)family + n_families > b->n_fam)
    return fail(WHALE_EINVAL, "families out of range");
  if (n_samples < 1 || cap < 1) return fail(WHALE_EINVAL, "n_samples and cap must be positive");
  if (b->last_mode < 0 || !b->last_store_all)
    return fail(WHALE_ESTATE, "no stored ℓ: evaluate with WHALE_KEEP_ELL (logpdf!) or with the gradient first");
  for (int32_t k = 0; k < n_families; ++k)
    if (!std::isfinite(b->pin_fam[family + k]))
      return fail(WHALE_EINVAL, "family " + std::to_string(family + k) + " has likelihood 0: nothing to backtrack");
  whale_model* m = b->model;
  whale_ctx* c = m->ctx;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t st = c->stream;
  const PlanHost& P = b->plan;
  if (!b->node_seg.p) {
    std::vector<int32_t> ns((size_t)b->n_fam * m->h.n, -1);
    for (uint32_t f = 0; f < b->n_fam; ++f)
      for (uint32_t s = P.fam_seg0[f]; s < P.fam_seg0[f] + P.fam_nseg[f]; ++s)
        ns[(size_t)f * m->h.n + P.seg[s].node] = (int32_t)s;
    std::vector<uint32_t> si(P.seg.size(), 0);
    for (size_t i = P.it_seg.size(); i-- > 0;) si[P.it_seg[i]] = (uint32_t)i;  // first item of each segment
    HIPCHK(upload(b->node_seg, ns, st));
    HIPCHK(upload(b->seg_item, si, st));
  }
  const int mode = b->last_mode;
  std::vector<uint8_t> f64(b->n_fam, 0);
  bool any64 = false;
  if (mode == WHALE_FP32_SCALED) {
    std::vector<uint32_t> flag(b->n_fam);
    HIPCHK(hipMemcpy(flag.data(), b->flag.p, sizeof(uint32_t) * b->n_fam, hipMemcpyDeviceToHost));
    for (uint32_t f = 0; f < b->n_fam; ++f) {
      f64[f] = flag[f] || (b->routed[f] && b->last_launch == WHALE_LAUNCH_BATCHED);
      any64 |= f64[f] != 0;
    }
    if (any64) HIPCHK(upload(b->fam64, f64, st));
  }
  BtDev D;
  const BatchDev B = b->dev();
  D.fam = B.fam;
  D.seg = B.seg;
  D.it_gid = B.it_gid;
  D.seg_item = b->seg_item.as<uint32_t>();
  D.node_seg = b->node_seg.as<int32_t>();
  D.spl_off = b->spl_off.as<uint32_t>();
  D.spl_g = b->spl_g.as<uint32_t>();
  D.split_p = B.split_p;
  D.clade_size = B.clade_size;
  D.ell = b->ell.p;
  D.ell64 = static_cast<const double*>(b->work_fallback().ell);
  D.E = mode == WHALE_FP64_PLAIN ? nullptr : b->E.as<int32_t>();
  D.fam64 = any64 ? b->fam64.as<uint8_t>() : nullptr;
  D.ell_float = mode == WHALE_FP32_SCALED ? 1 : 0;
  const ModelDev M = m->dev();
  // lanes in chunks whose node and stack buffers stay within 256 MiB
  const uint64_t per_lane = 16ull * (uint64_t)cap;
  const uint64_t lanes_total = (uint64_t)n_families * n_samples;
  const uint64_t fam_chunk = std::max<uint64_t>(1, (256ull << 20) / (per_lane * n_samples));
  const uint64_t lanes_cap = std::min<uint64_t>(lanes_total, fam_chunk * n_samples);
  // per walk where its nodes were packed; the packing cursor; the node counts
  HIPCHK(b->bt_counts.alloc(8 * (lanes_cap + 1) + 4 * lanes_cap));
  HIPCHK(b->bt_nodes.alloc(per_lane * lanes_cap));
  HIPCHK(b->bt_stack.alloc(per_lane * lanes_cap));
  for (uint64_t f0 = 0; f0 < (uint64_t)n_families; f0 += fam_chunk) {
    const uint32_t nf = (uint32_t)std::min<uint64_t>(fam_chunk, n_families - f0);
    const uint64_t lanes = (uint64_t)nf * n_samples;
    uint32_t max_items = 0;
    for (uint64_t k = 0; k < nf; ++k) max_items = std::max(max_items, P.fam[family + f0 + k].n_items);
    uint64_t* const d_first = b->bt_counts.as<uint64_t>();
    int32_t* const d_counts = (int32_t*)(d_first + lanes + 1);
    HIPCHK(launch_fill_u32(st, (uint32_t*)(d_first + lanes), 0u, 2));
    HIPCHK(launch_backtrack(st, D, M, (uint32_t)(family + f0), nf, (uint32_t)n_samples, seed, (uint32_t)cap, d_counts,
                            b->bt_nodes.as<int32_t>(), b->bt_stack.as<int32_t>(), max_items));
    // the nodes that the walks hold, packed where their stacks were
    HIPCHK(launch_bt_pack(st, lanes, d_counts, b->bt_nodes.as<int32_t>(), (uint32_t)cap, d_first,
                          d_first + lanes, b->bt_stack.as<int32_t>()));
    std::vector<uint64_t> first(lanes + 1);
    HIPCHK(hipMemcpyAsync(first.data(), d_first, 8 * (lanes + 1), hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(counts + f0 * n_samples, d_counts, 4 * lanes, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    std::vector<int32_t> packed(4 * (size_t)first[lanes]);
    if (!packed.empty()) {
      HIPCHK(hipMemcpyAsync(packed.data(), b->bt_stack.p, 4 * packed.size(), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
    }
    for (uint64_t k = 0; k < lanes; ++k) {
      const int32_t n = counts[f0 * n_samples + k];
      if (n > 0)
        std::memcpy(nodes + (f0 * n_samples + k) * 4 * (uint64_t)cap, packed.data() + 4 * (size_t)first[k],
                    16 * (size_t)n);
    }
  }
  return WHALE_OK;
}

int whale_download_ell(whale_batch* b, int32_t f, double* out, int64_t cap, int64_t* n_out) {
  if (!b || !n_out) return fail(WHALE_EINVAL, "NULL argument");
  if (f < 0 || (uint32_t)f >= b->n_fam) return fail(WHALE_EINVAL, "family out of range");
  if (b->last_mode < 0 || !b->last_store_all)
    return fail(WHALE_ESTATE, "no stored ℓ: evaluate with WHALE_KEEP_ELL or with the gradient first");
  const whale_model* m = b->model;
  const PlanHost& P = b->plan;
  const FamDev& F = P.fam[f];
  // reference layout sizes: per node id, (k+1) x |compat|
  std::vector<int> segof(m->h.n, -1);
  for (uint32_t s = P.fam_seg0[f]; s < P.fam_seg0[f] + P.fam_nseg[f]; ++s) segof[P.seg[s].node] = (int)s;
  int64_t total = 0;
  for (int e = 0; e < m->h.n; ++e)
    if (segof[e] >= 0) total += (int64_t)m->h.nodes[e].R * P.seg[segof[e]].nc;
  *n_out = total;
  if (!out || cap < total) return WHALE_OK;
  int mode = b->last_mode;
  HIPCHK(hipSetDevice(m->ctx->device));
  const char* base = (const char*)b->ell.p;
  if (mode == WHALE_FP32_SCALED) {
    uint32_t flagged = 0;
    HIPCHK(hipMemcpy(&flagged, b->flag.as<uint32_t>() + f, sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (flagged || (b->routed[f] && b->last_launch == WHALE_LAUNCH_BATCHED)) {
      mode = WHALE_FP64_SCALED;
      base = (const char*)b->work_fallback().ell;
    }
  }
  const size_t rs = mode == WHALE_FP32_SCALED ? 4 : 8;
  uint64_t cells = (f + 1 < (int32_t)b->n_fam ? P.fam[f + 1].ell0 : P.ell_cells) - F.ell0;
  std::vector<unsigned char> raw(cells * rs);
  std::vector<int32_t> E(F.n_clades, 0);
  HIPCHK(hipMemcpy(raw.data(), base + F.ell0 * rs, raw.size(), hipMemcpyDeviceToHost));
  if (mode != WHALE_FP64_PLAIN)
    HIPCHK(hipMemcpy(E.data(), b->E.as<int32_t>() + F.clade0, sizeof(int32_t) * F.n_clades, hipMemcpyDeviceToHost));
  // compatible clades of each segment, in increasing clade id (the same order as the reference's compat)
  int64_t k = 0;
  for (int e = 0; e < m->h.n; ++e) {
    int s = segof[e];
    if (s < 0) continue;
    const SegDev& sg = P.seg[s];
    // items of segment s are contiguous and it_seg is non-decreasing; they carry the clade ids
    std::vector<uint32_t> cl(sg.nc);
    uint32_t it0 = (uint32_t)(std::lower_bound(P.it_seg.begin(), P.it_seg.end(), (uint32_t)s) - P.it_seg.begin());
    for (uint32_t j = 0; j < sg.nc; ++j) cl[j] = P.it_gid[it0 + j];
    const int R = m->h.nodes[e].R;
    for (uint32_t j = 0; j < sg.nc; ++j) {
      for (int r = 0; r < R; ++r) {
        double v = 0.0;
        if (r < (int)sg.R) {
          size_t cell = sg.ell + (size_t)r * sg.nc + j;
          if (rs == 4) v = (double)reinterpret_cast<const float*>(raw.data())[cell];
          else v = reinterpret_cast<const double*>(raw.data())[cell];
          if (mode != WHALE_FP64_PLAIN && v != 0.0) v = std::ldexp(v, E[cl[j]]);
        }
        out[k++] = v;
      }
    }
  }
  return WHALE_OK;
}

}  // extern "C"
