// Execution plan of a batch of gene families, shared by the host compiler
// (host.cpp) and the device kernels (dp.hpp).
//
// The reference evaluates one family by walking the species-tree nodes in
// wm.order and, per node, every compatible clade and every time slice
// (src/core.jl:31-37, 83-128).  The plan regroups that work for one 64-lane
// wavefront, or a team of them, per family:
//
//   segment  a (family, node) pair whose compatible-clade set C_e is not
//            empty; its ℓ block is R_e x |C_e| values, row-major (one row =
//            all compatible clades at one slice), so row writes coalesce.
//   stage    all segments of one family at the same height of the species
//            tree (leaves first).  Segments of a stage are independent; their
//            clades form the stage's items, processed row by row in lockstep.
//            Segments that share a clade (possible only on MUL trees) are put
//            in different stages.
//   item     one (segment, compatible clade) pair, numbered within the stage.
//   slot     one lane's share of one item.  An item's value is a sum over its
//            splits (forward) or over the splits it is a part of (reverse
//            sweep); its terms are dealt to one slot, or to up to 16 adjacent
//            lanes of a 16-lane row when there are more than kSlotRecs.  The
//            last of them ("lead") holds the item's value.  Every sum is a
//            gather from the stage's row buffers in LDS followed by at most
//            four lane shifts: no atomics, and the order of the terms does not
//            depend on the launch.  64 slots make a chunk, one wave's work in
//            one pass; chunks are filled longest items first, so the lanes of
//            a chunk have similar term counts.
//   root     the last stage of every family: all clades, one row, processed
//            in levels (the root term uses the root's own smaller clades,
//            src/core.jl:151-158); its slots are listed level by
//            level, an item's lanes within 16 slots from a multiple of 16.
#pragma once
#include <stdint.h>

namespace whale {

constexpr uint32_t kNone = 0xffffffffu;

struct NodeDev {       // per model node, index = reference id - 1
  int32_t kind;        // WHALE_NODE_*
  int32_t child0;
  int32_t child1;
  int32_t tab;         // first row of this node in the slice tables
  int32_t R;           // rows = k + 1
  int32_t wgd;         // q index or -1
  int32_t parent;      // parent index or -1
  int32_t pad;
  double leafP;        // leafℙ
  double delta;        // slice length
};

struct FamDev {
  uint32_t n_clades;
  uint32_t n_stages;     // non-root stages
  uint32_t stage0;       // first stage (absolute)
  uint32_t item0;        // first item (absolute)
  uint32_t clade0;       // first clade (absolute): clade sizes, exponents
  uint32_t split0;       // first split (absolute)
  uint32_t lvl0;         // root level boundaries: lvl_f/lvl_b[lvl0 .. lvl0 + n_lvl], slots from root_fs / root_bs
  uint32_t n_lvl;
  uint32_t max_items;    // largest non-root stage (the root stage holds all n_clades)
  uint32_t max_slots;    // most slots of any non-root stage, either direction
  uint32_t root_seg;     // absolute segment of the root
  uint32_t root_fs;      // first forward slot of the root (absolute)
  uint32_t root_bs;      // first reverse slot of the root (absolute)
  uint32_t root_nfs;     // the root's slots
  uint32_t root_nbs;
  uint32_t root_recs;    // records of the root (the family's last)
  uint32_t rec0;         // first record (absolute); the family's records are contiguous, its entries start at 2 rec0
  uint32_t n_recs;       // records of all its stages and its root
  uint32_t n_items;      // items of its non-root stages
  uint64_t ell0;         // first ℓ cell (absolute)
  uint64_t ibar0;        // first ī cell (absolute)
};

struct StageDev {
  uint32_t item0;        // absolute first item
  uint32_t n_items;
  uint32_t r_max;        // largest R among its segments
  uint32_t seg0;         // absolute first segment
  uint32_t n_segs;
  uint32_t fs0;          // absolute first forward slot
  uint32_t n_fs;
  uint32_t bs0;          // absolute first reverse slot
  uint32_t n_bs;
  uint32_t pad;
};

struct SegDev {
  uint32_t node;         // model node index
  uint32_t nc;           // |C_e|
  uint32_t R;            // rows stored (1 for the root)
  uint32_t item0;        // stage-local index of the segment's first item
  uint32_t ell;          // first ℓ cell relative to FamDev::ell0
  uint32_t ibar;         // first ī cell relative to FamDev::ibar0 (slot k of child k: + k*nc), kNone if none
};

// what a lane needs of its item's segment and node: two 16-byte loads
struct alignas(16) SegRun {
  uint32_t ell;          // SegDev::ell - item0, so the cell of stage item i at row r is ell + i + r*nc (mod 2^32)
  uint32_t nc;
  uint32_t R;
  uint32_t tab;          // first row of the node in the slice tables
  uint32_t kn;           // node kind | node << 2
  uint32_t c0;           // child0 (leaf: the node itself)
  uint32_t c1;           // child1; a WGD node: its q index
  uint32_t ibar;         // SegDev::ibar - item0
};

// Slots: two arrays per direction, over all slots of the batch.
//   s4[s] = {a, b, c, d}
//     a, b   ℓ cells (relative to ell0) of child0's and child1's top rows for
//            the slot's clade, or -1 (a WGD node's one child stands in both)
//     c      item | position within the item's slots << 16 | kSlotLead
//     d      forward: clade | stage-local segment << 16
//            reverse: ī cell (relative to ibar0) holding d logL / d top-row value
//   s2[s] = {start, count | (reverse: stage-local segment << 16)}
//            the slot's terms: records rec0 + start .. (forward) or entries
//            2 rec0 + start .. (reverse)
// Unused lanes have no terms and no lead.
// Records (one per split of an item's clade): rec_ops[r] = l1 | l2 << 16,
// stage-local items of the two parts; rec_p[r] = p.
// Entries (two per record, listed by part): ent_ops[k] = owner | other << 16,
// the stage-local items owning the record and of its other part; ent_p[k] = p.
constexpr uint32_t kSlotLead = 1u << 20;
constexpr uint32_t kSlotRecs = 4;       // terms a slot holds before an item takes another lane
constexpr uint32_t kSlotLanes = 16;     // most lanes of one item
constexpr uint32_t kChunk = 64;

}  // namespace whale
