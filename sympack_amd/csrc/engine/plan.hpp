// Device execution plan for the supernodal factorization and solve.
//
// The plan is built once per symbolic structure on the host and uploaded to
// HBM.  It fixes:
//  * the factor layout: one contiguous arena holding every supernode's panel
//    (all rows of its structure x its columns), column-major with leading
//    dimension = number of structure rows, so a column of a panel is a
//    contiguous run of HBM;
//  * relative-index maps, so the Schur-update kernel scatters into ancestor
//    panels without searching block lists;
//  * the assembly map from the caller's CSC entries to arena offsets;
//  * etree-level task lists for every batched kernel launch.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "../analysis/analysis.hpp"

namespace spk {

constexpr int kTile = 64;    // update tile edge (rows x cols)
constexpr int kStep = 160;   // panel columns factored per step (diagonal block <= 160 x 160)
constexpr int kSub = 16;     // sub-block edge inside a diagonal block (MFMA 16x16 tiles)
constexpr int kTrsmRows = 64;  // panel rows per fused block factor + TRSM workgroup (16 per wave)
constexpr int kTrsmRowsWide = 128;  // panel rows per k_ptrsm workgroup (8 waves of 16 rows)
// supernodes that fit one wave (k_narrow<N>, N = 8 or 16: at most N columns and
// 64 - N rows below) get a launch of their own above this many
constexpr int64_t kNarrowMany = 256;
constexpr int kSchurKC = 32;   // k columns per LDS chunk of the Schur update
// Schur launches with fewer tasks than this (one per CU of the 256) split
// each task's k chunks over several workgroups; more splitting costs more in
// extra scatter than it gains in latency
constexpr int64_t kSplitTarget = 256;

// LDS bucket of a diagonal block with nb 16-column sub-blocks: kernels are
// compiled for nb <= 1, 2, 4, 6, 10.
inline int diag_bucket(int nb) { return nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : nb <= 6 ? 6 : 10; }

struct SnInfo {            // mirrored on the device (16-byte aligned)
  int64_t off;             // panel offset in the arena (elements)
  int64_t upd;             // offset into tcol/tmap for the panel's off-diagonal rows
  int32_t r;               // structure rows (= panel leading dimension)
  int32_t w;               // width (columns)
  int32_t fc;              // first column, 0-based, permuted numbering
  int32_t lx;              // offset of the structure in lindx0
};

struct Task4 {
  int32_t a, b, c, d;
};

// One panel of the solve: columns [c0, c0 + w), w <= kStep, of a supernode
// with the rows of its structure from c0 on (so a supernode of at most kStep
// columns is one panel, a wider one a chain of them).
struct SolvePanel {        // mirrored on the device
  int64_t off;             // arena offset of the panel's first diagonal entry
  int32_t ld;              // leading dimension (rows of the whole supernode)
  int32_t r;               // rows, w of them diagonal
  int32_t w;
  int32_t fc;              // first column, 0-based, permuted numbering
  int32_t lx;              // offset of the panel's first row in lindx0
  int32_t pad;
};

// Schur updates along chains.  A separator wider than the supernode limit is
// a chain of supernodes, each the main child of the next, and the rows of
// every member below the chain's columns are rows of the chain's last member
// E.  A member applies its update at its own level only inside the chain's
// columns; the rest is applied once for the whole chain, at E's level, as
// one product over the columns of all members.  Each target entry outside
// the chain is then written once per chain instead of once per member, and
// the product runs over a long k.
//
// The update that a supernode H computes at its level (its "head") is
//   C(a,b) = sum over its segments of  S(a,:) S(b,:)^T   (LDL: S D S^T)
// for H's off-diagonal rows a >= b, b < bcut.  Segment 0 is H itself; a row
// a of H is row shift + a of the segment's panel, or mmap[moff + a] where
// moff >= 0 (-1: the segment has no such row).
struct SchurSeg {          // mirrored on the device
  int64_t off;             // panel offset of the segment's supernode
  int64_t moff;            // offset of the row map in mmap, -1: shift
  int32_t ld;              // its panel's leading dimension (rows)
  int32_t w;               // its width (k columns)
  int32_t shift;
  int32_t sn;
};
struct SchurHead {         // mirrored on the device; one per supernode with an update
  int32_t seg0, nseg;      // segments [seg0, seg0 + nseg)
  int32_t bcut;            // output columns (off-diagonal rows b) below bcut only
  int32_t nq, nq16;        // k chunks of kSchurKC / of 16 columns over all segments
  // output columns below excl lie in panels that no other supernode of the
  // same etree level (the same launch) updates: no atomics needed there
  int32_t excl;
  int32_t split;           // k parts of its 64 x 64 tiles, tasks of their own
  int32_t pad;
};

// One run of consecutive off-diagonal rows [gb, ge) of supernode I whose
// rows are columns of the same ancestor J.  The relative indices of all of
// I's off-diagonal rows a >= gb inside struct(J) are
// rel[base + a - gb] (a in [gb, m_I)); they, and the scatter bases tcol /
// tmap of the rows [gb, ge), are filled on the device from this table
// (binary search of each row in struct(J)).
struct RelGroup {          // mirrored on the device
  int64_t base;
  int32_t I, J, gb, ge;
};

// Host and device code (the plan is counted on the host, the task lists are
// written on the device by the same formulas).
#if defined(__HIPCC__)
#define SPK_HD __host__ __device__
#else
#define SPK_HD
#endif

// Schur output tiles (ti, tj), tj <= ti, tj < ntj, of one supernode (ntj =
// the column-tile count, fewer than the row tiles where the head's columns
// are cut): those of the row tiles before ti.
SPK_HD inline int64_t schur_tiles_before(int64_t ti, int64_t ntj) {
  return ti <= ntj ? ti * (ti + 1) / 2 : ntj * (ntj + 1) / 2 + (ti - ntj) * ntj;
}

// A Schur task is {sn, ti, tj | part << kTileBits, head}: a non-negative field
// holds parts below kMaxParts.
constexpr int kTileBits = 20, kTileMask = (1 << kTileBits) - 1;
constexpr int64_t kMaxParts = int64_t(1) << (31 - kTileBits);

// Per supernode with a Schur update: where its tasks go in
// the four Schur task arrays (64 x 64 tiles in plan order and longest first,
// 128 x 128 tiles in plan order and longest first); nt x ntj and ntw x ntjw
// row x column tiles.
struct SchurEmit {         // mirrored on the device
  int64_t first[4];
  int32_t I, nt, ntj, ntw;
  int32_t ntjw, head;      // head: index of its SchurHead (the tasks' d)
  int32_t split, pad;      // as in the SchurHead
};

struct LaunchRange {
  int kind;          // 0 diagonal factor, 7 panel TRSM, 9 both fused, 1 in-panel update,
                     // 2 Schur update,
                     // 3 forward diag, 4 forward off-diag, 5 backward off-diag, 6 backward diag,
                     // 10 forward / 11 backward partitioned-inverse solve, 12 its preparation
  int64_t first;     // first task in that kind's task array
  int64_t count;     // number of tasks (= grid size)
  int aux = 0;       // kinds 0, 7, 9, 3, 6: diagonal-block bucket (diag_bucket; kind 0: -N = k_narrow<N>);
                     // kind 2: k-chunk split factor (0 or 1 = none)
  int level = 0;     // etree level of the launch (factor sequence)
  int alt = 0;       // kind 2: bit 0 = tasks in longest-first order, bit 1 = 128 x 128
                     // tiles, bit 2 = one wave per 64 x 64 tile (k_schur_w1)
  int64_t first_w = 0, count_w = 0;  // kind 2: the level's 128 x 128 tile tasks
  int nqmin = 0;     // kind 2: fewest k chunks of any task of the range
  int nsegmax = 0;   // kind 2: most segments of any task of the range
};

struct Plan {
  int32_t n = 0, nsuper = 0;
  int64_t arena_elems = 0;
  std::vector<SnInfo> sn;
  std::vector<int32_t> lindx0;     // 0-based structure rows (permuted numbering)
  std::vector<int32_t> level;      // etree height of every supernode
  int32_t nlevels = 0;
  // Schur scatter maps (per off-diagonal row b of supernode I):
  // target address of element (a,b) = tcol[upd+b] + rel[tmap[upd+b] + a].
  // tcol, tmap (upd_size entries each) and rel (rel_size entries) exist on
  // the device only, built from rel_groups.
  std::vector<RelGroup> rel_groups;
  int64_t upd_size = 0, rel_size = 0;
  // assembly: arena offset of every caller CSC entry (-1 = superseded duplicate)
  std::vector<int64_t> amap;
  std::vector<int32_t> perm0;      // perm0[new] = old, 0-based
  // task arrays
  std::vector<Task4> potrf_tasks;  // {sn, step, inverse-tile offset, 0}
  std::vector<Task4> narrow_tasks; // {sn, 0, inverse-tile offset, 0}: whole panels of k_narrow
  std::vector<Task4> trsm_tasks;   // {sn, step, row_tile, inverse-tile offset}
  int64_t inv_tiles = 0;           // 16x16 inverse diagonal tiles written by the factor
  std::vector<int64_t> inv_base;   // per supernode: first inverse tile (tile t of 16-column block t)
  std::vector<Task4> inpanel_tasks;// {sn, step, ti, tj}
  std::vector<Task4> fused_tasks;  // {sn, row tiles, row_tile, inverse-tile offset}: block factor + TRSM
  // Schur tasks: 64x64 output tiles (and k parts).  Four arrays,
  // written on the device from schur_emit: 64 x 64 tiles in plan order; the
  // same with every launch range's supernodes ordered by their k chunks,
  // longest first (stable; workgroups are dispatched in index order);
  // 128 x 128 tiles in plan order and longest first.
  int64_t n_schur = 0, n_schur_wide = 0;
  std::vector<SchurEmit> schur_emit;
  std::vector<SchurHead> schur_heads;
  std::vector<SchurSeg> schur_segs;
  std::vector<int32_t> mmap;
  std::vector<int32_t> chain_end;      // per supernode: last member of its chain (itself: a chain of one)
  // per supernode: the parent (in the same chain) that takes over its update
  // beyond the parent's columns, -1 = none.  The parent has it as a second
  // segment; beyond the chain's columns the chain's last member has both.
  std::vector<int32_t> deferred_into;
  std::vector<LaunchRange> factor_seq;
  // Solve, level by level over the panels (a supernode's panels follow one
  // another; where every supernode is at most kStep wide the levels are the
  // etree's).
  std::vector<SolvePanel> panels;
  std::vector<Task4> sdiag_tasks;  // {panel, inverse-tile base, 0, 0}: diagonal-block solves
  std::vector<Task4> soffm_tasks;  // {panel, row_tile, 0, 0}: 64-row tiles of the rows below the block
  std::vector<LaunchRange> fwd_seq, bwd_seq;  // kind 3/6 aux: diag_bucket of the level
  // Partitioned-inverse solve, for plans without a supernode wider than kStep
  // (a panel is then a supernode; lists empty otherwise):
  // G = [I; L_off] L_diag^{-1} of every panel (its
  // shape and offsets, in an arena of its own) is prepared once per
  // factorization; then each level costs one forward launch
  // [X_p; dY] = G_p Y_p and one backward launch X_p = G_p^T [X_p; -X_rows].
  // Tasks {panel, 64-row tile, inverse-tile base, 0} over all rows of every
  // panel; kinds 10/11 per level, kind 12 (preparation) per diagonal-block
  // bucket, aux = bucket.
  std::vector<Task4> gtiles;
  std::vector<LaunchRange> gfwd_seq, gbwd_seq, gprep_seq;
  // dependency-driven solve (one persistent launch per sweep), available when
  // every supernode fits one diagonal block (w <= kStep).  Tasks
  // {kind, sn, row tile, first target}: forward D(s) = 0 / O(s,rt) = 1 in
  // postorder, backward R(s,rt) = 2 / B(s) = 3 in reverse postorder; the
  // targets of O(s,rt) / R(s,rt), df_tgt[d .. end), are the supernodes
  // owning the tile's rows.
  bool df_ok = false;  // the lists can be built (build_dataflow_lists)
  // algorithmic counts
  double schur_flops = 0, inpanel_flops = 0, diag_flops = 0;
  int64_t schur_entries = 0;       // lower-triangle entries scattered
  int max_w = 0;
  int64_t max_panel = 0;           // largest panel, r * w elements
};

// Build the plan from the symbolic analysis and the caller's CSC pattern
// (lower triangle, any base).  merge_updates: 0 every supernode applies its
// whole update at its own level; 1 chains of supernodes at least kSchurKC
// wide, and inside a chain a child's update taken over by its parent where
// both levels have enough tiles to fill the GPU; 2 both wherever the
// structure allows.
void build_plan(const Symbolic& s, Int n, const Ptr* colptr, const Idx* rowind, int baseval,
                Plan& p, int merge_updates = 1);

// Task lists of the dependency-driven solve (switched off on the device):
// built on demand from the plan, not by build_plan.
struct DataflowLists {
  std::vector<Task4> fwd, bwd;
  std::vector<int32_t> fwd_end, bwd_end;
  std::vector<int32_t> tgt;          // shared by O and R tasks (same tiles)
  std::vector<int32_t> dcnt0;        // per supernode: O tasks that update its rows
  std::vector<int32_t> rcnt0;        // per supernode: its row tiles
};
DataflowLists build_dataflow_lists(const Plan& p);

// Checks the dependency-driven solve lists by running them in ticket order
// on one worker: every wait must already be satisfied when its task is
// reached (so with any number of workers taking tickets in order, the
// oldest unfinished task can always proceed), every counter must reach zero
// and every task's targets must be the owners of its rows.  Returns an
// empty string or the first violation.
std::string validate_solve_plan(const Plan& p);

}  // namespace spk
