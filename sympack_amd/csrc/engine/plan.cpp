// Host construction of the device plan (see plan.hpp).
#include "plan.hpp"

#include <algorithm>
#include <climits>
#include <stdexcept>
#include <exception>
#include <thread>

namespace spk {

namespace {
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Splits a level's items into launches by diagonal-block bucket.  A kernel
// compiled for wide blocks holds up to 119 KB of LDS or 40 operand registers
// also where the block is narrow, so one wide supernode on a level of
// hundreds of narrow ones makes them all slow: narrower buckets get a launch
// of their own when they have more than `enough` work units, otherwise they
// ride along with the next wider one (a launch costs 3-5 us).  315^2, level
// 1, 1,793 supernodes of one 16-column block and one of ten: block factors
// and TRSM 131 -> 66 us, forward sweep 37 -> 14 us.
struct BucketGroup {
  int bucket;
  std::vector<Int> items;
};
// The next bucket has to be four times as wide: 627 supernodes of two blocks
// beside one of six cost 37 us together and 61 us apart.  Solve of 315^2, one
// right-hand side: 222 us, 231 from twice as wide on, 235 never; 30^3 7-point 234,
// 242, 234; eight other structures within 2% either way.
template <class BucketOf, class UnitsOf>
std::vector<BucketGroup> bucket_groups(const std::vector<Int>& items, int64_t enough, BucketOf&& bucket_of,
                                       UnitsOf&& units_of) {
  std::vector<BucketGroup> out;
  BucketGroup cur{1, {}};
  int64_t units = 0;
  for (int bk : {1, 2, 4, 6, 10}) {
    bool any = false;
    for (Int I : items) any |= bucket_of(I) == bk;
    if (!any) continue;
    if (units > enough && bk >= 4 * cur.bucket) {
      out.push_back(std::move(cur));
      cur.items.clear();
      units = 0;
    }
    cur.bucket = bk;
    for (Int I : items)
      if (bucket_of(I) == bk) {
        cur.items.push_back(I);
        units += units_of(I);
      }
  }
  if (!cur.items.empty()) out.push_back(std::move(cur));
  return out;
}
}  // namespace

void build_plan(const Symbolic& s, Int n, const Ptr* colptr, const Idx* rowind, int baseval,
                Plan& p, int merge_updates) {
  p = Plan();
  p.n = n;
  const Int ns = s.nsuper();
  p.nsuper = ns;
  p.sn.resize(ns);
  p.lindx0.resize(s.lindx.size());
  for (size_t i = 0; i < s.lindx.size(); ++i) p.lindx0[i] = s.lindx[i] - 1;
  p.perm0.resize(n);
  for (Int i = 0; i < n; ++i) p.perm0[i] = s.ord.perm[i] - 1;

  // panels, column-major, leading dimension r
  int64_t off = 0, upd = 0;
  for (Int I = 0; I < ns; ++I) {
    SnInfo& si = p.sn[I];
    si.fc = s.xsuper[I] - 1;
    si.w = s.xsuper[I + 1] - s.xsuper[I];
    si.lx = (int32_t)(s.xlindx[I] - 1);
    si.r = (int32_t)(s.xlindx[I + 1] - s.xlindx[I]);
    si.off = off;
    si.upd = upd;
    off += (int64_t)si.r * si.w;
    upd += si.r - si.w;
    p.max_w = std::max(p.max_w, (int)si.w);
    p.max_panel = std::max(p.max_panel, (int64_t)si.r * si.w);
  }
  p.arena_elems = off;

  // etree heights (children have smaller indices than parents: postorder)
  p.level.assign(ns, 0);
  for (Int I = 0; I < ns; ++I) {
    Int par = s.sparent[I];
    if (par > 0) p.level[par - 1] = std::max(p.level[par - 1], p.level[I] + 1);
  }
  p.nlevels = 0;
  for (Int I = 0; I < ns; ++I) p.nlevels = std::max(p.nlevels, p.level[I] + 1);

  // row -> supernode (0-based) and position maps for the relative indices
  std::vector<int32_t> row_sup(n);
  for (Int i = 0; i < n; ++i) row_sup[i] = s.supMembership[i] - 1;

  // Assembly map: caller entry (row,col) of the lower triangle goes to
  // (max,min) of the permuted indices; later duplicates win.  It runs on its
  // own thread beside the scatter maps and the merges (it writes only amap
  // and reads the structure).
  // Common case: every column's rows are strictly increasing and none lies
  // above the diagonal, so no two entries share a pair; each entry then
  // finds its row in its target supernode's structure by itself (the
  // diagonal block directly, the rows below by binary search), on several
  // threads over column ranges of equal entry counts.
  // Otherwise entries are bucketed by their permuted column (stable, in
  // entry order); each supernode marks the positions of its structure rows
  // once, so every entry finds its row in O(1).  Two entries land on the same
  // arena offset exactly when they share the permuted pair, i.e. the bucket
  // and the row, and the earlier one is dropped.
  bool amap_error = false;
  std::exception_ptr amap_exc;
  std::thread amap_thread([&]() {
    try {
    const Ptr nnz = colptr[n] - baseval;
    p.amap.resize(nnz);
    {
      const int nth = (int)std::max<unsigned>(1, std::min<unsigned>(8, std::thread::hardware_concurrency()));
      std::vector<Int> split(nth + 1, n);
      split[0] = 0;
      for (int t = 1; t < nth; ++t)
        split[t] = (Int)(std::lower_bound(colptr, colptr + n, (Ptr)(nnz * t / nth) + baseval) - colptr);
      std::vector<char> unclean(nth, 0), missing(nth, 0);
      auto work = [&](int t) {
        for (Int c = split[t]; c < split[t + 1]; ++c) {
          const int32_t pcol = s.ord.invp[c] - 1;
          Idx prev = -1;
          for (Ptr q = colptr[c] - baseval; q < colptr[c + 1] - baseval; ++q) {
            const Idx r = rowind[q] - baseval;
            if (r < c || r <= prev) {
              unclean[t] = 1;
              return;
            }
            prev = r;
            const int32_t prow = s.ord.invp[r] - 1;
            const int32_t pr = std::max(prow, pcol), pc = std::min(prow, pcol);
            const SnInfo& sj = p.sn[row_sup[pc]];
            int32_t pos = pr - sj.fc;
            if (pos >= sj.w) {
              const int32_t* b = &p.lindx0[sj.lx] + sj.w;
              const int32_t* e = &p.lindx0[sj.lx] + sj.r;
              const int32_t* f = std::lower_bound(b, e, pr);
              if (f == e || *f != pr) {
                missing[t] = 1;
                return;
              }
              pos = (int32_t)(f - &p.lindx0[sj.lx]);
            }
            p.amap[q] = sj.off + (int64_t)(pc - sj.fc) * sj.r + pos;
          }
        }
      };
      std::vector<std::thread> pool;
      for (int t = 1; t < nth; ++t) pool.emplace_back(work, t);
      work(0);
      for (auto& th : pool) th.join();
      bool any_unclean = false;
      for (int t = 0; t < nth; ++t) {
        any_unclean |= unclean[t] != 0;
        amap_error |= missing[t] != 0;
      }
      if (!any_unclean || amap_error) return;
    }
    std::vector<int32_t> apos(n, -1);
    {
      std::fill(p.amap.begin(), p.amap.end(), -1);
      std::vector<Ptr> bstart(n + 1, 0), order(nnz);
      std::vector<int32_t> trow_of(nnz);
      for (Int c = 0; c < n; ++c)
        for (Ptr q = colptr[c] - baseval; q < colptr[c + 1] - baseval; ++q) {
          const int32_t pr = s.ord.invp[rowind[q] - baseval] - 1, pc = s.ord.invp[c] - 1;
          trow_of[q] = std::max(pr, pc);
          ++bstart[std::min(pr, pc) + 1];
        }
      for (Int i = 0; i < n; ++i) bstart[i + 1] += bstart[i];
      {
        std::vector<Ptr> fill(bstart.begin(), bstart.end() - 1);
        for (Int c = 0; c < n; ++c)
          for (Ptr q = colptr[c] - baseval; q < colptr[c + 1] - baseval; ++q) {
            const int32_t pr = s.ord.invp[rowind[q] - baseval] - 1, pc = s.ord.invp[c] - 1;
            order[fill[std::min(pr, pc)]++] = q;
          }
      }
      std::vector<int32_t> seen(n, -1);
      std::vector<Ptr> last(n, -1);
      for (Int J = 0; J < ns; ++J) {
        const SnInfo& sj = p.sn[J];
        const int32_t* stJ = &p.lindx0[sj.lx];
        for (int32_t q = 0; q < sj.r; ++q) apos[stJ[q]] = q;
        for (int32_t tcol = sj.fc; tcol < sj.fc + sj.w; ++tcol)
          for (Ptr t = bstart[tcol]; t < bstart[tcol + 1]; ++t) {
            const Ptr q = order[t];
            const int32_t trow = trow_of[q];
            const int32_t pp = apos[trow];
            if (pp < 0) {
              amap_error = true;
              return;
            }
            p.amap[q] = sj.off + (int64_t)(tcol - sj.fc) * sj.r + pp;
            if (seen[trow] == tcol) p.amap[last[trow]] = -1;  // an earlier entry of the same pair
            seen[trow] = tcol;
            last[trow] = q;
          }
        for (int32_t q = 0; q < sj.r; ++q) apos[stJ[q]] = -1;
      }
    }
    } catch (...) {
      amap_exc = std::current_exception();
    }
  });
  struct Joiner {  // joins on every exit, also when the code below throws
    std::thread& t;
    ~Joiner() {
      if (t.joinable()) t.join();
    }
  } amap_joiner{amap_thread};

  // Schur scatter maps.  For off-diagonal row b of I with target supernode J
  // (the supernode of column lindx[w+b]) the rows a >= first row of that
  // target group are all in struct(J); their positions there (rel) are
  // found on the device from one RelGroup per group.
  p.upd_size = upd;
  p.rel_groups.clear();
  p.rel_size = 0;
  std::vector<int64_t> group0(ns + 1, 0);  // first RelGroup of every supernode
  for (Int I = 0; I < ns; ++I) {
    group0[I] = (int64_t)p.rel_groups.size();
    const SnInfo& si = p.sn[I];
    const int32_t* st = &p.lindx0[si.lx];
    int32_t m = si.r - si.w;
    int32_t b = 0;
    while (b < m) {
      int32_t J = row_sup[st[si.w + b]];
      // group = consecutive off-diagonal rows falling in J's columns (the
      // columns of J are consecutive numbers: the group ends at the first
      // row past J's last column)
      int32_t gb = b;
      const int32_t jend = p.sn[J].fc + p.sn[J].w;
      b = (int32_t)(std::lower_bound(st + si.w + b, st + si.r, jend) - (st + si.w));
      p.rel_groups.push_back({p.rel_size, I, J, gb, b});
      p.rel_size += m - gb;
    }
  }
  group0[ns] = (int64_t)p.rel_groups.size();

  // Chains (see SchurSeg).  The parent P of C is the supernode of C's first
  // off-diagonal row; the rows of struct(C) inside P's columns form a prefix
  // of length n1, the remaining rows r2 all lie in struct(P).  C continues
  // its chain into P when its remaining rows cover most of P's (the chain's
  // products then carry few zero rows: 1% of the flops on 3D nested
  // dissection grids) and no other child of P comes near it in rows: where
  // two separators of similar size meet, their parent's columns are outside
  // both chains.  Members narrower than one k chunk are left out in mode 1:
  // a segment costs a whole chunk's staging.  The two limits decide little:
  // factor of 48^3 4.73 ms, 4.77 and 4.74 with 0.25 and 0.8 for siblings, 60^3
  // 27-point 12.05, 12.09 and 12.03; 0.7 and 0.95 of fill change nothing beyond
  // 0.3% there, on LDL^T 60^3 or under AMD.
  constexpr double kChainMinFill = 0.85, kChainMaxSibling = 0.5;
  std::vector<int32_t> par(ns, -1), n1(ns, 0);
  std::vector<int32_t> link(ns, -1), prev(ns, -1);  // next / previous member of the chain
  if (merge_updates > 0) {
    std::vector<int32_t> big(ns, -1), second(ns, 0);  // per parent: child with most rows, next one's rows
    auto rows_of = [&](Int I) { return p.sn[I].r - p.sn[I].w; };
    for (Int I = 0; I < ns; ++I) {
      const SnInfo& si = p.sn[I];
      const int32_t m = si.r - si.w;
      if (m <= 0) continue;
      const int32_t* st = &p.lindx0[si.lx + si.w];
      const Int P = row_sup[st[0]];
      par[I] = P;
      n1[I] = (int32_t)(std::lower_bound(st, st + m, p.sn[P].fc + p.sn[P].w) - st);
      if (big[P] < 0 || m > rows_of(big[P])) {
        if (big[P] >= 0) second[P] = std::max(second[P], rows_of(big[P]));
        big[P] = I;
      } else {
        second[P] = std::max(second[P], m);
      }
    }
    for (Int P = 0; P < ns; ++P) {
      const Int C = big[P];
      if (C < 0) continue;
      const int32_t mC = rows_of(C), mP = rows_of(P), r2 = mC - n1[C];
      if (merge_updates < 2 && p.sn[C].w < kSchurKC) continue;
      if (second[P] > kChainMaxSibling * mC || r2 < kChainMinFill * mP) continue;
      // the remaining rows must be rows of P
      const int32_t* c = &p.lindx0[p.sn[C].lx + p.sn[C].w] + n1[C];
      const int32_t* q = &p.lindx0[p.sn[P].lx + p.sn[P].w];
      if (!std::includes(q, q + mP, c, c + r2)) continue;
      link[C] = P;
      prev[P] = C;
    }
  }
  p.chain_end.resize(ns);
  for (Int I = ns - 1; I >= 0; --I) p.chain_end[I] = link[I] >= 0 ? p.chain_end[link[I]] : I;

  // Inside a chain, a child's update beyond its parent's columns can be taken
  // over by the parent as a second segment; a supernode that takes one over
  // is not itself taken over.  That moves work to the parent's level and
  // lengthens its tiles' k loop, which only pays where both levels have
  // enough tiles to keep every CU busy (3 workgroups per CU x 256 CUs); near
  // the root, where a level holds one or two supernodes, it would lengthen
  // the critical path instead.
  constexpr int32_t kMergeMinRows = 32;
  const int64_t kMergeMinLevelTiles = merge_updates >= 2 ? 0 : 768;
  std::vector<int64_t> level_tiles(p.nlevels, 0);
  for (Int I = 0; I < ns; ++I) {
    const int64_t t = ceil_div(p.sn[I].r - p.sn[I].w, kTile);
    level_tiles[p.level[I]] += t * (t + 1) / 2;
  }
  p.deferred_into.assign(ns, -1);
  std::vector<int32_t> absorbs(ns, -1);  // per supernode: the child it takes over
  for (Int P = 0; P < ns; ++P) {  // children precede parents
    const Int C = prev[P];
    if (C < 0 || p.sn[P].r <= p.sn[P].w || absorbs[C] >= 0) continue;
    if (level_tiles[p.level[P]] < kMergeMinLevelTiles || level_tiles[p.level[C]] < kMergeMinLevelTiles) continue;
    if ((p.sn[C].r - p.sn[C].w) - n1[C] < kMergeMinRows) continue;
    absorbs[P] = C;
    p.deferred_into[C] = P;
  }

  // heads and their segments
  p.schur_heads.reserve(ns);
  p.schur_segs.reserve(2 * (size_t)ns);
  auto add_segment = [&](Int H, Int S) {
    const SnInfo& sh = p.sn[H];
    const SnInfo& sg = p.sn[S];
    const int32_t mH = sh.r - sh.w;
    SchurSeg g{};
    g.off = sg.off;
    g.moff = -1;
    g.ld = sg.r;
    g.w = sg.w;
    g.sn = S;
    const int32_t* st = &p.lindx0[sg.lx];
    const int32_t first = (int32_t)(std::lower_bound(st + sg.w, st + sg.r, sh.fc + sh.w) - st);
    g.shift = first;  // S has exactly H's rows there, or:
    if (sg.r - first != mH) {
      g.moff = (int64_t)p.mmap.size();
      p.mmap.resize(p.mmap.size() + mH);
      int32_t* map = &p.mmap[g.moff];
      const int32_t* rows = &p.lindx0[sh.lx + sh.w];  // sorted, as st is
      int32_t q = first;
      for (int32_t a = 0; a < mH; ++a) {
        const bool has = q < sg.r && st[q] == rows[a];
        map[a] = has ? q : -1;
        q += has;
      }
    }
    p.schur_segs.push_back(g);
    p.schur_heads.back().nseg++;
    p.schur_heads.back().nq += (int32_t)ceil_div(sg.w, kSchurKC);
    p.schur_heads.back().nq16 += (int32_t)ceil_div(sg.w, 16);
  };
  std::vector<int32_t> head_of(ns, -1);
  for (Int I = 0; I < ns; ++I) {
    const SnInfo& si = p.sn[I];
    const int32_t m = si.r - si.w;
    if (m <= 0) continue;
    head_of[I] = (int32_t)p.schur_heads.size();
    SchurHead h{};
    h.seg0 = (int32_t)p.schur_segs.size();
    h.bcut = m;
    if (p.deferred_into[I] >= 0) {
      h.bcut = n1[I];
    } else if (p.chain_end[I] != I) {
      const SnInfo& se = p.sn[p.chain_end[I]];
      const int32_t* st = &p.lindx0[si.lx + si.w];
      h.bcut = (int32_t)(std::lower_bound(st, st + m, se.fc + se.w) - st);
    }
    p.schur_heads.push_back(h);
    add_segment(I, I);
    if (p.chain_end[I] == I)
      for (Int C = prev[I]; C >= 0; C = prev[C]) add_segment(I, C);
    else if (absorbs[I] >= 0)
      add_segment(I, absorbs[I]);
  }

  amap_thread.join();
  if (amap_exc) std::rethrow_exception(amap_exc);
  if (amap_error) throw std::logic_error("matrix entry outside the symbolic structure");

  // inverse diagonal tiles: ceil(w/16) per supernode, contiguous, so block t
  // of step st is tile inv_base + 10 st + t
  p.inv_base.assign(ns, 0);
  for (Int I = 0; I < ns; ++I) {
    p.inv_base[I] = p.inv_tiles;
    p.inv_tiles += ceil_div(p.sn[I].w, kSub);
  }

  // ---- factorization task lists, level by level ----
  std::vector<std::vector<Int>> by_level(p.nlevels);
  for (Int I = 0; I < ns; ++I) by_level[p.level[I]].push_back(I);
  std::vector<int32_t> writers(ns, 0);  // per panel: supernodes of the level that update it
  for (int L = 0; L < p.nlevels; ++L) {
    const auto& sns = by_level[L];
    auto each_target = [&](Int I, auto&& f) {
      if (head_of[I] < 0) return;
      const int32_t cut = p.schur_heads[head_of[I]].bcut;
      for (int64_t g = group0[I]; g < group0[I + 1] && p.rel_groups[g].gb < cut; ++g)
        if (!f(p.rel_groups[g])) break;
    };
    for (Int I : sns) each_target(I, [&](const RelGroup& g) { return ++writers[g.J], true; });
    for (Int I : sns)
      each_target(I, [&](const RelGroup& g) {
        SchurHead& h = p.schur_heads[head_of[I]];
        if (writers[g.J] != 1) return false;
        h.excl = std::min(g.ge, h.bcut);
        return true;
      });
    for (Int I : sns) each_target(I, [&](const RelGroup& g) { return writers[g.J] = 0, true; });
    const size_t level_first = p.factor_seq.size();
    // Levels of single-step supernodes with at most kFuseMaxTasks row
    // tiles in all: one fused block-factor + TRSM launch (every row-tile
    // workgroup factors the block again) instead of two dependent launches.
    constexpr int64_t kFuseMaxTasks = 256;
    int64_t fuse_tasks = 0;
    // Supernodes that fit one wave, in launches of their own where they are
    // many or all that is left of the level (otherwise they ride along with
    // the wider ones).  Few that are all of a level, factor against the fused
    // block factor and TRSM: 40^2 RCM, at most 8 wide, 1613 against 2070 us, 64^2
    // 267 against 291, 8^2 63.5 against 61.5.
    std::vector<Int> block_sns = sns;
    for (int N : {8, 16}) {
      const auto mid = std::stable_partition(block_sns.begin(), block_sns.end(), [&](Int I) {
        return p.sn[I].w > N || p.sn[I].r - p.sn[I].w > 64 - N;
      });
      const int64_t nn = block_sns.end() - mid;
      if (nn == 0 || (nn <= kNarrowMany && mid != block_sns.begin())) continue;
      LaunchRange nr{0, (int64_t)p.narrow_tasks.size(), nn, -N};
      for (auto it = mid; it != block_sns.end(); ++it) {
        const SnInfo& si = p.sn[*it];
        p.narrow_tasks.push_back({*it, 0, (int32_t)p.inv_base[*it], 0});
        p.diag_flops += (double)si.w * si.w * si.w / 3.0 + (double)si.w * si.w * (si.r - si.w);
      }
      p.factor_seq.push_back(nr);
      block_sns.erase(mid, block_sns.end());
    }
    int smax = 0;
    for (Int I : block_sns) smax = std::max<int>(smax, (int)ceil_div(p.sn[I].w, kStep));
    if (smax == 1)
      for (Int I : block_sns) fuse_tasks += std::max<int64_t>(1, ceil_div(p.sn[I].r - p.sn[I].w, kTrsmRows));
    if (smax == 1 && fuse_tasks <= kFuseMaxTasks) {
      LaunchRange fr{9, (int64_t)p.fused_tasks.size(), 0};
      int nbmax = 1;
      for (Int I : block_sns) {
        const SnInfo& si = p.sn[I];
        const int bs = si.w;
        nbmax = std::max(nbmax, (int)ceil_div(bs, kSub));
        const int64_t rows_below = si.r - bs;
        const int32_t inv_off = (int32_t)p.inv_base[I];
        const int64_t nt = std::max<int64_t>(1, ceil_div(rows_below, kTrsmRows));
        for (int64_t rt = 0; rt < nt; ++rt)
          p.fused_tasks.push_back({I, (int32_t)nt, (int32_t)rt, inv_off});
        p.diag_flops += (double)bs * bs * bs / 3.0 + (double)bs * bs * rows_below;
      }
      fr.aux = diag_bucket(nbmax);
      fr.count = (int64_t)p.fused_tasks.size() - fr.first;
      p.factor_seq.push_back(fr);
      smax = 0;  // nothing left for the per-step launches below
    }
    for (int st = 0; st < smax; ++st) {
      LaunchRange ur{1, (int64_t)p.inpanel_tasks.size(), 0};
      std::vector<Int> active;
      for (Int I : block_sns)
        if (st * kStep < p.sn[I].w) active.push_back(I);
      auto bucket_of = [&](Int I) {
        return diag_bucket((int)ceil_div(std::min(kStep, p.sn[I].w - st * kStep), kSub));
      };
      constexpr int64_t kOneRound = 256;  // blocks that CUs with one workgroup each take at once
      for (const BucketGroup& g : bucket_groups(active, kOneRound, bucket_of, [](Int) { return 1; })) {
        LaunchRange pr{0, (int64_t)p.potrf_tasks.size(), 0};
        LaunchRange tr{7, (int64_t)p.trsm_tasks.size(), 0};
        for (Int I : g.items) {
          const SnInfo& si = p.sn[I];
          int nsteps = (int)ceil_div(si.w, kStep);
          int c0 = st * kStep, bs = std::min(kStep, si.w - c0);
          int64_t rows_below = si.r - c0 - bs;
          int32_t inv_off = (int32_t)(p.inv_base[I] + (int64_t)st * (kStep / kSub));
          p.potrf_tasks.push_back({I, st, inv_off, 0});
          for (int64_t rt = 0; rt < ceil_div(rows_below, kTrsmRowsWide); ++rt)
            p.trsm_tasks.push_back({I, st, (int32_t)rt, inv_off});
          p.diag_flops += (double)bs * bs * bs / 3.0 + (double)bs * bs * rows_below;
          if (st < nsteps - 1) {
            int rb = c0 + bs;  // trailing rows/cols start
            int64_t nrow = si.r - rb, ncol = si.w - rb;
            int64_t ntr = ceil_div(nrow, kTile), ntc = ceil_div(ncol, kTile);
            for (int64_t ti = 0; ti < ntr; ++ti)
              for (int64_t tj = 0; tj < ntc && tj <= ti; ++tj)
                p.inpanel_tasks.push_back({I, st, (int32_t)ti, (int32_t)tj});
            // flops of the lower-trapezoid update with k = bs
            p.inpanel_flops += (double)bs * ((double)ncol * (ncol + 1) + 2.0 * (nrow - ncol) * ncol);
          }
        }
        pr.aux = tr.aux = g.bucket;
        pr.count = (int64_t)p.potrf_tasks.size() - pr.first;
        tr.count = (int64_t)p.trsm_tasks.size() - tr.first;
        if (pr.count) p.factor_seq.push_back(pr);
        if (tr.count) p.factor_seq.push_back(tr);
      }
      ur.count = (int64_t)p.inpanel_tasks.size() - ur.first;
      if (ur.count) p.factor_seq.push_back(ur);
    }
    // Schur tasks: counted here, written on the device (schur_emit)
    LaunchRange sr{2, p.n_schur, 0};
    sr.first_w = p.n_schur_wide;
    const size_t emit_first = p.schur_emit.size();
    // A head with a long k loop (a chain's last member) is split into parts of
    // at least kPartChunks chunks, so that every resident workgroup gets
    // about four: 1,827 tiles of 60 chunks on 1,024 slots (60^3 27-point,
    // level 36) 541 us whole, 529 us in two parts.  Whole factorizations move
    // by 1% either way: with 10, 20, 40 and no parts 27-point 60^3 12.06, 12.05,
    // 12.13, 12.15 ms, 27-point 40^3 2.70, 2.73, 2.73, 2.73, 48^3 4.73, 4.73, 4.68,
    // 4.68.
    constexpr int64_t kPartChunks = 20, kSlots = 1024;
    int64_t units = 0;  // chunks of all tiles of the level
    for (Int I : sns) {
      if (head_of[I] < 0) continue;
      const SchurHead& h = p.schur_heads[head_of[I]];
      units += h.nq * schur_tiles_before(ceil_div(p.sn[I].r - p.sn[I].w, kTile), ceil_div(h.bcut, kTile));
    }
    const int64_t part_chunks = std::max(kPartChunks, units / (4 * kSlots));
    int nqmin = INT_MAX, nqmax = 0;
    for (Int I : sns) {
      const SnInfo& si = p.sn[I];
      int64_t m = si.r - si.w;
      if (m <= 0) continue;
      SchurHead& h = p.schur_heads[head_of[I]];
      h.split = (int32_t)std::min(kMaxParts, std::max<int64_t>(1, h.nq / part_chunks));
      SchurEmit e{};
      e.I = I;
      e.nt = (int32_t)ceil_div(m, kTile);
      e.ntj = (int32_t)ceil_div(h.bcut, kTile);
      e.ntw = (int32_t)ceil_div(m, 2 * kTile);
      e.ntjw = (int32_t)ceil_div(h.bcut, 2 * kTile);
      e.head = head_of[I];
      e.split = h.split;
      p.schur_entries += (int64_t)h.bcut * m - (int64_t)h.bcut * (h.bcut - 1) / 2;
      e.first[0] = p.n_schur;
      e.first[2] = p.n_schur_wide;
      p.n_schur += schur_tiles_before(e.nt, e.ntj) * e.split;
      p.n_schur_wide += schur_tiles_before(e.ntw, e.ntjw);
      nqmin = std::min(nqmin, h.nq / h.split);
      nqmax = std::max(nqmax, h.nq);
      sr.nsegmax = std::max(sr.nsegmax, h.nseg);
      p.schur_emit.push_back(e);
      // algorithmic flops stay those of the supernode's whole update, wherever
      // its parts are computed
      p.schur_flops += (double)si.w * (double)m * (double)(m + 1);
    }
    sr.count = p.n_schur - sr.first;
    sr.count_w = p.n_schur_wide - sr.first_w;
    sr.nqmin = sr.count ? nqmin : 0;
    // longest-first order: the level's supernodes by k chunks, longest first,
    // stable (a counting sort on the chunk count, a small integer), each
    // supernode's tiles in their plan order
    {
      std::vector<int64_t> cnt(nqmax + 2, 0);
      for (size_t q = emit_first; q < p.schur_emit.size(); ++q) ++cnt[nqmax - p.schur_heads[p.schur_emit[q].head].nq + 1];
      for (int i = 1; i <= nqmax + 1; ++i) cnt[i] += cnt[i - 1];
      std::vector<size_t> order(p.schur_emit.size() - emit_first);
      for (size_t q = emit_first; q < p.schur_emit.size(); ++q)
        order[cnt[nqmax - p.schur_heads[p.schur_emit[q].head].nq]++] = q;
      int64_t f1 = sr.first, f3 = sr.first_w;
      for (size_t q : order) {
        SchurEmit& e = p.schur_emit[q];
        e.first[1] = f1;
        e.first[3] = f3;
        f1 += schur_tiles_before(e.nt, e.ntj) * e.split;
        f3 += schur_tiles_before(e.ntw, e.ntjw);
      }
    }
    // longest first: the same as plan order where all tasks are as long; 64 x
    // 64 tiles: 128 x 128 ones read half the operands but fill the last round
    // of workgroups worse (60^3 27-point, whole Schur: 8.58 against 9.95 ms;
    // 80^3 LDL^T: 39.8 against 43.0 ms; ahead by 3% on three of its levels)
    sr.alt = 1;
    if (sr.count && sr.count < kSplitTarget) {
      // few output tiles: each task's k chunks are split over S workgroups
      // (partial sums meet in the atomic scatter), S <= the fewest chunks of
      // any task of the level so that no part is empty
      sr.aux = (int)std::max<int64_t>(1, std::min<int64_t>(nqmin, kSplitTarget / sr.count));
    }
    if (sr.count) p.factor_seq.push_back(sr);
    for (size_t q = level_first; q < p.factor_seq.size(); ++q) p.factor_seq[q].level = L;
  }

  // ---- solve panels and their levels ----
  std::vector<int32_t> slevel;       // per panel
  std::vector<int32_t> inv_of;       // per panel: first inverse tile
  std::vector<int32_t> child_top(ns, 0);  // per supernode: first level above its children's panels
  for (Int I = 0; I < ns; ++I) {     // children precede parents
    const SnInfo& si = p.sn[I];
    int32_t L = child_top[I];
    for (int32_t c0 = 0; c0 < si.w; c0 += kStep, ++L) {
      p.panels.push_back({si.off + (int64_t)c0 * si.r + c0, si.r, si.r - c0, std::min(kStep, si.w - c0), si.fc + c0,
                          si.lx + c0, 0});
      inv_of.push_back((int32_t)(p.inv_base[I] + c0 / kSub));
      slevel.push_back(L);
    }
    if (si.r > si.w) {
      int32_t& top = child_top[row_sup[p.lindx0[si.lx + si.w]]];
      top = std::max(top, L);
    }
  }
  const Int np = (Int)p.panels.size();
  int32_t nslevels = 0;
  for (int32_t L : slevel) nslevels = std::max(nslevels, L + 1);
  std::vector<std::vector<Int>> panels_at(nslevels);
  for (Int q = 0; q < np; ++q) panels_at[slevel[q]].push_back(q);
  auto bucket_of = [&](Int q) { return diag_bucket((int)ceil_div(p.panels[q].w, kSub)); };

  // ---- solve task lists ----
  // Per level: one diagonal task per panel, one off-diagonal task per 64-row
  // tile below the diagonal block, and for the partitioned inverse (where no
  // supernode is wider than a panel) one task per 64-row tile of the whole
  // panel.
  const bool inverse = p.max_w <= kStep;
  struct SolveGroup {
    LaunchRange diag, offd, part;
  };
  std::vector<SolveGroup> groups;  // levels bottom-up
  constexpr int64_t kManyTiles = 512;
  for (int L = 0; L < nslevels; ++L)
    for (const BucketGroup& g : bucket_groups(panels_at[L], kManyTiles, bucket_of,
                                              [&](Int q) { return ceil_div(p.panels[q].r, kTile); })) {
      SolveGroup sg{{3, (int64_t)p.sdiag_tasks.size(), 0, g.bucket, L},
                    {4, (int64_t)p.soffm_tasks.size(), 0, g.bucket, L},
                    {10, (int64_t)p.gtiles.size(), 0, g.bucket, L}};
      for (Int q : g.items) {
        const SolvePanel& sp = p.panels[q];
        p.sdiag_tasks.push_back({q, inv_of[q], 0, 0});
        for (int64_t rt = 0; rt < ceil_div(sp.r - sp.w, kTile); ++rt) p.soffm_tasks.push_back({q, (int32_t)rt, 0, 0});
        for (int64_t rt = 0; inverse && rt < ceil_div(sp.r, kTile); ++rt)
          p.gtiles.push_back({q, (int32_t)rt, inv_of[q], 0});
      }
      sg.diag.count = (int64_t)p.sdiag_tasks.size() - sg.diag.first;
      sg.offd.count = (int64_t)p.soffm_tasks.size() - sg.offd.first;
      sg.part.count = (int64_t)p.gtiles.size() - sg.part.first;
      groups.push_back(sg);
    }
  // forward: levels bottom-up, diagonal solves then off-diagonal updates;
  // backward: levels top-down, off-diagonal gathers then diagonal solves
  for (const SolveGroup& g : groups) {
    p.fwd_seq.push_back(g.diag);
    if (g.offd.count) p.fwd_seq.push_back(g.offd);
    if (inverse) p.gfwd_seq.push_back(g.part);
  }
  for (auto g = groups.rbegin(); g != groups.rend(); ++g) {
    LaunchRange d = g->diag, o = g->offd, q = g->part;
    d.kind = 6;
    o.kind = 5;
    q.kind = 11;
    if (o.count) p.bwd_seq.push_back(o);
    p.bwd_seq.push_back(d);
    if (inverse) p.gbwd_seq.push_back(q);
  }
  // preparation of the partitioned inverse: the same tiles, regrouped by the
  // bucket of their own panel (appended after the level-ordered tiles)
  for (int bk : {1, 2, 4, 6, 10}) {
    LaunchRange r{12, (int64_t)p.gtiles.size(), 0, bk, -1};
    for (Int q = 0; q < np; ++q) {
      if (!inverse || bucket_of(q) != bk) continue;
      for (int64_t rt = 0; rt < ceil_div(p.panels[q].r, kTile); ++rt)
        p.gtiles.push_back({q, (int32_t)rt, inv_of[q], 0});
    }
    r.count = (int64_t)p.gtiles.size() - r.first;
    if (r.count) p.gprep_seq.push_back(r);
  }

  // the dependency-driven solve's lists are built on demand (build_dataflow_lists)
  p.df_ok = p.max_w <= kStep;
}


DataflowLists build_dataflow_lists(const Plan& p) {
  DataflowLists L;
  if (!p.df_ok) return L;
  const Int ns = p.nsuper;
  std::vector<int32_t> row_sup(p.n);
  for (Int I = 0; I < ns; ++I)
    for (int32_t c = p.sn[I].fc; c < p.sn[I].fc + p.sn[I].w; ++c) row_sup[c] = I;

    L.dcnt0.assign(ns, 0);
    L.rcnt0.assign(ns, 0);
    std::vector<int32_t> last_seen(ns, -1);
    std::vector<int64_t> dtask(ns, 0);  // forward D task of every supernode
    int32_t stamp = 0;
    for (Int I = 0; I < ns; ++I) {
      const SnInfo& si = p.sn[I];
      const int32_t m = si.r - si.w;
      const int32_t nt = (int32_t)ceil_div(m, kTile);
      L.rcnt0[I] = nt;
      dtask[I] = (int64_t)L.fwd.size();
      L.fwd.push_back({0, I, 0, 0});
      L.fwd_end.push_back(0);
      for (int32_t rt = 0; rt < nt; ++rt) {
        const int32_t first = (int32_t)L.tgt.size();
        ++stamp;
        for (int32_t a = rt * kTile; a < std::min<int32_t>(m, (rt + 1) * kTile); ++a) {
          const int32_t T = row_sup[p.lindx0[si.lx + si.w + a]];
          if (last_seen[T] != stamp) {
            last_seen[T] = stamp;
            L.tgt.push_back(T);
            ++L.dcnt0[T];
          }
        }
        L.fwd.push_back({1, I, rt, first});
        L.fwd_end.push_back((int32_t)L.tgt.size());
      }
    }
    // backward: the same tiles in reverse postorder, waiting for the owners
    // of their rows
    for (Int I = ns - 1; I >= 0; --I) {
      for (int32_t rt = 0; rt < L.rcnt0[I]; ++rt) {
        const int64_t q = dtask[I] + 1 + rt;
        L.bwd.push_back({2, I, rt, L.fwd[q].d});
        L.bwd_end.push_back(L.fwd_end[q]);
      }
      L.bwd.push_back({3, I, 0, 0});
      L.bwd_end.push_back(0);
    }
  return L;
}

std::string validate_solve_plan(const Plan& p) {
  if (!p.df_ok) return std::string();
  const DataflowLists L = build_dataflow_lists(p);
  const Int ns = p.nsuper;
  std::vector<int32_t> dcnt = L.dcnt0, rcnt = L.rcnt0;
  std::vector<char> dflag(ns, 0), bflag(ns, 0);
  std::vector<int32_t> row_sup(p.n, -1);
  for (Int I = 0; I < ns; ++I)
    for (int32_t c = 0; c < p.sn[I].w; ++c) row_sup[p.sn[I].fc + c] = I;
  auto owners_ok = [&](const Task4& t, int32_t end) -> bool {
    const SnInfo& si = p.sn[t.b];
    const int32_t m = si.r - si.w;
    std::vector<int32_t> want;
    for (int32_t a = t.c * kTile; a < std::min<int32_t>(m, (t.c + 1) * kTile); ++a) {
      const int32_t T = row_sup[p.lindx0[si.lx + si.w + a]];
      if (std::find(want.begin(), want.end(), T) == want.end()) want.push_back(T);
    }
    std::vector<int32_t> got(L.tgt.begin() + t.d, L.tgt.begin() + end);
    std::sort(want.begin(), want.end());
    std::sort(got.begin(), got.end());
    return want == got;
  };
  for (size_t q = 0; q < L.fwd.size(); ++q) {
    const Task4& t = L.fwd[q];
    if (t.a == 0) {
      if (dcnt[t.b] != 0) return "forward D(" + std::to_string(t.b) + ") reached with pending updates";
      dflag[t.b] = 1;
    } else if (t.a == 1) {
      if (!dflag[t.b]) return "forward O(" + std::to_string(t.b) + ") before its diagonal solve";
      if (!owners_ok(t, L.fwd_end[q])) return "forward O(" + std::to_string(t.b) + ") targets";
      for (int32_t k = t.d; k < L.fwd_end[q]; ++k) --dcnt[L.tgt[k]];
    } else {
      return "bad forward task kind";
    }
  }
  for (Int I = 0; I < ns; ++I)
    if (dcnt[I] != 0 || !dflag[I]) return "forward counters not drained";
  for (size_t q = 0; q < L.bwd.size(); ++q) {
    const Task4& t = L.bwd[q];
    if (t.a == 2) {
      for (int32_t k = t.d; k < L.bwd_end[q]; ++k)
        if (!bflag[L.tgt[k]]) return "backward R(" + std::to_string(t.b) + ") before an owner is solved";
      if (!owners_ok(t, L.bwd_end[q])) return "backward R(" + std::to_string(t.b) + ") targets";
      --rcnt[t.b];
    } else if (t.a == 3) {
      if (rcnt[t.b] != 0) return "backward B(" + std::to_string(t.b) + ") reached with pending tiles";
      bflag[t.b] = 1;
    } else {
      return "bad backward task kind";
    }
  }
  for (Int I = 0; I < ns; ++I)
    if (rcnt[I] != 0 || !bflag[I]) return "backward counters not drained";
  return std::string();
}

}  // namespace spk
