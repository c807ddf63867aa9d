// Host plan of the dK/dV launch: its tiling, and how its units are shared among
// the workgroups. No GPU code, so that it can be compiled and checked alone.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstring>

namespace kf {

// Key-stationary tiling shared by dkdv_kernel, the fixup and the host.
constexpr int kBNK = 128;  // keys per tile
constexpr int kBMQ = 64;   // query rows per unit

__host__ __device__ inline int dkdv_qstart(int kt, bool causal) {
  // Under the upper-left causal mask, query i sees key j iff j <= i, so no
  // query before the tile's first key (kt * 128) contributes.
  return causal ? kt * (kBNK / kBMQ) : 0;
}
__host__ __device__ inline int dkdv_nq(int kt, int nqt, bool causal) {
  const int n = nqt - dkdv_qstart(kt, causal);
  return n > 0 ? n : 0;
}
// Key tiles that hold any visible (query, key) pair: all of them, or under
// the causal mask those before ceil(nqt / 2) (dkdv_nq is zero from there).
__host__ __device__ inline int dkdv_seen_tiles(int nqt, int nkt, bool causal) {
  // dkdv_nq(kt) = nqt - 2 kt under the causal mask: zero from ceil(nqt / 2).
  const int m = causal ? (nqt + 1) / 2 : nkt;
  return m < nkt ? m : nkt;
}
// Order of the key tiles within a KV group: position pos holds tile
// dkdv_tile_at(pos). The seen tiles alternate from both ends (0, m - 1, 1,
// m - 2, ...), so that under the causal mask a long tile row is followed by
// a short one; tiles that see no query come last. With the causal triangle's
// rows, 256 - 8 kt units at config 3, each pair then costs about two
// workgroups, and the stream-K boundaries cut every pair once, in its long
// tile: at most two shares per tile and two segments per workgroup.
__host__ __device__ inline int dkdv_tile_at(int pos, int m) {
  if (pos >= m) return pos;
  return (pos & 1) ? m - 1 - (pos >> 1) : pos >> 1;
}
__host__ __device__ inline int dkdv_pos_of(int kt, int m) {
  if (kt >= m) return kt;
  return kt < (m + 1) / 2 ? 2 * kt : 2 * (m - 1 - kt) + 1;
}
// Stream-K shares: workgroup w owns units [start[w], start[w + 1]). The host
// places the boundaries by cost rather than by unit count: every key-tile row
// a workgroup enters (a "segment") costs about kSegmentCost units on top of
// its units (loading the keys' K/V rows, filling the LDS ring, flushing the
// accumulators), and the short rows of the causal triangle's far end would
// otherwise pile many segments onto the last workgroups.
constexpr int kMaxDkdvWG = 512;
struct DkdvSplit {
  int start[kMaxDkdvWG + 1];
};
// Stream-K bookkeeping from the host: total units and the workgroup count.
inline int64_t dkdv_total_units(int ngroups, int G, int nqt, int nkt, bool causal) {
  int64_t U = 0;
  for (int kt = 0; kt < nkt; ++kt) U += (int64_t)ngroups * G * dkdv_nq(kt, nqt, causal);
  return U;
}

// Cost-weighted stream-K boundaries (see DkdvSplit). A segment start costs
// kSegmentCost8 / 8 units: on the MI355X at config 3 a sweep of the weight
// put the shortest launch at 4.5 to 6 units, and after a segment's loads
// came to overlap the previous segment's flush, 3 and 4 units were still
// 1-2% slower than 5. With the long-short tile order and cuts charged to the
// share that makes them, 3, 7 and 10 units were 0.4-1.2% slower than 5.
constexpr int kSegmentCost8 = 40;
// Cut tile rows also cost their fp32 partials, stored by the dK/dV launch and
// summed by a fixup launch of its own. Shares of whole consecutive rows cost
// neither, and are taken when that leaves the longest share no more than this
// (8ths of a unit, by head-dim tile / 32 - 1) above an even one. Measured, us
// for dK/dV and fixup, cut -> whole rows: B=4 H=12 S=1000 D=64 causal 41.4 ->
// 27.9 (longest share 26.1 units against 21.0), B=4 H=16 S=512 D=128 causal
// 39.4 -> 24.1 (13.0, 10.0), B=4 H=12 S=2048 D=64 causal 90.7 -> 76.7 (81.2,
// 66.0), B=1 H=8 S=2000 D=128 52.3 -> 64.3 (37.4, 18.5). Over 19 shapes the cuts
// cost 11 to 31 units at D = 128 and 14 to 32 at D = 64.
constexpr int kFixupCost8[4] = {112, 112, 104, 88};
constexpr int kMaxWholeRows = 1024;
// Places the boundaries of nwg shares and returns the number of tile rows that
// one cuts (shared tiles). `fixup8`: what cuts cost besides their segment
// starts (kFixupCost8).
inline int dkdv_split(DkdvSplit& sp, int ngroups, int G, int nqt, int nkt, bool causal, int nwg, int fixup8) {
  int64_t rows_cost = 0, all_units = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    const int64_t units = (int64_t)G * dkdv_nq(kt, nqt, causal);
    if (units) rows_cost += (int64_t)ngroups * (8 * units + kSegmentCost8);
    all_units += (int64_t)ngroups * units;
  }
  const int mseen = dkdv_seen_tiles(nqt, nkt, causal);
  // Boundaries at equal cost over the rows in unit order (KV group outer,
  // key tiles in dkdv_tile_at order inner). A boundary inside a tile row
  // starts one more segment (the next share enters the row part-way); with
  // cut_cost = kSegmentCost8 that segment start is charged to the share
  // that makes it, and `total` must then include the cuts. Returns the
  // number of cuts; `shared` counts the rows cut at least once.
  auto place = [&](DkdvSplit& out, int64_t total, int64_t cut_cost, int& shared_rows) {
    int w = 1, cuts = 0;
    int64_t base = 0, cost = 0;
    shared_rows = 0;
    out.start[0] = 0;
    for (int g = 0; g < ngroups && w < nwg; ++g) {
      for (int pos = 0; pos < nkt && w < nwg; ++pos) {
        const int64_t units = (int64_t)G * dkdv_nq(dkdv_tile_at(pos, mseen), nqt, causal);
        if (!units) continue;
        const int64_t row_cost = 8 * units + kSegmentCost8;
        int row_cuts = 0;
        int64_t prev = 0;  // boundaries never move backwards
        while (w < nwg) {
          const int64_t target = (total * w + nwg - 1) / nwg;
          if (target > cost + row_cost + row_cuts * cut_cost) break;
          int64_t into = (target - cost - kSegmentCost8 - row_cuts * cut_cost + 7) / 8;
          into = into < prev ? prev : (into > units ? units : into);
          prev = into;
          out.start[w++] = (int)(base + into);
          if (into > 0 && into < units) ++row_cuts;
        }
        shared_rows += row_cuts > 0 ? 1 : 0;
        cuts += row_cuts;
        cost += row_cost + row_cuts * cut_cost;
        base += units;
      }
    }
    while (w < nwg) out.start[w++] = (int)all_units;
    out.start[nwg] = (int)all_units;
    return cuts;
  };
  // The plain placement first; then the cut-charged one, started from the
  // plain cut count and kept when it reaches a fixed point (at config 3
  // at once: the long tile of each pair is cut once, half a segment later).
  int shared = 0;
  int cuts = place(sp, rows_cost, 0, shared);
  DkdvSplit refined;
  for (int pass = 0; pass < 3; ++pass) {
    int rshared = 0;
    const int rcuts = place(refined, rows_cost + (int64_t)cuts * kSegmentCost8, kSegmentCost8, rshared);
    if (rcuts == cuts) {
      sp = refined;
      shared = rshared;
      break;
    }
    cuts = rcuts;
  }
  // Shares of whole rows, the longest of them as short as consecutive rows
  // allow: a bound on a share's cost is feasible if filling shares up to it
  // needs no more than nwg of them.
  const int rows = ngroups * mseen;
  if (shared > 0 && mseen == nkt && rows <= kMaxWholeRows) {
    auto pack = [&](DkdvSplit& out, int64_t bound) {
      int w = 0;
      int64_t base = 0, in = 0;
      out.start[0] = 0;
      for (int g = 0; g < ngroups; ++g)
        for (int pos = 0; pos < nkt; ++pos) {
          const int64_t units = (int64_t)G * dkdv_nq(dkdv_tile_at(pos, mseen), nqt, causal);
          const int64_t c = 8 * units + kSegmentCost8;
          if (c > bound) return false;
          if (in + c > bound) {
            if (++w == nwg) return false;
            out.start[w] = (int)base;
            in = 0;
          }
          in += c;
          base += units;
        }
      while (++w <= nwg) out.start[w] = (int)all_units;
      return true;
    };
    int64_t lo = rows_cost / nwg, hi = lo + fixup8;
    DkdvSplit whole;
    if (pack(whole, hi)) {
      shared = 0;
      while (hi - lo > 8) {
        sp = whole;
        const int64_t mid = (lo + hi) / 2;
        if (pack(whole, mid)) hi = mid; else { lo = mid; whole = sp; }
      }
      sp = whole;
    }
  }
  return shared;
}

// Shares of a problem: one per CU, or fewer where they would hold less than
// `least` units each: a share then costs more in its segment starts and in the
// fp32 partials that the fixup sums (one per share and row it touches) than its
// units take. A multiple of 8, for the XCD mapping, and not below one share per
// tile row: whole rows cost no partials.
inline int dkdv_share_count(int cus, int64_t units, int64_t rows, int least) {
  const int64_t n = ((units / least > rows ? units / least : rows) + 7) / 8 * 8;
  return n < 8 ? (cus < 8 ? cus : 8) : n < cus ? (int)n : cus;
}

// Least units per share. With 8 there are fewer partials, which pays where the
// rows stay whole or each is cut into at least kManyShares; rows cut into few
// long shares leave the launch waiting for the longest, and take 4.
// Measured over 300 shapes, us for dK/dV and fixup, one share per CU / 8 units
// / 4: few shares a row, B=3 Hq=16 Hkv=8 S=533 D=128 causal 35.4 / 40.5 / 35.9,
// B=1 Hq=16 Hkv=4 S=433 D=64 causal 4 ahead of 8 by 26%; many, B=1 Hq=8 Hkv=1
// 1393 x 467 D=72 98.9 / 34.0 / 39.5, B=1 Hq=4 Hkv=1 S=1739 D=80 causal 64.3 /
// 34.5 / 36.9; whole rows, B=4 H=4 S=872 D=112 causal 34.0 / 28.0 / 35.6.
// Geometric mean against one share per CU without whole rows: always 8 0.836,
// always 4 0.833, this rule 0.825, the worst shape 1.16, 1.05 and 1.04; over 500
// further shapes always 8 0.828 and 1.17, this rule 0.821 and 1.07.
constexpr int kShareUnits = 8, kCutShareUnits = 4, kManyShares = 3;

struct DkdvPlan {
  DkdvSplit split;
  int nwg;     // shares: workgroups of the launch
  int shared;  // tile rows in more than one share
};

// The plan of a problem on `cus` CUs. Kept per thread for the last problem: a
// training step plans its launches and their fixup alike, layer after layer.
inline const DkdvPlan& dkdv_plan(int ngroups, int G, int nqt, int nkt, bool causal, int cus, int fixup8) {
  struct Key {
    int ngroups, G, nqt, nkt, causal, cus, fixup8;
  };
  thread_local Key last{-1, 0, 0, 0, 0, 0, 0};
  thread_local DkdvPlan plan;
  const Key k{ngroups, G, nqt, nkt, causal ? 1 : 0, cus, fixup8};
  if (memcmp(&k, &last, sizeof k) == 0) return plan;
  const int64_t units = dkdv_total_units(ngroups, G, nqt, nkt, causal);
  const int64_t rows = (int64_t)ngroups * dkdv_seen_tiles(nqt, nkt, causal);
  plan.nwg = dkdv_share_count(cus, units, rows, kShareUnits);
  plan.shared = dkdv_split(plan.split, ngroups, G, nqt, nkt, causal, plan.nwg, fixup8);
  if (plan.shared > 0 && plan.nwg < kManyShares * rows) {
    const int nwg = dkdv_share_count(cus, units, rows, kCutShareUnits);
    if (nwg > plan.nwg) {
      plan.nwg = nwg;
      plan.shared = dkdv_split(plan.split, ngroups, G, nqt, nkt, causal, nwg, fixup8);
    }
  }
  last = k;
  return plan;
}

}  // namespace kf
