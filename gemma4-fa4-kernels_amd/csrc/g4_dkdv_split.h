// Split dK/dV launch: the (query, key tile) steps of a problem that does not
// fill the GPU with whole key tiles, cut into equal runs over its CUs.
//
// The dK/dV kernels are key-tile major: one workgroup per key tile (or pair of
// tiles) and KV head, the query rows walked one after the other.  One
// 1000-token global sequence has 16 tiles x 4 KV heads, so 32 workgroups of
// pairs walk 272 steps each while 224 CUs idle.  Here the steps of every tile
// are laid end to end (KV head, sequence, key tile, then the tile's own step
// order), each tile preceded by kTileCost steps' worth of set-up, and
// workgroup g of n takes the g-th equal part.  A tile that lies whole inside
// one part is written as bf16 as before; the parts of a cut tile go to the
// workspace as fp32 (two slots per workgroup: the end of a tile begun in an
// earlier part, the start of one that a later part goes on with), and a
// second launch adds them in part order.  The cuts follow from the problem
// alone, so results repeat bitwise.
#pragma once

#include <algorithm>

#include "g4_kernels.h"

namespace g4 {

// Work of a key tile beyond its steps (operand fragments, first copies, the
// epilogue), in steps.
constexpr int kSplitTileCost = 5;
// A cut this close (steps) to a tile's edge is moved onto the edge.
constexpr int kSplitMinSteps = 2;
// Parts of fewer steps than this are not worth a workgroup and its partials.
constexpr int kSplitMinPart = 16;

// A step here against one of the launch by whole tiles, and the second launch
// with the partials' traffic in steps (see dkdv_split_bytes).
constexpr double kSplitStep = 1.3;
constexpr int kSplitSumSteps = 7;

// Sum over t in [0, kt) of max(0, m t + a), m even.
inline int split_ramp(int kt, int m, int a) {
  const int t0 = a > 0 ? 0 : (-a) / m + 1;
  const int n = kt - t0;
  return n <= 0 ? 0 : m / 2 * n * (t0 + kt - 1) + a * n;
}

// Steps of one sequence's key tiles (bn keys each) without vision spans, for
// the host's choice of the launch: tile t is reached by the 32-query rows
// [max(0, m t - e), min(nrows, m t + h0)), m = bn / 32.
struct SplitSeq {
  int nt, nrows, m, e, h0, grp;
  bool windowed;
  void init(int lq, int lk, int bn, int window, int grp_) {
    const int off = lk - lq;
    grp = grp_;
    nt = (lk + bn - 1) / bn;
    nrows = lq > 0 ? (lq + 31) / 32 : 0;
    m = bn / 32;
    e = -((-off) >> 5);                        // ceil(off / 32)
    windowed = window > 0;
    h0 = (bn + window - 1 - off + 31) >> 5;    // ceil((bn - 1 + window - off) / 32)
  }
  // Cost of the tiles [0, kt).
  int before(int kt) const {
    if (nrows == 0) return kt * kSplitTileCost;
    int rows = windowed ? split_ramp(kt, m, h0) - split_ramp(kt, m, h0 - nrows) : kt * nrows;
    rows -= split_ramp(kt, m, -e);
    return rows * grp + kt * kSplitTileCost;
  }
};

// Head dim 256: the two launches' times from their schedules.  An average over
// the CUs does not tell them apart (packed sequences of one length, split /
// whole: 8 x 300 tokens 0.78, 12 x 300 1.21, 16 x 300 0.93): which items share a
// CU, and how many tiles a part touches, follow from the counts, so both
// schedules are walked.  The sequences are the longest first, then the others at
// their mean length (their own are on the device); with vision IDs every
// sequence is taken to hold one image of at most 700 tokens per 4000, which
// lengthens the tiles it lies in.  Both against 138 measured problems of 2 to 64
// sequences: 5% and 6%.
struct SplitTiles256 {
  static constexpr int kMax = 4 * kSplitParts;  // items of a problem that may split
  int steps[2][kMax];  // of a key tile of the longest sequence, of another one
  int nt[2];           // their key tiles
  int nseq, hkv;

  void fill(int which, int lq, int lk, int window, int grp, bool images) {
    const int off = lk - lq, nrows = lq > 0 ? (lq + 31) / 32 : 0;
    nt[which] = std::min((lk + 127) / 128, kMax);
    for (int t = 0; t < nt[which]; ++t) {
      int lo = std::max(128 * t - off, 0) >> 5;
      const int last = std::min(128 * t + 127, lk - 1);  // key
      const int hi = window > 0 ? std::min(nrows, ((last + window - 1 - off) >> 5) + 1) : nrows;
      if (images) {
        const int size = std::min(lk / 2, 700);
        for (int at = lk / 4; at + lk / 2 <= lk && at <= last; at += 4000)
          if (at + size > 128 * t) lo = std::min(lo, std::max(at - off, 0) >> 5);
      }
      steps[which][t] = std::max(hi - lo, 0) * grp;
    }
  }
  int tile_steps(int s, int t) const { return steps[s > 0][t]; }

  // Whole tiles, one workgroup each.  An XCD takes a run of the items and the
  // hardware deals it to four shader engines of eight CUs in turn, in order: an
  // item waits for a CU of its engine, and the later ones for it.
  double whole() const {
    const int per_kvh = nseq * nt[0], items = per_kvh * hkv;
    double worst = 0;
    for (int x = 0; x < (hkv % 8 == 0 ? 1 : 8); ++x) {
      const int lo = x * (items / 8) + std::min(x, items % 8);
      const int hi = lo + items / 8 + (x < items % 8 ? 1 : 0);
      double busy[4][8] = {}, now = 0;
      for (int i = lo; i < hi; ++i) {
        const int rank = i % per_kvh, s = rank / nt[0], r = rank % nt[0];
        const int t = r & 1 ? r >> 1 : nt[0] - 1 - (r >> 1);  // zigzag
        double* cu = std::min_element(busy[(i - lo) & 3], busy[(i - lo) & 3] + 8);
        now = std::max(now, *cu);
        *cu = now + (t < nt[s > 0] ? tile_steps(s, t) + 7 : 0.3);
        worst = std::max(worst, *cu);
      }
    }
    return 1.88 * worst - 5;  // us
  }
  // Equal parts: a tile that a part touches costs it five steps, whether it runs
  // all of it or not.
  double split() const {
    int cost = 0;
    for (int s = 0; s < nseq; ++s)
      for (int t = 0; t < nt[s > 0]; ++t) cost += tile_steps(s, t) + kSplitTileCost;
    if (cost == 0) return 0;
    const int64_t total = (int64_t)cost * hkv;
    const int n = (int)std::min<int64_t>(kSplitParts, std::max<int64_t>(total / kSplitMinPart, 1));
    const int walk = n % hkv == 0 ? n / hkv : n;  // (then the KV heads' parts are alike)
    int s = 0, t = 0, worst = 0;
    int64_t at = 0;  // where tile (s, t) begins
    while (nt[s > 0] == 0) ++s;
    for (int g = 0; g < walk; ++g) {
      const int64_t from = total * g / n, to = total * (g + 1) / n;
      int sum = 0;
      for (;;) {
        const int c = tile_steps(s, t);
        const int64_t end = at + c + kSplitTileCost;
        int lo = (int)std::max<int64_t>(from - at - kSplitTileCost, 0);
        int hi = (int)std::min<int64_t>(std::max<int64_t>(to - at - kSplitTileCost, 0), c);
        if (lo < kSplitMinSteps) lo = 0;
        if (hi < kSplitMinSteps && to < end) hi = 0;
        if (lo > 0 && c - lo < kSplitMinSteps) lo = c;
        if (c - hi < kSplitMinSteps) hi = c;
        if (hi > lo || (lo == 0 && hi == c)) sum += hi - lo + kSplitTileCost;
        if (to < end) break;
        at = end;
        ++t;
        while (t >= nt[s > 0]) {
          t = 0;
          if (++s == nseq) s = 0;  // the next KV head
        }
        if (at >= to) break;
      }
      worst = std::max(worst, sum);
    }
    return 2.48 * worst + 10;  // us
  }
};

// Where a part begins: unit = KV head * tiles + index of the key tile in the
// sequences' order (kvh, s, kt), after num of its den steps.  A cut at or past
// the last part is the end of the problem.
struct SplitCut {
  int unit, num, den, parts;
  int kvh, s, kt, pad;
};

// Workspace: two slots of a partial tile per part, then the cuts.
constexpr size_t kDkdvSplitBytes =
    2 * (size_t)kSplitParts * kSplitSlotFloats * 4 +
    ((kSplitParts + 1) * sizeof(SplitCut) + 255) / 256 * 256;

// Most key tiles of a split problem: four items per CU, an item holding up to
// two of them.
constexpr int kSplitMaxTiles = 2 * 4 * kSplitParts;

// LDS of split_cuts.
struct SplitScratch {
  int cost[kSplitMaxTiles + 1];  // inclusive prefix, from cost[0] = 0
  int seq[65];                   // packed: first tile of each sequence
  int wave[8];
};

// The cuts g and g + 1, by all kNT threads of a workgroup (the same values in
// every workgroup, so neighbours agree).  A tile's steps are exact: the query
// range of key_tile_query_range, with the tile's first key's span start for
// its vision spans (a span that begins inside the tile starts no earlier than
// the tile; the query reach used when an ID repeats does not decrease from key
// to key).
template <int kNT>
__device__ inline void split_cuts(const BwdParams& a, int bn, int g, SplitScratch G4_LDS* sc,
                                  SplitCut& from, SplitCut& to) {
  const g4_problem& p = a.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool packed = p.cu_seqlens_q != nullptr;
  const bool vis = p.vision_ids != nullptr && p.bidirectional_vision;
  const int hkv = p.num_kv_heads, grp = p.num_q_heads / hkv;
  const int nt0 = (p.seqlen_k + bn - 1) / bn;  // fixed: every sequence's tiles
  auto scan = [&](int x) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    return x;
  };
  if (packed && tid < 64) {
    const int n = lane < p.num_seqs
                      ? (p.cu_seqlens_k[lane + 1] - p.cu_seqlens_k[lane] + bn - 1) / bn
                      : 0;
    sc->seq[lane + 1] = scan(n);
    if (lane == 0) sc->seq[0] = 0;
  }
  __syncthreads();
  const int tiles = min(packed ? sc->seq[p.num_seqs] : p.num_seqs * nt0, kSplitMaxTiles);
  auto locate = [&](int t, int& s, int& kt) {
    if (!packed) {
      s = t / nt0;
      kt = t - s * nt0;
      return;
    }
    s = 0;  // the last sequence whose first tile is at most t (empty ones before it)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
      if (s + o < p.num_seqs && sc->seq[s + o] <= t) s += o;
    kt = t - sc->seq[s];
  };
  // Each thread's run of tiles, then a scan over the threads.
  const int per = (tiles + kNT - 1) / kNT;
  int sum = 0;
  for (int i = 0; i < per; ++i) {
    const int t = tid * per + i;
    if (t >= tiles) break;
    int s, kt;
    locate(t, s, kt);
    const Seq sq = resolve_seq(p, s);
    const int j0 = kt * bn, off = sq.lk - sq.lq;
    int lo, hi;
    key_tile_query_range(j0, min(j0 + bn, sq.lk) - 1, sq.lq, off, p.window,
                         vis ? a.span_lo[sq.ktok + j0] : 0x7fffffff, lo, hi);
    const int rows = hi > lo ? (hi + 31) / 32 - lo / 32 : 0;
    sum += rows * grp + kSplitTileCost;
    sc->cost[t + 1] = sum;
  }
  int incl = scan(sum);
  if (lane == 63) sc->wave[wave] = incl;
  __syncthreads();
  incl -= sum;
  for (int w = 0; w < wave; ++w) incl += sc->wave[w];
  for (int i = 0; i < per; ++i) {
    const int t = tid * per + i;
    if (t >= tiles) break;
    sc->cost[t + 1] += incl;
  }
  if (tid == 0) sc->cost[0] = 0;
  __syncthreads();
  const int cost = sc->cost[tiles], total = cost * hkv;
  const int n = min(kSplitParts, max(total / kSplitMinPart, 1));
  auto cut = [&](int at) {
    SplitCut c{hkv * tiles, 0, 1, n, hkv, 0, 0, 0};
    if (at < n && cost > 0) {
      const int pos = (int)((int64_t)total * at / n);
      c.kvh = pos / cost;
      const int rem = pos - c.kvh * cost;
      int lo = 0, hi = tiles;  // cost[lo] <= rem < cost[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (sc->cost[mid] <= rem)
          lo = mid;
        else
          hi = mid;
      }
      c.den = sc->cost[lo + 1] - sc->cost[lo] - kSplitTileCost;
      c.num = rem - sc->cost[lo] - kSplitTileCost;
      if (c.num < kSplitMinSteps) c.num = 0;
      if (c.num > 0 && c.den - c.num < kSplitMinSteps) {
        c.num = 0;
        if (++lo == tiles) {
          lo = 0;
          ++c.kvh;
        }
      }
      c.unit = c.kvh * tiles + lo;
      locate(lo, c.s, c.kt);
    }
    c = {__builtin_amdgcn_readfirstlane(c.unit), __builtin_amdgcn_readfirstlane(c.num),
         __builtin_amdgcn_readfirstlane(c.den), __builtin_amdgcn_readfirstlane(c.parts),
         __builtin_amdgcn_readfirstlane(c.kvh), __builtin_amdgcn_readfirstlane(c.s),
         __builtin_amdgcn_readfirstlane(c.kt), 0};
    return c;
  };
  from = cut(g);
  to = cut(g + 1);
}

// Step of a tile of nsteps steps at a cut: num, as nsteps is den.  (Taken as a
// share, so that the parts of a tile would meet whatever its nsteps.)
__device__ __forceinline__ int split_step(const SplitCut& b, int nsteps) {
  return (int)((int64_t)b.num * nsteps / (b.den > 0 ? b.den : 1));
}

}  // namespace g4
