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
