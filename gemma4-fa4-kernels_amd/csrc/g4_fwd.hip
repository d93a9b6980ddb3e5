// Forward attention kernel for gfx950: O = softmax(Q K^T + mask) V, fp32 LSE.
//
// One workgroup owns BM = 32 * NQG queries of one query head and walks the key
// tiles its mask-aware range admits (query_tile_key_range).  Each wave owns
// 32 queries and a DH = D / DSPLIT slice of the head dimension:
//   S^T (keys x queries) = K Q^T on MFMA with the query fragments in VGPRs and
//   K read from LDS; with DSPLIT = 2 the two d-slices of a query group
//   exchange their partial S^T through LDS and add them.  Because lanes own
//   queries, the softmax row max / sum are register reductions plus one
//   cross-half shuffle.  P is rounded to bf16 and fed straight from the
//   accumulator registers as the B operand of O^T += V^T P^T, with V^T read
//   from the natural-layout V tile by transposing LDS reads.
// K and V tiles are copied global -> LDS asynchronously (one 16-byte chunk per
// lane) one tile ahead of the compute.
#include <algorithm>

#include "g4_kernels.h"

namespace g4 {

template <int D, int BN, int DSPLIT, int NQG, bool VDOUBLE>
struct FwdCfg {
  static constexpr int kNW = NQG * DSPLIT;
  static constexpr int kNT = kNW * 64;
  static constexpr int kBM = NQG * 32;
  static constexpr int kDH = D / DSPLIT;
  static constexpr int kCPR = D / 8;  // 16-byte chunks per row
  static constexpr int kTileBytes = BN * D * 2;
  static constexpr int kLoadsPerWave = BN * kCPR / (64 * kNW);
  static constexpr int kKB = BN / 32;  // 32-key blocks per tile
  static constexpr int kXBytes = DSPLIT > 1 ? kNW * kKB * 4096 : 0;
  static constexpr int kVBufs = VDOUBLE ? 2 : 1;
  static constexpr int kLdsK = 0;
  static constexpr int kLdsV = kLdsK + 2 * kTileBytes;
  static constexpr int kLdsX = kLdsV + kVBufs * kTileBytes;
  static constexpr int kLdsMeta = kLdsX + kXBytes;  // [buf][vid x 64 | doc x 64] int32
  static constexpr int kLdsRed = kLdsMeta + 2 * 512;
  static constexpr int kLdsBytes = kLdsRed + 16 * 4;
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
  static_assert(kDH % 128 == 0, "head-dim slice must be a multiple of 128");
};

// Async copy of the vision / document IDs of keys [j0, j0 + 64) of a sequence
// (clamped to its last key; keys past the end are masked by index).
__device__ __forceinline__ void issue_meta(const g4_problem& p, const Seq& sq, int j0,
                                           char G4_LDS* dst, int lane, bool vid, bool doc) {
  // uniform base at the tile's first (clamped) key, small per-lane offsets
  const int j0c = min(j0, sq.lk - 1);
  const int64_t base = sq.ktok + j0c;
  const uint32_t off = (uint32_t)(min(j0 + lane, sq.lk - 1) - j0c) * 4u;
  if (vid) b2l4(p.vision_ids + base, off, dst);
  if (doc) b2l4(p.document_ids + base, off, dst + 256);
}

// Largest score excess (log2 units) over a row's running maximum that the
// online softmax absorbs without rescaling the O accumulators.
constexpr float kRescaleLog2 = 8.0f;

// META: key metadata kinds compiled in (bit 0 vision IDs, bit 1 document IDs).
// KS: wave groups that share the key tiles, each taking every KS-th one.
template <int D, int BN, int DSPLIT, int NQG, bool VDOUBLE, int META, int OCC = 1, int KS = 1>
struct FwdKernel {
  using C = FwdCfg<D, BN, DSPLIT, NQG, VDOUBLE>;
  static constexpr int kNB = C::kDH / 32;  // 32-wide head-dim blocks per wave
  static constexpr int kNC = C::kDH / 16;  // 16-deep head-dim steps per wave

  char G4_LDS* smem;
  const g4_problem* p;
  Seq sq;
  int tid, lane, wave, dh, h32;
  int my_a, my_vid, my_doc;
  bool has_vid, has_doc, has_meta;
  int a0;
  const __bf16* kbase;
  const __bf16* vbase;
  int64_t kstride, vstride;
  RowReader<C::kCPR> krd;
  // Head dim 512 keeps the compiler's wait before the P.V reads: with it the
  // 8192-token causal forward measured 2.81 ms, without it 2.91 ms.
  TrReader<C::kCPR, (D != 512)> vrd;
  TileCopier<C::kCPR, BN, C::kNW, (OCC * KS > 1)> kcp, vcp;
  bf16x8 qf[kNC];
  f32x16 o_acc[kNB];
  float m_run, l_run;

  __device__ __forceinline__ void issue_k(int row0, int buf) {
    char G4_LDS* dst = smem + C::kLdsK + buf * C::kTileBytes;
    if (row0 + BN <= sq.lk)
      kcp.issue(kbase + row0 * kstride, dst);
    else
      kcp.issue_clamped(kbase + row0 * kstride, kstride, sq.lk - row0, dst, wave, lane);
  }
  __device__ __forceinline__ void issue_v(int row0, int buf) {
    char G4_LDS* dst = smem + C::kLdsV + buf * C::kTileBytes;
    if (row0 + BN <= sq.lk)
      vcp.issue(vbase + row0 * vstride, dst);
    else
      vcp.issue_clamped(vbase + row0 * vstride, vstride, sq.lk - row0, dst, wave, lane);
  }

  template <int KB, int CP>
  __device__ __forceinline__ void s_step(const char G4_LDS* kt, f32x16& acc) const {
    if constexpr (CP < kNC) {
      // slice dh starts at chunk dh * kDH / 8 (a multiple of 16)
      bf16x8 kf = krd.template read<KB * 32, 0, CP>(kt);
      acc = mfma32(kf, qf[CP], acc);
      s_step<KB, CP + 1>(kt, acc);
    }
  }

  template <int KB, int HK, int B>
  __device__ __forceinline__ void pv_step(const char G4_LDS* vt, const bf16x8& pb) {
    if constexpr (B < kNB) {
      bf16x8 vf = vrd.template read<KB * 32 + 16 * HK, 0, B>(vt);
      o_acc[B] = mfma32(vf, pb, o_acc[B]);
      pv_step<KB, HK, B + 1>(vt, pb);
    }
  }

  // Branch-free Gemma predicate on the lane's 16 * kKB scores (keys kb0 + ...).
  // Causal part: lo_w <= j <= min(a, Sk - 1); vision part: same non-negative
  // block, j >= lo_w, j < Sk; document part: equal IDs.
  __device__ __forceinline__ void apply_mask(int cur, f32x16 (&sacc)[C::kKB], int kb0) const {
    const int lo_w = p->window > 0 ? my_a - p->window + 1 : -0x40000000;
    const int hi_c = min(my_a, sq.lk - 1);
    const int* km = (const int*)(smem + C::kLdsMeta + cur * 512);
#pragma unroll
    for (int kb = 0; kb < C::kKB; ++kb)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int jl0 = kb * 32 + 8 * r4 + 4 * h32;
        i32x4 vk = {-1, -1, -1, -1}, dk = {0, 0, 0, 0};
        if (has_meta) {
          vk = *(const i32x4*)(km + jl0);
          dk = *(const i32x4*)(km + 64 + jl0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = kb0 + jl0 + e;
          const bool in_w = j >= lo_w;
          const bool causal = in_w & (j <= hi_c);
          const bool vis = has_vid & (my_vid >= 0) & (vk[e] == my_vid) & in_w & (j < sq.lk);
          const bool doc_ok = !has_doc | (dk[e] == my_doc);
          const bool ok = (causal | vis) & doc_ok;
          sacc[kb][r4 * 4 + e] = ok ? sacc[kb][r4 * 4 + e] : kNegInf;
        }
      }
  }

  // AHEAD (double-buffered V, no key metadata): K runs two tiles ahead
  // instead of one; K(it + 2) is issued into this step's K buffer once every
  // wave is done reading it, so about two tiles of copies stay in flight (the
  // split-key forward, whose steps are short next to a tile's fetch).  The
  // caller issues K(0), V(0) and K(1) first.
  template <bool AHEAD = false>
  __device__ __forceinline__ void step(int cur, int it, int ntiles, int t_first) {
    static_assert(!AHEAD || (VDOUBLE && META == 0 && KS == 1), "K-ahead steps");
    const int kb0 = (t_first + it * KS) * BN;
    // This wave's copies of K (and, double-buffered, V) for this tile have
    // landed; the barrier publishes every wave's copies and ends all reads of
    // the buffers refilled below.  (AHEAD: K(it + 1), issued last, may still
    // be in flight.)
    if constexpr (AHEAD) {
      if (it + 1 < ntiles)
        vm_wait<C::kLoadsPerWave>();
      else
        vm_wait<0>();
    } else if constexpr (VDOUBLE) {
      vm_wait<0>();
    } else {
      vm_wait<C::kLoadsPerWave>();
    }
    barrier_lds();
    if constexpr (AHEAD) {
      if (it + 1 < ntiles) issue_v(kb0 + BN, cur ^ 1);
    } else if (it + 1 < ntiles) {
      issue_k(kb0 + KS * BN, cur ^ 1);
      if (has_meta && wave == 0) issue_meta(*p, sq, kb0 + KS * BN, smem + C::kLdsMeta + (cur ^ 1) * 512, lane, has_vid, has_doc);
      if constexpr (VDOUBLE) issue_v(kb0 + KS * BN, cur ^ 1);
    }

    // S^T partial over this wave's head-dim slice.
    f32x16 sacc[C::kKB];
    const char G4_LDS* kt = smem + C::kLdsK + cur * C::kTileBytes;
    __builtin_amdgcn_sched_barrier(0);
    mfma_prio_begin();
    __builtin_amdgcn_sched_barrier(0);
    sacc[0] = f32x16{};
    s_step<0, 0>(kt, sacc[0]);
    if constexpr (C::kKB > 1) {
      sacc[1] = f32x16{};
      s_step<1, 0>(kt, sacc[1]);
    }
    mfma_pipeline_hint<C::kKB * kNC, 3, 1>();

    __builtin_amdgcn_sched_barrier(0);
    mfma_prio_end();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (DSPLIT > 1) {
      // Publish the partial, then add the partner slice's partial.
      char G4_LDS* xb = smem + C::kLdsX;
#pragma unroll
      for (int kb = 0; kb < C::kKB; ++kb)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          f32x4 v = {sacc[kb][q4 * 4], sacc[kb][q4 * 4 + 1], sacc[kb][q4 * 4 + 2],
                     sacc[kb][q4 * 4 + 3]};
          *(f32x4 G4_LDS*)(xb + (((wave * C::kKB + kb) * 4 + q4) * 64 + lane) * 16) = v;
        }
      // Single V buffer: this tile's V copies were issued after the previous
      // PV phase, before the K copies of the next tile.
      if constexpr (!VDOUBLE) vm_wait<C::kLoadsPerWave>();
      barrier_lds();
      const int pw = wave ^ 1;
#pragma unroll
      for (int kb = 0; kb < C::kKB; ++kb)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          f32x4 v =
              *(const f32x4 G4_LDS*)(xb + (((pw * C::kKB + kb) * 4 + q4) * 64 + lane) * 16);
          // add in slice order so both slices hold bit-identical scores
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float mine = sacc[kb][q4 * 4 + e];
            sacc[kb][q4 * 4 + e] = dh == 0 ? mine + v[e] : v[e] + mine;
          }
        }
    } else if constexpr (!VDOUBLE) {
      vm_wait<C::kLoadsPerWave>();
      barrier_lds();
    }
    if constexpr (AHEAD) {
      // every wave is done reading K(it): after the partial exchange's
      // barrier, or with one wave, once its own S chain has its operands
      if (it + 2 < ntiles) issue_k(kb0 + 2 * BN, cur);
    }

    // Mask (only on tiles the mask does not fully admit), then online softmax
    // in the log2 domain (softmax scale is 1.0; log2 e is folded into the
    // exponent's FMA, and the row maximum is scaled once: rounding is
    // monotonic, so max(s) * log2 e rounds to the maximum of the scaled scores).
    const bool full = !has_doc && (kb0 + BN <= sq.lk) && (kb0 + BN - 1 <= a0) &&
                      (p->window <= 0 || kb0 > a0 + C::kBM - 1 - p->window);
    if (!full) {
      __builtin_amdgcn_sched_barrier(0);
      apply_mask(cur, sacc, kb0);
      __builtin_amdgcn_sched_barrier(0);
    }
    float mx = kNegInf;
#pragma unroll
    for (int kb = 0; kb < C::kKB; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sacc[kb][r]);
    mx = fmaxf(mx, wave_xor32(mx)) * kLog2e;
    // The running maximum only moves when a row's scores exceed it by more
    // than kRescaleLog2 (P <= 2^kRescaleLog2 meanwhile, exact in fp32 and in
    // bf16 range), so the O accumulators are rescaled rarely after the first
    // admitted tile instead of on most tiles.
    const float m_new = mx > m_run + kRescaleLog2 ? mx : m_run;
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float rs = 0.f;
    bf16x8 pb[C::kKB][2];
#pragma unroll
    for (int kb = 0; kb < C::kKB; ++kb)
#pragma unroll
      for (int hk = 0; hk < 2; ++hk)
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          float pv = fast_exp2(__builtin_fmaf(sacc[kb][hk * 8 + m], kLog2e, -m_use));
          rs += pv;
          pb[kb][hk][m] = (__bf16)pv;
        }
    l_run = l_run * alpha + rs;
    m_run = m_new;
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int b = 0; b < kNB; ++b) o_acc[b] *= alpha;
    }

    // O^T += V^T P^T with V^T from transposing reads of the V tile.
    const char G4_LDS* vt = smem + C::kLdsV + (VDOUBLE ? cur : 0) * C::kTileBytes;
    __builtin_amdgcn_sched_barrier(0);
    mfma_prio_begin();
    __builtin_amdgcn_sched_barrier(0);
    pv_step<0, 0, 0>(vt, pb[0][0]);
    pv_step<0, 1, 0>(vt, pb[0][1]);
    if constexpr (C::kKB > 1) {
      pv_step<1, 0, 0>(vt, pb[1][0]);
      pv_step<1, 1, 0>(vt, pb[1][1]);
    }
    mfma_pipeline_hint<C::kKB * 2 * kNB, 6, 2>();

    __builtin_amdgcn_sched_barrier(0);
    mfma_prio_end();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!VDOUBLE) {
      // Single V buffer: every wave must finish its PV reads before refill.
      barrier_lds();
      if (it + 1 < ntiles) issue_v(kb0 + KS * BN, 0);
    }
  }
};

// Work item L of a forward grid: heads outermost (KV head, then the grid's
// query tiles, then the query heads of the group), query tiles sequence by
// sequence.  A compact grid (FwdParams::compact) enumerates only the tiles
// that exist; otherwise every sequence has ntq slots, the ones past its end
// empty.
struct FwdItem {
  int kvh, qh, s, local, nt;
  // False for an item past the last tile of a compact grid.
  __device__ __forceinline__ bool decode(const FwdParams& a, int L, int bm) {
    const g4_problem& p = a.p;
    const int grp = p.num_q_heads / p.num_kv_heads;
    SeqTiles tiles;
    if (a.compact) tiles.init(p.cu_seqlens_q, a.num_seqs, bm);
    const int per_kvh = (a.compact ? tiles.total : a.num_seqs * a.ntq) * grp;
    kvh = L / per_kvh;
    if (kvh >= p.num_kv_heads) return false;
    const int rem = L % per_kvh;
    const int rank = rem / grp;
    qh = kvh * grp + rem % grp;
    if (a.compact) {
      tiles.find(rank, s, local, nt);
    } else {
      s = rank / a.ntq;
      local = rank % a.ntq;
      nt = a.ntq;
    }
    return true;
  }
  // The item of this workgroup in a launch of one item per workgroup.
  __device__ static __forceinline__ int of_block(const FwdParams& a) {
    return a.desc_order ? xcd_remap_desc(blockIdx.x, gridDim.x,
                                          a.p.num_q_heads / a.p.num_kv_heads)
                        : xcd_remap(blockIdx.x, gridDim.x);
  }
  // The index in the full (num_seqs x ntq) grid of the item for the same
  // query tile (the two grids order a sequence's tiles over nt and over ntq).
  __device__ __forceinline__ int full_index(const FwdParams& a) const {
    const int grp = a.p.num_q_heads / a.p.num_kv_heads;
    const int r = unzigzag(zigzag(local, nt), a.ntq);
    return (kvh * a.num_seqs * a.ntq + s * a.ntq + r) * grp + qh % grp;
  }
};

// Item of the rescaling pass after the wide kernel: 64 queries (tile qt) of one
// head of sequence s.
struct FixupItem {
  static constexpr int kBM = 64;
  int s, qt, qh;
};

// The rescaling pass's items, in the order of blocks of four tiles (a sequence's
// last ones first; then sequence and KV head), their tiles from the last on and
// the heads of a tile.  Flagged items are few and lie anywhere (one head, one row
// of every head, one sequence), and each walks a whole key range, so no fixed
// share of all items balances the workgroups: every workgroup reads the flags (4
// bytes per 32 queries and head), and the flagged items are dealt in order,
// forwards in the even rounds and backwards in the odd ones (a round's last item
// costs least).  Neighbours (an XCD's 32 workgroups take 32 in a row) then walk the
// same keys at the same time: 8192 tokens with every row flagged, tiles taken in
// zigzag order instead 7.9 ms, one tile of all KV heads 5.6.
struct FixupScan {
  static constexpr int kTiles = 4;   // tiles of a block: one thread's in a step
  static constexpr int kMine = 64;   // a step's items of one workgroup, at most
  static constexpr int kLdsBytes = kMine * 16 + 64;
  const FwdParams& a;
  int grp;
  int64_t segs, blocks;
  __device__ __forceinline__ explicit FixupScan(const FwdParams& x) : a(x) {
    grp = a.p.num_q_heads / a.p.num_kv_heads;
    segs = (int64_t)a.num_seqs * a.p.num_kv_heads;
    blocks = segs * ((a.ntq + kTiles - 1) / kTiles);
  }
  // Block u: tiles t0 .. t0 + 3 of sequence s.
  __device__ __forceinline__ void locate(int64_t u, int& s, int& t0, int& kvh) const {
    const int hkv = a.p.num_kv_heads, nb = (a.ntq + kTiles - 1) / kTiles;
    if (blocks < (int64_t(1) << 31)) {  // (32-bit divisions, a tenth of the 64-bit ones' cost)
      const uint32_t t = (uint32_t)u / (uint32_t)segs, g = (uint32_t)u - t * (uint32_t)segs;
      s = (int)(g / (uint32_t)hkv);
      kvh = (int)(g - (uint32_t)s * (uint32_t)hkv);
      t0 = (nb - 1 - (int)t) * kTiles;
      return;
    }
    const int64_t t = u / segs, g = u - t * segs;
    s = (int)(g / hkv);
    kvh = (int)(g - (int64_t)s * hkv);
    t0 = (nb - 1 - (int)t) * kTiles;
  }
  // Heads of a block's tiles with a row that the wide kernel could not finish, a
  // bit each: 8 bits per tile, the last tile's lowest.  (GRP at compile time, so
  // that the loads are in flight together.)
  template <int GRP>
  __device__ __forceinline__ unsigned heads(int64_t u) const {
    if (u >= blocks) return 0;
    int s, t0, kvh;
    locate(u, s, t0, kvh);
    const g4_problem& p = a.p;
    const int nq32 = (p.seqlen_q + 31) / 32;
    const int lq = p.cu_seqlens_q ? p.cu_seqlens_q[s + 1] - p.cu_seqlens_q[s] : p.seqlen_q;
    const int* f = a.raise_flags + (int64_t)s * nq32 * p.num_q_heads + kvh * GRP;
    constexpr int kVec = GRP < 4 ? GRP : 4;
    typedef int vec __attribute__((ext_vector_type(kVec)));
    vec x[2 * kTiles][GRP / kVec];
#pragma unroll
    for (int i = 0; i < 2 * kTiles; ++i)
#pragma unroll
      for (int j = 0; j < GRP / kVec; ++j)
        x[i][j] = *(const vec*)(f + (int64_t)min(t0 * 2 + i, nq32 - 1) * p.num_q_heads + j * kVec);
    unsigned any = 0;
#pragma unroll
    for (int i = 0; i < 2 * kTiles; ++i) {
      int m = 0;
#pragma unroll
      for (int j = 0; j < GRP; ++j) m |= x[i][j / kVec][j % kVec];
      // 32-query groups past the sequence's end hold nothing
      any |= (t0 * 2 + i) * 32 < lq ? (unsigned)m << 8 * (kTiles - 1 - i / 2) : 0u;
    }
    return any;
  }
  __device__ __forceinline__ unsigned heads(int64_t u) const {
    switch (grp) {
      case 1: return heads<1>(u);
      case 2: return heads<2>(u);
      case 4: return heads<4>(u);
      default: return heads<8>(u);
    }
  }
  // Runs run(item) for every flagged item of this workgroup; all threads call
  // it.  lds: kLdsBytes that run() leaves alone.
  template <class Run>
  __device__ __forceinline__ void each(char G4_LDS* lds, Run run) const {
    i32x4 G4_LDS* list = (i32x4 G4_LDS*)lds;
    int G4_LDS* wave_sum = (int G4_LDS*)(lds + kMine * 16);  // [step parity][wave]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
    const int n = gridDim.x, me = xcd_remap(blockIdx.x, n);
    auto number = [&](int64_t round) { return round * n + (round & 1 ? n - 1 - me : me); };
    int64_t before = 0;  // flagged items of the earlier steps
    int par = 0;
    for (int64_t u0 = 0; u0 < blocks; u0 += nt, par ^= 1) {
      const unsigned any = heads(u0 + tid);
      const int cnt = __popc(any);
      int incl = cnt;
      if (__ballot(cnt != 0)) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(incl, o, 64);
          if (lane >= o) incl += y;
        }
      }
      if (lane == 63) wave_sum[par * 8 + wave] = incl;
      barrier_lds();  // (and the previous step's list has been read)
      int total = 0;
      int64_t rank = before + incl - cnt;
      for (int w = 0; w < nt / 64; ++w) {
        const int x = wave_sum[par * 8 + w];
        if (w < wave) rank += x;
        total += x;
      }
      total = __builtin_amdgcn_readfirstlane(total);
      if (total == 0) continue;
      const int64_t round0 = before / n, end = before + total;
      for (unsigned m = any; m; m &= m - 1, ++rank) {
        const int64_t round = rank / n;
        if (rank != number(round)) continue;
        const int bit = __ffs(m) - 1;
        int s, t0, kvh;
        locate(u0 + tid, s, t0, kvh);
        list[round - round0] = i32x4{s, t0 + kTiles - 1 - bit / 8, kvh * grp + bit % 8, 0};
      }
      barrier_lds();
      for (int64_t round = round0; round * n < end; ++round) {
        const int64_t r = number(round);
        if (r < before || r >= end) continue;
        const i32x4 it = list[round - round0];
        run(FixupItem{__builtin_amdgcn_readfirstlane(it[0]), __builtin_amdgcn_readfirstlane(it[1]),
                      __builtin_amdgcn_readfirstlane(it[2])});
      }
      before = end;
    }
  }
};

// Workgroups of a forward grid of bm-query tiles; sets b->compact.  A packed
// batch of 2..64 sequences enumerates only its tiles: at most
// sum ceil(len / bm) <= (total_q + num_seqs (bm - 1)) / bm per head, against
// num_seqs x ntq for the grid sized by the longest sequence.
static int64_t fwd_grid(FwdParams* b, int bm, bool allow_compact) {
  const g4_problem& p = b->p;
  b->ntq = (p.seqlen_q + bm - 1) / bm;
  b->compact = 0;
  b->desc_order = 0;
  int64_t tiles = (int64_t)b->num_seqs * b->ntq;
  if (allow_compact && p.cu_seqlens_q != nullptr && b->num_seqs > 1 && b->num_seqs <= 64) {
    const int64_t bound = (p.total_q + (int64_t)b->num_seqs * (bm - 1)) / bm;
    if (bound < tiles) {
      tiles = bound;
      b->compact = 1;
    }
  }
  const int64_t n = tiles * p.num_q_heads;
  // Heaviest first within each XCD: the zigzag ranks of a sequence alternate
  // heavy and light only if ntq is even (rank parity = tile-rank parity).
  const int grp = p.num_q_heads / p.num_kv_heads;
  if (allow_compact && !b->compact && b->ntq % 2 == 0 && n % (16 * grp) == 0) b->desc_order = 1;
  return n;
}

// Two groups of waves of one workgroup with the same queries and every second
// key tile each (KS = 2).
template <class C>
struct FwdKeyGroups {
  static constexpr int kGroupLds = (C::kLdsBytes + 1023) / 1024 * 1024;
  static constexpr int kNB = C::kDH / 32;
  static constexpr int kHalf = kNB / 2 * 4096;               // half of a wave's accumulators
  static constexpr int kLdsState = 2 * C::kNW * kHalf;       // [group][wave][m, l][lane] fp32
  static constexpr int kLdsBytes = std::max(2 * kGroupLds, kLdsState + 2 * C::kNW * 512);
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");

  // Group G finishes half G of the head dim: it sends the other half of its
  // accumulators, and its m and l, through LDS, and with M the larger m,
  // O = sum 2^(m_g - M) O_g / sum 2^(m_g - M) l_g.
  template <int G, class K>
  __device__ static __forceinline__ void finish(const FwdParams& a, K& ker, char* smem_all, int s,
                                                int qh, int my_i, bool q_valid) {
    char G4_LDS* smem = (char G4_LDS*)smem_all;
    const int lane = ker.lane, wave = ker.wave;
    const float l_mine = ker.l_run + wave_xor32(ker.l_run);
    barrier_lds();  // both groups are done with their tiles
    char G4_LDS* send = smem + (G * C::kNW + wave) * kHalf + lane * 16;
    const char G4_LDS* recv = smem + ((1 - G) * C::kNW + wave) * kHalf + lane * 16;
    float G4_LDS* st = (float G4_LDS*)(smem + kLdsState);
#pragma unroll
    for (int b = 0; b < kNB / 2; ++b)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f32x16& x = ker.o_acc[(1 - G) * (kNB / 2) + b];
        *(f32x4 G4_LDS*)(send + (b * 4 + r4) * 1024) =
            f32x4{x[r4 * 4], x[r4 * 4 + 1], x[r4 * 4 + 2], x[r4 * 4 + 3]};
      }
    st[(G * C::kNW + wave) * 128 + lane] = ker.m_run;
    st[(G * C::kNW + wave) * 128 + 64 + lane] = l_mine;
    barrier_lds();
    const float m_other = st[((1 - G) * C::kNW + wave) * 128 + lane];
    const float l_other = st[((1 - G) * C::kNW + wave) * 128 + 64 + lane];
    const float m = fmaxf(ker.m_run, m_other);
    const float m_use = m == kNegInf ? 0.f : m;
    const float f_mine = fast_exp2(ker.m_run - m_use), f_other = fast_exp2(m_other - m_use);
    const float l_tot = l_mine * f_mine + l_other * f_other;
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (!q_valid) return;
    __bf16* orow = a.o + tok_off(ker.sq, s, ker.sq.qtok, my_i, a.ol) +
                   (int64_t)qh * a.ol.head_stride + G * (C::kDH / 2) + 4 * ker.h32;
#pragma unroll
    for (int b = 0; b < kNB / 2; ++b)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f32x16& x = ker.o_acc[G * (kNB / 2) + b];
        const f32x4 y = *(const f32x4 G4_LDS*)(recv + (b * 4 + r4) * 1024);
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = (__bf16)((x[r4 * 4 + e] * f_mine + y[e] * f_other) * inv);
        *(bf16x4*)(orow + b * 32 + 8 * r4) = v;
      }
    if (G == 0 && ker.h32 == 0)
      a.lse[lse_off(a.p, ker.sq, s, qh, my_i)] =
          l_tot > 0.f ? (m + fast_log2(l_tot)) * kLn2 : kNegInf;
  }
};

// One work item L of the forward (one query tile of one head).
// FIXUP: the item `fix` of the rescaling pass (L is not used).
// OCC: workgroups per CU the register budget is sized for.
// KS = 2: two groups of waves, each with LDS of its own, take the even and the
// odd key tiles; their states are combined at the end.
template <int D, int BN, int DSPLIT, int NQG, bool VDOUBLE, int META, bool FIXUP, int OCC,
          int KS = 1>
__device__ __forceinline__ void fwd_item(const FwdParams& a, char* smem_all, int L,
                                         FixupItem fix = {}) {
  using K = FwdKernel<D, BN, DSPLIT, NQG, VDOUBLE, META, OCC, KS>;
  using C = typename K::C;
  static_assert(KS == 1 || (KS == 2 && DSPLIT == 1 && VDOUBLE && !FIXUP && META != 3),
                "key groups");
  K ker;
  int kg = 0;  // this wave's group
  char* smem_raw = smem_all;
  if constexpr (KS > 1) {
    kg = __builtin_amdgcn_readfirstlane(threadIdx.x / C::kNT);
    smem_raw += kg * FwdKeyGroups<C>::kGroupLds;
  }
  ker.smem = (char G4_LDS*)smem_raw;
  ker.p = &a.p;
  const g4_problem& p = a.p;

  ker.tid = KS > 1 ? threadIdx.x % C::kNT : threadIdx.x;
  ker.lane = ker.tid & 63;
  ker.wave = __builtin_amdgcn_readfirstlane(ker.tid >> 6);
  const int qg = ker.wave / DSPLIT;
  ker.dh = ker.wave % DSPLIT;
  ker.h32 = ker.lane >> 5;
  const int l32 = ker.lane & 31;

  // ---- work item -------------------------------------------------------
  FwdItem it;
  int kvh, qh, s, qt;
  if constexpr (FIXUP) {
    kvh = fix.qh / (p.num_q_heads / p.num_kv_heads);
    qh = fix.qh;
    s = fix.s;
    qt = fix.qt;
  } else {
    if (!it.decode(a, L, C::kBM)) return;
    kvh = it.kvh;
    qh = it.qh;
    s = it.s;
    qt = zigzag(it.local, it.nt);
  }

  ker.sq = resolve_seq(p, s);
  const Seq& sq = ker.sq;
  const int i0 = qt * C::kBM;
  if (i0 >= sq.lq) return;
  const int off = sq.lk - sq.lq;  // query i sits at key position i + off
  ker.a0 = i0 + off;
  const int a_last_valid = min(i0 + C::kBM, sq.lq) - 1 + off;
  ker.has_vid = (META & 1) && p.vision_ids != nullptr && p.bidirectional_vision;
  ker.has_doc = (META & 2) && p.document_ids != nullptr;
  ker.has_meta = ker.has_vid || ker.has_doc;

  // ---- key range (mask-aware tile scheduler) -------------------------------
  int span_max = -1;
  if (ker.has_vid) {
    int* red = (int*)(smem_raw + C::kLdsRed);
    int v = -1;
    for (int t = ker.tid; t < C::kBM; t += C::kNT) {
      int i = i0 + t;
      if (i < sq.lq) v = max(v, a.span_hi[sq.ktok + i + off]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    if (ker.lane == 0) red[ker.wave] = v;
    barrier_lds();
#pragma unroll
    for (int w = 0; w < C::kNW; ++w) span_max = max(span_max, red[w]);
  }
  int klo, khi;
  query_tile_key_range(ker.a0, a_last_valid, sq.lk, p.window, span_max, klo, khi);
  int t_first = klo / BN;
  int ntiles = (khi + BN - 1) / BN - t_first;
  const int all_tiles = ntiles;
  if constexpr (KS > 1) {  // this group's
    t_first += kg;
    ntiles = max((all_tiles - kg + KS - 1) / KS, 0);
  }
  // ---- document uniformity -------------------------------------------------
  // The range spans whole 64-key tiles (a superset of the visited tiles for
  // BN <= 64), so both launches of a split problem evaluate it identically.
  if (p.document_ids != nullptr && (ker.has_doc || a.doc_pass == 1)) {
    const bool uni = doc_uniform<C::kNW>(
        p.document_ids, sq.ktok, sq.lk, min(klo / 64 * 64, ker.a0),
        max((khi + 63) / 64 * 64, a_last_valid + 1), ker.tid, ker.lane, ker.wave,
        (int*)(smem_raw + C::kLdsRed));
    if (a.doc_pass == 1 && !uni) {
      // left to the second pass
      // (its index in the full grid, which pass 2 decodes)
      if (ker.tid == 0 && a.doc_list != nullptr)
        a.doc_list[atomicAdd(a.doc_list_n, 1u)] = it.full_index(a);
      return;
    }
    if (a.doc_pass == 2 && uni) return;
    if (uni) {
      ker.has_doc = false;
      ker.has_meta = ker.has_vid;
    }
  }

  // ---- operand bases, address tables ---------------------------------------
  ker.kbase = a.k + tok_off(sq, s, sq.ktok, 0, a.kl) + (int64_t)kvh * a.kl.head_stride;
  ker.vbase = a.v + tok_off(sq, s, sq.ktok, 0, a.vl) + (int64_t)kvh * a.vl.head_stride;
  ker.kstride = a.kl.token_stride;
  ker.vstride = a.vl.token_stride;
  ker.krd.init(ker.lane, ker.dh * C::kDH * 2);
  ker.vrd.init(ker.lane, ker.dh * C::kDH * 2);
  ker.kcp.init(ker.kstride, ker.wave, ker.lane);
  ker.vcp.init(ker.vstride, ker.wave, ker.lane);

  // ---- query fragments (B operand of S^T = K Q^T) -------------------------
  const int my_i = i0 + qg * 32 + l32;  // this lane's query
  ker.my_a = my_i + off;
  const bool q_valid = my_i < sq.lq;
  {
    const __bf16* qrow = a.q + tok_off(sq, s, sq.qtok, min(my_i, sq.lq - 1), a.ql) +
                         (int64_t)qh * a.ql.head_stride + ker.dh * C::kDH + ker.h32 * 8;
#pragma unroll
    for (int c = 0; c < K::kNC; ++c) {
      bf16x8 x = ld_global16(qrow + c * 16);
      ker.qf[c] = q_valid ? x : bf16x8{};
    }
  }
  ker.my_vid = -1;
  ker.my_doc = 0;
  if (ker.has_vid && q_valid) ker.my_vid = p.vision_ids[sq.ktok + ker.my_a];
  if (ker.has_doc && q_valid) ker.my_doc = p.document_ids[sq.ktok + ker.my_a];

  // ---- prologue: tile 0 (issue order K, key metadata, V) -----------------
  if (ntiles > 0) {
    ker.issue_k(t_first * BN, 0);
    if (ker.has_meta && ker.wave == 0) issue_meta(p, sq, t_first * BN, ker.smem + C::kLdsMeta, ker.lane, ker.has_vid, ker.has_doc);
    ker.issue_v(t_first * BN, 0);
  }

#pragma unroll
  for (int b = 0; b < K::kNB; ++b) ker.o_acc[b] = f32x16{};
  ker.m_run = kNegInf;
  ker.l_run = 0.f;

  // Two tiles per iteration, so each step's buffers are compile-time.
  // (Two tiles per iteration with compile-time buffers measured slower: the
  // unrolled loop spills.)
  for (int it = 0; it < ntiles; ++it) ker.step(it & 1, it, ntiles, t_first);
  if constexpr (KS > 1) {
    // a step has one barrier; the second group may have a step less
    if (kg > 0 && all_tiles > 0 && all_tiles % KS) barrier_lds();
    if (kg == 0)
      FwdKeyGroups<C>::template finish<0>(a, ker, smem_all, s, qh, my_i, q_valid);
    else
      FwdKeyGroups<C>::template finish<1>(a, ker, smem_all, s, qh, my_i, q_valid);
    return;
  }

  // ---- epilogue: normalise, write O and LSE ---------------------------------
  const float l_tot = ker.l_run + wave_xor32(ker.l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (q_valid) {
    __bf16* orow = a.o + tok_off(sq, s, sq.qtok, my_i, a.ol) + (int64_t)qh * a.ol.head_stride;
#pragma unroll
    for (int b = 0; b < K::kNB; ++b) {
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int d = ker.dh * C::kDH + b * 32 + 8 * r4 + 4 * ker.h32;
        const f32x16& acc = ker.o_acc[b];
        bf16x4 v = {(__bf16)(acc[r4 * 4] * inv), (__bf16)(acc[r4 * 4 + 1] * inv),
                    (__bf16)(acc[r4 * 4 + 2] * inv), (__bf16)(acc[r4 * 4 + 3] * inv)};
        *(bf16x4*)(orow + d) = v;
      }
    }
    if (ker.dh == 0 && ker.h32 == 0) {
      a.lse[lse_off(p, sq, s, qh, my_i)] =
          l_tot > 0.f ? (ker.m_run + fast_log2(l_tot)) * kLn2 : kNegInf;
    }
  }
}

template <int D, int BN, int DSPLIT, int NQG, bool VDOUBLE, int META, bool FIXUP = false,
          int OCC = 1, int KS = 1>
__global__ void __launch_bounds__(NQG * DSPLIT * KS * 64, OCC) fwd_kernel(FwdParams a) {
  using C = FwdCfg<D, BN, DSPLIT, NQG, VDOUBLE>;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  if constexpr (META == 3 && !FIXUP) {
    // Second document pass with the first pass's list: the listed items,
    // strided over a resident grid (an item leaves no tile copy in flight;
    // the barrier retires its LDS reads).  One call site, so the item is
    // inlined once.
    const bool listed = a.doc_pass == 2 && a.doc_list != nullptr;
    const int n = listed ? (int)__builtin_amdgcn_readfirstlane(*a.doc_list_n) : (int)blockIdx.x + 1;
    for (int t = blockIdx.x; t < n; t += gridDim.x) {
      if (t != (int)blockIdx.x) barrier_lds();
      const int L = listed ? __builtin_amdgcn_readfirstlane(a.doc_list[t])
                           : FwdItem::of_block(a);
      fwd_item<D, BN, DSPLIT, NQG, VDOUBLE, META, FIXUP, OCC>(a, smem_raw, L);
    }
  } else if constexpr (FIXUP) {
    // Rescaling pass.  Flags are rare, so the pass is its reading of them: one
    // workgroup per item spent 119 us on 33792 workgroups of 32 packed sequences
    // (32768 tokens).
    static_assert(C::kBM == FixupItem::kBM, "rescaling tiles");
    FixupScan(a).each((char G4_LDS*)smem_raw + C::kLdsBytes, [&](const FixupItem& it) {
      barrier_lds();  // the previous item's LDS reads are done
      fwd_item<D, BN, DSPLIT, NQG, VDOUBLE, META, FIXUP, OCC>(a, smem_raw, 0, it);
    });
  } else {
    fwd_item<D, BN, DSPLIT, NQG, VDOUBLE, META, FIXUP, OCC, KS>(a, smem_raw,
                                                                FwdItem::of_block(a));
  }
}

// ===========================================================================
// Split-key forward for few queries per KV head (decode).
//
// One workgroup per (sequence, KV head, chunk of split_keys keys): its 32
// rows are the query rows of the KV head's group, row r = query head
// kvh * grp + r / Sq, query r % Sq (grp * Sq <= 32; the rest are zero rows),
// so each K / V tile is read once for the whole group, and the chunks spread a
// long key range over the GPU.  The steps are FwdKernel's (one 32-row group,
// head dim split over D / 256 waves); the workgroup writes its rows' partial
// state (O not normalised, running maximum m in log2 units, row sum l) and
// merge_split_kernel combines the chunks: with M the largest m,
// O = sum 2^(m_c - M) O_c / sum 2^(m_c - M) l_c.
// ===========================================================================

template <int D>
using SplitKernel = FwdKernel<D, 32, D / 256, 1, true, 0, (D == 256 ? 2 : 1)>;

template <int D>
__global__ void __launch_bounds__(D / 4, (D == 256 ? 2 : 1)) fwd_split_kernel(FwdParams a) {
  using K = SplitKernel<D>;
  using C = typename K::C;
  constexpr int BN = 32;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  K ker;
  ker.smem = (char G4_LDS*)smem_raw;
  ker.p = &a.p;
  const g4_problem& p = a.p;
  ker.tid = threadIdx.x;
  ker.lane = ker.tid & 63;
  ker.wave = __builtin_amdgcn_readfirstlane(ker.tid >> 6);
  ker.dh = ker.wave;
  ker.h32 = ker.lane >> 5;
  const int r = ker.lane & 31;

  // ---- item: (sequence, KV head) group g, chunk c ---------------------------
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int n = a.split_chunks;
  const int g = L / n, c = L % n;
  const int s = g / p.num_kv_heads, kvh = g % p.num_kv_heads;
  const int grp = p.num_q_heads / p.num_kv_heads;
  const int rows = grp * p.seqlen_q;  // row stride of the partial buffers
  ker.sq = resolve_seq(p, s);
  const Seq& sq = ker.sq;
  const int lq = sq.lq;
  if (lq <= 0) return;
  const int off = sq.lk - lq;
  const bool valid = r < grp * lq;
  const int qh = kvh * grp + (valid ? r / lq : 0);
  const int qi = valid ? r % lq : 0;
  ker.my_a = qi + off;
  ker.a0 = off;  // the first query's position (the full-tile test's lower bound)
  ker.has_vid = ker.has_doc = ker.has_meta = false;
  ker.my_vid = -1;
  ker.my_doc = 0;

  // ---- this chunk's key tiles ------------------------------------------------
  int klo, khi;
  query_tile_key_range(off, off + lq - 1, sq.lk, p.window, -1, klo, khi);
  const int per = a.split_keys / BN;
  const int t_first = klo / BN + c * per;
  const int t_end = min((khi + BN - 1) / BN, t_first + per);
  const int ntiles = khi > klo ? max(t_end - t_first, 0) : 0;

  ker.kbase = a.k + tok_off(sq, s, sq.ktok, 0, a.kl) + (int64_t)kvh * a.kl.head_stride;
  ker.vbase = a.v + tok_off(sq, s, sq.ktok, 0, a.vl) + (int64_t)kvh * a.vl.head_stride;
  ker.kstride = a.kl.token_stride;
  ker.vstride = a.vl.token_stride;
  ker.krd.init(ker.lane, ker.dh * C::kDH * 2);
  ker.vrd.init(ker.lane, ker.dh * C::kDH * 2);
  ker.kcp.init(ker.kstride, ker.wave, ker.lane);
  ker.vcp.init(ker.vstride, ker.wave, ker.lane);
  {
    const __bf16* qrow = a.q + tok_off(sq, s, sq.qtok, qi, a.ql) +
                         (int64_t)qh * a.ql.head_stride + ker.dh * C::kDH + ker.h32 * 8;
#pragma unroll
    for (int cc = 0; cc < K::kNC; ++cc) {
      bf16x8 x = ld_global16(qrow + cc * 16);
      ker.qf[cc] = valid ? x : bf16x8{};
    }
  }
  if (ntiles > 0) {
    ker.issue_k(t_first * BN, 0);
    ker.issue_v(t_first * BN, 0);
    if (ntiles > 1) ker.issue_k((t_first + 1) * BN, 1);
  }
#pragma unroll
  for (int b = 0; b < K::kNB; ++b) ker.o_acc[b] = f32x16{};
  ker.m_run = kNegInf;
  ker.l_run = 0.f;
  for (int it = 0; it < ntiles; ++it) ker.template step<true>(it & 1, it, ntiles, t_first);

  // ---- partial rows ---------------------------------------------------------
  const float l_tot = ker.l_run + wave_xor32(ker.l_run);
  if (valid) {
    const int64_t row = ((int64_t)g * n + c) * rows + r;
    float* po = a.part + row * D;
#pragma unroll
    for (int b = 0; b < K::kNB; ++b)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int d = ker.dh * C::kDH + b * 32 + 8 * r4 + 4 * ker.h32;
        const f32x16& x = ker.o_acc[b];
        *(f32x4*)(po + d) = f32x4{x[r4 * 4], x[r4 * 4 + 1], x[r4 * 4 + 2], x[r4 * 4 + 3]};
      }
    if (ker.dh == 0 && ker.h32 == 0) {
      float* ml = a.part + (int64_t)p.num_seqs * p.num_kv_heads * n * rows * D + row * 2;
      ml[0] = ker.m_run;
      ml[1] = l_tot;
    }
  }
}

// One workgroup per (sequence, KV head, row): the row's maximum over its
// chunks first, then wave w sums chunks w, w + 4, ... (four chunks' loads in
// flight per lane), and wave 0 adds the four waves' sums in order.  (One
// 64-lane workgroup walking the chunks one by one took 73 us at 128 chunks.)
template <int D>
__global__ void __launch_bounds__(256) merge_split_kernel(FwdParams a) {
  constexpr int E = D / 64;  // elements per lane: 4 (D = 256) or 8 (D = 512)
  constexpr int kW = 4;      // waves
  __shared__ float red_m[kW], red_l[kW];
  __shared__ float stage[kW - 1][E][64];
  const g4_problem& p = a.p;
  const int grp = p.num_q_heads / p.num_kv_heads;
  const int rows = grp * p.seqlen_q;
  const int n = a.split_chunks;
  const int g = blockIdx.x / rows, r = blockIdx.x % rows;
  const int s = g / p.num_kv_heads, kvh = g % p.num_kv_heads;
  const Seq sq = resolve_seq(p, s);
  if (r >= grp * sq.lq) return;
  const int qh = kvh * grp + r / sq.lq, qi = r % sq.lq;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* ml = a.part + (int64_t)p.num_seqs * p.num_kv_heads * n * rows * D;
  const int64_t row0 = (int64_t)g * n * rows + r;  // chunk c: row0 + c * rows
  float mx = kNegInf;
  for (int c = threadIdx.x; c < n; c += kW * 64) {
    const float* e = ml + (row0 + (int64_t)c * rows) * 2;
    if (e[1] > 0.f) mx = fmaxf(mx, e[0]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) red_m[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
  float acc[E] = {};
  float l = 0.f;
#pragma unroll 4
  for (int c = wave; c < n; c += kW) {
    const int64_t row = row0 + (int64_t)c * rows;
    const float lc = ml[row * 2 + 1];
    // an empty chunk (no keys for this row) wrote l = 0 and O = 0
    const float w = lc > 0.f ? fast_exp2(ml[row * 2] - mx) : 0.f;
    l += w * lc;
    const float* po = a.part + row * D;
#pragma unroll
    for (int h = 0; h < E / 4; ++h) {
      const f32x4 x = *(const f32x4*)(po + h * 256 + 4 * lane);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[4 * h + u] += w * x[u];
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int e = 0; e < E; ++e) stage[wave - 1][e][lane] = acc[e];
    if (lane == 0) red_l[wave] = l;
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < kW; ++w) {
    l += red_l[w];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] += stage[w - 1][e][lane];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  __bf16* orow = a.o + tok_off(sq, s, sq.qtok, qi, a.ol) + (int64_t)qh * a.ol.head_stride;
#pragma unroll
  for (int h = 0; h < E / 4; ++h)
    *(bf16x4*)(orow + h * 256 + 4 * lane) =
        bf16x4{(__bf16)(acc[4 * h] * inv), (__bf16)(acc[4 * h + 1] * inv),
               (__bf16)(acc[4 * h + 2] * inv), (__bf16)(acc[4 * h + 3] * inv)};
  if (lane == 0)
    a.lse[lse_off(p, sq, s, qh, qi)] = l > 0.f ? (mx + fast_log2(l)) * kLn2 : kNegInf;
}

template <int D>
static hipError_t launch_fwd_split(const FwdParams& a, hipStream_t stream) {
  using C = typename SplitKernel<D>::C;
  static_assert(C::kNT == D / 4, "one wave per 256 of the head dim");
  static LdsAttr attr;
  hipError_t e = attr.ensure((const void*)fwd_split_kernel<D>, C::kLdsBytes);
  if (e != hipSuccess) return e;
  const int64_t groups = (int64_t)a.num_seqs * a.p.num_kv_heads;
  const int64_t rows = (int64_t)(a.p.num_q_heads / a.p.num_kv_heads) * a.p.seqlen_q;
  const int64_t items = groups * a.split_chunks;
  if (items <= 0) return hipSuccess;
  hipLaunchKernelGGL(fwd_split_kernel<D>, dim3((unsigned)items), dim3(C::kNT), C::kLdsBytes,
                     stream, a);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(merge_split_kernel<D>, dim3((unsigned)(groups * rows)), dim3(256), 0, stream,
                     a);
  return hipGetLastError();
}

// ===========================================================================
// Decode at head dim 512 with equal parts.
//
// As the split-key forward above (32 rows of one KV head's group), but what
// bounds a decode step is how evenly, and with how many bytes in flight, the CUs
// read the cache.  So the key tiles of all (sequence, KV head) segments lie end
// to end and part g of n takes the g-th equal run of them, whatever the
// sequences' lengths, and two workgroups share a CU (one K and one V tile each
// in LDS, 72 KB), one's copies in flight while the other computes.  A part
// writes its rows' state over each segment it touches to slot g + segment, and
// merge_decode_kernel combines a segment's slots.  Before / after, both
// launches: 1 x 8192 keys 29.2 / 26.9 us, 1 x 131072 249 / 199, 16 x 4K-8K
// 204 / 149 (5.1 TB/s), 16 x 8192 238 / 197, 32 x 1000 66 / 55.
// (Measured and not kept: the next segment's first copies and queries issued
// from the last tile's step, 16 x 8192 219 us: the step grows and spills.  At
// head dim 256 no gain: 32 x 1024 110 us against 105, 16 x 700 40 against 39.)
// ===========================================================================

template <int D>
struct DecodeCfg {
  static constexpr int kNW = D / 256;  // waves, each a 256-wide head-dim slice
  static constexpr int kBN = 32;
  static constexpr int kCPR = D / 8;
  static constexpr int kTile = kBN * D * 2;
  static constexpr int kNC = 16;  // 16-deep S steps of a slice
  static constexpr int kNB = 8;   // 32-wide O blocks of a slice
  static constexpr int kLdsK = 0;
  static constexpr int kLdsV = kTile;
  static constexpr int kLdsX = 2 * kTile;  // partial S of each wave
  static constexpr int kLdsBytes = kLdsX + kNW * 4096;
  static_assert(kNW == 2, "each wave adds the one other slice's partial S");
};

// The key tiles of the segments, end to end: sequence-major, KV head, tile.  Of up
// to 64 packed sequences lane s holds sequence s, so that the cumulative arrays
// are read once and not again at each step from a position to its keys (about a
// microsecond each time, with nothing else to do).  (HELD at compile time: tested
// in the kernel it cost one unpacked 8000-token cache 0.5 us of 26.8.)
template <bool HELD>
struct DecodeMap {
  const g4_problem* p;
  int total;  // tiles of all segments
  int q0, k0, lq, lk, first, n, start;  // the lane's sequence

  struct Keys {
    int first, n;  // tiles a sequence's queries reach
  };
  __device__ __forceinline__ Keys range(int lq, int lk) const {
    if (lq <= 0) return {0, 0};
    int lo, hi;
    query_tile_key_range(lk - lq, lk - 1, lk, p->window, -1, lo, hi);
    return {lo / 32, hi > lo ? (hi + 31) / 32 - lo / 32 : 0};
  }
  __device__ __forceinline__ Keys keys(int s) const {
    if constexpr (HELD)
      return {__builtin_amdgcn_readlane(first, s), __builtin_amdgcn_readlane(n, s)};
    if (p->cu_seqlens_q == nullptr) return range(p->seqlen_q, p->seqlen_k);
    return range(p->cu_seqlens_q[s + 1] - p->cu_seqlens_q[s],
                 p->cu_seqlens_k[s + 1] - p->cu_seqlens_k[s]);
  }
  __device__ __forceinline__ Seq seq(int s) const {
    if constexpr (!HELD) return resolve_seq(*p, s);
    Seq r;
    r.packed = true;
    r.lq = __builtin_amdgcn_readlane(lq, s);
    r.lk = __builtin_amdgcn_readlane(lk, s);
    r.qtok = __builtin_amdgcn_readlane(q0, s);
    r.ktok = __builtin_amdgcn_readlane(k0, s);
    return r;
  }
  __device__ __forceinline__ static int scan(int x) {
    const int lane = __lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    return x;
  }
  __device__ __forceinline__ void init(const g4_problem& prob) {
    p = &prob;
    if constexpr (HELD) {
      const int s = min((int)__lane_id(), p->num_seqs - 1);
      q0 = p->cu_seqlens_q[s];
      k0 = p->cu_seqlens_k[s];
      lq = p->cu_seqlens_q[s + 1] - q0;
      lk = p->cu_seqlens_k[s + 1] - k0;
      const Keys r = range(lq, lk);
      first = r.first;
      n = (int)__lane_id() < p->num_seqs ? r.n : 0;
      const int end = scan(n);
      start = (end - n) * p->num_kv_heads;
      total = __builtin_amdgcn_readlane(end, 63) * p->num_kv_heads;
      return;
    }
    if (p->cu_seqlens_q == nullptr) {
      total = keys(0).n * p->num_seqs * p->num_kv_heads;
      return;
    }
    int sum = 0;
    for (int s = __lane_id(); s < p->num_seqs; s += 64) sum += keys(s).n;
    total = __builtin_amdgcn_readlane(scan(sum), 63) * p->num_kv_heads;
  }
  // Sequence s that holds position pos < total, and its first position.
  __device__ __forceinline__ void find(int pos, int& s, int& first_pos) const {
    const int hkv = p->num_kv_heads;
    if constexpr (HELD) {
      s = __builtin_amdgcn_readfirstlane(__popcll(__ballot(start + n * hkv <= pos)));
      first_pos = __builtin_amdgcn_readlane(start, s);
      return;
    }
    if (p->cu_seqlens_q == nullptr) {
      const int per = keys(0).n * hkv;
      s = pos / per;
      first_pos = s * per;
      return;
    }
    first_pos = 0;
    for (int base = 0; base < p->num_seqs; base += 64) {
      const int mine = base + (int)__lane_id();
      const int cnt = mine < p->num_seqs ? keys(mine).n * hkv : 0;
      const int incl = scan(cnt) + first_pos;
      const int end = __builtin_amdgcn_readlane(incl, 63);
      if (pos < end) {
        const int at = __builtin_amdgcn_readfirstlane(__popcll(__ballot(incl <= pos)));
        s = base + at;
        first_pos = __builtin_amdgcn_readlane(incl - cnt, at);
        return;
      }
      first_pos = end;
    }
    s = p->num_seqs;  // (pos >= total)
  }
  // First position of sequence s.
  __device__ __forceinline__ int start_of(int s) const {
    if constexpr (HELD) return __builtin_amdgcn_readlane(start, s);
    if (p->cu_seqlens_q == nullptr) return s * keys(0).n * p->num_kv_heads;
    int sum = 0;
    for (int t = __lane_id(); t < s; t += 64) sum += keys(t).n;
    return __builtin_amdgcn_readlane(scan(sum), 63) * p->num_kv_heads;
  }
  // First position of part g of n.
  __device__ __forceinline__ int bound(int g, int n) const {
    return (int)((int64_t)total * g / n);
  }
  // The part of n that holds position pos.
  __device__ __forceinline__ int part_of(int pos, int n) const {
    int g = (int)((int64_t)pos * n / total);
    while (bound(g + 1, n) <= pos) ++g;
    while (bound(g, n) > pos) --g;
    return g;
  }
};

template <int D>
struct DecodeKernel {
  using C = DecodeCfg<D>;
  using Copier = TileCopier<C::kCPR, C::kBN, C::kNW>;
  static constexpr int kPer = Copier::kPer;  // copy instructions of a tile per wave
  char G4_LDS* smem;
  const FwdParams* a;
  Seq sq;
  int lane, dh, h32, r;
  int off, lq, my_a;
  const __bf16* kbase;
  const __bf16* vbase;
  RowReader<C::kCPR> krd;
  TrReader<C::kCPR> vrd;
  Copier kcp, vcp;
  bf16x8 qf[C::kNC];
  f32x16 o_acc[C::kNB];
  float m_run, l_run;

  __device__ __forceinline__ void issue(const Copier& cp, const __bf16* base, int64_t stride,
                                        int row0, int lds) {
    if (row0 + C::kBN <= sq.lk)
      cp.issue(base + row0 * stride, smem + lds);
    else
      cp.issue_clamped(base + row0 * stride, stride, sq.lk - row0, smem + lds);
  }
  __device__ __forceinline__ void issue_k(int t) {
    issue(kcp, kbase, a->kl.token_stride, t * C::kBN, C::kLdsK);
  }
  __device__ __forceinline__ void issue_v(int t) {
    issue(vcp, vbase, a->vl.token_stride, t * C::kBN, C::kLdsV);
  }

  // Key tile t; its K and V copies are in flight (K issued first).
  __device__ __forceinline__ void step(int t, bool more) {
    const int kb0 = t * C::kBN;
    vm_wait<kPer>();
    barrier_lds();  // K(t) has landed in every wave
    f32x16 sv = f32x16{};
    __builtin_amdgcn_sched_barrier(0);
    row_steps<C::kNC, 4>(krd, smem + C::kLdsK, sv, qf);
    __builtin_amdgcn_sched_barrier(0);
    char G4_LDS* xb = smem + C::kLdsX;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      *(f32x4 G4_LDS*)(xb + ((dh * 4 + q4) * 64 + lane) * 16) =
          f32x4{sv[q4 * 4], sv[q4 * 4 + 1], sv[q4 * 4 + 2], sv[q4 * 4 + 3]};
    barrier_lds();
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const f32x4 v = *(const f32x4 G4_LDS*)(xb + (((dh ^ 1) * 4 + q4) * 64 + lane) * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) sv[q4 * 4 + e] += v[e];  // (the same sum in both slices)
    }
    if (more) issue_k(t + 1);  // every wave is done with K(t)

    const int window = a->p.window;
    const bool full = kb0 + C::kBN <= sq.lk && kb0 + C::kBN - 1 <= off &&
                      (window <= 0 || kb0 > off + lq - 1 - window);
    if (!full) {
      const int lo_w = window > 0 ? my_a - window + 1 : -0x40000000;
      const int hi_c = min(my_a, sq.lk - 1);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int j = kb0 + 8 * (e >> 2) + 4 * h32 + (e & 3);
        sv[e] = j >= lo_w && j <= hi_c ? sv[e] : kNegInf;
      }
    }
    float mx = sv[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, sv[e]);
    mx = fmaxf(mx, wave_xor32(mx)) * kLog2e;
    const float m_new = mx > m_run + kRescaleLog2 ? mx : m_run;
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float rs = 0.f;
    bf16x8 pb[2];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float pv = fast_exp2(__builtin_fmaf(sv[e], kLog2e, -m_use));
      rs += pv;
      pb[e >> 3][e & 7] = (__bf16)pv;
    }
    l_run = l_run * alpha + rs;
    m_run = m_new;
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int b = 0; b < C::kNB; ++b) o_acc[b] *= alpha;
    }
    if (more)
      vm_wait<kPer>();
    else
      vm_wait<0>();
    barrier_lds();  // V(t) has landed in every wave
    __builtin_amdgcn_sched_barrier(0);
    acc_steps<C::kNB, 4>(vrd, smem + C::kLdsV, pb, o_acc);
    __builtin_amdgcn_sched_barrier(0);
    barrier_lds();  // every wave is done with V(t)
    if (more) issue_v(t + 1);
  }
};

template <int D, bool HELD>
__global__ void __launch_bounds__(D / 4) fwd_decode_kernel(FwdParams a) {
  using K = DecodeKernel<D>;
  using C = typename K::C;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const g4_problem& p = a.p;
  K ker;
  ker.smem = (char G4_LDS*)smem_raw;
  ker.a = &a;
  ker.lane = threadIdx.x & 63;
  ker.dh = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  ker.h32 = ker.lane >> 5;
  ker.r = ker.lane & 31;
  ker.krd.init(ker.lane, ker.dh * 512);
  ker.vrd.init(ker.lane, ker.dh * 512);
  ker.kcp.init(a.kl.token_stride, ker.dh, ker.lane);
  ker.vcp.init(a.vl.token_stride, ker.dh, ker.lane);
  const int grp = p.num_q_heads / p.num_kv_heads;
  const int rows = grp * p.seqlen_q;  // row stride of the partial slots

  const int g = xcd_remap(blockIdx.x, gridDim.x);
  DecodeMap<HELD> map;
  map.init(p);
  const int n = min(a.split_chunks, map.total);  // (every part holds a tile)
  if (g >= n) return;
  int pos = map.bound(g, n);
  const int end = map.bound(g + 1, n);
  int s, start;
  map.find(pos, s, start);
  while (pos < end) {
    const auto keys = map.keys(s);
    if (keys.n == 0) {
      ++s;
      continue;
    }
    const int kvh = (pos - start) / keys.n;
    const int t_lo = (pos - start) - kvh * keys.n;
    const int t_hi = min(keys.n, t_lo + end - pos);
    ker.sq = map.seq(s);
    const Seq& sq = ker.sq;
    ker.lq = sq.lq;
    ker.off = sq.lk - sq.lq;
    const bool valid = ker.r < grp * sq.lq;
    const int qh = kvh * grp + (valid ? ker.r / sq.lq : 0);
    const int qi = valid ? ker.r % sq.lq : 0;
    ker.my_a = qi + ker.off;
    ker.kbase = a.k + tok_off(sq, s, sq.ktok, 0, a.kl) + (int64_t)kvh * a.kl.head_stride;
    ker.vbase = a.v + tok_off(sq, s, sq.ktok, 0, a.vl) + (int64_t)kvh * a.vl.head_stride;
    const __bf16* qrow = a.q + tok_off(sq, s, sq.qtok, qi, a.ql) +
                         (int64_t)qh * a.ql.head_stride + ker.dh * 256 + ker.h32 * 8;
#pragma unroll
    for (int cc = 0; cc < C::kNC; ++cc) ker.qf[cc] = ld_global16(qrow + cc * 16);
    ker.issue_k(keys.first + t_lo);
    ker.issue_v(keys.first + t_lo);
#pragma unroll
    for (int cc = 0; cc < C::kNC; ++cc) ker.qf[cc] = valid ? ker.qf[cc] : bf16x8{};
#pragma unroll
    for (int b = 0; b < C::kNB; ++b) ker.o_acc[b] = f32x16{};
    ker.m_run = kNegInf;
    ker.l_run = 0.f;
    for (int t = t_lo; t < t_hi; ++t) ker.step(keys.first + t, t + 1 < t_hi);

    // ---- this part's rows of the segment: slot g + segment -------------------
    const float l_tot = ker.l_run + wave_xor32(ker.l_run);
    if (valid) {
      const int64_t row = ((int64_t)g + s * p.num_kv_heads + kvh) * rows + ker.r;
      float* po = a.part + row * D;
#pragma unroll
      for (int b = 0; b < C::kNB; ++b)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int d = ker.dh * 256 + b * 32 + 8 * r4 + 4 * ker.h32;
          const f32x16& x = ker.o_acc[b];
          *(f32x4*)(po + d) = f32x4{x[r4 * 4], x[r4 * 4 + 1], x[r4 * 4 + 2], x[r4 * 4 + 3]};
        }
      if (ker.dh == 0 && ker.h32 == 0) {
        float* ml = a.part + (int64_t)a.split_slots * rows * D + row * 2;
        ml[0] = ker.m_run;
        ml[1] = l_tot;
      }
    }
    pos += t_hi - t_lo;
    if (kvh + 1 == p.num_kv_heads && t_hi == keys.n) {
      start += keys.n * p.num_kv_heads;
      ++s;
    }
  }
}

// One workgroup per (sequence, KV head, row, Q-th of the head dim).  What
// bounds it is the chain of loads (a part's rows come from other XCDs, about
// 2 us each time): the parts' maxima and sums are read at once and their weights
// kept in LDS, then every thread's share of the O rows is in flight together
// (kP parts per load instruction of the workgroup), and the kP sums are added
// in order.  128 parts of an 8K cache: 17 us when each wave walked every fourth
// part, reading its maximum, sum and row one after the other; 6.2 us like this.
// Q = 4 while the rows alone are fewer workgroups than CUs (16 sequences, 512
// rows of about ten parts: Q = 4 12.8 us, Q = 1 9.0).
template <int D, int Q, bool HELD>
__global__ void __launch_bounds__(256) merge_decode_kernel(FwdParams a) {
  constexpr int kCols = D / Q;          // columns of a workgroup
  constexpr int kLanes = kCols / 4;     // 16-byte loads of one part's row
  constexpr int kP = 256 / kLanes;      // parts per load instruction
  constexpr int kMaxParts = 512;
  __shared__ float wts[kMaxParts];
  __shared__ float red_m[4], red_l[4];
  __shared__ float stage[kP][kCols];
  const g4_problem& p = a.p;
  const int grp = p.num_q_heads / p.num_kv_heads;
  const int rows = grp * p.seqlen_q;
  const int quarter = blockIdx.x % Q;
  const int seg = blockIdx.x / Q / rows, r = blockIdx.x / Q % rows;
  const int s = seg / p.num_kv_heads, kvh = seg % p.num_kv_heads;
  DecodeMap<HELD> map;
  map.init(p);
  const Seq sq = map.seq(s);
  if (r >= grp * sq.lq) return;
  const int qh = kvh * grp + r / sq.lq, qi = r % sq.lq;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles = map.keys(s).n;
  int g0 = 0, n = 0;
  if (tiles > 0) {
    const int first = map.start_of(s) + kvh * tiles;
    const int parts = min(a.split_chunks, map.total);
    g0 = map.part_of(first, parts);
    n = min(map.part_of(first + tiles - 1, parts) - g0 + 1, kMaxParts);
  }
  const float* ml = a.part + (int64_t)a.split_slots * rows * D;
  const int64_t row0 = ((int64_t)g0 + seg) * rows + r;  // part c: row0 + c * rows
  constexpr int kOwn = kMaxParts / 256;
  float m_c[kOwn], l_c[kOwn];
  float mx = kNegInf;
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    const int c = tid + 256 * i;
    m_c[i] = kNegInf;
    l_c[i] = 0.f;
    if (c < n) {
      const float* e = ml + (row0 + (int64_t)c * rows) * 2;
      m_c[i] = e[0];
      l_c[i] = e[1];
      // (a part without keys for this row wrote l = 0 and O = 0)
      if (l_c[i] > 0.f) mx = fmaxf(mx, m_c[i]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) red_m[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
  float l = 0.f;
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    const int c = tid + 256 * i;
    const float w = l_c[i] > 0.f ? fast_exp2(m_c[i] - mx) : 0.f;
    if (c < n) wts[c] = w;
    l += w * l_c[i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
  if (lane == 0) red_l[wave] = l;
  __syncthreads();
  l = (red_l[0] + red_l[1]) + (red_l[2] + red_l[3]);
  const int sub = tid / kLanes, col = tid % kLanes;
  const float* po = a.part + row0 * D + quarter * kCols + col * 4;
  f32x4 acc = {};
#pragma unroll 16
  for (int c = sub; c < n; c += kP) acc += wts[c] * *(const f32x4*)(po + (int64_t)c * rows * D);
  *(f32x4*)&stage[sub][col * 4] = acc;
  __syncthreads();
  if (tid >= kLanes) return;
  acc = f32x4{};
#pragma unroll
  for (int u = 0; u < kP; ++u) acc += *(const f32x4*)&stage[u][tid * 4];
  const float inv = l > 0.f ? 1.f / l : 0.f;
  __bf16* orow = a.o + tok_off(sq, s, sq.qtok, qi, a.ol) + (int64_t)qh * a.ol.head_stride +
                 quarter * kCols;
  *(bf16x4*)(orow + tid * 4) = bf16x4{(__bf16)(acc[0] * inv), (__bf16)(acc[1] * inv),
                                      (__bf16)(acc[2] * inv), (__bf16)(acc[3] * inv)};
  if (quarter == 0 && tid == 0)
    a.lse[lse_off(p, sq, s, qh, qi)] = l > 0.f ? (mx + fast_log2(l)) * kLn2 : kNegInf;
}

template <int D, bool HELD>
static hipError_t launch_fwd_decode(const FwdParams& a, hipStream_t stream) {
  using C = DecodeCfg<D>;
  static LdsAttr attr;
  hipError_t e = attr.ensure((const void*)fwd_decode_kernel<D, HELD>, C::kLdsBytes);
  if (e != hipSuccess) return e;
  const int64_t rows = (int64_t)a.num_seqs * a.p.num_q_heads * a.p.seqlen_q;
  hipLaunchKernelGGL((fwd_decode_kernel<D, HELD>), dim3((unsigned)a.split_chunks),
                     dim3(C::kNW * 64), C::kLdsBytes, stream, a);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (rows < 256)
    hipLaunchKernelGGL((merge_decode_kernel<D, 4, HELD>), dim3((unsigned)(rows * 4)), dim3(256), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((merge_decode_kernel<D, 1, HELD>), dim3((unsigned)rows), dim3(256), 0,
                       stream, a);
  return hipGetLastError();
}

// ===========================================================================
// Software-pipelined forward for wide heads without key metadata.
//
// A workgroup owns 128 query rows of one KV head: 128 / grp consecutive queries
// with the grp query heads of its group, query-major (row r is query r / grp,
// head r % grp).  Rows of fewer queries end closer to one causal end than 128
// queries of one head do: with GQA 8 a tile walks on average half a key tile
// past its rows' ends instead of two (1000 tokens: 16.1 key tiles a workgroup
// against 18), and a chunk of 16 new tokens is one tile per KV head, not 32
// nearly empty ones.
// Four waves, one per SIMD, each owning 32 rows and the whole head dim, so
// no partial scores are exchanged and one K / V tile serves 128 rows.  Per
// key tile the loop runs two regions:
//   A: S^T(t+1) = K(t+1) Q^T on MFMA, interleaved with the softmax of tile t
//      (VALU) and with the async copies of K(t+2) and V(t+1);
//   B: O^T += V(t)^T P(t)^T on MFMA.
// One barrier per tile: it publishes K(t+1) and V(t) and retires every read
// of the buffers refilled in the next region A.
//
// The O accumulators (256 AGPRs per lane) are never rescaled.  A row's
// running maximum m is set by its first admitted tile; later tiles use the
// same m as long as their maximum stays below m + kRaiseLog2 (log2 units), so
// P = exp2(s - m) <= 2^kRaiseLog2 is exact in fp32 and in bf16 range and O, l
// stay far from fp32 overflow.  A row whose scores jump higher (by more than
// kRaiseLog2 * ln 2 within the row) marks its head in its wave's slot of
// raise_flags; launch_fwd then reruns the 64-query tile of that head with the
// rescaling kernel.
//
// SPLIT: few query rows over a long cached prefix (500 new tokens after 12000
// are 128 workgroups; 16 are 4) do not fill the GPU.  Each tile's key tiles are
// then cut into kv_chunks equal chunks, one workgroup each, which write their
// rows' unnormalised O, maximum and sum to the workspace for
// merge_wide_kernel.  Chunk-major within a KV head, so that the workgroups of
// an XCD walk the same keys.
// ===========================================================================

constexpr float kRaiseLog2 = 48.0f;

template <int D>
struct WideCfg {
  static constexpr int kNW = 4;
  static constexpr int kNT = kNW * 64;
  static constexpr int kBM = kNW * 32;
  static constexpr int kBN = 32;
  static constexpr int kCPR = D / 8;
  static constexpr int kTile = kBN * D * 2;
  static constexpr int kNC = D / 16;  // 16-deep steps of S^T
  static constexpr int kNB = D / 32;  // 32-wide head-dim blocks of O^T
  static constexpr int kLdsK = 0;
  static constexpr int kLdsV = 2 * kTile;
  static constexpr int kLdsBytes = 4 * kTile;
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
};

template <int D>
struct FwdWide {
  using C = WideCfg<D>;
  static constexpr int kNC = C::kNC;
  static constexpr int kNB = C::kNB;
  static constexpr int BN = C::kBN;
  // Operand reads in flight in the S and P.V chains: one wave per SIMD has no
  // other wave to cover LDS latency (2.79 ms on config 2 with the scheduler's
  // one read per MFMA, 2.66 with two in flight, 2.56-2.59 with three or four).
  static constexpr int kAhead = 4;

  char G4_LDS* smem;
  Seq sq;
  int lane, wave, h32;
  int a0, a_last, window, lo_w, hi_c;  // positions of the tile's first / last query
  const __bf16* kbase;
  const __bf16* vbase;
  int64_t kstride, vstride;
  RowReader<C::kCPR> krd;
  TrReader<C::kCPR, false> vrd;  // as FwdKernel's at head dim 512
  TileCopier<C::kCPR, BN, C::kNW> kcp, vcp;
  bf16x8 qf[kNC];
  f32x16 o_acc[kNB];
  float m_run, l_run;
  bool raise;  // a later tile exceeded this row's maximum by more than kRaiseLog2

  __device__ __forceinline__ void issue_k(int row0, int buf) {
    char G4_LDS* dst = smem + C::kLdsK + buf * C::kTile;
    if (row0 + BN <= sq.lk)
      kcp.issue(kbase + row0 * kstride, dst);
    else
      kcp.issue_clamped(kbase + row0 * kstride, kstride, sq.lk - row0, dst);
  }
  __device__ __forceinline__ void issue_v(int row0, int buf) {
    char G4_LDS* dst = smem + C::kLdsV + buf * C::kTile;
    if (row0 + BN <= sq.lk)
      vcp.issue(vbase + row0 * vstride, dst);
    else
      vcp.issue_clamped(vbase + row0 * vstride, vstride, sq.lk - row0, dst);
  }

  // Softmax of one tile's raw scores (keys kb0 + ...) into bf16 P.
  __device__ __forceinline__ void softmax(f32x16& s, int kb0, bf16x8 (&pb)[2]) {
    const bool full = (kb0 + BN <= sq.lk) && (kb0 + BN - 1 <= a0) &&
                      (window <= 0 || kb0 > a_last - window);
    if (!full) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = kb0 + 8 * (r >> 2) + 4 * h32 + (r & 3);
        const bool ok = (j >= lo_w) & (j <= hi_c);
        s[r] = ok ? s[r] : kNegInf;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, wave_xor32(mx)) * kLog2e;
    if (m_run == kNegInf) m_run = mx;  // first admitted tile of the row (or still none)
    raise |= mx > m_run + kRaiseLog2;
    const float m_use = m_run == kNegInf ? 0.f : m_run;
    float rs = 0.f;
#pragma unroll
    for (int hk = 0; hk < 2; ++hk)
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const float pv = fast_exp2(__builtin_fmaf(s[hk * 8 + m], kLog2e, -m_use));
        rs += pv;
        pb[hk][m] = (__bf16)pv;
      }
    l_run += rs;
  }
};

// Query tile at rank r among a sequence's n: zigzag over groups of 8 adjacent
// tiles (heaviest first within a group), the group that may be short first.
// An XCD's run of ranks then holds light and heavy tiles alike, and neighbours
// cost about the same: the hardware deals workgroups to the shader engines of
// an XCD in turn, and with heavy and light tiles alternating one by one half of
// the engines took the heavy ones while the others waited (32 packed sequences,
// 32768 tokens: CUs busy 71% of the launch, 2.81 ms; in groups, and with the
// rows leaving through LDS, 2.16 ms).
constexpr int kWideGroup = 8;
__device__ __forceinline__ int wide_tile(int r, int n) {
  const int ng = (n + kWideGroup - 1) / kWideGroup;
  const int first = n - (ng - 1) * kWideGroup;  // tiles of the last group
  if (r < first) return n - 1 - r;
  const int x = r - first;
  return zigzag(1 + x / kWideGroup, ng) * kWideGroup + kWideGroup - 1 - x % kWideGroup;
}

// Tiles of a run of WideItem::decode_equal (1: 8192 tokens 1% slower, 3 x 2000
// tokens alike; 8: 3 x 2000 tokens 1% slower), and of a batch on one XCD.
constexpr int kEqualRun = 4;
constexpr int kEqualBatch = 64;

// Query tile of a wide workgroup: KV head kvh, key chunk, sequence s, tile qt.
struct WideItem {
  int kvh, chunk, s, qt;
  int row_tile;  // (KV head, tile) index of the partial rows
  __device__ __forceinline__ bool decode(const FwdParams& a, int L, int queries) {
    SeqTiles tiles;
    if (a.compact) tiles.init(a.p.cu_seqlens_q, a.num_seqs, queries);
    const int per_kvh = a.compact ? tiles.total : a.num_seqs * a.ntq;
    const int n = a.kv_chunks;
    kvh = L / (per_kvh * n);
    if (kvh >= a.p.num_kv_heads) return false;
    chunk = L / per_kvh % n;
    const int rank = L % per_kvh;
    row_tile = kvh * per_kvh + rank;
    int local, nt;
    if (a.compact) {
      tiles.find(rank, s, local, nt);
    } else {
      s = rank / a.ntq;
      local = rank % a.ntq;
      nt = a.ntq;
    }
    qt = wide_tile(local, nt);
    return true;
  }
  // Item of workgroup b of a launch without a split over sequences of equal
  // length.  The (sequence, KV head) segments fall into as many equal sets as
  // XCDs allow (the largest power of two up to 8 that divides them), each set
  // on an equal number of XCDs, which take kEqualRun adjacent tiles at a time, the
  // last tiles first: heavy ones begin first, light ones fill the end, and an XCD's
  // neighbours cost alike and share K and V.  A set of several segments takes them
  // in batches of about two rounds of its CUs, the runs of a batch's segments in
  // turn, so that no segment's heavy tiles begin when the others' light ones end (one
  // segment after the other 8 heads of 4 x 2048 tokens, GQA 1, took 234 us, in zigzag
  // ranks 212, so 180; all segments in one batch lose the shared K and V: 32 heads of
  // 5 x 1300 517 us, 468 in batches).  Within a run the tiles rotate from run to run: the
  // hardware deals neighbours to the four shader engines of an XCD in turn, and each
  // would get the same tile of every segment.  Up to kEqualRun tiles in all, the
  // segments' last tiles come first, then the ones before (16 x 500, 8 heads 93 / 76).
  __device__ __forceinline__ bool decode_equal(const FwdParams& a, int b) {
    constexpr int kXcd = 8;
    const int segs = a.num_seqs * a.p.num_kv_heads;
    const int sets = min(segs & -segs, kXcd), per_set = segs / sets, xcds = kXcd / sets;
    const int x = b % kXcd, p = b / kXcd, sub = x & (xcds - 1), turn = p / kEqualRun;
    int r = (turn * xcds + (turn & 1 ? xcds - 1 - sub : sub)) * kEqualRun + p % kEqualRun;
    if (r >= per_set * a.ntq) return false;
    int seg = x / xcds * per_set;
    if (per_set > 1) {
      const int batches = max(per_set * a.ntq / (kEqualBatch * xcds), 1);
      const int batch = (per_set + batches - 1) / batches;
      seg += r / (batch * a.ntq) * batch;
      r %= batch * a.ntq;
      const int n = min(batch, (x / xcds + 1) * per_set - seg);  // segments of this batch
      const int full = a.ntq / kEqualRun * kEqualRun * n, rem = a.ntq % kEqualRun;
      if (a.ntq <= kEqualRun) {
        seg += r % n;
        r /= n;
      } else if (r < full) {
        const int run = r / kEqualRun;
        seg += run % n;
        r = run / n * kEqualRun + (r + run) % kEqualRun;
      } else {
        r -= full;
        seg += r / rem;
        r = a.ntq - rem + (r + (rem == 2 ? r / rem / 2 : 0)) % rem;
      }
    }
    qt = a.ntq - 1 - r;
    s = seg / a.p.num_kv_heads;
    kvh = seg - s * a.p.num_kv_heads;
    chunk = row_tile = 0;
    return true;
  }
  // Workgroups of that launch.
  static int64_t equal_blocks(int64_t segs, int64_t ntq) {
    const int64_t sets = std::min<int64_t>(segs & -segs, 8), xcds = 8 / sets;
    const int64_t runs = (segs / sets * ntq + kEqualRun - 1) / kEqualRun;
    return 8 * ((runs + xcds - 1) / xcds) * kEqualRun;
  }
};

// Raise-flag slot of the 32-row wave whose first query is q (a multiple of
// 32 / grp): the grp waves of a 32-query group take the slots of the group and
// KV head, each with a bit per query head of its rows (raise_heads).
__device__ __forceinline__ int64_t raise_slot(const g4_problem& p, int s, int q, int kvh,
                                              int grp) {
  const int nq32 = (p.seqlen_q + 31) / 32;
  return ((int64_t)s * nq32 + q / 32) * p.num_q_heads + kvh * grp + q % 32 * grp / 32;
}

// The query heads (bit = head of the group) with a marked row among a wave's 32:
// row r, on lanes r and r + 32, is of head r % grp.
__device__ __forceinline__ int raise_heads(bool marked, int grp) {
  const unsigned long long m = __ballot(marked);
  unsigned x = (unsigned)m | (unsigned)(m >> 32);
  for (int o = 16; o >= grp; o >>= 1) x |= x >> o;
  return (int)(x & ((1u << grp) - 1));
}

// The MFMA fragments of a 32-row tile's rows.
template <int CP, int NC, class RR>
__device__ __forceinline__ void row_fragments(const RR& rrd, const char G4_LDS* t,
                                              bf16x8 (&frag)[NC]) {
  if constexpr (CP < NC) {
    frag[CP] = rrd.template read<0, 0, CP>(t);
    row_fragments<CP + 1>(rrd, t, frag);
  }
}

// Floats of a chunk's partial rows: 128 x D of O in register order (per wave,
// 1 KB per store), then the rows' maximum and sum.
template <int D>
constexpr int64_t kWidePartFloats = 128 * D + 256;

template <int D, bool SPLIT>
__global__ void __launch_bounds__(256, 1) fwd_wide_kernel(FwdParams a) {
  using K = FwdWide<D>;
  using C = typename K::C;
  constexpr int BN = C::kBN;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  K ker;
  ker.smem = (char G4_LDS*)smem_raw;
  const g4_problem& p = a.p;
  const int tid = threadIdx.x;
  ker.lane = tid & 63;
  ker.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ker.h32 = ker.lane >> 5;
  const int l32 = ker.lane & 31;

  const int grp = p.num_q_heads / p.num_kv_heads;
  const int gsh = __builtin_ctz(grp);  // grp is 1, 2, 4 or 8
  const int queries = C::kBM >> gsh;   // of a tile
  WideItem it;
  if (!SPLIT && a.equal_order) {
    if (!it.decode_equal(a, blockIdx.x)) return;
  } else {
    const int L = a.desc_order ? xcd_remap_desc(blockIdx.x, gridDim.x, kWideGroup)
                               : xcd_remap(blockIdx.x, gridDim.x);
    if (!it.decode(a, L, queries)) return;
  }
  const int kvh = it.kvh, s = it.s;

  ker.sq = resolve_seq(p, s);
  const Seq& sq = ker.sq;
  const int i0 = it.qt * queries;
  if (i0 >= sq.lq) return;
  const int off = sq.lk - sq.lq;
  ker.a0 = i0 + off;
  ker.a_last = ker.a0 + queries - 1;
  const int a_last_valid = min(i0 + queries, sq.lq) - 1 + off;
  ker.window = p.window;

  int klo, khi;
  query_tile_key_range(ker.a0, a_last_valid, sq.lk, p.window, -1, klo, khi);
  int t_first = klo / BN;
  int ntiles = (khi + BN - 1) / BN - t_first;
  if constexpr (SPLIT) {
    const int lo = ntiles * it.chunk / a.kv_chunks;
    ntiles = ntiles * (it.chunk + 1) / a.kv_chunks - lo;
    t_first += lo;
  }

  ker.kbase = a.k + tok_off(sq, s, sq.ktok, 0, a.kl) + (int64_t)kvh * a.kl.head_stride;
  ker.vbase = a.v + tok_off(sq, s, sq.ktok, 0, a.vl) + (int64_t)kvh * a.vl.head_stride;
  ker.kstride = a.kl.token_stride;
  ker.vstride = a.vl.token_stride;
  ker.krd.init(ker.lane, 0);
  ker.vrd.init(ker.lane, 0);
  ker.kcp.init(ker.kstride, ker.wave, ker.lane);
  ker.vcp.init(ker.vstride, ker.wave, ker.lane);

  const int w_q = i0 + ((ker.wave * 32) >> gsh);  // the wave's first query
  const int my_i = w_q + (l32 >> gsh);
  const int qh = kvh * grp + (l32 & (grp - 1));
  const int my_a = my_i + off;
  const bool q_valid = my_i < sq.lq;
  ker.lo_w = p.window > 0 ? my_a - p.window + 1 : -0x40000000;
  ker.hi_c = min(my_a, sq.lk - 1);
  // Query fragments: each wave copies its rows whole into a quarter of the tile
  // area and reads them as it reads K.  (Loaded from memory as fragments, every
  // lane of an instruction is in another line, 64 cycles each: 9000 cycles, and
  // as many for one query as for 16.)
  const int nrows = max(min(32 >> gsh, sq.lq - w_q), 0) << gsh;  // the rows of this wave
  {
    static_assert(C::kNW * 32 * D * 2 <= C::kLdsBytes && C::kCPR == 64, "staged rows");
    char G4_LDS* stage = ker.smem + ker.wave * 32 * D * 2;
    const __bf16* qbase = a.q + tok_off(sq, s, sq.qtok, w_q, a.ql) +
                          (int64_t)(kvh * grp) * a.ql.head_stride;
#pragma unroll 4
    for (int r = 0; r < nrows; ++r)
      b2l16(qbase + (r >> gsh) * a.ql.token_stride + (r & (grp - 1)) * a.ql.head_stride,
            swz_slot(r, ker.lane) * 16u, stage + r * 1024);
    vm_wait<0>();
    row_fragments<0>(ker.krd, stage, ker.qf);
#pragma unroll
    for (int c = 0; c < K::kNC; ++c) ker.qf[c] = q_valid ? ker.qf[c] : bf16x8{};
    barrier_lds();  // every wave has read its rows
  }
  ker.m_run = kNegInf;
  ker.l_run = 0.f;
  ker.raise = false;
#pragma unroll
  for (int b = 0; b < K::kNB; ++b) ker.o_acc[b] = f32x16{};

  f32x16 s_cur = {};
  if (ntiles > 0) {
    // Prologue: K(0), V(0), K(1); S(0).
    ker.issue_k(t_first * BN, 0);
    ker.issue_v(t_first * BN, 0);
    if (ntiles > 1) {
      ker.issue_k((t_first + 1) * BN, 1);
      vm_wait<decltype(ker.kcp)::kPer>();
    } else {
      vm_wait<0>();
    }
    barrier_lds();
    __builtin_amdgcn_sched_barrier(0);
    row_steps<K::kNC, K::kAhead>(ker.krd, ker.smem + C::kLdsK, s_cur, ker.qf);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int it = 0; it < ntiles; ++it) {
    const int cur = it & 1, nxt = cur ^ 1;
    const int kb0 = (t_first + it) * BN;
    // K(it + 1) and V(it) have landed in every wave; every wave is done with
    // the K buffer of tile it and the V buffer of tile it - 1.
    vm_wait<0>();
    barrier_lds();
    __builtin_amdgcn_sched_barrier(0);

    // ---- region A: S(it + 1) || softmax(it) || copies K(it + 2), V(it + 1)
    if (it + 2 < ntiles) ker.issue_k(kb0 + 2 * BN, cur);
    if (it + 1 < ntiles) ker.issue_v(kb0 + BN, nxt);
    f32x16 s_nxt = {};
    bf16x8 pb[2];
    if (it + 1 < ntiles) {
      row_steps<K::kNC, K::kAhead>(ker.krd, ker.smem + C::kLdsK + nxt * C::kTile, s_nxt,
                                   ker.qf);
      ker.softmax(s_cur, kb0, pb);
    } else {
      ker.softmax(s_cur, kb0, pb);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- region B: O^T += V(it)^T P(it)^T
    const char G4_LDS* vt = ker.smem + C::kLdsV + cur * C::kTile;
    acc_steps<K::kNB, K::kAhead>(ker.vrd, vt, pb, ker.o_acc);
    __builtin_amdgcn_sched_barrier(0);
    s_cur = s_nxt;
  }

  const bool raise = ker.raise && q_valid;
  const float l_tot = ker.l_run + wave_xor32(ker.l_run);
  if constexpr (SPLIT) {
    float* part = a.part + ((int64_t)it.row_tile * a.kv_chunks + it.chunk) * kWidePartFloats<D>;
    f32x4* po = (f32x4*)part + ker.wave * (K::kNB * 4 * 64) + ker.lane;
#pragma unroll
    for (int b = 0; b < K::kNB; ++b)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f32x16& x = ker.o_acc[b];
        po[(b * 4 + r4) * 64] = f32x4{x[r4 * 4], x[r4 * 4 + 1], x[r4 * 4 + 2], x[r4 * 4 + 3]};
      }
    if (ker.h32 == 0) {
      // (a sum of -1 marks the row for the rescaling pass)
      float* ml = part + 128 * D + 2 * (ker.wave * 32 + l32);
      ml[0] = ker.m_run;
      ml[1] = raise ? -1.f : l_tot;
    }
    return;
  }

  // Every wave reports the heads whose rows need the rescaling pass; the last
  // tile also clears the slots of its 32-query group past the tile.
  const int heads = raise_heads(raise, grp);
  if (ker.lane == 0 && w_q / 32 * 32 < sq.lq)
    a.raise_flags[raise_slot(p, s, w_q, kvh, grp)] = heads;
  const int i1 = i0 + queries;
  if (i1 >= sq.lq && i1 % 32 != 0 && tid < grp && tid >= i1 % 32 * grp / 32)
    a.raise_flags[raise_slot(p, s, i1 / 32 * 32, kvh, grp) + tid] = 0;

  // The rows leave as whole lines through LDS (a lane's accumulators are one
  // row's 8-byte runs): each wave stages its 32 rows in a quarter of the tile
  // area, 16-byte chunks swizzled by row.  (Stored as they lie, an item spent
  // 9-10 us after its loop; a 20-tile item's loop takes 40.)
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  barrier_lds();  // every wave is done with the last tiles
  char G4_LDS* stage = ker.smem + ker.wave * 32 * D * 2;
#pragma unroll
  for (int b = 0; b < K::kNB; ++b)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const f32x16& acc = ker.o_acc[b];
      *(bf16x4 G4_LDS*)(stage + l32 * D * 2 + ((b * 4 + r4) ^ (l32 & 15)) * 16 + 8 * ker.h32) =
          bf16x4{(__bf16)(acc[r4 * 4] * inv), (__bf16)(acc[r4 * 4 + 1] * inv),
                 (__bf16)(acc[r4 * 4 + 2] * inv), (__bf16)(acc[r4 * 4 + 3] * inv)};
    }
  if (q_valid && ker.h32 == 0)
    a.lse[lse_off(p, sq, s, qh, my_i)] =
        l_tot > 0.f ? (ker.m_run + fast_log2(l_tot)) * kLn2 : kNegInf;
  // Eight rows at a time, their LDS reads in flight together.
  __bf16* const obase = a.o + tok_off(sq, s, sq.qtok, w_q, a.ol) +
                        (int64_t)(kvh * grp) * a.ol.head_stride + ker.lane * 8;
  static_assert(D * 2 == 64 * 16, "one 16-byte chunk per lane and row");
  for (int r0 = 0; r0 < nrows; r0 += 8) {
    bf16x8 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = *(const bf16x8 G4_LDS*)(stage + (r0 + j) * D * 2 +
                                     (ker.lane ^ ((r0 + j) & 15)) * 16);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = r0 + j;
      if (r < nrows)
        *(bf16x8*)(obase + (r >> gsh) * a.ol.token_stride + (r & (grp - 1)) * a.ol.head_stride) =
            v[j];
    }
  }
}

// O and LSE of a split tile's rows from its chunks.  Workgroup (tile, wave of
// 32 rows, quarter of the head dim): a thread keeps one row (its lane's), so
// the chunks' weights 2^(m_c - M) are formed once per thread; the partials are
// read in the order they were written (1 KB per wave instruction) and the
// rows leave through LDS.
template <int D>
__global__ void __launch_bounds__(256) merge_wide_kernel(FwdParams a) {
  using C = WideCfg<D>;
  constexpr int kCols = D / 4;              // columns of a workgroup
  constexpr int kPitch = kCols * 2 + 16;    // bytes of a staged row
  __shared__ __attribute__((aligned(16))) char stage[32 * kPitch];
  const g4_problem& p = a.p;
  const int grp = p.num_q_heads / p.num_kv_heads;
  const int gsh = __builtin_ctz(grp);
  const int queries = C::kBM >> gsh;
  const int n = a.kv_chunks;
  const int quarter = blockIdx.x & 3, w = (blockIdx.x >> 2) & 3;
  FwdParams one = a;  // the tile as the unsplit grid orders it
  one.kv_chunks = 1;
  WideItem it;
  if (!it.decode(one, blockIdx.x >> 4, queries)) return;
  const Seq sq = resolve_seq(p, it.s);
  const int i0 = it.qt * queries;
  if (i0 >= sq.lq) return;
  const int w_q = i0 + ((w * 32) >> gsh);
  const int tid = threadIdx.x, l32 = tid & 31, h32 = (tid >> 5) & 1, sub = tid >> 6;
  const int my_i = w_q + (l32 >> gsh);
  const int qh = it.kvh * grp + (l32 & (grp - 1));

  const float* part = a.part + (int64_t)it.row_tile * n * kWidePartFloats<D>;
  const float* ml = part + 128 * D + 2 * (w * 32 + l32);
  float mx = kNegInf;
  bool raise = false;
  for (int c = 0; c < n; ++c) {
    const float m = ml[c * kWidePartFloats<D>], l = ml[c * kWidePartFloats<D> + 1];
    raise |= l < 0.f;
    if (l > 0.f) mx = fmaxf(mx, m);
  }
  const int heads = raise_heads(raise && my_i < sq.lq, grp);
  if (quarter == 0 && tid == 0 && w_q / 32 * 32 < sq.lq)
    a.raise_flags[raise_slot(p, it.s, w_q, it.kvh, grp)] = heads;
  const int i1 = i0 + queries;
  if (quarter == 0 && w == 0 && i1 >= sq.lq && i1 % 32 != 0 && tid < grp &&
      tid >= i1 % 32 * grp / 32)
    a.raise_flags[raise_slot(p, it.s, i1 / 32 * 32, it.kvh, grp) + tid] = 0;
  if (w_q >= sq.lq) return;  // (a marked head's rows are written again by the rescaling pass)

  // this workgroup's 32-column blocks of the wave's register-order partial
  constexpr int kB = D / 32 / 4;  // blocks
  static_assert(kB * 4 * 64 == 4 * 256, "four 16-byte loads per thread and chunk");
  const f32x4* src = (const f32x4*)part + (w * (D / 32) + quarter * kB) * 4 * 64 + tid;
  f32x4 acc[4] = {};
  float l = 0.f;
#pragma unroll 4
  for (int c = 0; c < n; ++c) {
    const float lc = ml[c * kWidePartFloats<D> + 1];
    const float wt = lc > 0.f ? fast_exp2(ml[c * kWidePartFloats<D>] - mx) : 0.f;
    l += wt * lc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += wt * src[c * (kWidePartFloats<D> / 4) + i * 256];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  // element i of a thread: block i, register group sub, row l32, columns
  // 32 i + 8 sub + 4 h32 .. of the quarter
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *(bf16x4*)(stage + l32 * kPitch + (32 * i + 8 * sub + 4 * h32) * 2) =
        bf16x4{(__bf16)(acc[i][0] * inv), (__bf16)(acc[i][1] * inv), (__bf16)(acc[i][2] * inv),
               (__bf16)(acc[i][3] * inv)};
  if (quarter == 0 && tid < 32 && my_i < sq.lq)
    a.lse[lse_off(p, sq, it.s, qh, my_i)] = l > 0.f ? (mx + fast_log2(l)) * kLn2 : kNegInf;
  __syncthreads();
  const int row = tid >> 3;
  const int oi = w_q + (row >> gsh);
  if (oi >= sq.lq) return;
  __bf16* orow = a.o + tok_off(sq, it.s, sq.qtok, oi, a.ol) +
                 (int64_t)(it.kvh * grp + (row & (grp - 1))) * a.ol.head_stride + quarter * kCols;
#pragma unroll
  for (int i = 0; i < kCols / 64; ++i) {
    const int c = (tid & 7) + 8 * i;
    *(bf16x8*)(orow + c * 8) = *(const bf16x8*)(stage + row * kPitch + c * 16);
  }
}

// Tiles per KV head of a wide launch's grid (an upper bound for packed
// sequences): see fwd_grid.
static int64_t wide_tiles(const g4_problem& p, int queries, int* compact) {
  int64_t tiles = (int64_t)p.num_seqs * ((p.seqlen_q + queries - 1) / queries);
  *compact = 0;
  if (p.cu_seqlens_q != nullptr && p.num_seqs > 1 && p.num_seqs <= 64) {
    const int64_t bound = (p.total_q + (int64_t)p.num_seqs * (queries - 1)) / queries;
    if (bound < tiles) {
      tiles = bound;
      *compact = 1;
    }
  }
  return tiles;
}

// Key chunks per query tile of the wide forward: 1 (no split) or the count
// whose rounds of workgroups over the 256 CUs are shortest, in key tiles of one
// workgroup's walk (1.2 us): (chunk + kSetup) per round, plus the merge: its
// launch, a chain of loads that grows with the chunks, and the partials written
// and read, at about 10 TB/s as far as the caches hold them and 4 beyond.  At least
// kMinTiles key tiles a chunk.  Measured, 32 heads of 4 KV heads, whole / split
// us: 5 tokens over 200 keys 25.6 whole, 300 31 / 24, 512 42 / 27, 1000 65 / 30;
// 48 over 450 41 / 30; 100 over 600 48 / 36; 300 over 1500 98 / 60; 500 over 2000
// 129 / 91; 600 over 3000 186 whole.
int wide_chunks(const g4_problem& p) {
  if (p.head_dim != 512 || (p.vision_ids != nullptr && p.bidirectional_vision) ||
      p.document_ids != nullptr)
    return 1;
  constexpr int kSetup = 6, kMinTiles = 2, kCus = 256;
  constexpr double kTile = 1.2, kCached = 64e6;  // us; bytes of partials
  int compact;
  const int64_t items =
      wide_tiles(p, 128 / (p.num_q_heads / p.num_kv_heads), &compact) * p.num_kv_heads;
  const int64_t range = p.window > 0
                            ? std::min<int64_t>(p.seqlen_k, (int64_t)p.window + 128)
                            : p.seqlen_k;
  const int64_t nt = (range + 31) / 32;
  int best = 1;
  double best_cost = (double)((items + kCus - 1) / kCus) * (nt + kSetup);
  for (int64_t n = 2; n <= 64 && n * kMinTiles <= nt && n * items <= 4 * kCus; ++n) {
    const double bytes = (double)(items * n) * kWidePartFloats<512> * 4;
    const double moved = 2 * (std::min(bytes, kCached) / 10e6 +
                              std::max(bytes - kCached, 0.0) / 4e6);  // us
    const double merge = 5 + 0.3 * n + moved / kTile;
    const double cost =
        (double)((items * n + kCus - 1) / kCus) * ((nt + n - 1) / n + kSetup) + merge;
    if (cost < best_cost) {
      best_cost = cost;
      best = (int)n;
    }
  }
  return best;
}
size_t wide_split_bytes(const g4_problem& p) {
  const int n = wide_chunks(p);
  if (n == 1) return 0;
  int compact;
  const int64_t tiles = wide_tiles(p, 128 / (p.num_q_heads / p.num_kv_heads), &compact);
  return (size_t)tiles * p.num_kv_heads * n * kWidePartFloats<512> * 4;
}

template <int D>
static hipError_t launch_fwd_wide(const FwdParams& a, hipStream_t stream) {
  using C = WideCfg<D>;
  FwdParams b = a;
  const int grp = a.p.num_q_heads / a.p.num_kv_heads;
  const int queries = C::kBM / grp;
  b.ntq = (a.p.seqlen_q + queries - 1) / queries;
  const int64_t tiles = wide_tiles(a.p, queries, &b.compact) * a.p.num_kv_heads;
  const bool split = a.part != nullptr;
  b.kv_chunks = split ? wide_chunks(a.p) : 1;
  int64_t nblocks = tiles * b.kv_chunks;
  if (nblocks <= 0) return hipSuccess;
  // One sequence, or several of one length: WideItem::decode_equal.  In zigzag
  // ranks such a launch ended on heavy tiles unless its tiles came out even (32
  // heads of 4 KV heads, forward us, zigzag / equal order: 1200 tokens 126 / 89,
  // 2000 230 / 155, 2048 165 / 159, 3500 560 / 431, 5000 1024 / 850, 8192 2149 /
  // 2147, 3 x 2000 536 / 491).
  b.equal_order = !split && (a.p.cu_seqlens_q == nullptr || a.p.num_seqs == 1);
  if (b.equal_order)
    nblocks = WideItem::equal_blocks((int64_t)a.p.num_seqs * a.p.num_kv_heads, b.ntq);
  // heaviest first within each XCD (xcd_remap_desc): whole groups of ranks, and
  // group parity = parity within the sequence
  b.desc_order = !b.compact && b.ntq % (2 * kWideGroup) == 0 && nblocks % (16 * kWideGroup) == 0;
  void (*kern)(FwdParams) = split ? fwd_wide_kernel<D, true> : fwd_wide_kernel<D, false>;
  static LdsAttr attr[2];
  hipError_t e = attr[split].ensure((const void*)kern, C::kLdsBytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::kNT), C::kLdsBytes, stream, b);
  e = hipGetLastError();
  if (e != hipSuccess || !split) return e;
  hipLaunchKernelGGL(merge_wide_kernel<D>, dim3((unsigned)(tiles * 16)), dim3(256), 0, stream, b);
  return hipGetLastError();
}

// Key metadata kinds a problem carries (bit 0 vision IDs, bit 1 document IDs).
static int meta_kind(const g4_problem& p) {
  return ((p.vision_ids != nullptr && p.bidirectional_vision) ? 1 : 0) |
         (p.document_ids != nullptr ? 2 : 0);
}

// Workgroups of the rescaling pass: one per CU.
constexpr int kFixupGrid = 256;

// meta < 0: the problem's own metadata kinds; doc_pass: see FwdParams.
template <int D, int BN, int DSPLIT, int NQG, bool VDOUBLE, int OCC = 1>
static hipError_t launch_fwd_cfg(const FwdParams& a, hipStream_t stream, bool fixup = false,
                                 int meta_override = -1, int doc_pass = 0) {
  using C = FwdCfg<D, BN, DSPLIT, NQG, VDOUBLE>;
  const int meta = meta_override >= 0 ? meta_override : meta_kind(a.p);
  void (*kern)(FwdParams) =
      meta == 1   ? fwd_kernel<D, BN, DSPLIT, NQG, VDOUBLE, 1, false, OCC>
      : meta == 2 ? fwd_kernel<D, BN, DSPLIT, NQG, VDOUBLE, 2, false, OCC>
      : meta == 3 ? fwd_kernel<D, BN, DSPLIT, NQG, VDOUBLE, 3, false, OCC>
                  : fwd_kernel<D, BN, DSPLIT, NQG, VDOUBLE, 0, false, OCC>;
  if constexpr (D == 512)
    if (fixup) kern = fwd_kernel<D, BN, DSPLIT, NQG, VDOUBLE, 0, true, OCC>;
  const int variant = fixup ? 4 : meta;
  const int lds = C::kLdsBytes + (fixup ? FixupScan::kLdsBytes : 0);
  static LdsAttr attr[5];
  hipError_t e = attr[variant].ensure((const void*)kern, lds);
  if (e != hipSuccess) return e;
  FwdParams b = a;
  b.doc_pass = doc_pass;
  // (the rescaling pass and the listed second document pass decode full-grid indices)
  int64_t nblocks = fwd_grid(&b, C::kBM, !fixup && doc_pass != 2);
  if (nblocks <= 0) return hipSuccess;
  if (fixup) nblocks = std::min<int64_t>(nblocks, kFixupGrid);
  if (doc_pass == 2 && a.doc_list != nullptr) {
    // the first pass's list, over at most one resident grid
    static PersistentGrid grid;
    bool many = false;
    const int64_t g = grid.size((const void*)kern, C::kNT, C::kLdsBytes, nblocks, &many);
    if (g <= 0) return hipErrorInvalidValue;
    nblocks = many ? g : nblocks;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::kNT), lds, stream, b);
  return hipGetLastError();
}

constexpr int kCus = 256;

// Two groups of waves per query tile (KS = 2, head dim 256): one workgroup of
// 8 waves per CU in place of two of 4 waves.  With more tiles than CUs the two
// workgroups fill a CU by themselves, and drift apart, so that one's softmax
// meets the other's matrix steps; up to 256 tiles each would run alone on its
// CU, bound by its own chain of steps (32 of 1.25 us at 1024 keys, 0.43 us of
// them in the matrix cores).  Sharing the keys makes it 16 steps of 2.0 us and
// 1.3 us for the exchange, which pays from about 256 keys on: 32 heads over
// 1024 tokens 46.5 -> 38.6 us, 777 tokens 37.6 -> 31.9, 64 new tokens after
// 1023 cached (4 sequences) 45.7 -> 35.9, 400 tokens 23.5 -> 22.1; at 256
// 18.5 -> 18.3, at 128 13.6 -> 15.1.
static bool use_fwd_groups(const g4_problem& p, int64_t nblocks) {
  const int64_t keys =
      p.window > 0 ? std::min<int64_t>(p.seqlen_k, (int64_t)p.window + 127) : p.seqlen_k;
  return nblocks > 0 && nblocks <= kCus && keys > 256;
}

template <int META>
static hipError_t launch_fwd_groups(const FwdParams& a, int64_t nblocks, hipStream_t stream) {
  using C = FwdCfg<256, 32, 1, 4, true>;
  const auto kern = fwd_kernel<256, 32, 1, 4, true, META, false, 1, 2>;
  static LdsAttr attr;
  hipError_t e = attr.ensure((const void*)kern, FwdKeyGroups<C>::kLdsBytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(2 * C::kNT), FwdKeyGroups<C>::kLdsBytes,
                     stream, a);
  return hipGetLastError();
}

__global__ void clear_list_kernel(unsigned* n) {
  if (threadIdx.x == 0) *n = 0u;
}

hipError_t launch_fwd(const FwdParams& a, hipStream_t stream) {
  if (a.split_slots > 0)
    return a.p.cu_seqlens_q != nullptr && a.num_seqs <= 64 ? launch_fwd_decode<512, true>(a, stream)
                                                           : launch_fwd_decode<512, false>(a, stream);
  if (a.split_chunks > 0) {
    if (a.p.head_dim == 256) return launch_fwd_split<256>(a, stream);
    if (a.p.head_dim == 512) return launch_fwd_split<512>(a, stream);
    return hipErrorInvalidValue;
  }
  if (a.p.head_dim == 256) {
    // Two workgroups of 32-key tiles share a CU (the register file holds two
    // waves per SIMD).  With both vision and document IDs the mask state needs
    // one workgroup of 64-key tiles per CU, so such a problem is split: the
    // query tiles that see a single document run in the vision-only kernel,
    // the rest in the full-mask one.
    if (meta_kind(a.p) != 3) {
      FwdParams b = a;
      b.doc_pass = 0;
      const int64_t n = fwd_grid(&b, FwdCfg<256, 32, 1, 4, true>::kBM, true);
      if (use_fwd_groups(a.p, n)) {
        switch (meta_kind(a.p)) {
          case 1: return launch_fwd_groups<1>(b, n, stream);
          case 2: return launch_fwd_groups<2>(b, n, stream);
          default: return launch_fwd_groups<0>(b, n, stream);
        }
      }
      return launch_fwd_cfg<256, 32, 1, 4, true, 2>(a, stream);
    }
    static_assert(FwdCfg<256, 32, 1, 4, true>::kBM == FwdCfg<256, 64, 1, 4, true>::kBM,
                  "both passes must tile queries alike");
    if (a.doc_list_n != nullptr) {
      // pass 1 refills the list on every call (a fill kernel, not a memset
      // node, so the launch sequence can be captured in a graph)
      hipLaunchKernelGGL(clear_list_kernel, dim3(1), dim3(64), 0, stream, a.doc_list_n);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    hipError_t e = launch_fwd_cfg<256, 32, 1, 4, true, 2>(a, stream, false, /*meta=*/1,
                                                          /*doc_pass=*/1);
    if (e != hipSuccess) return e;
    return launch_fwd_cfg<256, 64, 1, 4, true, 1>(a, stream, false, /*meta=*/3,
                                                  /*doc_pass=*/2);
  }
  if (a.p.head_dim == 512) {
    if (meta_kind(a.p) != 0 || a.raise_flags == nullptr)
      return launch_fwd_cfg<512, 32, 2, 2, true>(a, stream);
    // Fast pass, then the rescaling kernel on the 64-query tiles of the heads it flagged.
    hipError_t e = launch_fwd_wide<512>(a, stream);
    if (e != hipSuccess) return e;
    return launch_fwd_cfg<512, 32, 2, 2, true>(a, stream, /*fixup=*/true);
  }
  return hipErrorInvalidValue;
}

}  // namespace g4
