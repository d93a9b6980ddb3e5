// K/V (and Q) preparation from a projection source, fused.
//
// Per (token, head) row z of head_dim D (512 for the global layer's shared
// K/V source and its queries, 256 for the sliding layers' queries and keys):
//   r  = (mean(z^2) + eps)^(-1/2)            (fp32 over the row)
//   n  = z r                                  (fp32)
//   V  = bf16(n)                              (RMSNorm without a weight)
//   kn = bf16(n w)                            (RMSNorm with the learned weight)
//   K  = kn with RoPE on its first R dims: K_i = kn_i cos_i + rot(kn)_i sin_i,
//        rot(x)_i = -x_{i+R/2} (i < R/2), x_{i-R/2} (R/2 <= i < R); the other
//        dims pass through.  K in fp32 (fp32 tables): fp32 products and sum,
//        no contraction.  K in bf16 (bf16 tables): each product and the sum
//        rounded to bf16, as bf16 tensor operations round them.
// Lane l of a row holds dims 8 l .. 8 l + 7 (one 16-byte load), so the row
// reduction is a lane reduction and rot(x) an exchange with lane l +- R / 16.
// HBM-bound: each row reads 2 D bytes of z and writes K and V (either may be
// left out).
//
// Backward (D = 512; fp32 throughout, dz rounded to bf16 once):
//   g_k  = adjoint of the RoPE applied to dK: i < R/2: dK_i cos_i + dK_{i+R/2} sin_{i+R/2};
//          R/2 <= i < R: dK_i cos_i - dK_{i-R/2} sin_{i-R/2}; pass dims dK_i
//   g_n  = g_k w + dV,   dw += g_k n  (summed over every row)
//   dz   = r g_n - (r^3 / D) z sum_j(g_n,j z_j)
// dw is summed per workgroup in a fixed order into workspace rows, then the
// rows are summed in a fixed order by a second kernel: no atomics, bitwise
// repeatable.
#include <algorithm>

#include "g4_kernels.h"

namespace g4 {
namespace {

constexpr int kPrepD = 512;
constexpr int kPrepWaves = 4;      // forward: rows in flight per workgroup
constexpr int kPrepBwdWaves = 16;  // backward: more rows per dweight partial row

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// Rows enumerate (batch, token, head) with the head fastest.  64-bit divisions
// and products were half of the forward's instructions, so below 2^31 rows and
// with strides below 2^32 elements the row index is split with multipliers from
// the host and an offset is three 32 x 32 + 64 bit multiply-adds (NARROW);
// anything larger keeps the 64-bit form, and so does the backward, where it
// made no difference (32.3 us for 32768 rows of 512 either way).  So do
// kWideRows rows or more with K in fp32: they no longer fit the caches and are
// bound by HBM (4 TB/s), which the faster issue disturbs (rows of 512, 64-bit /
// NARROW us: 65536 71.9 / 71.8, 131072 135.6 / 137.5, 262144 264 / 267, 524288
// 543 / 564; K in bf16 262144 203 / 201).
constexpr int64_t kWideRows = int64_t(1) << 17;
struct RowMap {
  uint32_t heads_mul, seq_mul;
  int heads_shift, seq_shift;
  bool narrow;
};

// n / d for n < 2^31 is (n * mul) >> (31 + shift), shift = ceil(log2 d),
// mul = floor(2^(31 + shift) / d) + 1: the multiplier is too large by less than
// one part in 2^31 / n, so the quotient is exact (Granlund and Montgomery).
void division(uint32_t d, uint32_t& mul, int& shift) {
  shift = 0;
  while ((uint64_t(1) << shift) < d) ++shift;
  mul = (uint32_t)((uint64_t(1) << (31 + shift)) / d + 1);
}

bool narrow_layout(const g4_layout& l) {
  return ((l.batch_stride | l.token_stride | l.head_stride) >> 32) == 0;
}

template <class... L>
RowMap row_map(const g4_kv_prep& p, const L&... layouts) {
  RowMap m{};
  const int64_t rows = (int64_t)p.num_batches * p.seqlen * p.num_heads;
  m.narrow = rows < (p.k_fp32 ? kWideRows : int64_t(1) << 31) && (p.cs_batch_stride >> 32) == 0 &&
             (narrow_layout(layouts) && ...);
  if (m.narrow) {
    division((uint32_t)p.num_heads, m.heads_mul, m.heads_shift);
    division((uint32_t)p.seqlen, m.seq_mul, m.seq_shift);
  }
  return m;
}

struct RowAddr {
  int64_t b, t, h;
};

__device__ __forceinline__ RowAddr row_of(const g4_kv_prep& p, int64_t row) {
  const int64_t bt = row / p.num_heads;
  return RowAddr{bt / p.seqlen, bt % p.seqlen, row % p.num_heads};
}

template <bool NARROW>
__device__ __forceinline__ RowAddr row_of(const g4_kv_prep& p, const RowMap& m, int64_t row) {
  if constexpr (NARROW) {
    const uint32_t n = (uint32_t)row;
    const uint32_t bt = (uint32_t)(((uint64_t)n * m.heads_mul) >> (31 + m.heads_shift));
    const uint32_t b = (uint32_t)(((uint64_t)bt * m.seq_mul) >> (31 + m.seq_shift));
    return RowAddr{b, bt - b * (uint32_t)p.seqlen, n - bt * (uint32_t)p.num_heads};
  }
  return row_of(p, row);
}

template <bool NARROW>
__device__ __forceinline__ int64_t product(int64_t i, int64_t stride) {
  return NARROW ? (int64_t)((uint64_t)(uint32_t)i * (uint32_t)stride) : i * stride;
}

template <bool NARROW = false>
__device__ __forceinline__ int64_t elem_off(const g4_layout& l, const RowAddr& a) {
  return product<NARROW>(a.b, l.batch_stride) + product<NARROW>(a.t, l.token_stride) +
         product<NARROW>(a.h, l.head_stride);
}

// Offset of a row's token in the cos / sin tables.
template <bool NARROW>
__device__ __forceinline__ int64_t table_off(const g4_kv_prep& p, const RowAddr& a) {
  return product<NARROW>(a.b, p.cs_batch_stride) + product<NARROW>(a.t, p.rotary_dim);
}

__device__ __forceinline__ void load8(const __bf16* p, float (&x)[8]) {
  const bf16x8 v = *(const bf16x8*)p;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (float)v[e];
}

__device__ __forceinline__ void store8(__bf16* p, const float (&x)[8]) {
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (__bf16)x[e];
  *(bf16x8*)p = v;
}

__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
  const f32x4 lo = *(const f32x4*)p;
  const f32x4 hi = *(const f32x4*)(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = lo[e];
    x[4 + e] = hi[e];
  }
}

// D / 8 lanes per row, 8 dims (one 16-byte load) per lane: a wave takes one row
// of 512 or two of 256.  Bound by instructions issued per row before it is by
// HBM, hence two rows of 256 per instruction, partners exchanged as bf16 pairs
// and the cheap row addresses: 32000 rows of 256 (K with RoPE) 14.9 -> 10.7 us,
// 16000 rows 9.2 -> 7.4, 32768 rows of 512 (K in fp32, and V) 30.9 -> 26.4, at
// 5 TB/s.
template <int D, bool NARROW>
__global__ void __launch_bounds__(kPrepWaves * 64) kv_prep_fwd_kernel(
    g4_kv_prep p, RowMap map, const __bf16* z, g4_layout zl, const float* w, const float* cosv,
    const float* sinv, void* k, g4_layout kl, __bf16* v, g4_layout vl, int64_t rows) {
  constexpr int LPR = D / 8;  // lanes per row
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t first = (int64_t)blockIdx.x * (kPrepWaves * 64 / LPR) + threadIdx.x / LPR;
  const int64_t step = (int64_t)gridDim.x * (kPrepWaves * 64 / LPR);
  const int rl = p.rotary_dim / 8;  // lanes holding rotary dims
  const int half = rl / 2;          // lane distance of the rotate-half partner
  float wl[8];
  load8(w + 8 * lane, wl);
  for (int64_t row = first; row < rows; row += step) {
    const RowAddr a = row_of<NARROW>(p, map, row);
    float x[8], c[8], s[8];
    load8(z + elem_off<NARROW>(zl, a) + 8 * lane, x);
    if (k != nullptr && lane < rl) {  // issued with z, before the row reduction waits for it
      const int64_t t = table_off<NARROW>(p, a) + 8 * lane;
      load8(cosv + t, c);
      load8(sinv + t, s);
    }
    // Row sum of the rounded squares.  At 256 the two halves of a lane's dims
    // are summed over the lanes apart and added last: the order of 64 lanes
    // with 4 dims each.
    float ss = 0.f, ss_hi = 0.f;
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int e = 0; e < 8; ++e) (D == 256 && e >= 4 ? ss_hi : ss) += x[e] * x[e];
    }
    if constexpr (D == 256) {
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) {
        ss += __shfl_xor(ss, o, 64);
        ss_hi += __shfl_xor(ss_hi, o, 64);
      }
      ss += ss_hi;
    } else {
      ss = wave_sum(ss);
    }
    const float r = 1.f / __fsqrt_rn(ss / (float)D + p.eps);
    float n[8];
    bf16x8 kb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      n[e] = x[e] * r;
      kb[e] = (__bf16)(n[e] * wl[e]);
    }
    if (v != nullptr) store8(v + elem_off<NARROW>(vl, a) + 8 * lane, n);
    if (k == nullptr) continue;
    // rotate-half partner values, two bf16 per exchange (every lane of the row takes part)
    const int partner = lane < half ? lane + half : lane - half;
    const i32x4 kw = __builtin_bit_cast(i32x4, kb);
    i32x4 pw;
#pragma unroll
    for (int e = 0; e < 4; ++e) pw[e] = __shfl(kw[e], partner, LPR);
    const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
    float kout[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) kout[e] = (float)kb[e];
    if (lane < rl) {
      // x * cos + rotate_half(x) * sin as two products and a sum, no fused
      // multiply-add; in bf16 each product is rounded before the sum (the
      // products of bf16 values are exact in fp32, so one rounding each)
#pragma clang fp contract(off)
      const float sign = lane < half ? -1.f : 1.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float a0 = kout[e] * c[e];
        float a1 = (sign * (float)pb[e]) * s[e];
        if (!p.k_fp32) {
          a0 = (float)(__bf16)a0;
          a1 = (float)(__bf16)a1;
        }
        kout[e] = a0 + a1;
      }
    }
    const int64_t off = elem_off<NARROW>(kl, a) + 8 * lane;
    if (p.k_fp32) {
      float* kp = (float*)k + off;
      *(f32x4*)kp = f32x4{kout[0], kout[1], kout[2], kout[3]};
      *(f32x4*)(kp + 4) = f32x4{kout[4], kout[5], kout[6], kout[7]};
    } else {
      store8((__bf16*)k + off, kout);
    }
  }
}

// cos / sin of a row's token for this lane's dims (lanes below R / 8 only).
__device__ __forceinline__ void load_rope(const g4_kv_prep& p, const float* cs, const RowAddr& a,
                                          int lane, float (&x)[8]) {
  const float* src = cs + a.b * p.cs_batch_stride + a.t * (int64_t)p.rotary_dim + 8 * lane;
  const f32x4 lo = *(const f32x4*)src;
  const f32x4 hi = *(const f32x4*)(src + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = lo[e];
    x[4 + e] = hi[e];
  }
}

// dK of this lane's dims, from a bf16 or fp32 gradient.
__device__ __forceinline__ void load_dk(const g4_kv_prep& p, const void* dk, int64_t off,
                                        float (&x)[8]) {
  if (p.k_fp32) {
    const float* q = (const float*)dk + off;
    const f32x4 lo = *(const f32x4*)q;
    const f32x4 hi = *(const f32x4*)(q + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = lo[e];
      x[4 + e] = hi[e];
    }
  } else {
    load8((const __bf16*)dk + off, x);
  }
}

__global__ void __launch_bounds__(kPrepBwdWaves * 64) kv_prep_bwd_kernel(
    g4_kv_prep p, const __bf16* z, g4_layout zl, const float* w, const float* cosv,
    const float* sinv, const void* dk, g4_layout dkl, const __bf16* dv, g4_layout dvl,
    __bf16* dz, g4_layout dzl, float* dw_part, int64_t rows) {
  __shared__ f32x4 red[kPrepBwdWaves][64][2];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t first = (int64_t)blockIdx.x * kPrepBwdWaves + wave;
  const int64_t step = (int64_t)gridDim.x * kPrepBwdWaves;
  const int rl = p.rotary_dim / 8;
  const int half = rl / 2;
  float wl[8], dwl[8];
  {
    const f32x4 lo = *(const f32x4*)(w + 8 * lane);
    const f32x4 hi = *(const f32x4*)(w + 8 * lane + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      wl[e] = lo[e];
      wl[4 + e] = hi[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) dwl[e] = 0.f;
  const int partner = lane < half ? lane + half : lane - half;
  for (int64_t row = first; row < rows; row += step) {
    const RowAddr a = row_of(p, row);
    float x[8], gk[8], gv[8], c[8], ps[8];  // cos of this lane's dims, sin of the partner's
    load8(z + elem_off(zl, a) + 8 * lane, x);
    load_dk(p, dk, elem_off(dkl, a) + 8 * lane, gk);
    load8(dv + elem_off(dvl, a) + 8 * lane, gv);
    if (lane < rl) {
      load_rope(p, cosv, a, lane, c);
      load_rope(p, sinv, a, partner, ps);
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
    ss = wave_sum(ss);
    const float r = 1.f / __fsqrt_rn(ss / (float)kPrepD + p.eps);
    // adjoint of the RoPE: the partner lane's dK times its sin
    float pg[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) pg[e] = __shfl(gk[e], partner, 64);
    if (lane < rl) {
      const float sign = lane < half ? 1.f : -1.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) gk[e] = gk[e] * c[e] + sign * pg[e] * ps[e];
    }
    float gn[8], dot = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float n = x[e] * r;
      gn[e] = gk[e] * wl[e] + gv[e];
      dwl[e] += gk[e] * n;
      dot += gn[e] * x[e];
    }
    dot = wave_sum(dot);
    const float coef = r * r * r * dot / (float)kPrepD;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = r * gn[e] - coef * x[e];
    store8(dz + elem_off(dzl, a) + 8 * lane, o);
  }
  // fixed-order sum of the waves' dw partials, one 512-float row per workgroup
  red[wave][lane][0] = f32x4{dwl[0], dwl[1], dwl[2], dwl[3]};
  red[wave][lane][1] = f32x4{dwl[4], dwl[5], dwl[6], dwl[7]};
  __syncthreads();
  if (wave == 0) {
    f32x4 s0 = red[0][lane][0], s1 = red[0][lane][1];
#pragma unroll
    for (int wv = 1; wv < kPrepBwdWaves; ++wv) {
      s0 += red[wv][lane][0];
      s1 += red[wv][lane][1];
    }
    float* dst = dw_part + (int64_t)blockIdx.x * kPrepD + 8 * lane;
    *(f32x4*)dst = s0;
    *(f32x4*)(dst + 4) = s1;
  }
}

// dw[d] = sum over workgroups of dw_part[b][d] in a fixed order: a block owns
// 8 columns; thread (g, c) sums rows b = g, g + 32, ... of column c in order,
// then thread g = 0 adds the 32 group sums in group order.
__global__ void __launch_bounds__(256) kv_prep_dw_kernel(const float* dw_part, int nparts,
                                                         float* dw) {
  __shared__ float part[32][8];
  const int c = threadIdx.x & 7, g = threadIdx.x >> 3;
  const int d = blockIdx.x * 8 + c;
  float s = 0.f;
  for (int b = g; b < nparts; b += 32) s += dw_part[(int64_t)b * kPrepD + d];
  part[g][c] = s;
  __syncthreads();
  if (g == 0) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) t += part[i][c];
    dw[d] = t;
  }
}

}  // namespace

// Workgroups of the backward (each writes one row of dweight partials):
// enough waves to keep HBM busy, few partial rows to sum.
int kv_prep_blocks(int64_t rows) {
  const int64_t want = (rows + kPrepBwdWaves - 1) / kPrepBwdWaves;
  return (int)std::min<int64_t>(want, 512);
}

size_t kv_prep_workspace_bytes(const g4_kv_prep& p) {
  const int64_t rows = (int64_t)p.num_batches * p.seqlen * p.num_heads;
  return (size_t)kv_prep_blocks(rows) * kPrepD * sizeof(float);
}

hipError_t launch_kv_prep_fwd(const g4_kv_prep& p, const void* z, g4_layout zl, const float* w,
                              const float* cosv, const float* sinv, void* k, g4_layout kl,
                              void* v, g4_layout vl, hipStream_t stream) {
  const int64_t rows = (int64_t)p.num_batches * p.seqlen * p.num_heads;
  if (rows <= 0) return hipSuccess;
  const int per_block = kPrepWaves * 512 / p.head_dim;
  const int blocks = (int)std::min<int64_t>((rows + per_block - 1) / per_block, 4096);
  const RowMap map = row_map(p, zl, k != nullptr ? kl : zl, v != nullptr ? vl : zl);
  const auto kernel = p.head_dim == 256
                          ? (map.narrow ? kv_prep_fwd_kernel<256, true> : kv_prep_fwd_kernel<256, false>)
                          : (map.narrow ? kv_prep_fwd_kernel<512, true> : kv_prep_fwd_kernel<512, false>);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kPrepWaves * 64), 0, stream, p, map,
                     (const __bf16*)z, zl, w, cosv, sinv, k, kl, (__bf16*)v, vl, rows);
  return hipGetLastError();
}

hipError_t launch_kv_prep_bwd(const g4_kv_prep& p, const void* z, g4_layout zl, const float* w,
                              const float* cosv, const float* sinv, const void* dk,
                              g4_layout dkl, const void* dv, g4_layout dvl, void* dz,
                              g4_layout dzl, float* dw, void* ws, hipStream_t stream) {
  const int64_t rows = (int64_t)p.num_batches * p.seqlen * p.num_heads;
  const int blocks = rows > 0 ? kv_prep_blocks(rows) : 0;
  if (blocks > 0) {
    hipLaunchKernelGGL(kv_prep_bwd_kernel, dim3(blocks), dim3(kPrepBwdWaves * 64), 0, stream, p,
                       (const __bf16*)z, zl, w, cosv, sinv, dk, dkl, (const __bf16*)dv, dvl,
                       (__bf16*)dz, dzl, (float*)ws, rows);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kv_prep_dw_kernel, dim3(kPrepD / 8), dim3(256), 0, stream,
                     (const float*)ws, blocks, dw);
  return hipGetLastError();
}

}  // namespace g4
