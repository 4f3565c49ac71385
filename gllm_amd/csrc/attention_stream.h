// Generic attention for few query rows per launch (decode, short chunks):
// paged attention and the dense-bias op for fp32 models, for bf16 / fp16
// models whose head dim the MFMA kernels do not take (not 64 or 128; up to
// 256), and for a 16-bit model over a cache of another dtype (f32, or the
// other 16-bit type).  Batches that fill the GPU with 128-column workgroups
// run on attention_tile.h.  fp32 arithmetic on v_mfma_f32_16x16x4_f32 with
// an exact online softmax (expf).  Compiled with -ffp-contract=off so the q
// rotation rounds each op like the reference
// (gllm/model/layers/attention.py:105-118): in fp32, or to the 16-bit model
// dtype after every op.
#pragma once
#include "common.h"
#include "generic.h"
#include "launch.h"

namespace gllm {

// A value of the model dtype stored in the cache dtype, as torch's
// .to(kv_dtype) rounds it (to nearest even; fp8: NaN -> 0x7f|sign).
template <typename KV> __device__ __forceinline__ KV to_kv(float x);
template <> __device__ __forceinline__ float to_kv<float>(float x) { return x; }
template <> __device__ __forceinline__ __bf16 to_kv<__bf16>(float x) {
  return __builtin_bit_cast(__bf16, (uint16_t)pack_bf16x2(x, 0.f));
}
template <> __device__ __forceinline__ _Float16 to_kv<_Float16>(float x) { return (_Float16)x; }
template <> __device__ __forceinline__ fp8e4m3 to_kv<fp8e4m3>(float x) { return fp8e4m3{fp8_byte(x)}; }

// 4 consecutive elements of one row, dims d .. d + 3: raw words in registers
// until use, then the fp32 values the reference's gather gives (dims past D: 0).
// V = 4 (D a multiple of 4): one load of all four, whatever the row's alignment
// (global loads need none); a chunk past dim D re-reads the row's last one.
// V = 2 (other D >= 4): the same, and last2 puts the dims of the chunk that
// dim D cuts in place.  V = 1 (D < 4): element by element.
template <typename KV> struct Raw4 { uint32_t w[sizeof(KV)]; };
template <typename KV, int V>
__device__ __forceinline__ Raw4<KV> ld_raw4(const KV* row, int d, int D) {
  Raw4<KV> r;
  if constexpr (V > 1) {
    __builtin_memcpy(&r, reinterpret_cast<const char*>(row + min(d, D - 4)), sizeof(r));
  } else {
#pragma unroll
    for (int i = 0; i < (int)sizeof(KV); ++i) r.w[i] = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int de = min(d + e, D - 1);
      if constexpr (sizeof(KV) == 4) r.w[e] = reinterpret_cast<const uint32_t*>(row)[de];
      else if constexpr (sizeof(KV) == 2) r.w[e / 2] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[de] << (16 * (e % 2));
      else r.w[0] |= (uint32_t)reinterpret_cast<const uint8_t*>(row)[de] << (8 * e);
    }
  }
  return r;
}
// The chunk of dims D - 2, D - 1 (D even), loaded as the row's last four.
template <typename KV>
__device__ __forceinline__ void last2(Raw4<KV>& r, bool last) {
  if constexpr (sizeof(KV) == 1) {
    r.w[0] = last ? r.w[0] >> 16 : r.w[0];
  } else {
#pragma unroll
    for (int i = 0; i < (int)sizeof(KV) / 2; ++i) r.w[i] = last ? r.w[i + sizeof(KV) / 2] : r.w[i];
  }
}
template <typename KV, typename QT>
__device__ __forceinline__ f32x4 widen4(const Raw4<KV>& r) {
  f32x4 x;
  if constexpr (std::is_same<KV, float>::value) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = __uint_as_float(r.w[i]);
  } else if constexpr (std::is_same<KV, fp8e4m3>::value) {
    float v[4];
    unpack_fp8x4(r.w[0], v);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x[2 * i] = E16<KV>::lo(r.w[i]);
      x[2 * i + 1] = E16<KV>::hi(r.w[i]);
    }
  }
  constexpr bool exact = std::is_same<QT, float>::value || std::is_same<KV, QT>::value ||
                         std::is_same<KV, fp8e4m3>::value;
  if constexpr (!exact) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = rnd<QT>(x[i]);
  }
  return x;
}

// The same four elements as two packed words of a 16-bit model dtype (exact:
// the gather's cast gives values of QT).
template <typename KV, typename QT>
__device__ __forceinline__ u32x2 pack4(const Raw4<KV>& r) {
  if constexpr (std::is_same<KV, QT>::value) {
    return u32x2{r.w[0], r.w[1]};
  } else if constexpr (std::is_same<KV, fp8e4m3>::value) {
    return u32x2{E16<QT>::template fp8x2<false>(r.w[0]), E16<QT>::template fp8x2<true>(r.w[0])};
  } else {
    const f32x4 x = widen4<KV, QT>(r);
    return u32x2{E16<QT>::pack2(x[0], x[1]), E16<QT>::pack2(x[2], x[3])};
  }
}

// One workgroup per (sequence, kv head, 16 columns); a column is a (query row,
// head of the group) pair, c = r G + g, so a decode step's G heads share one
// pass over the keys.  The NW waves take the keys 16 at a time in turn, K and V
// straight from memory into MFMA operand registers, PF sub-tiles ahead:
//   S^T = K Q^T, 16x16x4: lane (n, grp) loads dims 16t + 4grp .. + 3 of key n;
//     element e of the four is the k = grp operand of step (t, e), Q likewise.
//   O^T += V^T P^T: score j of a lane is key 4grp + j of column n, which is
//     already the B operand of step j; A is V[key 4grp + j][64u + 4n + e], so
//     one 4-element load per (j, u) feeds the four output blocks e.
// A 16-bit model's K, V and q are 16-bit values, so its S runs on the 16x16x32
// instruction (products exact, fp32 sums).  P stays in fp32, and so does P V: P in
// two 16-bit parts lost bits (fp16 parts of a small p are subnormal) and turned an
// infinity in V into a NaN, and three parts with V's infinities kept from the low
// ones cost as much as fp32 (bf16, 1 x 2048 keys, D = 96 and 256: 48 and 86 us).
// Head dims that are no multiple of 4, and rows at odd offsets, read whole chunks
// too: a 16-bit row of D = 50 loaded element by element into 256-dim registers took
// 352 us (fp32 638) for one row on 2048 keys, 22 (37) so.
// The waves' (max, sum, acc) merge through LDS at the end.  Latency-bound at
// short contexts (one round trip per PF sub-tiles), HBM-bound beyond.  Against
// one workgroup per (query head, query row) with VALU dot products, which read
// K/V once per query head (32 / 8 heads, fp32, us before -> after): 32
// sequences x 2 rows x 2048 keys 427 -> 48 at D = 64 (5.6 TB/s of K/V), 462 ->
// 118 at D = 128; 1 x 2 x 2048 54 -> 35; 8 x 16 x 256 213 -> 12.
// FUSED (a.k_new != null, at most kFusedRows query rows per sequence): the
// new tokens' K/V are written by this launch.  Every workgroup rotates and
// casts the sequence's new keys into LDS, the value the cache round trip gives
// (stored in KV, read back as QT); the sub-tiles cover the cached keys
// [0, ctx), and one wave takes the new ones from LDS as a last sub-tile.  The
// workgroup of the first column stores them at their slots (block table); no
// workgroup of the launch reads those slots.
constexpr int kFusedRows = 16;
template <typename KV, typename QT, int DP, int V>
struct StreamCfg {
  static constexpr int kBytes = DP * (int)sizeof(KV);      // K (or V) bytes per key
  static constexpr int kNW = kBytes > 512 || V == 1 ? 4 : 8; // waves that split the keys (registers)
  static constexpr int kQS = DP + 4;                       // floats per LDS row of q, the new keys and the merge
  static constexpr int kMerge = kNW * 16 * kQS;
  template <bool FUSED> static constexpr int stage() { return (16 + (FUSED ? 32 : 0)) * kQS; }
  template <bool FUSED> static constexpr int lds() { return kMerge > stage<FUSED>() ? kMerge : stage<FUSED>(); }
  // sub-tiles in flight beside the current one (registers; at DP 256 the waves
  // overlap each other's loads instead, and other head dims than multiples of
  // 4 are rare)
  static constexpr int kPF = V < 4 || DP == 256 ? 0 : (kBytes <= 256 ? 2 : 1);
};
template <bool DENSE, typename KV, typename QT, int DP, bool FUSED, int V>
__global__ void __launch_bounds__((64 * StreamCfg<KV, QT, DP, V>::kNW)) attn_stream_kernel(AttnArgs a) {
  using Cfg = StreamCfg<KV, QT, DP, V>;
  constexpr int NW = Cfg::kNW, PF = Cfg::kPF;
  constexpr int NT = DP / 16;             // K steps of 16 dims
  constexpr int NU = DP / 64;             // V column groups of 64 dims
  constexpr int QS = Cfg::kQS;
  constexpr bool k16 = sizeof(QT) == 2;   // 16-bit MFMA (above)
  // q of the columns, the new keys' K and V (FUSED); the merge reuses the area
  __shared__ __attribute__((aligned(16))) float lds[Cfg::template lds<FUSED>()];
  __shared__ float mml[NW][16][2];
  float (*const qs)[QS] = reinterpret_cast<float (*)[QS]>(lds);
  float (*const nk)[QS] = reinterpret_cast<float (*)[QS]>(lds + 16 * QS);
  float (*const nv)[QS] = reinterpret_cast<float (*)[QS]>(lds + 32 * QS);
  float (*const macc)[16][QS] = reinterpret_cast<float (*)[16][QS]>(lds);
  static_assert(kFusedRows == 16, "LDS layout");
  const int wgrp = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, grp = lane >> 4;
  const int D = a.head_dim, half = D / 2;
  const int G = a.num_q_heads / a.num_kv_heads;
  int ctx, qlen, L;
  int64_t row0;
  if (DENSE) {
    ctx = 0;
    qlen = a.dense_Tq;
    L = a.dense_T;
    row0 = (int64_t)b * a.dense_Tq;
  } else {
    if (b >= a.num_seqs) return;
    const SeqInfo si = a.seqs[b];
    ctx = si.ctx_len;
    qlen = si.q_len;
    L = ctx + qlen;
    row0 = si.q_row_start;
  }
  const int ncol = qlen * G, c0 = wgrp * 16;
  if (c0 >= ncol || (!DENSE && a.tile_min_q > 0 && qlen >= a.tile_min_q)) return;   // the latter: attn_tile_kernel's
  const int col = min(c0 + n, ncol - 1);
  const int r = col / G, g = col - r * G;
  const int r_last = (min(c0 + 16, ncol) - 1) / G;
  const int nkeys = DENSE ? L : (FUSED ? ctx : ctx + r_last + 1);
  const int vis = DENSE ? L - 1 : ctx + r;       // last visible key of the lane's column
  const int32_t* bt = DENSE ? nullptr : a.block_table + (int64_t)b * a.block_table_stride;
  const KV* kbase = DENSE ? (const KV*)a.k + (int64_t)b * a.k_batch_stride + (int64_t)kvh * D
                          : (const KV*)a.k_cache + (int64_t)kvh * D;
  const KV* vbase = DENSE ? (const KV*)a.v + (int64_t)b * a.v_batch_stride + (int64_t)kvh * D
                          : (const KV*)a.v_cache + (int64_t)kvh * D;
  const int64_t kstride = DENSE ? a.k_row_stride : a.cache_slot_stride;
  const int64_t vstride = DENSE ? a.v_row_stride : a.cache_slot_stride;
  const QT* brow = DENSE ? (const QT*)a.bias + (int64_t)b * a.bias_batch_stride + (int64_t)r * a.bias_row_stride
                         : nullptr;

  // this wave's sub-tiles: 16 keys from 16 (wave + NW t), t < ntw
  const int nsub = (nkeys + 15) >> 4;
  const int ntw = nsub > wave ? (nsub - wave + NW - 1) / NW : 0;
  // block id of the lane's key n of sub-tile t (fetched a sub-tile ahead of
  // its K/V); lanes of grp share it
  auto block_of = [&](int t) -> uint32_t {
    if (DENSE) return 0;
    const int key = min(16 * (wave + NW * t) + n, nkeys - 1);
    return (uint32_t)bt[div_bs((uint32_t)key, a.block_magic, a.block_shift)];
  };
  struct Tile {
    Raw4<KV> k[NT];
    Raw4<KV> v[4][NU];
    float bias[DENSE ? 4 : 1];
  };
  auto issue = [&](int t, uint32_t blk, Tile& x) {
    const int p0 = 16 * (wave + NW * t);
    const int key = min(p0 + n, nkeys - 1);      // keys past the end: masked, re-read the last
    int64_t row = key;
    if (!DENSE) {
      const uint32_t bi = div_bs((uint32_t)key, a.block_magic, a.block_shift);
      if (blk >= (uint64_t)a.num_blocks) blk = 0;   // never address outside the pool
      row = (int64_t)blk * a.block_size + (key - (int)bi * a.block_size);
    }
    const KV* kp = kbase + row * kstride;
#pragma unroll
    for (int u = 0; u < NT; ++u) x.k[u] = ld_raw4<KV, V>(kp, 16 * u + 4 * grp, D);
#pragma unroll
    for (int j = 0; j < 4; ++j) {                // row of key 4grp + j: lane 4grp + j of the first 16 holds it
      const int src = 4 * grp + j;
      const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)row, src, 64);
      const uint32_t hi = (uint32_t)__shfl((int)((uint64_t)row >> 32), src, 64);
      const KV* vp = vbase + (int64_t)(((uint64_t)hi << 32) | lo) * vstride;
#pragma unroll
      for (int u = 0; u < NU; ++u) x.v[j][u] = ld_raw4<KV, V>(vp, 64 * u + 4 * n, D);
    }
    if constexpr (DENSE) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x.bias[j] = (float)brow[min(p0 + 4 * grp + j, L - 1)];
    }
  };
  Tile ring[PF + 1];
  uint32_t blk[PF + 1];                          // blk[t % (PF + 1)]: the block id of sub-tile t
  if (ntw > 0) {
#pragma unroll
    for (int u = 0; u <= PF; ++u) blk[u] = block_of(u);
#pragma unroll
    for (int u = 0; u < PF; ++u) issue(u, blk[u], ring[u]);
  }

  // q, rotated, in the tile order of columns
  for (int e = tid; e < 16 * (DP / 2); e += 64 * NW) {
    const int cc = e / (DP / 2), j = e - cc * (DP / 2);      // pair (j, j + D/2)
    const int gc = min(c0 + cc, ncol - 1);
    const int rq = gc / G, gq = gc - rq * G;
    if (j < half) {
      const QT* qp = (const QT*)a.q + (row0 + rq) * a.q_row_stride + (int64_t)(kvh * G + gq) * D;
      float x1 = (float)qp[j], x2 = (float)qp[j + half];
      if (!DENSE && a.rope_mode != kRopeNone) {
        const int64_t crow = a.rope_mode == kRopeByPosition ? (int64_t)(ctx + rq) : row0 + rq;
        const float c = (float)((const QT*)a.rope_cos)[crow * a.rope_row_stride + j];
        const float s = (float)((const QT*)a.rope_sin)[crow * a.rope_row_stride + j];
        const float lo = rnd<QT>(__fsub_rn(rnd<QT>(__fmul_rn(x1, c)), rnd<QT>(__fmul_rn(x2, s))));
        const float hi = rnd<QT>(__fadd_rn(rnd<QT>(__fmul_rn(x1, s)), rnd<QT>(__fmul_rn(x2, c))));
        x1 = lo;
        x2 = hi;
      }
      qs[cc][j] = x1;
      qs[cc][j + half] = x2;
    } else {                                     // dims D .. DP - 1 (D = 2 half): zeros
      qs[cc][2 * j] = 0.f;
      qs[cc][2 * j + 1] = 0.f;
    }
  }
  if constexpr (FUSED) {
    // element pairs (token t, dims j and j + D/2)
    const bool writer = wgrp == 0;
    for (int e = tid; e < 16 * (DP / 2); e += 64 * NW) {
      const int t = e / (DP / 2), j = e - t * (DP / 2);
      if (t >= qlen) {                             // no such key: weight 0, V 0
        nv[t][2 * j] = nv[t][2 * j + 1] = 0.f;
        continue;
      }
      if (j >= half) {
        nk[t][2 * j] = nk[t][2 * j + 1] = 0.f;
        nv[t][2 * j] = nv[t][2 * j + 1] = 0.f;
        continue;
      }
      const int64_t row = row0 + t;
      const QT* kn = (const QT*)a.k_new + row * a.k_new_row_stride + (int64_t)kvh * D;
      const QT* vn = (const QT*)a.v_new + row * a.v_new_row_stride + (int64_t)kvh * D;
      float lo = (float)kn[j], hi = (float)kn[j + half];
      if (a.rope_mode != kRopeNone) {
        const int64_t crow = a.rope_mode == kRopeByPosition ? (int64_t)(ctx + t) : row;
        const float c = (float)((const QT*)a.rope_cos)[crow * a.rope_row_stride + j];
        const float sn = (float)((const QT*)a.rope_sin)[crow * a.rope_row_stride + j];
        const float x1 = lo, x2 = hi;
        lo = rnd<QT>(__fsub_rn(rnd<QT>(__fmul_rn(x1, c)), rnd<QT>(__fmul_rn(x2, sn))));
        hi = rnd<QT>(__fadd_rn(rnd<QT>(__fmul_rn(x1, sn)), rnd<QT>(__fmul_rn(x2, c))));
      }
      const KV k1 = to_kv<KV>(lo), k2 = to_kv<KV>(hi);
      const KV v1 = to_kv<KV>((float)vn[j]), v2 = to_kv<KV>((float)vn[j + half]);
      nk[t][j] = kvld<KV, QT>(&k1);
      nk[t][j + half] = kvld<KV, QT>(&k2);
      nv[t][j] = kvld<KV, QT>(&v1);
      nv[t][j + half] = kvld<KV, QT>(&v2);
      if (writer) {
        const int p = ctx + t;
        const uint32_t bi = div_bs((uint32_t)p, a.block_magic, a.block_shift);
        const uint32_t nb = (uint32_t)bt[bi];
        if (nb < (uint64_t)a.num_blocks) {   // never address outside the pool
          const int64_t off = ((int64_t)nb * a.block_size + (p - (int64_t)bi * a.block_size)) * a.cache_slot_stride +
                              (int64_t)kvh * D + j;
          KV* kc = (KV*)a.k_cache + off;
          KV* vc = (KV*)a.v_cache + off;
          kc[0] = k1; kc[half] = k2;
          vc[0] = v1; vc[half] = v2;
        }
      }
    }
  }
  __syncthreads();
  f32x4 qv[k16 ? 1 : NT];
  u32x4 qh[k16 ? NT / 2 : 1];             // 16-bit: dims 32t + 4grp .. + 3 and 32t + 16 + 4grp .. + 3
  if constexpr (k16) {
#pragma unroll
    for (int u = 0; u < NT / 2; ++u) {
      const float* q0 = &qs[n][32 * u + 4 * grp];
      qh[u] = u32x4{E16<QT>::pack2(q0[0], q0[1]), E16<QT>::pack2(q0[2], q0[3]), E16<QT>::pack2(q0[16], q0[17]),
                    E16<QT>::pack2(q0[18], q0[19])};
    }
  } else {
#pragma unroll
    for (int u = 0; u < NT; ++u) qv[u] = *reinterpret_cast<const f32x4*>(&qs[n][16 * u + 4 * grp]);
  }

  float m = kNegInf, l = 0.f;
  f32x4 o[NU][4];
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[u][e] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One sub-tile: kf(u) = K dims 16u + 4grp .. + 3 of key n, vf(j, u) = V dims
  // 64u + 4n .. + 3 of key 4grp + j (fp32 values, or packed words of a 16-bit
  // model); lim: keys 4grp + j <= lim are visible
  auto tile = [&](auto kf, auto vf, int lim, bool mask, const float* bias) {
    // two chains: half the length of the fp32 sums; from 128 dims on, the fp32
    // products' in two halves of the dims
    f32x4 s = {0.f, 0.f, 0.f, 0.f}, s1 = s, sh = s;
    if constexpr (k16) {
#pragma unroll
      for (int u = 0; u < NT / 2; ++u) {
        const u32x2 k0 = kf(2 * u), k1 = kf(2 * u + 1);
        f32x4& c = u & 1 ? s1 : s;
        c = E16<QT>::mfma16(u32x4{k0[0], k0[1], k1[0], k1[1]}, qh[u], c);
      }
    } else {
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        if (DP >= 128 && u == NT / 2) {
          sh = s + s1;
          s = s1 = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const f32x4 kk = kf(u);
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          s = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e], qv[u][e], s, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e + 1], qv[u][e + 1], s1, 0, 0, 0);
        }
      }
    }
    s += s1;
    if (!k16 && DP >= 128) s += sh;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] *= a.scale;
      if constexpr (DENSE) s[j] += bias[j];
      if (mask && 4 * grp + j > lim) s[j] = kNegInf;
    }
    float tm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    tm = max_xor32(max_xor16(tm));
    const float mn = fmaxf(m, tm);
    const float mu = mn == kNegInf ? 0.f : mn;   // every key so far masked: all weights 0
    const float alpha = expf(m - mu);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = expf(s[j] - mu);
    l = l * alpha + ((s[0] + s[1]) + (s[2] + s[3]));
    m = mn;
    // the sub-tile's P V from zero, then one FMA per output with the rescale
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      f32x4 w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 vv;
        if constexpr (k16) {
          const u32x2 x = vf(j, u);
          vv = f32x4{E16<QT>::lo(x[0]), E16<QT>::hi(x[0]), E16<QT>::lo(x[1]), E16<QT>::hi(x[1])};
        } else {
          vv = vf(j, u);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[e], s[j], w[e], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[u][e][i] = __builtin_fmaf(o[u][e][i], alpha, w[e][i]);
    }
  };
  const bool tail = D != DP;
  auto compute = [&](int t, Tile& x) {
    const int p0 = 16 * (wave + NW * t);
    if constexpr (V == 2) {
#pragma unroll
      for (int u = 0; u < NT; ++u) last2(x.k[u], 16 * u + 4 * grp + 2 == D);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int u = 0; u < NU; ++u) last2(x.v[j][u], 64 * u + 4 * n + 2 == D);
    }
    const int lim = min(vis, nkeys - 1) - p0;
    const bool mask = p0 + 16 > nkeys || (!DENSE && p0 + 15 > ctx);
    if constexpr (k16) {
      tile(
          [&](int u) {
            u32x2 kk = pack4<KV, QT>(x.k[u]);
            if (tail) {                          // an even D ends on a whole word
#pragma unroll
              for (int e = 0; e < 2; ++e) kk[e] = 16 * u + 4 * grp + 2 * e < D ? kk[e] : 0u;
            }
            return kk;
          },
          [&](int j, int u) { return pack4<KV, QT>(x.v[j][u]); }, lim, mask, x.bias);
    } else {
      tile(
          [&](int u) {
            f32x4 kk = widen4<KV, QT>(x.k[u]);
            if (tail) {
#pragma unroll
              for (int e = 0; e < 4; ++e) kk[e] = 16 * u + 4 * grp + e < D ? kk[e] : 0.f;
            }
            return kk;
          },
          [&](int j, int u) { return widen4<KV, QT>(x.v[j][u]); }, lim, mask, x.bias);
    }
  };
  // Loads are issued unconditionally in whole groups of PF + 1 sub-tiles (past
  // the last one every lane re-reads the last key's row, one line per load), so
  // their order is the same on every path and the waits keep PF sub-tiles in
  // flight; the tail issues nothing.
  int t0 = 0;
  for (; t0 + PF < ntw; t0 += PF + 1) {
#pragma unroll
    for (int u = 0; u <= PF; ++u) {
      const int t = t0 + u, w = (u + PF) % (PF + 1);
      issue(t + PF, blk[w], ring[w]);
      blk[u] = block_of(t + PF + 1);
      __builtin_amdgcn_sched_barrier(0);
      compute(t, ring[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (t0 + u < ntw) compute(t0 + u, ring[u]);
  if constexpr (FUSED) {
    // the new keys ctx .. ctx + qlen - 1 (row r sees the first r + 1), from LDS
    if (wave == nsub % NW) {
      auto get = [&](const float* p) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(p);
        if constexpr (k16) return u32x2{E16<QT>::pack2(x[0], x[1]), E16<QT>::pack2(x[2], x[3])};
        else return x;
      };
      tile([&](int u) { return get(&nk[min(n, qlen - 1)][16 * u + 4 * grp]); },
           [&](int j, int u) { return get(&nv[4 * grp + j][64 * u + 4 * n]); }, r, true, nullptr);
    }
  }
  l = sum_xor32(sum_xor16(l));

  // merge the waves' states (exact LSE merge; a wave without keys has
  // m = -inf and weight 0).  o[u][e][i] is dim 64u + 4(4grp + i) + e.
  __syncthreads();                        // every wave is done with q and the new keys
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(&macc[wave][n][64 * u + 16 * grp + 4 * i]) =
          f32x4{o[u][0][i], o[u][1][i], o[u][2][i], o[u][3][i]};
  if (grp == 0) {
    mml[wave][n][0] = m;
    mml[wave][n][1] = l;
  }
  __syncthreads();
  // thread: 4 dims of one column
  for (int e = tid; e < 16 * (DP / 4); e += 64 * NW) {
    const int cc = e / (DP / 4), d = 4 * (e - cc * (DP / 4));
    if (c0 + cc >= ncol || d >= D) continue;
    float M = kNegInf;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, mml[w][cc][0]);
    float lt = 0.f;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = mml[w][cc][0];
      const float wt = mw == kNegInf ? 0.f : expf(mw - M);
      lt += wt * mml[w][cc][1];
      x += wt * *reinterpret_cast<const f32x4*>(&macc[w][cc][d]);
    }
    const int rq = (c0 + cc) / G, gq = (c0 + cc) - rq * G;
    QT* op = (QT*)a.out + (row0 + rq) * a.out_row_stride + (int64_t)(kvh * G + gq) * D + d;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] /= lt;   // lt == 0 (every key masked) gives NaN, as torch's softmax
    if (a.vec_out) {                          // D a multiple of 4, rows aligned to 4 elements
      if constexpr (sizeof(QT) == 4) *reinterpret_cast<f32x4*>(op) = x;
      else st8(op, u32x2{E16<QT>::pack2(x[0], x[1]), E16<QT>::pack2(x[2], x[3])});
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (d + i < D) stq<QT>(op + i, x[i]);
    }
  }
}

template <bool DENSE, typename KV, typename QT, bool FUSED>
static hipError_t launch_stream_d(const AttnArgs& a, dim3 grid, hipStream_t st) {
  auto go = [&](auto dp, auto v) {
    constexpr int DP = decltype(dp)::value, V = decltype(v)::value;
    const dim3 block(64 * StreamCfg<KV, QT, DP, V>::kNW);
    hipLaunchKernelGGL((attn_stream_kernel<DENSE, KV, QT, DP, FUSED, V>), grid, block, 0, st, a);
  };
  auto by_dim = [&](auto v) {
    if (a.head_dim <= 64) go(std::integral_constant<int, 64>(), v);
    else if (a.head_dim <= 128) go(std::integral_constant<int, 128>(), v);
    else go(std::integral_constant<int, 256>(), v);
  };
  if (a.head_dim % 4 == 0) by_dim(std::integral_constant<int, 4>());
  else if (a.head_dim > 4) by_dim(std::integral_constant<int, 2>());
  else go(std::integral_constant<int, 64>(), std::integral_constant<int, 1>());
  return hipGetLastError();
}

// Cache dtype KV under model dtype QT (paged), or QT throughout (dense).
template <typename QT>
static hipError_t launch_stream_t(const AttnArgs& a, bool dense, dim3 grid, hipStream_t st) {
  if (dense) return launch_stream_d<true, QT, QT, false>(a, grid, st);
  auto go = [&](auto kv) {
    using KV = decltype(kv);
    return a.k_new ? launch_stream_d<false, KV, QT, true>(a, grid, st) : launch_stream_d<false, KV, QT, false>(a, grid, st);
  };
  switch (a.kv_dtype) {
    case kF32: return go(float{});
    case kBF16: return go(__bf16{});
    case kF16: return go(_Float16{});
    case kFP8: return go(fp8e4m3{});
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gllm
