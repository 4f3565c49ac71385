// Tiled generic attention: the prefill rows (paged) and the dense-bias op for
// what the bf16 / fp16 MFMA kernels do not take: fp32 models, 16-bit models
// whose head dim is not 64 or 128 (any even D up to 256), and a 16-bit model
// over a cache of another dtype.  Batches that cannot fill the GPU with its
// 128-column workgroups (decode, short chunks) run on attention_stream.h.
//
// All arithmetic is fp32 on v_mfma_f32_32x32x2_f32 (256 flops per clock and
// CU, the card's fp32 matrix rate), so fp32 models lose nothing and 16-bit
// models keep fp32 probabilities.  Bound: that MFMA rate.  Compiled with
// -ffp-contract=off so the q rotation rounds each op to the model dtype like
// the reference (gllm/model/layers/attention.py:105-118).
#pragma once
#include "common.h"
#include "generic.h"
#include "launch.h"

namespace gllm {

// 16 bytes of cached elements as the fp32 values the reference's gather gives
template <typename KV, typename QT>
__device__ __forceinline__ void widen16(u32x4 w, float* o) {
  if constexpr (std::is_same<KV, float>::value) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(w[i]);
  } else if constexpr (std::is_same<KV, fp8e4m3>::value) {
#pragma unroll
    for (int i = 0; i < 4; ++i) unpack_fp8x4(w[i], o + 4 * i);
  } else {
    unpack8<KV>(w, o);
  }
  constexpr bool exact = std::is_same<QT, float>::value || std::is_same<KV, QT>::value ||
                         std::is_same<KV, fp8e4m3>::value;
  if constexpr (!exact) {
#pragma unroll
    for (int i = 0; i < 16 / (int)sizeof(KV); ++i) o[i] = rnd<QT>(o[i]);
  }
}

// One 4-wave workgroup per (sequence, kv head, 128 columns); a column is one
// (query row, head of the group) pair, c = r G + g, so 32 columns of a wave
// are 32 / G neighbouring rows of all G heads: they share every K/V tile, and
// a wave's rows of a dense bias are few.  K/V tiles of 32 keys go HBM ->
// registers (a tile ahead) -> LDS as fp32, two buffers, one barrier per tile.
//   S^T = K Q^T: A = K rows (one ds_read_b128 feeds four MFMAs: lane half h
//     holds dims 8t + 4h .. + 3, Q's registers the same dims),
//   O^T += V^T P^T: the score register j of a lane is key 8(j/4) + 4h + j%4 of
//     column n, which is already a B operand (k = lane half), so P needs no
//     move; A = V[that key][32 db + n], one ds_read_b32.
// LDS rows are DP + 4 floats: 16 rows at one dim hit 16 distinct 16-byte bank
// groups.  Measured (fp32, 32 / 8 heads of 64, us; one workgroup per (head,
// row) before): 8 ragged prompts of 64-1024 tokens 7200 -> 182 (68 TFLOP/s of
// visible pairs), 32 x 256 rows on 2048 cached keys 52400 -> 1415 (97 TFLOP/s).  Online softmax in fp32 with the exact running max and expf.  DP: D rounded up to an instantiated size (dims past D
// are zeros).
template <bool DENSE, typename KV, typename QT, int DP>
__global__ void __launch_bounds__(256) attn_tile_kernel(AttnArgs a) {
  constexpr int NW = 4, BK = 32;
  constexpr int ST = DP + 4;                       // floats per LDS row
  constexpr int NO = DP / 32;
  constexpr int EPC = 16 / (int)sizeof(KV);        // elements per 16-byte chunk
  constexpr int TPK = 64 * NW / BK;                // threads per key row
  constexpr int NCH = (DP / EPC + TPK - 1) / TPK;  // chunks per thread and row
  __shared__ __attribute__((aligned(16))) float lds[2][2][BK][ST];   // [buffer][K, V][key][dim]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n = lane & 31, h = lane >> 5;
  const int D = a.head_dim, half = D / 2;
  const int G = a.num_q_heads / a.num_kv_heads;

  int seq, kvh, wgrp, ctx, qlen, TK;
  int64_t qstart;
  if (DENSE) {
    wgrp = gridDim.x - 1 - blockIdx.x;
    kvh = blockIdx.y;
    seq = blockIdx.z;
    ctx = 0;
    qlen = a.dense_Tq;
    TK = a.dense_T;
    qstart = (int64_t)seq * a.dense_Tq;
  } else {
    if (a.tile_items) {
      const WorkItem it = a.tile_items[blockIdx.x];
      seq = it.seq;
      kvh = it.a;
      wgrp = it.kind_b >> 8;
      ctx = it.ctx_len;
      qlen = it.q_len;
      qstart = it.q_row_start;
    } else {
      wgrp = gridDim.x - 1 - blockIdx.x;           // later rows (more keys) first
      kvh = blockIdx.y;
      seq = blockIdx.z;
      const SeqInfo si = a.seqs[seq];
      ctx = si.ctx_len;
      qlen = si.q_len;
      qstart = si.q_row_start;
      if (qlen < a.tile_min_q) return;             // attn_stream_kernel's
    }
    TK = ctx + qlen;
  }
  const int ncol = qlen * G;
  const int c0 = (wgrp * NW + wave) * 32;          // the wave's first column
  if (wgrp * NW * 32 >= ncol) return;
  const bool wact = c0 < ncol;
  const int col = min(c0 + n, ncol - 1);
  const int r = col / G, g = col - r * G;
  const bool col_ok = c0 + n < ncol;
  const int64_t qrow = qstart + r;
  const int qh = kvh * G + g;
  const int vis = DENSE ? TK - 1 : ctx + r;        // last visible key
  const int r_last = (min((wgrp + 1) * NW * 32, ncol) - 1) / G;
  const int kend = DENSE ? TK : ctx + r_last + 1;                             // the workgroup's keys
  const int kend_w = DENSE ? TK : ctx + (min(c0 + 32, ncol) - 1) / G + 1;     // the wave's
  const int kfull = DENSE ? TK : ctx + c0 / G + 1;                            // keys every row of the wave sees

  // ---- K/V staging: thread -> key kt of the tile, chunks ct, ct + TPK, ...
  const int kt = tid / TPK, ct = tid % TPK;
  const int32_t* bt = DENSE ? nullptr : a.block_table + (int64_t)seq * a.block_table_stride;
  const KV* kbase = DENSE ? (const KV*)a.k + (int64_t)seq * a.k_batch_stride + (int64_t)kvh * D
                          : (const KV*)a.k_cache + (int64_t)kvh * D;
  const KV* vbase = DENSE ? (const KV*)a.v + (int64_t)seq * a.v_batch_stride + (int64_t)kvh * D
                          : (const KV*)a.v_cache + (int64_t)kvh * D;
  const int64_t kstride = DENSE ? a.k_row_stride : a.cache_slot_stride;
  const int64_t vstride = DENSE ? a.v_row_stride : a.cache_slot_stride;
  auto block_of = [&](int t) -> uint32_t {         // block id of the thread's key of tile t
    if (DENSE) return 0;
    const int key = min(t * BK + kt, kend - 1);
    return (uint32_t)bt[div_bs((uint32_t)key, a.block_magic, a.block_shift)];
  };
  auto load_chunk = [&](const KV* row, int c) -> u32x4 {
    if (a.vec_rows) return ld16(row + c * EPC);    // rows and D in whole aligned 16-byte chunks
    u32x4 w = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < EPC; ++e) {
      if (c * EPC + e < D) {
        if constexpr (sizeof(KV) == 4) w[e] = reinterpret_cast<const uint32_t*>(row)[c * EPC + e];
        else if constexpr (sizeof(KV) == 2)
          w[e / 2] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[c * EPC + e] << (16 * (e % 2));
        else w[e / 4] |= (uint32_t)reinterpret_cast<const uint8_t*>(row)[c * EPC + e] << (8 * (e % 4));
      }
    }
    return w;
  };
  u32x4 kr[NCH], vr[NCH];
  const int clast = (D + EPC - 1) / EPC - 1;       // last chunk with real dims
  auto issue = [&](int t, uint32_t blk) {
    const int key = min(t * BK + kt, kend - 1);    // keys past the end: masked, re-read the last
    int64_t row = key;
    if (!DENSE) {
      const uint32_t bi = div_bs((uint32_t)key, a.block_magic, a.block_shift);
      if (blk >= (uint64_t)a.num_blocks) blk = 0;  // never address outside the pool
      row = (int64_t)blk * a.block_size + (key - (int)bi * a.block_size);
    }
    const KV* kp = kbase + row * kstride;
    const KV* vp = vbase + row * vstride;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = min(ct + i * TPK, clast);
      kr[i] = load_chunk(kp, c);
      vr[i] = load_chunk(vp, c);
    }
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = ct + i * TPK;
      if (c * EPC >= DP) continue;
      float kf[EPC], vf[EPC];
      widen16<KV, QT>(kr[i], kf);
      widen16<KV, QT>(vr[i], vf);
      const bool real = c <= clast;
#pragma unroll
      for (int u = 0; u < EPC; u += 4) {
        f32x4 kw = {kf[u], kf[u + 1], kf[u + 2], kf[u + 3]}, vw = {vf[u], vf[u + 1], vf[u + 2], vf[u + 3]};
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<f32x4*>(&lds[b][0][kt][c * EPC + u]) = real ? kw : z;
        *reinterpret_cast<f32x4*>(&lds[b][1][kt][c * EPC + u]) = real ? vw : z;
      }
    }
  };

  const int nt = (kend + BK - 1) / BK;
  uint32_t blk = block_of(0);
  issue(0, blk);
  blk = block_of(min(1, nt - 1));

  // ---- Q: rotated (each op rounded to the model dtype) into LDS, 128 columns
  // x DP in the tile buffers, then each lane's dims into registers
  {
    float* qs = &lds[0][0][0][0];
    constexpr int H2P = DP / 2;
    for (int e = tid; e < NW * 32 * H2P; e += 64 * NW) {
      const int cc = e / H2P, j = e - cc * H2P;    // pair (j, j + D/2) of the workgroup's column cc
      const int gc = min(wgrp * NW * 32 + cc, ncol - 1);
      const int rq = gc / G, gq = gc - rq * G;
      if (j < half) {
        const QT* qp = (const QT*)a.q + (qstart + rq) * a.q_row_stride + (int64_t)(kvh * G + gq) * D;
        float x1 = (float)qp[j], x2 = (float)qp[j + half];
        if (!DENSE && a.rope_mode != kRopeNone) {
          const int64_t crow = a.rope_mode == kRopeByPosition ? (int64_t)(ctx + rq) : qstart + rq;
          const float c = (float)((const QT*)a.rope_cos)[crow * a.rope_row_stride + j];
          const float s = (float)((const QT*)a.rope_sin)[crow * a.rope_row_stride + j];
          const float lo = rnd<QT>(__fsub_rn(rnd<QT>(__fmul_rn(x1, c)), rnd<QT>(__fmul_rn(x2, s))));
          const float hi = rnd<QT>(__fadd_rn(rnd<QT>(__fmul_rn(x1, s)), rnd<QT>(__fmul_rn(x2, c))));
          x1 = lo;
          x2 = hi;
        }
        qs[cc * ST + j] = x1;
        qs[cc * ST + j + half] = x2;
      } else {                                     // dims D .. DP - 1 (D = 2 half): zeros
        qs[cc * ST + 2 * j] = 0.f;
        qs[cc * ST + 2 * j + 1] = 0.f;
      }
    }
  }
  __syncthreads();
  f32x4 qv[DP / 8];
#pragma unroll
  for (int t = 0; t < DP / 8; ++t)
    qv[t] = *reinterpret_cast<const f32x4*>(&lds[0][0][0][0] + (wave * 32 + n) * ST + 8 * t + 4 * h);
  __syncthreads();
  put(0);

  float m = kNegInf, l = 0.f;
  f32x16 o[NO];
#pragma unroll
  for (int db = 0; db < NO; ++db)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[db][j] = 0.f;
  const QT* brow = DENSE ? (const QT*)a.bias + (int64_t)seq * a.bias_batch_stride + (int64_t)r * a.bias_row_stride
                         : nullptr;

  for (int t = 0; t < nt; ++t) {
    __syncthreads();                               // tile t in LDS; tile t - 1's buffer free
    if (t + 1 < nt) {
      issue(t + 1, blk);
      blk = block_of(min(t + 2, nt - 1));
    }
    const int p0 = t * BK;
    if (wact && p0 < kend_w) {
      const int b = t & 1;
      float bv[DENSE ? 16 : 1];
      if constexpr (DENSE) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int p = p0 + 8 * (j >> 2) + 4 * h + (j & 3);
          bv[j] = (float)brow[min(p, TK - 1)];
        }
      }
      // two chains: half the length of the fp32 sums; at 256 dims in two halves
      f32x16 s = f32x16{}, s1 = f32x16{}, sh = f32x16{};
#pragma unroll
      for (int u = 0; u < DP / 8; ++u) {
        if (DP == 256 && u == DP / 16) {
          sh = s + s1;
          s = s1 = f32x16{};
        }
        const f32x4 kv4 = *reinterpret_cast<const f32x4*>(&lds[b][0][n][8 * u + 4 * h]);
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv4[e], qv[u][e], s, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kv4[e + 1], qv[u][e + 1], s1, 0, 0, 0);
        }
      }
      s += s1;
      if (DP == 256) s += sh;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        s[j] *= a.scale;
        if constexpr (DENSE) s[j] += bv[j];
      }
      if (p0 + BK > kfull) {                       // causal edge / past the last key
        const int lim = vis - p0 - 4 * h;
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (8 * (j >> 2) + (j & 3) > lim) s[j] = kNegInf;
      }
      float tm = s[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) tm = fmaxf(tm, s[j]);
      tm = max_xor32(tm);
      const float mn = fmaxf(m, tm);
      const float mu = mn == kNegInf ? 0.f : mn;   // every key so far masked: all weights 0
      const float alpha = expf(m - mu);
      float ls = 0.f;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        s[j] = expf(s[j] - mu);
        ls += s[j];
      }
      l = l * alpha + ls;
      m = mn;
      // the tile's P V from zero, then one FMA per output with the rescale: the
      // fp32 sums stay 32 keys long, plus one term per tile
#pragma unroll
      for (int db = 0; db < NO; ++db) {
        f32x16 w;
#pragma unroll
        for (int j = 0; j < 16; ++j) w[j] = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j)
          w = __builtin_amdgcn_mfma_f32_32x32x2f32(lds[b][1][8 * (j >> 2) + 4 * h + (j & 3)][32 * db + n], s[j], w, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 16; ++j) o[db][j] = __builtin_fmaf(o[db][j], alpha, w[j]);
      }
    }
    if (t + 1 < nt) put((t + 1) & 1);
  }

  l = sum_xor32(l);
  if (!wact || !col_ok) return;
  QT* op = (QT*)a.out + qrow * a.out_row_stride + (int64_t)qh * D;
#pragma unroll
  for (int db = 0; db < NO; ++db)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      const int d = 32 * db + 8 * jq + 4 * h;
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[db][4 * jq + e] / l;   // l == 0 (every key masked) gives NaN, as torch's softmax
      if (a.vec_out) {                             // D a multiple of 4, rows aligned to 4 elements
        if (d < D) {
          if constexpr (sizeof(QT) == 4) *reinterpret_cast<f32x4*>(op + d) = f32x4{x[0], x[1], x[2], x[3]};
          else st8(op + d, u32x2{E16<QT>::pack2(x[0], x[1]), E16<QT>::pack2(x[2], x[3])});
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < D) stq<QT>(op + d + e, x[e]);
      }
    }
}

template <bool DENSE, typename KV, typename QT>
static hipError_t launch_tile_d(const AttnArgs& a, dim3 grid, hipStream_t st) {
  const dim3 block(256);
  if (a.head_dim <= 64) hipLaunchKernelGGL((attn_tile_kernel<DENSE, KV, QT, 64>), grid, block, 0, st, a);
  else if (a.head_dim <= 96) hipLaunchKernelGGL((attn_tile_kernel<DENSE, KV, QT, 96>), grid, block, 0, st, a);
  else if (a.head_dim <= 128) hipLaunchKernelGGL((attn_tile_kernel<DENSE, KV, QT, 128>), grid, block, 0, st, a);
  else if (a.head_dim <= 256) hipLaunchKernelGGL((attn_tile_kernel<DENSE, KV, QT, 256>), grid, block, 0, st, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <typename QT>
static hipError_t launch_tile_t(const AttnArgs& a, bool dense, dim3 grid, hipStream_t st) {
  if (dense) return launch_tile_d<true, QT, QT>(a, grid, st);
  switch (a.kv_dtype) {
    case kF32: return launch_tile_d<false, float, QT>(a, grid, st);
    case kBF16: return launch_tile_d<false, __bf16, QT>(a, grid, st);
    case kF16: return launch_tile_d<false, _Float16, QT>(a, grid, st);
    case kFP8: return launch_tile_d<false, fp8e4m3, QT>(a, grid, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gllm
