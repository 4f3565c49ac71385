// Generic attention (any model dtype over any cache dtype, even head dims up to
// 256): the fp32 model's kernels and the dispatch between them.  The 16-bit
// models' instantiations are units of their own (generic_attention_bf16.hip,
// generic_attention_f16.hip).
#ifndef GLLM_GENERIC_QT
#define GLLM_GENERIC_QT float
#define GLLM_GENERIC_LAUNCH launch_generic_f32
#define GLLM_GENERIC_DISPATCH 1
#endif

#include "attention_stream.h"
#include "attention_tile.h"

namespace gllm {

hipError_t GLLM_GENERIC_LAUNCH(const AttnArgs& a, bool tile, bool dense, dim3 grid, hipStream_t st) {
  return tile ? launch_tile_t<GLLM_GENERIC_QT>(a, dense, grid, st) : launch_stream_t<GLLM_GENERIC_QT>(a, dense, grid, st);
}

#ifdef GLLM_GENERIC_DISPATCH
hipError_t launch_generic_bf16(const AttnArgs& a, bool tile, bool dense, dim3 grid, hipStream_t st);
hipError_t launch_generic_f16(const AttnArgs& a, bool tile, bool dense, dim3 grid, hipStream_t st);

static hipError_t launch_kind(AttnArgs a, bool tile, bool dense, dim3 grid, hipStream_t st) {
  const size_t eq = a.dtype == kF32 ? 4 : 2;
  if (tile) {                                      // 16-byte chunks of K/V
    const size_t ek = dense ? eq : (a.kv_dtype == kF32 ? 4 : (a.kv_dtype == kFP8 ? 1 : 2));
    const auto rows = [&](const void* p, int64_t stride, int64_t batch) {
      return ((uintptr_t)p & 15) == 0 && (size_t)stride * ek % 16 == 0 && (size_t)batch * ek % 16 == 0;
    };
    a.vec_rows = (size_t)a.head_dim * ek % 16 == 0 &&
                 (dense ? rows(a.k, a.k_row_stride, a.k_batch_stride) && rows(a.v, a.v_row_stride, a.v_batch_stride)
                        : rows(a.k_cache, a.cache_slot_stride, 0) && rows(a.v_cache, a.cache_slot_stride, 0));
  }
  a.vec_out = a.head_dim % 4 == 0 && a.out_row_stride % 4 == 0 && ((uintptr_t)a.out & (4 * eq - 1)) == 0;
  switch (a.dtype) {
    case kF32: return launch_generic_f32(a, tile, dense, grid, st);
    case kBF16: return launch_generic_bf16(a, tile, dense, grid, st);
    case kF16: return launch_generic_f16(a, tile, dense, grid, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_attention_generic(AttnArgs a, bool dense, int B, int max_q, int max_stream_q, int64_t stream_rows,
                                    hipStream_t st) {
  if (B == 0 || max_q == 0) return hipSuccess;
  if (a.head_dim <= 0 || a.head_dim > 256) return hipErrorInvalidValue;
  const int G = a.num_q_heads / a.num_kv_heads;
  const auto grid = [&](int rows, int cols) {
    return dim3((unsigned)(((int64_t)rows * G + cols - 1) / cols), a.num_kv_heads, B);
  };
  if (dense) {
    const bool tile = max_q >= kTileMinRows && (int64_t)grid(max_q, kTileCols).x * a.num_kv_heads * B >= kTileMinWgs;
    return launch_kind(a, tile, true, grid(max_q, tile ? kTileCols : kStreamCols), st);
  }
  if (a.k_new) {
    // the fused KV write (at most kFusedRows rows): every sequence on the
    // stream kernel, which keeps the new keys in LDS
    a.tile_min_q = 0;
    max_stream_q = max_q;
  } else if (a.tile_min_q > 0 && max_q >= a.tile_min_q) {
    const dim3 g = a.tile_items ? dim3(a.n_tile_items) : grid(max_q, kTileCols);
    if (hipError_t e = launch_kind(a, true, false, g, st); e != hipSuccess) return e;
  }
  if (max_stream_q == 0) return hipSuccess;
  // Where most workgroups are empty (decodes beside a chunk: all but their first)
  // the column groups are an odd number: at an even stride the working ones all
  // fell to a few shader engines.  9 decodes and a chunk of 125 rows, bf16 D = 80,
  // 177 -> 42 us (apart 29 and 22); fp32 D = 64, 11 and two of 24-48 45 -> 22.  Sequences
  // of like length keep the even stride: two of 39-78 rows 14 -> 18 otherwise.
  dim3 g = grid(max_stream_q, kStreamCols);
  if (2 * stream_rows < (int64_t)B * max_stream_q) g.x |= 1;
  return launch_kind(a, false, false, g, st);
}
#endif  // GLLM_GENERIC_DISPATCH

}  // namespace gllm
