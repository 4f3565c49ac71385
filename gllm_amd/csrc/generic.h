// Element helpers of the generic attention kernels (attention_stream.h,
// attention_tile.h): any model dtype QT over any cache dtype KV, widened to
// fp32 for the arithmetic.
#pragma once
#include <type_traits>

#include "common.h"

namespace gllm {

template <typename KV> __device__ __forceinline__ float ldkv(const KV* p);
template <> __device__ __forceinline__ float ldkv<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ldkv<__bf16>(const __bf16* p) { return (float)*p; }
template <> __device__ __forceinline__ float ldkv<_Float16>(const _Float16* p) { return (float)*p; }
// fp8 e4m3fn cache: exact widening (the reference's .to(model dtype) after the gather)
template <> __device__ __forceinline__ float ldkv<fp8e4m3>(const fp8e4m3* p) { return __builtin_amdgcn_cvt_f32_fp8((int)p->bits, 0); }

// model dtype: loads widen exactly; each RoPE op rounds to it
template <typename QT> __device__ __forceinline__ float rnd(float x);
template <> __device__ __forceinline__ float rnd<float>(float x) { return x; }
template <> __device__ __forceinline__ float rnd<__bf16>(float x) { return round_bf16(x); }
template <> __device__ __forceinline__ float rnd<_Float16>(float x) { return (float)(_Float16)x; }
template <typename QT> __device__ __forceinline__ void stq(QT* p, float x);
template <> __device__ __forceinline__ void stq<float>(float* p, float x) { *p = x; }
template <> __device__ __forceinline__ void stq<__bf16>(__bf16* p, float x) {
  *reinterpret_cast<uint16_t*>(p) = (uint16_t)pack_bf16x2(x, 0.f);
}
template <> __device__ __forceinline__ void stq<_Float16>(_Float16* p, float x) { *p = (_Float16)x; }

// A cached value as the reference's gather reads it: cast to the model dtype
// (attention.py:169-170, .to(q.dtype)).  Exact when the cache holds the model
// dtype, fp8 e4m3fn (a subset of every model dtype) or feeds an fp32 model;
// rounded to nearest even for an f32 cache (or the other 16-bit type) under
// a 16-bit model.
template <typename KV, typename QT>
__device__ __forceinline__ float kvld(const KV* p) {
  constexpr bool exact = std::is_same<QT, float>::value || std::is_same<KV, QT>::value ||
                         std::is_same<KV, fp8e4m3>::value;
  const float x = ldkv<KV>(p);
  if constexpr (exact) return x;
  else return rnd<QT>(x);
}

}  // namespace gllm
