// Arithmetic of the gated RMSNorm (Qwen3_5RMSNormGated.forward, mindspeed_mm/fsdp/models/qwen3_5/modeling_qwen3_5.py:330-349)
// on one 16-byte piece of a row, shared by the stand-alone kernels and by the output kernel of the chunked rule when
// it applies the norm in its epilogue: both must round at the same places and add in the same order to agree bit
// for bit.
//     xn = x * rsqrt(mean(x^2) + eps)        (fp32, then cast to the input dtype)
//     y  = (weight * xn) * silu(gate)        (gate in fp32; result cast to the input dtype)
// ACT = 1 is the norm of the KDA layer (KimiK_3_MoeRMSNormGated.forward,
// mindspeed_mm/fsdp/models/kimi_k3/modeling_kimi_linear.py:83-96): the gate passes through a sigmoid that is cast to
// the input dtype before the product,
//     y  = (weight * xn) * cast(sigmoid(gate))
#pragma once
#include "gdn_common.h"

namespace gdn {

// 16-bit types: reciprocal instruction and one Newton step, which lands on the correctly rounded quotient but for ties (the
// first estimate is off by an ulp, the step squares that), in two thirds of the instructions of the IEEE division, which
// made these kernels bound by vector issue instead of memory.  The reciprocal is taken of a quarter of 1 + e^-p: the
// instruction flushes subnormal results, which a quarter never has.  v_div_fixup sets 0 where e^-p overflowed (the step
// gives 0 x inf there) and hands a NaN on.
template <typename T> __device__ __forceinline__ float sigmoid_(float p) {
  if constexpr (sizeof(T) == 4) {
    return 1.f / (1.f + __expf(-p));
  } else {
    const float d = fmaf(__expf(-p), 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(d), r4 = 0.25f * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, r, 1.f), r4, r4), d, 1.f);
  }
}

// round to T and back: the reference casts to the input dtype between the steps (16-bit types: two elements at a time)
template <typename T> __device__ __forceinline__ void round_piece(float* f) {
  if constexpr (sizeof(T) == 2) unpack16<T>(pack16<T>(f), f);
}

template <typename T, typename TW> __device__ __forceinline__ void load_weight(float* w, const TW* p) {
  constexpr int V = Elem<T>::kVec;
  if constexpr (sizeof(TW) == sizeof(T)) {
    const Vec16<TW> v = ld16(p);
#pragma unroll
    for (int e = 0; e < V; ++e) w[e] = v.get(e);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) w[e] = Elem<TW>::to_f(p[e]);
  }
}

// sum of the squares of a piece's elements, added in element order
template <typename T> __device__ __forceinline__ float piece_sumsq(const Vec16<T>& xv) {
  float f[Elem<T>::kVec], ss = 0.f;
  unpack16<T>(xv, f);
#pragma unroll
  for (int e = 0; e < Elem<T>::kVec; ++e) ss += f[e] * f[e];
  return ss;
}

// TW = T: weight in the input dtype, weight * xn is rounded to T as in the reference; TW = float: kept in fp32
template <typename T, typename TW, int ACT = 0>
__device__ __forceinline__ Vec16<T> rmsnorm_gated_piece(const Vec16<T>& xv, const Vec16<T>& gv, const float* w, float rstd) {
  constexpr int V = Elem<T>::kVec;
  float t[V], gf[V], s[V];
  unpack16<T>(xv, t);
  unpack16<T>(gv, gf);
#pragma unroll
  for (int e = 0; e < V; ++e) t[e] *= rstd;
  round_piece<T>(t);
#pragma unroll
  for (int e = 0; e < V; ++e) t[e] *= w[e];
  if constexpr (sizeof(TW) == sizeof(T)) round_piece<T>(t);
#pragma unroll
  for (int e = 0; e < V; ++e) s[e] = ACT == 0 ? gf[e] * sigmoid_<T>(gf[e]) : sigmoid_<T>(gf[e]);
  if constexpr (ACT != 0) round_piece<T>(s);
#pragma unroll
  for (int e = 0; e < V; ++e) t[e] *= s[e];
  return pack16<T>(t);
}

}  // namespace gdn
