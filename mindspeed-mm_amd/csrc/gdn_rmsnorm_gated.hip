// Gated RMSNorm: the step right after the gated delta rule in the reference layer
// (Qwen3_5RMSNormGated.forward, mindspeed_mm/fsdp/models/qwen3_5/modeling_qwen3_5.py:330-349, called at :897-900 on
// rows of head_v_dim elements):
//     xn = x * rsqrt(mean(x^2) + eps)        (fp32, then cast to the input dtype)
//     y  = (weight * xn) * silu(gate)        (gate in fp32; result cast to the input dtype)
// Row-wise and bandwidth-bound: forward reads x, gate and writes y; backward reads x, gate, dy and writes dx, dgate.
// The forward pass gives every workgroup 4 KB of each tensor and nothing more: handed out in order, such pieces keep what
// is in flight close together, which the memory rewards (1M rows of 128 bf16: 164 us = 4.9 TB/s with 2048 workgroups
// striding over the rows and element-wise conversions, 127 to 133 us = 6.1 to 6.3 TB/s now; the card's copy of 4 KB pieces reaches 6.2
// to 6.5, of 32 KB pieces 5.4).  The backward pass needs few partial sums of dweight and strides (276 -> 234 to 243 us).
// A row of N elements is held by N/VEC neighbouring lanes (16 bytes each); row sums use data-parallel-primitive moves.
// With gate_activation = 1 the gate passes through a sigmoid instead (the KDA layer's norm, KimiK_3_MoeRMSNormGated,
// mindspeed_mm/fsdp/models/kimi_k3/modeling_kimi_linear.py:75-96): s = cast(sigmoid(gate)).
// Backward, with t = weight * xn, s = silu(gate) or sigmoid(gate), xh = x * rstd in fp32:
//     dgate = dy t s'(gate)     dt = dy s     dweight = sum_rows dt xn     dxn = dt weight
//     dx = rstd (dxn - xh mean(dxn xh))
// dweight is accumulated per thread over the rows it visits, reduced inside the workgroup through LDS and written as one
// partial row per workgroup; rmsnorm_gated_dw_reduce_kernel adds the partials in a fixed order (bitwise reproducible).
#include "gdn_common.h"
#include "gdn_profile.h"
#include "gdn_rmsnorm_gated.h"

namespace gdn {

template <int LPR> __device__ __forceinline__ float row_lanes_sum(float v) {
  if constexpr (LPR <= 32) {
    return lane_group_sum<LPR>(v);
  } else {
    v = lane_group_sum<32>(v);
    return v + __shfl_xor(v, 32);
  }
}

// TW = T: weight in the input dtype, weight * xn is rounded to T as in the reference; TW = float: kept in fp32
template <typename T, typename TW, int LPR, int ACT>
__global__ __launch_bounds__(kThreads) void rmsnorm_gated_fwd_kernel(const T* __restrict__ x, const T* __restrict__ gate,
                                                                     const TW* __restrict__ weight, T* __restrict__ y,
                                                                     float* __restrict__ rstd_out, int64_t rows,
                                                                     float eps) {
  constexpr int V = Elem<T>::kVec, N = LPR * V, RPB = kThreads / LPR;
  const int c = threadIdx.x % LPR;
  float w[V];
  load_weight<T, TW>(w, weight + c * V);
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  const bool ok = row < rows;        // every lane takes part in the row sums: lanes past the end repeat the last row
  const int64_t at = (ok ? row : rows - 1) * N + c * V;
  const Vec16<T> xv = ld16_stream(x + at), gv = ld16_stream(gate + at);
  const float ss = row_lanes_sum<LPR>(piece_sumsq<T>(xv));
  const float rstd = rsqrtf(ss * (1.f / N) + eps);
  const Vec16<T> out = rmsnorm_gated_piece<T, TW, ACT>(xv, gv, w, rstd);
  if (ok) {
    __builtin_nontemporal_store(out.raw, reinterpret_cast<u32x4*>(y + at));
    if (c == 0) rstd_out[row] = rstd;
  }
}

template <typename T, typename TW, int LPR, int ACT>
__global__ __launch_bounds__(kThreads) void rmsnorm_gated_bwd_kernel(
    const T* __restrict__ x, const T* __restrict__ gate, const TW* __restrict__ weight,
    const float* __restrict__ rstd_in, const T* __restrict__ dy, T* __restrict__ dx, T* __restrict__ dgate,
    float* __restrict__ part, int64_t rows) {
  constexpr int V = Elem<T>::kVec, N = LPR * V, RPB = kThreads / LPR;
  __shared__ float red[kThreads * V];
  const int c = threadIdx.x % LPR, rg = threadIdx.x / LPR;
  float w[V], dwa[V];
  load_weight<T, TW>(w, weight + c * V);
#pragma unroll
  for (int e = 0; e < V; ++e) dwa[e] = 0.f;
  const int64_t step = (int64_t)gridDim.x * RPB, stop = (rows + RPB - 1) / RPB * RPB;
  int64_t row = (int64_t)blockIdx.x * RPB + rg;
  // a trip's rows are requested one trip ahead; rows past the end repeat the last one with nothing added or stored
  Vec16<T> xv, gv, dv;
  float rstd;
  auto request = [&](int64_t r) {
    const int64_t rc = r < rows ? r : rows - 1, at = rc * N + c * V;
    xv = ld16_stream(x + at);
    gv = ld16_stream(gate + at);
    dv = ld16_stream(dy + at);
    rstd = rstd_in[rc];
  };
  request(row);
  for (; row < stop; row += step) {   // uniform trip count: every lane takes part in the row sums
    const bool ok = row < rows;
    float xh[V], xn[V], t[V], gf[V], d[V], sg[V], dxn[V], dgo[V], dot = 0.f;
    const float rs = ok ? rstd : 0.f;
    unpack16<T>(xv, xh);
    unpack16<T>(gv, gf);
    unpack16<T>(dv, d);
    request(row + step);
#pragma unroll
    for (int e = 0; e < V; ++e) { xh[e] *= rs; xn[e] = xh[e]; }
    round_piece<T>(xn);
#pragma unroll
    for (int e = 0; e < V; ++e) t[e] = w[e] * xn[e];
    if constexpr (sizeof(TW) == sizeof(T)) round_piece<T>(t);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      sg[e] = sigmoid_<T>(gf[e]);
      dgo[e] = ACT == 0 ? d[e] * t[e] * sg[e] * (1.f + gf[e] * (1.f - sg[e])) : d[e] * t[e] * sg[e] * (1.f - sg[e]);
    }
    if constexpr (ACT != 0) round_piece<T>(sg);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float dt = ACT == 0 ? d[e] * gf[e] * sg[e] : d[e] * sg[e];
      xn[e] *= dt;
      dxn[e] = dt * w[e];
      dot += dxn[e] * xh[e];
    }
    dot = row_lanes_sum<LPR>(dot) * (1.f / N);
#pragma unroll
    for (int e = 0; e < V; ++e) dxn[e] = rs * (dxn[e] - xh[e] * dot);
    if (ok) {
      const int64_t at = row * N + c * V;
#pragma unroll
      for (int e = 0; e < V; ++e) dwa[e] += xn[e];
      __builtin_nontemporal_store(pack16<T>(dxn).raw, reinterpret_cast<u32x4*>(dx + at));
      __builtin_nontemporal_store(pack16<T>(dgo).raw, reinterpret_cast<u32x4*>(dgate + at));
    }
  }
  // workgroup partial of dweight: add the RPB row groups in a fixed order
#pragma unroll
  for (int e = 0; e < V; ++e) red[threadIdx.x * V + e] = dwa[e];
  __syncthreads();
  for (int i = threadIdx.x; i < N; i += kThreads) {
    const int cc = i / V, e = i % V;
    float s = 0.f;
    for (int r = 0; r < RPB; ++r) s += red[(r * LPR + cc) * V + e];
    part[(int64_t)blockIdx.x * N + i] = s;
  }
}

// one workgroup per column: strided partial sums per thread, then a fixed-order tree through LDS
__global__ __launch_bounds__(kThreads) void rmsnorm_gated_dw_reduce_kernel(const float* __restrict__ part,
                                                                           float* __restrict__ dw, int nparts, int N) {
  __shared__ float red[kThreads];
  const int i = blockIdx.x;
  float s = 0.f;
  for (int p = threadIdx.x; p < nparts; p += kThreads) s += part[(int64_t)p * N + i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int m = kThreads / 2; m > 0; m >>= 1) {
    if ((int)threadIdx.x < m) red[threadIdx.x] += red[threadIdx.x + m];
    __syncthreads();
  }
  if (threadIdx.x == 0) dw[i] = red[0];
}

// Two workgroups per CU, each a trip ahead with its requests.  Five streams share the memory: what counts is that the
// rows in flight stay close together (2048 workgroups: 5.3 TB/s, 1024: 5.2, 768: 5.5, 512: 5.75, 384: 5.25, 256: 5.0 at
// 1M rows of 128 bf16).  Three per CU for 16-bit tensors of up to 100 MB, which the memory-side cache holds in part (262144
// rows, with the reduction: 70 to 72 -> 69 us; 131072: 39 -> 37.5; 524288, 134 MB: 121 -> 126; fp32, 67 MB: 64 -> 66).
template <typename T> static int rmsnorm_bwd_blocks(int64_t rows, int rpb) {
  const int64_t need = (rows + rpb - 1) / rpb, tensor = need * (kThreads * 16);
  const int most = sizeof(T) == 2 && tensor <= 100 * 1000 * 1000 ? 768 : 512;
  return (int)(need < most ? (need > 0 ? need : 1) : most);
}

template <typename T, typename TW, int LPR>
static int rmsnorm_fwd_launch(const void* x, const void* gate, const void* weight, void* y, float* rstd, int64_t rows,
                              float eps, int act, hipStream_t st) {
  constexpr int N = LPR * Elem<T>::kVec, RPB = kThreads / LPR;
  constexpr int64_t most = GDN_MAX_LAUNCH_THREADS / kThreads * RPB;   // rows of one launch (4 KB of x to a workgroup: 68 GB)
  for (int64_t r = 0; r < rows; r += most) {
    const int64_t n = rows - r < most ? rows - r : most;
    auto launch = [&](auto kern) {
      GDN_LAUNCH(kKernRmsNormFwd, st, kern, dim3((unsigned)((n + RPB - 1) / RPB)), dim3(kThreads), 0, st, (const T*)x + r * N,
                 (const T*)gate + r * N, (const TW*)weight, (T*)y + r * N, rstd + r, n, eps);
    };
    if (act == 0) launch(rmsnorm_gated_fwd_kernel<T, TW, LPR, 0>);
    else launch(rmsnorm_gated_fwd_kernel<T, TW, LPR, 1>);
  }
  return (int)hipGetLastError();
}

template <typename T, typename TW, int LPR>
static int rmsnorm_bwd_launch(const void* x, const void* gate, const void* weight, const float* rstd, const void* dy,
                              void* dx, void* dgate, float* dw, float* part, int64_t rows, int act, hipStream_t st) {
  constexpr int N = LPR * Elem<T>::kVec;
  const int nb = rmsnorm_bwd_blocks<T>(rows, kThreads / LPR);
  if (act == 0)
    GDN_LAUNCH(kKernRmsNormBwd, st, (rmsnorm_gated_bwd_kernel<T, TW, LPR, 0>), dim3(nb), dim3(kThreads), 0, st, (const T*)x,
               (const T*)gate, (const TW*)weight, rstd, (const T*)dy, (T*)dx, (T*)dgate, part, rows);
  else
    GDN_LAUNCH(kKernRmsNormBwd, st, (rmsnorm_gated_bwd_kernel<T, TW, LPR, 1>), dim3(nb), dim3(kThreads), 0, st, (const T*)x,
               (const T*)gate, (const TW*)weight, rstd, (const T*)dy, (T*)dx, (T*)dgate, part, rows);
  GDN_LAUNCH(kKernRmsNormReduce, st, rmsnorm_gated_dw_reduce_kernel, dim3(N), dim3(kThreads), 0, st,
             (const float*)part, dw, nb, N);
  return (int)hipGetLastError();
}

// lanes per row for a row of N elements of `elem` bytes, or 0 if the size is not supported
static int rmsnorm_lpr(int N, int elem) {
  const int vec = 16 / elem;
  if (N <= 0 || N % vec != 0) return 0;
  const int lpr = N / vec;
  return (lpr == 4 || lpr == 8 || lpr == 16 || lpr == 32 || lpr == 64) ? lpr : 0;
}

}  // namespace gdn

#define GDN_RMS_DISPATCH(CALL)                                                          \
  switch (lpr) {                                                                        \
    case 4: return CALL(4);                                                             \
    case 8: return CALL(8);                                                             \
    case 16: return CALL(16);                                                           \
    case 32: return CALL(32);                                                           \
    default: return CALL(64);                                                           \
  }

extern "C" int gdn_rmsnorm_gated_fwd(const void* x, const void* gate, const void* weight, void* y, float* rstd,
                                     int64_t rows, int N, float eps, int dtype, int weight_dtype, int gate_activation,
                                     void* stream) {
  using namespace gdn;
  if (!x || !gate || !weight || !y || !rstd) return -1;
  if (rows < 0) return -2;
  if (dtype != 0 && dtype != 1) return -4;
  if (weight_dtype != 0 && weight_dtype != dtype) return -4;
  if (gate_activation != 0 && gate_activation != 1) return -4;
  const int lpr = rmsnorm_lpr(N, dtype == 0 ? 4 : 2);
  if (lpr == 0) return -3;
  if (rows == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == 0) {
#define CALL(L_) rmsnorm_fwd_launch<float, float, L_>(x, gate, weight, y, rstd, rows, eps, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  } else if (weight_dtype == 1) {
#define CALL(L_) rmsnorm_fwd_launch<bf16_t, bf16_t, L_>(x, gate, weight, y, rstd, rows, eps, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  } else {
#define CALL(L_) rmsnorm_fwd_launch<bf16_t, float, L_>(x, gate, weight, y, rstd, rows, eps, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  }
}

extern "C" int64_t gdn_rmsnorm_gated_bwd_workspace_bytes(int64_t rows, int N) {
  (void)rows;
  return (int64_t)2048 * (N > 0 ? N : 1) * (int64_t)sizeof(float);
}

extern "C" int gdn_rmsnorm_gated_bwd(const void* x, const void* gate, const void* weight, const float* rstd,
                                     const void* dy, void* dx, void* dgate, float* dweight, void* workspace,
                                     int64_t workspace_bytes, int64_t rows, int N, int dtype, int weight_dtype,
                                     int gate_activation, void* stream) {
  using namespace gdn;
  if (!x || !gate || !weight || !rstd || !dy || !dx || !dgate || !dweight || !workspace) return -1;
  if (rows < 0) return -2;
  if (dtype != 0 && dtype != 1) return -4;
  if (weight_dtype != 0 && weight_dtype != dtype) return -4;
  if (gate_activation != 0 && gate_activation != 1) return -4;
  const int lpr = rmsnorm_lpr(N, dtype == 0 ? 4 : 2);
  if (lpr == 0) return -3;
  if (workspace_bytes < gdn_rmsnorm_gated_bwd_workspace_bytes(rows, N)) return -5;
  hipStream_t st = (hipStream_t)stream;
  float* part = static_cast<float*>(workspace);
  if (rows == 0) {   // dweight = 0: the reduction over zero partials
    GDN_LAUNCH(kKernRmsNormReduce, st, rmsnorm_gated_dw_reduce_kernel, dim3(N), dim3(kThreads), 0, st,
               (const float*)part, dweight, 0, N);
    return (int)hipGetLastError();
  }
  if (dtype == 0) {
#define CALL(L_) rmsnorm_bwd_launch<float, float, L_>(x, gate, weight, rstd, dy, dx, dgate, dweight, part, rows, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  } else if (weight_dtype == 1) {
#define CALL(L_) rmsnorm_bwd_launch<bf16_t, bf16_t, L_>(x, gate, weight, rstd, dy, dx, dgate, dweight, part, rows, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  } else {
#define CALL(L_) rmsnorm_bwd_launch<bf16_t, float, L_>(x, gate, weight, rstd, dy, dx, dgate, dweight, part, rows, gate_activation, st)
    GDN_RMS_DISPATCH(CALL)
#undef CALL
  }
}
