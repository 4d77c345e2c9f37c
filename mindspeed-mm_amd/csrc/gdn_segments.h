// Sequences cut into segments for the two recurrences.
//
// A recurrence is affine in the state it starts from: over a run of chunks S_out = A S_in + B with A [K,K] and B [K,V].
// With few (sequence, head) pairs -- heads sharded over ranks, one long sequence -- the plain kernels fill a fraction of
// the device (8 heads of 128 columns: 32 of 256 compute units) and take one dependent step per chunk of the sequence.
// Each sequence is then cut into P segments and a pass has three launches:
//   1. the map of every segment but the last: the recurrence kernel with V + K columns, started from [0 | I] and with
//      the inputs of the last K columns zero, leaves [B | A] in fp32; nothing else is written
//   2. segment_chain_kernel: the state each segment starts from, P - 1 dependent fp32 products
//   3. the recurrence kernel proper, every segment from its own start
// The reverse recurrence does the same from the other end.  2 n / P dependent steps instead of n.  32768 tokens, 8 heads
// of 128, 8 segments: maps 98 us, chain 21, recurrence 92 (205 together) where the uncut recurrence takes 561; reverse maps 120,
// chain 21, recurrence 164 beside the refill; forward and backward 1430 -> 728 us.  The error against float64 is the uncut
// recurrence's (4160 to 16384 tokens, 2 to 8 heads, four seeds each: o 4.745e-3 and 4.745e-3 with decays near 1 over a whole
// segment, final state 3.79e-3 and 3.78e-3, dk 5.63e-3 and 5.63e-3, dg 5.19e-3 to 5.68e-3 uncut, 5.14e-3 to 5.65e-3 cut, smaller in
// two of four cases).
#pragma once
#include "gdn_common.h"

namespace gdn {

// chunks to a segment of a sequence of `nchunks`
__device__ __forceinline__ int segment_chunks(int nchunks, int segs) { return (nchunks + segs - 1) / segs; }

// the run of chunks a workgroup of a recurrence kernel walks
struct SegmentRun {
  int n, p;            // sequence, segment
  int64_t bos;         // first token
  int len, nchunks;    // tokens and chunks of the run
  int64_t chunk_base;  // its first chunk
};
// ns counts (sequence, segment) pairs of which a launch has `per_seq` to a sequence, beginning at segment `first`
__device__ __forceinline__ SegmentRun segment_run(int ns, int per_seq, int first, int segs, const int64_t* cu,
                                                  const int* chunk_offsets, int T_len) {
  SegmentRun s;
  s.n = ns / per_seq;
  s.p = first + ns % per_seq;
  s.bos = cu ? cu[s.n] : (int64_t)s.n * T_len;
  s.len = cu ? (int)(cu[s.n + 1] - s.bos) : T_len;
  s.nchunks = (s.len + kChunk - 1) / kChunk;
  s.chunk_base = cu ? chunk_offsets[s.n] : (int64_t)s.n * ((T_len + kChunk - 1) / kChunk);
  if (segs > 1) {   // equal runs, the last ones of a short sequence shorter or empty
    const int per = segment_chunks(s.nchunks, segs), c0 = imin(s.p * per, s.nchunks);
    s.nchunks = imin(per, s.nchunks - c0);
    s.len = s.nchunks > 0 ? imin(s.len - c0 * kChunk, s.nchunks * kChunk) : 0;
    s.bos += (int64_t)c0 * kChunk;
    s.chunk_base += c0;
  }
  return s;
}

// start[p + 1] = A_p start[p] + B_p along the segments of a sequence (REVERSE: start[p - 1] = A_p start[p] + B_p), from
// `first` (null: zero).  map: f32 [N, P-1, Hv, K, V + K], the segments 0 .. P-2 (REVERSE: 1 .. P-1); start: f32
// [N, P, Hv, K, V].  An empty segment has no map: the state passes it as it is, infinities included (0 x inf in a product
// with the identity would be NaN).  A workgroup owns 16 columns of one head's states, wave w their rows
// 16 w .. 16 w + 15.  Bound by latency: a step is 32 fp32 matrix instructions per wave behind one barrier, its map
// requested a step ahead (3.2 us a step; requested two steps ahead it takes the same).
template <int DK, bool REVERSE>
__global__ __launch_bounds__(4 * DK) void segment_chain_kernel(const float* __restrict__ map, const float* __restrict__ first,
                                                               float* __restrict__ start, const int64_t* __restrict__ cu,
                                                               int T_len, int segs, int Hv, int V) {
  constexpr int LD = DK + 4, NM = DK / 16;
  __shared__ __align__(16) float hs[2][16 * LD];   // the running state, column-major
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, j = lane >> 4;
  const int n = blockIdx.x / Hv, h = blockIdx.x % Hv, v0 = 16 * blockIdx.y, ld = V + DK;
  const int row0 = 16 * wave + 4 * j;              // the lane's rows row0 .. row0 + 3 of column c
  auto start_at = [&](int p) { return start + ((((int64_t)n * segs + p) * Hv + h) * DK + row0) * V + v0 + c; };
  const int nchunks = ((cu ? (int)(cu[n + 1] - cu[n]) : T_len) + kChunk - 1) / kChunk;
  const int live = nchunks > 0 ? (nchunks - 1) / segment_chunks(nchunks, segs) + 1 : 0;   // segments with chunks
  auto applies = [&](int s) { return s < segs && (REVERSE ? segs - s : s - 1) < live; };
  f32x4 A[NM], B, S;
  auto request = [&](int s) {                      // the map applied in step s = 1 .. segs - 1
    const int i = n * (segs - 1) + (REVERSE ? segs - 1 - s : s - 1);
    const float* m = map + ((int64_t)i * Hv + h) * DK * ld;
#pragma unroll
    for (int k = 0; k < NM; ++k) A[k] = *reinterpret_cast<const f32x4*>(m + (int64_t)(16 * wave + c) * ld + V + 16 * k + 4 * j);
#pragma unroll
    for (int r = 0; r < 4; ++r) B[r] = m[(int64_t)(row0 + r) * ld + v0 + c];
  };
  if (applies(1)) request(1);
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = first ? first[(((int64_t)n * Hv + h) * DK + row0 + r) * V + v0 + c] : 0.f;
  for (int s = 1;; ++s) {
    float* out = start_at(REVERSE ? segs - s : s - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(int64_t)r * V] = S[r];
    if (s == segs) break;
    if (!applies(s)) {
      if (applies(s + 1)) request(s + 1);
      continue;
    }
    float* hb = hs[s & 1];
    *reinterpret_cast<f32x4*>(hb + c * LD + row0) = S;
    __syncthreads();
    // k runs in the order the lanes hold it: lane group j feeds k = 16 m + 4 j + e to instruction (m, e)
    f32x4 a0 = B, a1 = {0.f, 0.f, 0.f, 0.f}, now[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) now[k] = A[k];
    if (applies(s + 1)) request(s + 1);
#pragma unroll
    for (int k = 0; k < NM; ++k) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(hb + c * LD + 16 * k + 4 * j);
      a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(now[k][0], x[0], a0, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(now[k][1], x[1], a1, 0, 0, 0);
      a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(now[k][2], x[2], a0, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(now[k][3], x[3], a1, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = a0[r] + a1[r];
  }
}

}  // namespace gdn
