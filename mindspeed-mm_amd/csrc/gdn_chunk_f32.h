// The two recurrences of the chunked rule in fp32 (the 16-bit types: chunk_state_kernel, chunk_state_bwd_kernel).
//
// Bound by the chain of dependent matrix products: an fp32 matrix instruction does an eighth of a bf16 one's work per
// cycle, and a wave that owns 32 state columns spends 11 (K = 64) to 19 (K = 128) products of 32 x 32 x 32, 1024 cycles
// each, on a chunk, while few heads leave most of the chip idle.  Here four waves share 16 CW columns and split the *rows*
// of every product: wave w owns tokens 16 w .. 16 w + 15 of a chunk and rows 16 w + 64 i .. of the state, in 16 x 16 x 4
// instructions of 32 cycles, and the waves hand each other S, z and V' (dS, dV' and R) through LDS, column by column, where
// an accumulator's four rows are the 16 bytes another wave reads as four steps of its contraction.  A chunk is then 48
// (K = 64) to 80 instructions per wave and column tile instead of 176 to 304 that take twice as long.
// Forward / backward recurrence, us, waves that own 32 columns -> this: 512 tokens, 4 heads, K = V = 64 54 / 90 -> 20 / 28,
// K = V = 128 116 / 141 -> 27 / 40; 2 x 1024 tokens, 32 heads of 128 241 / 286 -> 86 / 129; 4 x 512, 32 heads, V = 256
// 137 / 290 -> 128 / 242.  Of a chunk's 2.2 us (K = 64) the instructions are 0.65; the rest are the waits of the three
// exchanges and the address arithmetic and issue of the next chunk's requests.  Error against float64, 512 tokens, K = 64: o
// 5.8e-7 -> 5.5e-7, final state 6.0e-7 -> 5.8e-7, dq 5.5e-7 -> 5.2e-7, dh0 2.8e-7 -> 2.1e-7.
//
// Order of the contraction: lane group j = lane / 16 feeds k = 16 m + 4 j + e to instruction (m, e), so that operands are
// read 16 bytes at a time.  Tiles arrive in fragment order, 32 x 32 values as [8 pieces of 4 columns][32 rows][4 columns]:
// 16-byte rows of a piece are contraction steps of the tile as it lies, single values those of its transpose.  What is read
// as it lies only (Tm forward; Q^T and Aq backward) goes from memory to the registers of the one wave that needs it; K and,
// backward, Tm pass through LDS, the rows of piece p rotated by p, which puts a transposed read's 64 values on 64 banks.
#pragma once
#include "gdn_common.h"
#include "gdn_segments.h"

namespace gdn {

constexpr int kF32Threads = 256;

template <int DK, int CW> struct StateF32Smem {   // in floats
  static constexpr int cols = 16 * CW, ldk = DK + 4, ldt = 64 + 4;   // padded columns: 16 of them start on 16 x 4 banks
  static constexpr int off_k = 0, off_s = off_k + 64 * DK, off_z = off_s + cols * ldk;
  static constexpr int off_v = off_z + cols * ldt, bytes = (off_v + cols * ldt) * 4;
  static_assert(bytes <= 160 * 1024, "one CU's LDS");
};
template <int DK, int CW> struct StateBwdF32Smem {
  static constexpr int cols = 16 * CW, ldk = DK + 4, ldt = 64 + 4;
  static constexpr int off_k = 0, off_tm = off_k + 64 * DK, off_s = off_tm + 3 * 1024;
  static constexpr int off_do = off_s + cols * ldk, off_dv = off_do + cols * ldt;
  static constexpr int off_r = off_dv + cols * ldt, off_row = off_r + cols * ldt;   // scale e^G [64]
  static constexpr int bytes = (off_row + 64) * 4;
  static_assert(bytes <= 160 * 1024, "one CU's LDS");
};

// place of 16-byte row `row` of piece `p` of tile `t`, in 16-byte units, rows rotated by p
__device__ __forceinline__ int f32_rot_slot(int t, int p, int row) { return t * 256 + p * 32 + ((row + p) & 31); }

// pieces [0, N) of 16 bytes, N a multiple of the threads, global -> registers -> LDS, rows of a piece rotated;
// LOWER: three kept tiles (0,0), (1,0), (1,1) of the four that memory has places for
template <int N, bool LOWER> struct F32Pieces {
  static constexpr int kPer = N / kF32Threads;
  static_assert(N % kF32Threads == 0, "the same number of pieces for every thread");
  f32x4 r[kPer];
  __device__ __forceinline__ void request(const float* src, int tid) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = tid + i * kF32Threads, t = c / 256;
      r[i] = *reinterpret_cast<const f32x4*>(src + ((LOWER && t > 0 ? t + 1 : t) * 256 + c % 256) * 4);
    }
  }
  __device__ __forceinline__ void place(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = tid + i * kF32Threads, q = c % 256;
      reinterpret_cast<f32x4*>(lds)[f32_rot_slot(c / 256, q / 32, q % 32)] = r[i];
    }
  }
};

// B operands of M steps of 16 of a contraction, from columns of `ld` floats in LDS.  All of a product's operands are read
// before its first instruction: read one step at a time each step would wait for the LDS once more.
template <int M, int CW> __device__ __forceinline__ void f32_load(f32x4 (&b)[M][CW], const float* cols, int ld) {
  const int c = threadIdx.x & 15, j = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) b[m][ct] = *reinterpret_cast<const f32x4*>(cols + (16 * ct + c) * ld + 16 * m + 4 * j);
}
// One step: C[16 x 16] += A B for CW column tiles; a: the lane's 4 values of its row of A.  Two accumulators take turns (an
// instruction that adds to the previous one's result waits for it).
template <int CW> __device__ __forceinline__ void f32_step(f32x4 (&acc)[2][CW], f32x4 a, const f32x4 (&b)[CW]) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
      acc[e & 1][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[ct][e], acc[e & 1][ct], 0, 0, 0);
}
// steps of a triangular product that a wave has no part in: B cleared (A there repeats a step of the wave's own rows), for a
// branch around a step costs more than the step
template <int CW> __device__ __forceinline__ void f32_keep(f32x4 (&b)[CW], bool keep) {
#pragma unroll
  for (int ct = 0; ct < CW; ++ct)
#pragma unroll
    for (int e = 0; e < 4; ++e) b[ct][e] = keep ? b[ct][e] : 0.f;
}
template <int CW> __device__ __forceinline__ void f32_zero(f32x4 (&acc)[2][CW]) {
#pragma unroll
  for (int ct = 0; ct < CW; ++ct) acc[0][ct] = acc[1][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
}
// a rotated tile set's rows row0 + lane % 16 of tile t, contraction steps 16 (m & 1) .. of its columns
__device__ __forceinline__ f32x4 f32_rows(const float* lds, int t, int m, int row0) {
  const int j = (threadIdx.x & 63) >> 4;
  return reinterpret_cast<const f32x4*>(lds)[f32_rot_slot(t, 4 * (m & 1) + j, row0 + (threadIdx.x & 15))];
}
// acc += K S for the wave's 16 tokens, 64 key channels' operands at a time
template <int DK, int CW>
__device__ __forceinline__ void f32_rows_product(f32x4 (&acc)[2][CW], const float* Ks, const float* Sx, int ldk, int wave) {
#pragma unroll
  for (int mb = 0; mb < DK / 16; mb += 4) {
    f32x4 ka[4], sb[4][CW];
#pragma unroll
    for (int m = 0; m < 4; ++m) ka[m] = f32_rows(Ks, ((mb + m) >> 1) * 2 + (wave >> 1), m, 16 * (wave & 1));
    f32_load(sb, Sx + 16 * mb, ldk);
    GDN_SCHED_FENCE();
#pragma unroll
    for (int m = 0; m < 4; ++m) f32_step<CW>(acc, ka[m], sb[m]);
  }
}
// the transposed read: column col0 + lane % 16 (of 32) of tile t, contraction steps 16 (m & 1) .. of its rows
__device__ __forceinline__ f32x4 f32_cols(const float* lds, int t, int m, int col0) {
  const int j = (threadIdx.x & 63) >> 4, col = col0 + (threadIdx.x & 15), p = col >> 2;
  f32x4 a;
#pragma unroll
  for (int e = 0; e < 4; ++e) a[e] = lds[f32_rot_slot(t, p, 16 * (m & 1) + 4 * j + e) * 4 + (col & 3)];
  return a;
}
// the same as f32_rows from a tile in memory
__device__ __forceinline__ f32x4 f32_rows_mem(const float* tile, int m, int row0, int tid) {
  return reinterpret_cast<const f32x4*>(tile)[(4 * (m & 1) + ((tid & 63) >> 4)) * 32 + row0 + (tid & 15)];
}
__device__ __forceinline__ f32x4 f32_ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// Per chunk: y = K S; z = beta (v - e^G y); V' = Tm z; S <- e^{G_last} S + K^T (e^{G_last - G} V').
// vf, hf: V' and the state before each chunk, in fragment order.
template <int DK, int CW>
__global__ __launch_bounds__(kF32Threads) GDN_WAVES_PER_SIMD(2) void chunk_state_f32_kernel(
    const float* __restrict__ kaf, const float* __restrict__ ai, const float* __restrict__ v, const float* __restrict__ G,
    const float* __restrict__ bt, const float* __restrict__ h0, float* __restrict__ ht, float* __restrict__ vf,
    float* __restrict__ hf, const int64_t* __restrict__ cu, const int* __restrict__ chunk_offsets, int T_len, int Hqk, int Hv,
    int V, int64_t v_stride) {
  using SM = StateF32Smem<DK, CW>;
  constexpr int NKT = DK / 32, RT = DK / 64;   // RT: row tiles of the state per wave
  float* const lds = reinterpret_cast<float*>(gdn_smem);
  float *Ks = lds + SM::off_k, *Sx = lds + SM::off_s, *Zx = lds + SM::off_z, *Vx = lds + SM::off_v;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x / Hv, h = blockIdx.x % Hv, v0 = 16 * CW * blockIdx.y;
  const SegmentRun run = segment_run(n, 1, 0, 1, cu, chunk_offsets, T_len);
  const int row = 16 * wave + 4 * j;           // the lane's tokens of a chunk: row .. row + 3

  f32x4 S[RT][CW];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[rt][ct][r] = h0 != nullptr ? h0[(((int64_t)n * Hv + h) * DK + 64 * rt + row + r) * V + v0 + 16 * ct + c] : 0.f;

  struct Set {
    F32Pieces<16 * DK, false> k;
    f32x4 t[4];                                // the wave's rows of Tm
    float v[CW][4];
    f32x4 g, b;
    float gl;
  };
  auto request = [&](int ch_, Set& p, int on) {   // on: -1, or 0: every lane asks for what the first one does, and no one uses it
    const int tid_ = tid & on, c_ = c & on, row_ = row & on;
    const int nvalid = imin(kChunk, run.len - ch_ * kChunk);
    const int64_t ch = (run.chunk_base + ch_) * Hv + h, tok0 = run.bos + (int64_t)ch_ * kChunk;
    p.k.request(kaf + ((run.chunk_base + ch_) * Hqk + h / (Hv / Hqk)) * (64 * DK), tid_);
#pragma unroll
    for (int m = 0; m < 4; ++m)   // steps above the diagonal repeat the last one and are not used
      p.t[m] = f32_rows_mem(ai + ch * 4096 + (2 * (wave >> 1) + (imin(m, wave) >> 1)) * 1024, m, 16 * (wave & 1), tid_);
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        p.v[ct][r] = v[(tok0 + imin(row_ + r, nvalid - 1)) * v_stride + (int64_t)h * V + v0 + 16 * ct + c_];
    p.g = f32_ld4(G + ch * 64 + row_);
    p.b = f32_ld4(bt + ch * 64 + row_);
    p.gl = G[ch * 64 + 63];
  };
  auto step = [&](int ci, Set& p, auto more) {   // more: a chunk follows (K = 64)
    const int64_t ch = (run.chunk_base + ci) * Hv + h;
    const int nvalid = imin(kChunk, run.len - ci * kChunk);
    p.k.place(Ks, tid);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) {
        *reinterpret_cast<f32x4*>(Sx + (16 * ct + c) * SM::ldk + 64 * rt + row) = S[rt][ct];
        const int k0 = 64 * rt + row, col = v0 + 16 * ct + c;   // the state before the chunk
        *reinterpret_cast<f32x4*>(hf + (((ch * (V / 32) + col / 32) * NKT + k0 / 32) * 256 + (k0 % 32) / 4 * 32 + col % 32) * 4) = S[rt][ct];
      }
    f32x4 bt4, eg4, ed4, tm[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) tm[m] = p.t[m];
    float vv[CW][4];
    const float eg = __expf(p.gl);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bt4[r] = p.b[r];
      eg4[r] = __expf(p.g[r]);
      ed4[r] = __expf(p.gl - p.g[r]);
    }
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) vv[ct][r] = p.v[ct][r];
    GDN_LDS_BARRIER();   // (not __syncthreads(), which would wait for the stores of S)
    // Behind the last chunk there is nothing to ask for, and asking for that chunk once more cost a sequence of one chunk up
    // to a quarter of its time.  64 sequences of 64 tokens, 32 heads, us: K = V = 64 67 -> 60 with a last step of its own; K =
    // V = 128, where that spills (4 x 1024 tokens 132 -> 182), 206 -> 167 with every lane asking for the same line (130).
    if constexpr (DK == 128) request(imin(ci + 1, run.nchunks - 1), p, ci + 1 < run.nchunks ? -1 : 0);
    else if constexpr (decltype(more)::value) request(ci + 1, p, -1);
    f32x4 acc[2][CW], kt[RT][4], xb[4][CW];
    // y = K S
    f32_zero<CW>(acc);
    f32_rows_product<DK, CW>(acc, Ks, Sx, SM::ldk, wave);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)   // K^T, for the last product
#pragma unroll
      for (int m = 0; m < 4; ++m) kt[rt][m] = f32_cols(Ks, (2 * rt + (wave >> 1)) * 2 + (m >> 1), m, 16 * (wave & 1));
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      f32x4 z;
#pragma unroll
      for (int r = 0; r < 4; ++r) z[r] = row + r < nvalid ? bt4[r] * (vv[ct][r] - eg4[r] * (acc[0][ct][r] + acc[1][ct][r])) : 0.f;
      *reinterpret_cast<f32x4*>(Zx + (16 * ct + c) * SM::ldt + row) = z;
    }
    GDN_LDS_BARRIER();
    // V' = Tm z, lower triangular
    f32_load(xb, Zx, SM::ldt);
    f32_zero<CW>(acc);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f32_keep<CW>(xb[m], m <= wave);
      f32_step<CW>(acc, tm[m], xb[m]);
    }
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      const f32x4 x = acc[0][ct] + acc[1][ct];
      const int col = v0 + 16 * ct + c;
      *reinterpret_cast<f32x4*>(vf + (((ch * (V / 32) + col / 32) * 2 + row / 32) * 256 + (row % 32) / 4 * 32 + col % 32) * 4) = x;
      *reinterpret_cast<f32x4*>(Vx + (16 * ct + c) * SM::ldt + row) = x * ed4;
    }
    GDN_LDS_BARRIER();
    // S <- e^{G_last} S + K^T (e^{G_last - G} V')
    f32_load(xb, Vx, SM::ldt);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      f32_zero<CW>(acc);
#pragma unroll
      for (int m = 0; m < 4; ++m) f32_step<CW>(acc, kt[rt][m], xb[m]);
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) S[rt][ct] = eg * S[rt][ct] + (acc[0][ct] + acc[1][ct]);
    }
    GDN_LDS_BARRIER();   // K and S in LDS are consumed
  };
  if (run.nchunks > 0) {
    Set set;
    request(0, set, -1);
    const int steps = DK == 128 ? run.nchunks : run.nchunks - 1;
    for (int ci = 0; ci < steps; ++ci) step(ci, set, std::true_type{});
    if constexpr (DK != 128) step(steps, set, std::false_type{});
  }
  if (ht != nullptr) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CW; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) ht[(((int64_t)n * Hv + h) * DK + 64 * rt + row + r) * V + v0 + 16 * ct + c] = S[rt][ct][r];
  }
}

// Per chunk, last to first: dV' = e^{G_last - G} (K dS) + (scale Aq)^T dO; R = Tm^T dV';
// dS <- e^{G_last} dS + Q^T (scale e^G dO) - K^T (beta e^G R).  dvf, dhf: dV' and the gradient of the state after a chunk.
template <int DK, int CW>
__global__ __launch_bounds__(kF32Threads) GDN_WAVES_PER_SIMD(DK == 64 ? 2 : 1) void chunk_state_bwd_f32_kernel(
    const float* __restrict__ kaf, const float* __restrict__ qtf, const float* __restrict__ ai, const float* __restrict__ aqf,
    const float* __restrict__ dO, const float* __restrict__ G, const float* __restrict__ bt, const float* __restrict__ dht,
    float* __restrict__ dh0, float* __restrict__ dvf, float* __restrict__ dhf, const int64_t* __restrict__ cu,
    const int* __restrict__ chunk_offsets, int T_len, int Hqk, int Hv, int V, float scale) {
  using SM = StateBwdF32Smem<DK, CW>;
  constexpr int NKT = DK / 32, RT = DK / 64;
  float* const lds = reinterpret_cast<float*>(gdn_smem);
  float *Ks = lds + SM::off_k, *Tms = lds + SM::off_tm, *Sx = lds + SM::off_s, *Dx = lds + SM::off_do;
  float *Vx = lds + SM::off_dv, *Rx = lds + SM::off_r, *Es = lds + SM::off_row;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, j = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x / Hv, h = blockIdx.x % Hv, v0 = 16 * CW * blockIdx.y;
  const SegmentRun run = segment_run(n, 1, 0, 1, cu, chunk_offsets, T_len);
  const int row = 16 * wave + 4 * j;

  f32x4 dS[RT][CW];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        dS[rt][ct][r] = dht != nullptr ? dht[(((int64_t)n * Hv + h) * DK + 64 * rt + row + r) * V + v0 + 16 * ct + c] : 0.f;

  struct Set {
    F32Pieces<16 * DK, false> k;
    F32Pieces<768, true> t;
    f32x4 a[4];                                // the wave's rows of Aq^T
    float d[CW][4];
    f32x4 g, b;
    float gl;
  };
  auto request = [&](int ch_, Set& p) {
    const int nvalid = imin(kChunk, run.len - ch_ * kChunk);
    const int64_t ch = (run.chunk_base + ch_) * Hv + h, tok0 = run.bos + (int64_t)ch_ * kChunk;
    p.k.request(kaf + ((run.chunk_base + ch_) * Hqk + h / (Hv / Hqk)) * (64 * DK), tid);
    p.t.request(ai + ch * 4096, tid);
#pragma unroll
    for (int m = 0; m < 4; ++m)   // the tiles of Aq are stored by columns: its transpose as it lies
      p.a[m] = f32_rows_mem(aqf + ch * 4096 + (2 * (imax(m, wave) >> 1) + (wave >> 1)) * 1024, m, 16 * (wave & 1), tid);
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        p.d[ct][r] = dO[((tok0 + imin(row + r, nvalid - 1)) * Hv + h) * V + v0 + 16 * ct + c];
    p.g = f32_ld4(G + ch * 64 + row);
    p.b = f32_ld4(bt + ch * 64 + row);
    p.gl = G[ch * 64 + 63];
  };
  auto step = [&](int ci, Set& p, auto more) {   // more: requests follow
    const int64_t ch = (run.chunk_base + ci) * Hv + h;
    const int nvalid = imin(kChunk, run.len - ci * kChunk);
    p.k.place(Ks, tid);
    p.t.place(Tms, tid);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) {
        const int k0 = 64 * rt + row, col = v0 + 16 * ct + c;
        *reinterpret_cast<f32x4*>(Sx + (16 * ct + c) * SM::ldk + k0) = dS[rt][ct];
        *reinterpret_cast<f32x4*>(dhf + (((ch * (V / 32) + col / 32) * NKT + k0 / 32) * 256 + (k0 % 32) / 4 * 32 + col % 32) * 4) = dS[rt][ct];
      }
    f32x4 ed4, nb4, se4, at[4], qt[RT][4];   // e^{G_last - G}, -beta e^G, scale e^G
    const float eg = __expf(p.gl);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ed4[r] = __expf(p.gl - p.g[r]);
      nb4[r] = row + r < nvalid ? -p.b[r] * __expf(p.g[r]) : 0.f;
      se4[r] = scale * __expf(p.g[r]);
    }
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = row + r < nvalid ? p.d[ct][r] : 0.f;
      *reinterpret_cast<f32x4*>(Dx + (16 * ct + c) * SM::ldt + row) = x;
    }
    if (c == 0) *reinterpret_cast<f32x4*>(Es + row) = se4;
#pragma unroll
    for (int m = 0; m < 4; ++m) at[m] = p.a[m];
    GDN_LDS_BARRIER();   // (not __syncthreads(), which would wait for the stores of dS)
    {   // Q^T of this chunk, needed last, then what the next one begins with
      const float* qc = qtf + ((run.chunk_base + ci) * Hqk + h / (Hv / Hqk)) * (64 * DK);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int m = 0; m < 4; ++m) qt[rt][m] = f32_rows_mem(qc + ((2 * rt + (wave >> 1)) * 2 + (m >> 1)) * 1024, m, 16 * (wave & 1), tid);
    }
    if constexpr (decltype(more)::value) request(imax(ci - 1, 0), p);
    f32x4 acc[2][CW], aq[2][CW], kt[RT][4], tt[4], db[4][CW], xb[4][CW];
    // dV'
    f32_zero<CW>(acc);
    f32_zero<CW>(aq);
    f32_rows_product<DK, CW>(acc, Ks, Sx, SM::ldk, wave);
    f32_load(db, Dx, SM::ldt);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f32x4 x[CW];
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) x[ct] = db[m][ct];
      f32_keep<CW>(x, m >= wave);
      f32_step<CW>(aq, at[m], x);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)   // Tm^T; steps before the diagonal repeat its own and are not used
      tt[m] = f32_cols(Tms, (imax(m, wave) >> 1) + (wave >> 1), m, 16 * (wave & 1));
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      const f32x4 x = ed4 * (acc[0][ct] + acc[1][ct]) + (aq[0][ct] + aq[1][ct]);
      const int col = v0 + 16 * ct + c;
      *reinterpret_cast<f32x4*>(dvf + (((ch * (V / 32) + col / 32) * 2 + row / 32) * 256 + (row % 32) / 4 * 32 + col % 32) * 4) = x;
      *reinterpret_cast<f32x4*>(Vx + (16 * ct + c) * SM::ldt + row) = x;
    }
    GDN_LDS_BARRIER();
    // R = Tm^T dV', upper triangular
    f32_load(xb, Vx, SM::ldt);
    f32_zero<CW>(acc);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f32_keep<CW>(xb[m], m >= wave);
      f32_step<CW>(acc, tt[m], xb[m]);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        kt[rt][m] = f32_cols(Ks, (2 * rt + (wave >> 1)) * 2 + (m >> 1), m, 16 * (wave & 1));
        qt[rt][m] *= f32_ld4(Es + 16 * m + 4 * j);   // scale e^G rides on Q^T
      }
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
      *reinterpret_cast<f32x4*>(Rx + (16 * ct + c) * SM::ldt + row) = nb4 * (acc[0][ct] + acc[1][ct]);
    GDN_LDS_BARRIER();
    // dS <- e^{G_last} dS + Q^T (scale e^G dO) + K^T (-beta e^G R)
    f32_load(xb, Rx, SM::ldt);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      f32_zero<CW>(acc);
#pragma unroll
      for (int m = 0; m < 4; ++m) f32_step<CW>(acc, qt[rt][m], db[m]);
#pragma unroll
      for (int m = 0; m < 4; ++m) f32_step<CW>(acc, kt[rt][m], xb[m]);
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) dS[rt][ct] = eg * dS[rt][ct] + (acc[0][ct] + acc[1][ct]);
    }
    GDN_LDS_BARRIER();   // the tiles and dS, R in LDS are consumed
  };
  if (run.nchunks > 0) {
    Set set;
    request(run.nchunks - 1, set);
    // K = 128: the last step without requests (64 sequences of 64 tokens, 32 heads of 128: 320 -> 278 us; 17 of 500: 556 -> 547).
    // K = 64 repeats the requests of its last chunk: the step twice spills there (64 sequences of 64 tokens, 32 heads of 64: 86 -> 137 us).
    constexpr int kLast = DK == 64 ? 0 : 1;
    for (int ci = run.nchunks - 1; ci >= kLast; --ci) step(ci, set, std::true_type{});
    if constexpr (kLast == 1) step(0, set, std::false_type{});
  }
  if (dh0 != nullptr) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CW; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) dh0[(((int64_t)n * Hv + h) * DK + 64 * rt + row + r) * V + v0 + 16 * ct + c] = dS[rt][ct][r];
  }
}

// Columns to a workgroup: 16 while the compute units hold all of those workgroups at once (per_unit each: 2, but 1 for the
// reverse recurrence with K = 128, whose registers fill a unit), else 32, which read the tiles half as often; the same bits.
// 512 tokens, K = V, 16 / 32 columns, us, by the workgroups of 16 columns.  Forward, 64: 256 22 / 30, 512 31 / 33, 768 46 / 46,
// 1024 62 / 49; 128: 256 31 / 44, 384 41 / 46, 512 44 / 47, 768 65 / 65, 1024 81 / 69.  Reverse, 64: 256 33 / 45, 512 46 / 48,
// 768 69 / 68, 1024 93 / 72; 128: 256 44 / 63, 384 81 / 67, 512 84 / 68.
inline bool f32_sixteen_columns(int64_t sequences, int Hv, int V, int compute_units, int per_unit) {
  return sequences * Hv * (V / 16) <= (int64_t)per_unit * compute_units;
}

}  // namespace gdn
