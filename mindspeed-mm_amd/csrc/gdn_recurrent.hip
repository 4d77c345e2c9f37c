// Fused recurrent gated delta rule (decode).  Per (sequence b, value head h) and token t:
//     S <- e^{g} S;  delta = beta (v - S^T k);  S <- S + k delta^T;  o = scale S^T q
// (reference math: mindspeed_mm/fsdp/models/qwen3_5/modeling_qwen3_5.py:478-517).
//
// The kernel is bound by streaming the fp32 state [K,V] (64 KB at K=V=128) through HBM once in, once
// out (a batch of 256 with 32 heads: 1.08 GB in 183 us = 5.9 TB/s on states that no cache holds, 162 us = 6.7 TB/s where the
// memory-side cache holds a part of them; 217 and 163 us with the loads left to themselves).  256 threads own a [K, BV] column
// slab of one state, a workgroup one slab, or in a decode step with its convolution 1, 2 or 4; a slab lives in registers for
// all T tokens of the call.  With S_old the state before the token,
//     S^T k = e^g (S_old^T k),   S^T q = e^g (S_old^T q) + (k.q) delta
// so both contractions are taken in ONE pass over the registers, then the rank-1 update is applied.
// No MFMA: 6 flop per 8 bytes of state traffic, far below the matrix-core ridge.
//
// q, k, v are read with a token stride, so they can be the column ranges of the convolution's [tokens, D] output, and
// the gates can be formed here from the layer's projections (g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b)
// rounded to b's dtype as the layer's `b.sigmoid()` is; modeling_qwen3_5.py:833-841) instead of being passed in: a
// decode step of the layer is then the convolution update followed by this kernel, with no copies in between, or, where
// launch_decode_step takes the sizes, this kernel alone (CONV).
#include "gdn_chunk.h"
#include "gdn_common.h"
#include "gdn_profile.h"

namespace gdn {

struct RecurrentGates {   // either g, beta (fp32 [tokens,Hv]) or the projections a, b [tokens,Hv] and A_log, dt_bias [Hv]
  const float* g;
  const float* beta;
  const void* a;
  const void* b;
  const void* A_log;
  const void* dt_bias;
};

// A decode step's convolution update, where the kernel does it too: one token per sequence, S = W taps, the rows of
// conv_state [B,D,W] and weight [D,W] one vector load each, D = 2 Hqk K + Hv V.
struct RecurrentConv {
  const void* hidden;   // [B,D]
  void* state;
  const void* weight;
  const void* bias;     // [D] or null
  int silu;
};

// n consecutive values, n * sizeof(T) <= 16 bytes, in one load; aligned as their type is, not as the load is wide
template <typename T, int n> __device__ __forceinline__ void load_run(float* dst, const T* p) {
  constexpr int bytes = n * (int)sizeof(T);
  static_assert(bytes == 2 || bytes == 4 || bytes == 8 || bytes == 16, "2 to 16 bytes");
  float f[Elem<T>::kVec];
  Vec16<T> x = zero16<T>();
  __builtin_memcpy(&x.raw, p, bytes);
  unpack16<T>(x, f);
#pragma unroll
  for (int e = 0; e < n; ++e) dst[e] = f[e];
}

// A workgroup's slab is BV columns of one state, 4 of them per thread in RPT rows.  Everything a token needs is requested
// at once: the slab, k and q (each wave normalises them by itself and keeps them in a part of the LDS of its own), v and
// the gates; the only barrier of a token lies between the waves' partial sums over the rows.
// The sums over the rows run in one order whatever BV is, so that a sequence's bits do not depend on the size of its batch,
// which decides BV: 32 chains of the rows r, r + 32, ..., r = g + 8 m; then over m = 0 .. 3 in pairs, over the two g of a
// wave, over the waves.  A thread holds BV / 32 of the m; the others and the second g are lanes of its wave.
// waves per SIMD the registers have to allow: left to itself the compiler takes 280 for some of the smaller slabs
constexpr int recurrent_waves(int dk, int bv) { return dk * bv <= 128 * 128 ? 4 : 2; }

// How the states are loaded.  kStream passes by the caches, which hold states that fit them (kCached) from one step to the
// next.  Larger ones pass through the 256 MB memory-side cache for nothing and cost bandwidth on their way; kMixed leaves it
// a fixed part of them, of every kKeepPeriod workgroups (about what the device has in flight) the first kKept, so that hits
// and memory work side by side: 256 sequences of 32 heads (512 MB), the same states every step 162 us (kCached 163, kStream
// 184), two or three sets of states in turn 162 (217, 183), six sets 183 (217, 182).
enum class StateLoads { kCached, kStream, kMixed };
constexpr int kKeepPeriod = 512, kKept = 80;

// CONV = 0: q, k, v come from memory.  CONV = n: a decode step with its convolution update in one launch.  A workgroup is n
// groups of 256 threads, a slab each, and covers all slabs of all value heads of one q/k head: it alone reads and rolls the
// convolution states of its channels, so no other workgroup can meet them half done.  Its threads form the convolution's
// outputs, a channel at a time, and leave them in LDS while the slabs are on their way.
template <typename T, typename TP, int DK, int BV, StateLoads LOADS, int CONV = 0>
__global__ __launch_bounds__(256 * (CONV ? CONV : 1), recurrent_waves(DK, BV)) void recurrent_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int64_t sq, int64_t sk, int64_t sv,
    RecurrentGates gates, const float* state_in, float* state_out, T* __restrict__ o, const int64_t* __restrict__ cu,
    int T_len, int Hqk, int Hv, int V, float scale, int use_l2norm, RecurrentConv conv) {
  constexpr int UN = CONV ? CONV : 1;   // slabs of the workgroup
  constexpr int CG = BV / 4;            // column groups (4 fp32 = 16 bytes each)
  constexpr int MC = BV / 32;           // chains of rows held by a thread
  constexpr int NJ = DK / 32;           // rows of a chain
  constexpr int EPL = DK / 64;          // elements of k and q per lane for the norms
  static_assert(MC == 1 || MC == 2 || MC == 4, "tile shape");
  __shared__ float red_[UN][2][4][CG][8], kq_rows_[UN][4][DK][2];
  __shared__ float conv_out[CONV ? 2 * DK + UN * BV : 1];   // q, k, then v of the value heads in their order

  const int unit = CONV ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  auto& red = red_[unit];
  auto& kq_rows = kq_rows_[unit];
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int cg = tid % CG, lrow = lane / CG;
  const int row0 = 2 * wave + lrow / (4 / MC) + 8 * MC * (lrow % (4 / MC));
  // the thread's rows are row0 + 32 j + 8 m
  // the slabs of a state are neighbours in the launch order: what is in flight then stays close together in memory
  const int nslab = V / BV, slab = blockIdx.x * UN + unit, bh = slab / nslab, b = bh / Hv, h = bh % Hv, hq = h / (Hv / Hqk);
  const int v0 = (slab % nslab) * BV + cg * 4;
  const int64_t sbase = ((int64_t)bh * DK + row0) * V + v0;

  // the convolution's operands are requested ahead of the slab and used behind its requests
  constexpr int W = 4, NCH = 2 * DK + UN * BV, CPT = CONV ? (NCH + 256 * UN - 1) / (256 * UN) : 1;   // channels per thread
  typedef uint32_t RowVec __attribute__((ext_vector_type(W * (int)sizeof(T) / 4)));
  union Row { RowVec v; T e[W]; };
  Row cs[CPT], cw[CPT];
  T cx[CPT], cb[CPT];
  auto channel = [&](int i) {   // (column of the convolution's output, place in conv_out) of the thread's i-th channel
    const int c = imin((int)threadIdx.x + 256 * UN * i, NCH - 1);
    return c < DK ? hq * DK + c : c < 2 * DK ? (Hqk + hq) * DK + c - DK : 2 * Hqk * DK + hq * (Hv / Hqk) * V + c - 2 * DK;
  };
  if constexpr (CONV != 0) {
    const int D = 2 * Hqk * DK + Hv * V;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int d = channel(i);
      cs[i].v = *reinterpret_cast<const RowVec*>(static_cast<const T*>(conv.state) + ((int64_t)b * D + d) * W);
      cw[i].v = *reinterpret_cast<const RowVec*>(static_cast<const T*>(conv.weight) + (int64_t)d * W);
      cx[i] = static_cast<const T*>(conv.hidden)[(int64_t)b * D + d];
      if (conv.bias != nullptr) cb[i] = static_cast<const T*>(conv.bias)[d];
    }
    GDN_SCHED_FENCE();
  }
  // the arithmetic of the stand-alone update (conv1d_update_kernel): the same bits
  auto convolve = [&]() {
    const int D = 2 * Hqk * DK + Hv * V;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = (int)threadIdx.x + 256 * UN * i;
      float st[W + 1], a = conv.bias != nullptr ? Elem<T>::to_f(cb[i]) : 0.f;
#pragma unroll
      for (int j = 0; j < W; ++j) st[j] = Elem<T>::to_f(cs[i].e[j]);
      st[W] = Elem<T>::to_f(cx[i]);
#pragma unroll
      for (int w = 0; w < W; ++w) a += st[1 + w] * Elem<T>::to_f(cw[i].e[w]);
      if (c < NCH) {
        conv_out[c] = Elem<T>::to_f(Elem<T>::from_f(conv.silu ? a * sigmoidf_(a) : a));
        Row r;
#pragma unroll
        for (int j = 0; j < W; ++j) r.e[j] = Elem<T>::from_f(st[1 + j]);
        *reinterpret_cast<RowVec*>(static_cast<T*>(conv.state) + ((int64_t)b * D + channel(i)) * W) = r.v;
      }
    }
  };

  f32x4 S[NJ][MC];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int m = 0; m < MC; ++m) S[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (state_in != nullptr) {
    auto load = [&](auto stream) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int m = 0; m < MC; ++m) {
          const f32x4* p = reinterpret_cast<const f32x4*>(state_in + sbase + (int64_t)(32 * j + 8 * m) * V);
          if constexpr (decltype(stream)::value) S[j][m] = __builtin_nontemporal_load(p);
          else S[j][m] = *p;
        }
      if constexpr (CONV != 0) {
        // here, inside the branch of the loads, at whose end the compiler waits for them; and nothing of it between the
        // requests (47 registers spilled with slabs of 128 columns)
        asm volatile("" ::: "memory");
        GDN_SCHED_FENCE();
        convolve();
        asm volatile("" ::: "memory");
      }
    };
    if constexpr (LOADS == StateLoads::kCached) {
      load(std::false_type{});
    } else if (LOADS == StateLoads::kStream || blockIdx.x % (kKeepPeriod / UN) >= kKept / UN) {
      load(std::true_type{});
    } else {
      asm volatile("" ::: "memory");   // or the compiler makes one branch of the two, and its loads plain
      load(std::false_type{});
      asm volatile("" ::: "memory");
    }
  } else if constexpr (CONV != 0) {
    convolve();
  }
  if constexpr (CONV != 0) GDN_LDS_BARRIER();

  // packed input (cu given): "sequence" b owns the tokens cu[b] .. cu[b+1] of the one batch row
  const int64_t tok0 = cu != nullptr ? cu[b] : (int64_t)b * T_len;
  const int ntok = cu != nullptr ? (int)(cu[b + 1] - cu[b]) : T_len;
  for (int t = 0; t < ntok; ++t) {
    const int64_t tok = tok0 + t;
    float ke[EPL], qe[EPL], vv[4];
    if constexpr (CONV != 0) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) { qe[e] = conv_out[lane * EPL + e]; ke[e] = conv_out[DK + lane * EPL + e]; }
#pragma unroll
      for (int c = 0; c < 4; ++c) vv[c] = conv_out[2 * DK + unit * BV + cg * 4 + c];
    } else {
      load_run<T, EPL>(ke, k + tok * sk + hq * DK + lane * EPL);
      load_run<T, EPL>(qe, q + tok * sq + hq * DK + lane * EPL);
      load_run<T, 4>(vv, v + tok * sv + h * V + v0);
    }
    float eg, bt;
    if (gates.a == nullptr) {
      eg = __expf(gates.g[tok * Hv + h]);
      bt = gates.beta[tok * Hv + h];
    } else {
      const float x = Elem<T>::to_f(static_cast<const T*>(gates.a)[tok * Hv + h]) +
                      Elem<TP>::to_f(static_cast<const TP*>(gates.dt_bias)[h]);
      const float sp = x > 20.f ? x : log1pf(expf(x));
      eg = __expf(-expf(Elem<TP>::to_f(static_cast<const TP*>(gates.A_log)[h])) * sp);   // as __expf(g) of a passed-in g
      const float sg = 1.f / (1.f + expf(-Elem<T>::to_f(static_cast<const T*>(gates.b)[tok * Hv + h])));
      bt = Elem<T>::to_f(Elem<T>::from_f(sg));
    }
    // ---- optional l2 norm of k and q; q carries the scale ----
    float tk = 0.f, tq = 0.f, kq = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) { tk += ke[e] * ke[e]; tq += qe[e] * qe[e]; kq += ke[e] * qe[e]; }
    tk = wave_sum_dpp(tk);
    tq = wave_sum_dpp(tq);
    kq = wave_sum_dpp(kq);
    float rk = 1.f, rq = scale;
    if (use_l2norm) { rk = rsqrtf(tk + 1e-6f); rq = scale * rsqrtf(tq + 1e-6f); }
    kq *= rk * rq;
    float (*kw)[2] = kq_rows[wave];
    GDN_WAVE_LDS_SYNC();   // the previous token's reads are done
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      kw[lane * EPL + e][0] = ke[e] * rk;
      kw[lane * EPL + e][1] = qe[e] * rq;
    }
    GDN_WAVE_LDS_SYNC();

    // ---- one pass over the slab: S_old^T k and S_old^T q ----
    f32x4 ck[MC], cq[MC];
#pragma unroll
    for (int m = 0; m < MC; ++m) ck[m] = cq[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        const float kk = kw[row0 + 32 * j + 8 * m][0], qq = kw[row0 + 32 * j + 8 * m][1];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          ck[m][c] = fmaf(S[j][m][c], kk, ck[m][c]);
          cq[m][c] = fmaf(S[j][m][c], qq, cq[m][c]);
        }
      }
    f32x4 pk = ck[0], pq = cq[0];
    if constexpr (MC == 2) { pk = ck[0] + ck[1]; pq = cq[0] + cq[1]; }
    if constexpr (MC == 4) { pk = (ck[0] + ck[1]) + (ck[2] + ck[3]); pq = (cq[0] + cq[1]) + (cq[2] + cq[3]); }
#pragma unroll
    for (int m = CG; m < 64; m <<= 1) {
#pragma unroll
      for (int c = 0; c < 4; ++c) { pk[c] += __shfl_xor(pk[c], m); pq[c] += __shfl_xor(pq[c], m); }
    }
    float (*rd)[CG][8] = red[t & 1];   // two sets: one is read while the next token's is written
    if (lane < CG) {
#pragma unroll
      for (int c = 0; c < 4; ++c) { rd[wave][cg][c] = pk[c]; rd[wave][cg][4 + c] = pq[c]; }
    }
    GDN_LDS_BARRIER();
    float delta[4], ov[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float skv = rd[0][cg][c] + rd[1][cg][c] + rd[2][cg][c] + rd[3][cg][c];
      const float sqv = rd[0][cg][4 + c] + rd[1][cg][4 + c] + rd[2][cg][4 + c] + rd[3][cg][4 + c];
      delta[c] = bt * fmaf(-eg, skv, vv[c]);
      ov[c] = fmaf(eg, sqv, kq * delta[c]);
    }
    // ---- rank-1 update in registers ----
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        const float kk = kw[row0 + 32 * j + 8 * m][0];
#pragma unroll
        for (int c = 0; c < 4; ++c) S[j][m][c] = fmaf(kk, delta[c], eg * S[j][m][c]);
      }
    if (wave == 0 && lrow == 0) {
      T* op = o + (tok * Hv + h) * V + v0;
      if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<f32x4*>(op) = f32x4{ov[0], ov[1], ov[2], ov[3]};
      } else {
        *reinterpret_cast<u32x2*>(op) = u32x2{f32x2_to_bf16x2(ov[0], ov[1]), f32x2_to_bf16x2(ov[2], ov[3])};
      }
    }
  }

  if (state_out != nullptr) {
    GDN_WAIT_VMEM();   // once, where the compiler waits before every store (195 -> 184 us at 256 sequences of 32 heads)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int m = 0; m < MC; ++m)   // streaming store: the slab is not read again by this kernel
        __builtin_nontemporal_store(S[j][m], reinterpret_cast<f32x4*>(state_out + sbase + (int64_t)(32 * j + 8 * m) * V));
  }
}

template <typename T, typename TP>
static int launch_recurrent(const void* q, const void* k, const void* v, int64_t sq, int64_t sk, int64_t sv,
                            const RecurrentGates& gates, const float* state_in, float* state_out, void* o, int B,
                            int T_len, int Hqk, int Hv, int K, int V, float scale, int use_l2norm, hipStream_t stream,
                            const int64_t* cu = nullptr) {
  // Times in us, the same states every step / three sets of states in turn.
  // 32 columns per workgroup while wider slabs would leave CUs without one (32 heads: one sequence 8.1 -> 7.1, 16 sequences
  // 18 against 14), else 128, or 64 where V asks for it (V = 64, 32 sequences: 15.3 / 15.2 with 32 columns, 11.9 / 14.6).
  // K = 256: 64 (V = 128, 1 GB of states 326 / 382, 128 columns 340 / 390), but 128 for states in the memory-side cache
  // (64 MB 26.2 -> 24.3) and for rows of several such slabs beyond it (V = 256, 1 GB 349 / 403 -> 330 / 381).
  // Loads: kCached between the L2s' 32 MB and the memory-side cache's 256 MB (128 MB 45 / 47; kStream 49), kMixed beyond, save
  // for K = 64 in 128 columns, where the kept part earns nothing (512 MB 179 against 175).
  // Beyond: two workgroups per CU instead of four (by the LDS they ask for), less memory in flight at once: 512 MB 198 -> 184
  // with kStream.  Three for slabs of 16 KB (K = V = 64, 512 MB 169 / 171 -> 161 / 164).
  constexpr int64_t MB = 1 << 20;
  const int64_t bytes = (int64_t)B * Hv * K * V * 4;
  const bool beyond = bytes >= 256 * MB, cached = bytes > 32 * MB && !beyond;
  const int full = V % 128 != 0 || (K == 256 && !cached && !(beyond && V % 256 == 0)) ? 64 : 128;
  const int bv = (int64_t)B * Hv * (V / full) <= device_compute_units() ? 32 : full;
  const int lds = !beyond ? 0 : K * full > 64 * 64 ? 45000 : 30000;
  auto launch = [&](auto kern) {
    GDN_LAUNCH(kKernRecurrent, stream, kern, dim3((unsigned)((int64_t)B * Hv * (V / bv))), dim3(kThreads), lds, stream,
               (const T*)q, (const T*)k, (const T*)v, sq, sk, sv, gates, state_in, state_out, (T*)o, cu, T_len, Hqk, Hv, V,
               scale, use_l2norm, RecurrentConv{});
    return (int)hipGetLastError();
  };
#define GDN_REC(DK_, BV_, LOADS_) return launch(recurrent_kernel<T, TP, DK_, BV_, StateLoads::LOADS_>)
#define GDN_REC_WIDTH(DK_, BV_, BEYOND_)               \
  if (K == DK_ && bv == BV_) {                         \
    if (beyond) GDN_REC(DK_, BV_, BEYOND_);            \
    if (cached) GDN_REC(DK_, BV_, kCached);            \
    GDN_REC(DK_, BV_, kStream);                        \
  }
  if (K == 64 && bv == 32) GDN_REC(64, 32, kStream);
  if (K == 128 && bv == 32) GDN_REC(128, 32, kStream);
  if (K == 256 && bv == 32) GDN_REC(256, 32, kStream);
  GDN_REC_WIDTH(64, 64, kMixed)
  GDN_REC_WIDTH(64, 128, kStream)
  GDN_REC_WIDTH(128, 64, kMixed)
  GDN_REC_WIDTH(128, 128, kMixed)
  GDN_REC_WIDTH(256, 64, kMixed)
  if (K == 256 && cached) GDN_REC(256, 128, kCached);
  if (K == 256) GDN_REC(256, 128, kMixed);
#undef GDN_REC_WIDTH
#undef GDN_REC
  return -3;
}

// A decode step with its convolution update in one launch; -3 for what needs the two launches: other key widths, and heads
// whose slabs do not add up to 1, 2 or 4 groups of threads.
// 16 q/k and 32 value heads of 128, 24 layers in turn, us a step in a graph / of an eager program, two launches -> one.  Small
// batches save the host's share of a launch, not time on the device: 1 sequence 6.3 / 18.3 -> 8.1 / 10.2 (in the profiler 2.7 +
// 5.1 -> 8.8), 4 sequences 8.2 / 17.9 -> 8.9 / 10.2, 16: 15.9 / 18.0 -> 15.1 / 15.3, 32: 33.5 -> 24.9, 64: 60.3 -> 52.8, 128: 105.0
// -> 105.6.  The same states every step, 48 sequences 39.5 -> 36.6, 128: 93.5 -> 89.5, 256: 179.0 -> 167.6; three sets of states
// in turn, 256: 198.4 -> 197.8.
// Slabs of 64 columns up to 32 MB of states, where few workgroups hold many waves each (1 sequence 9.7, with slabs of 128
// columns 11.7), but 128 where 64 would make eight slabs to a workgroup (64 value heads, 1 sequence eager 17.8 -> 12.7, 8
// 18.3 -> 16.9); beyond, 128 columns and two workgroups a CU (17 sequences 21 -> 16, 256: 208 -> 167).  Loads: kStream to
// 128 MB (64 sequences, five sets of states in turn, 53 against 56 with kCached; 32: 25 and 26), then kCached (112 sequences,
// the same states every step, 81 against 86), kMixed from 256 MB on as in the rule alone.
// Four slabs of 128 columns (four value heads to a q/k head) end at 128 MB: their 1024 threads have a CU to themselves, where
// nothing loads while they compute, and past that size two launches are faster.  16 q/k and 64 value heads, us, one launch /
// two: twelve sets of states in turn 64 MB 27 / 34, 128 MB 52 / 61, 160 MB 78 / 75, 256 MB 111 / 105, 512 MB 212 / 200; the same
// states every step 96 MB 41 / 39, 160 MB 64 / 60, 256 MB 100 / 92, 512 MB 188 / 176.
template <typename T, typename TP>
static int launch_decode_step(const RecurrentConv& conv, const RecurrentGates& gates, float* state, void* o, int B, int Hqk,
                              int Hv, int K, int V, float scale, hipStream_t stream) {
  constexpr int64_t MB = 1 << 20;
  const int64_t bytes = (int64_t)B * Hv * K * V * 4;
  const int bv = bytes > 32 * MB || (Hv / Hqk * (V / 64) > 4 && V % 128 == 0) ? 128 : 64;
  if (K != 128 || V % bv != 0 || (int64_t)B * Hqk > 0x7fffffff) return -3;
  const int64_t units = (int64_t)(Hv / Hqk) * (V / bv);
  if (units == 4 && bytes > 128 * MB) return -3;
  auto launch = [&](auto kern) {
    GDN_LAUNCH(kKernRecurrent, stream, kern, dim3((unsigned)(B * Hqk)), dim3((unsigned)(kThreads * units)), 0, stream,
               (const T*)nullptr, (const T*)nullptr, (const T*)nullptr, 0, 0, 0, gates, (const float*)state, state, (T*)o,
               (const int64_t*)nullptr, 1, Hqk, Hv, V, scale, 1, conv);
    return (int)hipGetLastError();
  };
#define GDN_STEP(UN_)                                                                                        \
  if (units == UN_) {                                                                                        \
    if (bv == 64) return launch(recurrent_kernel<T, TP, 128, 64, StateLoads::kStream, UN_>);                 \
    if (bytes <= 128 * MB) return launch(recurrent_kernel<T, TP, 128, 128, StateLoads::kStream, UN_>);       \
    if constexpr (UN_ != 4) {                                                                                \
      if (bytes < 256 * MB) return launch(recurrent_kernel<T, TP, 128, 128, StateLoads::kCached, UN_>);      \
      return launch(recurrent_kernel<T, TP, 128, 128, StateLoads::kMixed, UN_>);                             \
    }                                                                                                        \
  }
  GDN_STEP(1)
  GDN_STEP(2)
  GDN_STEP(4)
#undef GDN_STEP
  return -3;
}

static int recurrent_check(int B, int T, int Hqk, int Hv, int V) {
  if (B <= 0 || T < 0 || Hqk <= 0 || Hv <= 0 || Hv % Hqk != 0) return -2;
  if (V % 64 != 0 || V <= 0) return -3;
  return 0;
}

}  // namespace gdn

extern "C" int gdn_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                 const float* state_in, float* state_out, void* o, int B, int T, int Hqk, int Hv,
                                 int K, int V, float scale, int use_qk_l2norm, int dtype, void* stream) {
  using namespace gdn;
  if (!q || !k || !v || !g || !beta || !o) return -1;
  if (int e = recurrent_check(B, T, Hqk, Hv, V)) return e;
  if (T == 0 && state_out == nullptr) return 0;
  hipStream_t s = (hipStream_t)stream;
  const RecurrentGates gates{g, beta, nullptr, nullptr, nullptr, nullptr};
  const int64_t nq = (int64_t)Hqk * K, nv = (int64_t)Hv * V;
  if (dtype == 0)
    return launch_recurrent<float, float>(q, k, v, nq, nq, nv, gates, state_in, state_out, o, B, T, Hqk, Hv, K, V, scale,
                                          use_qk_l2norm, s);
  if (dtype == 1)
    return launch_recurrent<bf16_t, float>(q, k, v, nq, nq, nv, gates, state_in, state_out, o, B, T, Hqk, Hv, K, V, scale,
                                           use_qk_l2norm, s);
  return -4;
}

extern "C" int gdn_recurrent_fwd_packed(const void* q, const void* k, const void* v, const float* g, const float* beta,
                                        const float* state_in, float* state_out, void* o, const int64_t* cu_seqlens,
                                        int N, int T, int Hqk, int Hv, int K, int V, float scale, int use_qk_l2norm,
                                        int dtype, void* stream) {
  using namespace gdn;
  if (!q || !k || !v || !g || !beta || !o || !cu_seqlens) return -1;
  if (int e = recurrent_check(N, T, Hqk, Hv, V)) return e;
  hipStream_t s = (hipStream_t)stream;
  const RecurrentGates gates{g, beta, nullptr, nullptr, nullptr, nullptr};
  const int64_t nq = (int64_t)Hqk * K, nv = (int64_t)Hv * V;
  if (dtype == 0)
    return launch_recurrent<float, float>(q, k, v, nq, nq, nv, gates, state_in, state_out, o, N, T, Hqk, Hv, K, V, scale,
                                          use_qk_l2norm, s, cu_seqlens);
  if (dtype == 1)
    return launch_recurrent<bf16_t, float>(q, k, v, nq, nq, nv, gates, state_in, state_out, o, N, T, Hqk, Hv, K, V, scale,
                                           use_qk_l2norm, s, cu_seqlens);
  return -4;
}

extern "C" int gdn_recurrent_fwd_qkv(const void* qkv, int64_t token_stride, const void* a, const void* b,
                                     const void* A_log, const void* dt_bias, const float* state_in, float* state_out,
                                     void* o, int B, int T, int Hqk, int Hv, int K, int V, float scale,
                                     int use_qk_l2norm, int dtype, int param_dtype, void* stream) {
  using namespace gdn;
  if (!qkv || !a || !b || !A_log || !dt_bias || !o) return -1;
  if (int e = recurrent_check(B, T, Hqk, Hv, V)) return e;
  if (dtype != 0 && dtype != 1) return -4;
  if (param_dtype != 0 && param_dtype != dtype) return -4;
  const int64_t nq = (int64_t)Hqk * K, nv = (int64_t)Hv * V, vec = dtype == 0 ? 4 : 8, es = dtype == 0 ? 4 : 2;
  if (token_stride < 2 * nq + nv || token_stride % vec != 0 || ((uintptr_t)qkv & 15) != 0) return -6;
  if (T == 0 && state_out == nullptr) return 0;
  hipStream_t s = (hipStream_t)stream;
  const RecurrentGates gates{nullptr, nullptr, a, b, A_log, dt_bias};
  const char* base = static_cast<const char*>(qkv);
  const void *q = base, *k = base + nq * es, *v = base + 2 * nq * es;
  if (dtype == 0)
    return launch_recurrent<float, float>(q, k, v, token_stride, token_stride, token_stride, gates, state_in, state_out,
                                          o, B, T, Hqk, Hv, K, V, scale, use_qk_l2norm, s);
  if (param_dtype == 1)
    return launch_recurrent<bf16_t, bf16_t>(q, k, v, token_stride, token_stride, token_stride, gates, state_in,
                                            state_out, o, B, T, Hqk, Hv, K, V, scale, use_qk_l2norm, s);
  return launch_recurrent<bf16_t, float>(q, k, v, token_stride, token_stride, token_stride, gates, state_in, state_out,
                                         o, B, T, Hqk, Hv, K, V, scale, use_qk_l2norm, s);
}

extern "C" int gdn_decode_step(const void* hidden, void* conv_state, const void* conv_weight, const void* conv_bias,
                               const void* a, const void* b, const void* A_log, const void* dt_bias, float* state, void* o,
                               int B, int Hqk, int Hv, int K, int V, int W, int activation, float scale, int dtype,
                               int param_dtype, void* stream) {
  using namespace gdn;
  if (!hidden || !conv_state || !conv_weight || !a || !b || !A_log || !dt_bias || !state || !o) return -1;
  if (int e = recurrent_check(B, 1, Hqk, Hv, V)) return e;
  if (dtype != 0 && dtype != 1) return -4;
  if (param_dtype != 0 && param_dtype != dtype) return -4;
  const int row = W * (dtype == 0 ? 4 : 2);
  if (W != 4 || (((uintptr_t)conv_state | (uintptr_t)conv_weight) & (row - 1)) != 0 || ((uintptr_t)state & 15) != 0) return -3;
  hipStream_t s = (hipStream_t)stream;
  const RecurrentConv conv{hidden, conv_state, conv_weight, conv_bias, activation};
  const RecurrentGates gates{nullptr, nullptr, a, b, A_log, dt_bias};
  if (dtype == 0) return launch_decode_step<float, float>(conv, gates, state, o, B, Hqk, Hv, K, V, scale, s);
  if (param_dtype == 1) return launch_decode_step<bf16_t, bf16_t>(conv, gates, state, o, B, Hqk, Hv, K, V, scale, s);
  return launch_decode_step<bf16_t, float>(conv, gates, state, o, B, Hqk, Hv, K, V, scale, s);
}
