// chunk_bwd_local16_kernel: what chunk_bwd_local_kernel does, for 16-bit types; with KDA its main loop alone.
//
// With z = beta (v - e^G . K S), V' = (I + L)^-1 z and R = Tm^T dV' = dz (Tm = (I + L)^-1), the gradient of L is
// -strict_tril(R V'^T), that of a triangular solve's matrix; no product with Tm is needed beyond R:
//   dv = beta R          P = -R S^T          dM = -strict_tril(R V'^T) . Gam
//   ds = scale tril(dO V'^T . Gam)           dQ = scale e^G . (dO S^T) + ds K
//   dK1 = e^{G_last-G} . (V' dS'^T) + ds^T Q          dK = dK1 + beta (e^G P + dM K) + dM^T (beta K)
//   dbeta = <R,v> + <e^G P + dM K, k>        dG as in chunk_bwd_local_kernel
// (chunk_bwd_local_kernel forms dM as -(Tm^T strict_tril(dW Kb^T + dV' Vb^T) Tm^T) . Gam with dW = -dV' S^T, the reference's
// way: six more 64-wide products behind four more barriers, each rounding what it hands on.)
//
// A workgroup of eight waves, two to a CU and so four waves to a SIMD, per (chunk, q/k group); the value heads of the group
// follow one after the other and their dq, dk add up, rounded to 16 bits from head to head.  Wave w owns the K
// columns [16 w, 16 w + 16) of dQ, dK, P and one or two of the ten 16x16 tiles on and below the diagonal of the 64x64
// matrices.  All products are v_mfma_f32_16x16x32_bf16; lane n + 16 g holds row (A) or column (B) n of a tile and eight values
// of the contraction index, accumulator register e the row 4 g + e of column n.
//   R and dv of 128 columns of V first, a 16-token tile to a wave at a time, R left in LDS as A operands;
//   main loop over 32-column V blocks: V', S and dS' lie the other way round and are read with the transposing LDS read; the
//     contraction index V runs 8 g .. 8 g + 7;
//   epilogue: contractions over tokens take them in the order 32 b + {4 g + e, 16 + 4 g + e}, which is that of two packed
//     accumulator tiles; the 64x64 matrices pass between the waves as bf16 matrices in LDS (Mat64), written in 8-byte units
//     straight from accumulators and read along their rows or, with the transposing read, along their columns.
// Bound by bytes and vector instructions together: 2 x 8192 tokens, 16 q/k and 32 value heads of 128 move 1.96 GB in 390 to
// 411 us (4.8 to 5.0 TB/s; the main loop alone, which is all that KDA runs, 6.2), where one launch per
// value head of the four-wave kernel, which waited (two waves to a SIMD), moved 2.04 GB in 466; 4 x 1024 tokens 139 -> 106,
// 32768 tokens of 8 heads 234 -> 193; K = 64, 2 x 8192 tokens, 16 heads of 64 142 -> 133, 32 value heads of 256 616 -> 555 (half
// of the waves have no K columns there and repeat the others' main loop).  (With four spilled values, each of which waits for all
// requests in flight when it is read back: 422, 111, 203.)  What is read once passes the L2 by: kept in it, 422, 111, 204, KDA
// 302 -> 352, 65536 tokens of 64 heads of 256 4990 -> 5200.
#pragma once
#include "gdn_chunk.h"
#include "gdn_common.h"
#include "gdn_slab.h"

namespace gdn {

// 16 bytes of zeros: the source of rows past the end of a sequence
static __device__ __attribute__((aligned(16))) const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

namespace bl16 {

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ void mma(f32x4& c, u32x4 a, u32x4 b) { Slab16::mma_half(c, a, b); }
__device__ __forceinline__ u32x4 join(u32x2 a, u32x2 b) { return u32x4{a[0], a[1], b[0], b[1]}; }
__device__ __forceinline__ u32x2 pack1(const f32x4& a) { return u32x2{f32x2_to_bf16x2(a[0], a[1]), f32x2_to_bf16x2(a[2], a[3])}; }
// two accumulator tiles (tokens 0..15 and 16..31 of a block of 32) as an operand whose contraction index is their row
__device__ __forceinline__ u32x4 pack2(const f32x4& a, const f32x4& b) { return join(pack1(a), pack1(b)); }
// element (tile i of the two, register e) of such an operand
__device__ __forceinline__ float at(u32x4 f, int i, int e) {
  const uint32_t w = f[2 * i + (e >> 1)];
  return __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
}

// orders of the contraction index: as the 16-byte pieces of a row hold it, as packed accumulators do, as the pieces of a
// fragment-order tile do
enum Order { kRows, kAccs, kPiece };

// The lane's place n + 16 g, and the addresses that follow from it.  Each phase of the kernel makes its own (here()), out of
// the compiler's sight: formed once for the whole kernel, these addresses would take more registers than a wave has.
struct Lane {
  int id, n, g, w;   // w: the wave
  static __device__ __forceinline__ Lane here() {
    int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GDN_KEEP_HERE(l);
    GDN_KEEP_HERE_UNIFORM(w);
    return Lane{l, l & 15, l >> 4, w};
  }
  // the wave's tiles of the lower triangle: index w, for the last two waves also 8, 9; (ti, tj) in the order of the rows
  __device__ __forceinline__ int tiles() const { return w >= 6 ? 2 : 1; }
  __device__ __forceinline__ int ti(int x) const { return x == 1 || w >= 6 ? 3 : w >= 3 ? 2 : w >= 1 ? 1 : 0; }
  __device__ __forceinline__ int tj(int x) const { return x == 1 ? imin(w - 4, 3) : w - ti(0) * (ti(0) + 1) / 2; }
  __device__ __forceinline__ int first(Order o, int i) const {   // the first of the four values i of the eight that the lane holds
    return o == kRows ? 8 * g + 4 * i : o == kAccs ? 4 * g + 16 * i : 16 * (g >> 1) + 4 * (g & 1) + 8 * i;
  }
  // From a 32x32 tile in fragment order in LDS that holds X as (lane <-> row, registers <-> column): columns 16 t .. 16 t + 15
  // as lanes, rows as contraction index.  `half`: the tile is a copy of the blocks of column half t alone.
  __device__ __forceinline__ const bf16_t* turned_at(const bf16_t* tile, int t, Order o, int i, bool half = false) const {
    const int e = n >> 2, q = n & 3, b = 2 * t + (q & 1);
    return tile + ((half ? (q & 1) : b) * 32 + ((first(o, i) + e + 4 * b) & 31)) * 8 + 4 * (q >> 1);
  }
  __device__ __forceinline__ u32x4 turned(const bf16_t* tile, int t, Order o) const {
    const bf16_t* p[2] = {turned_at(tile, t, o, 0), turned_at(tile, t, o, 1)};
    u32x4 x;
    lds_read_tr16_pairs<1>(p, &x);
    return x;
  }
  // the tile as it lies: rows `row` as lanes, contraction index kPiece
  __device__ __forceinline__ u32x4 lying(const bf16_t* tile, int row) const {
    return *reinterpret_cast<const u32x4*>(tile + (32 * g + ((row + 4 * g) & 31)) * 8);
  }
};

// A bf16 matrix [R][64] in LDS, rows of sixteen 8-byte units.  The unit u of row r lies at u ^ key(r): sixteen rows' units
// of one column (reads along rows, writes of accumulators) and four rows' times four units (transposing reads) then fall
// on all banks.
struct Mat64 {
  bf16_t* p;
  static __device__ __forceinline__ int key(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
  __device__ __forceinline__ bf16_t* unit(int r, int u) const { return p + r * 64 + ((u ^ key(r)) * 4); }
  // accumulator tile (ti, tj) of a matrix X, stored transposed: row j, unit of the rows i
  __device__ __forceinline__ void put(Lane l, int ti, int tj, u32x2 x) const { *reinterpret_cast<u32x2*>(unit(16 * tj + l.n, 4 * ti + l.g)) = x; }
  // rows 16 t .. 16 t + 15 as lanes, columns of block kb as contraction index in the order kAccs
  __device__ __forceinline__ u32x4 along(Lane l, int t, int kb) const {
    const int r = 16 * t + l.n, u = 8 * kb + l.g;
    return join(*reinterpret_cast<const u32x2*>(unit(r, u)), *reinterpret_cast<const u32x2*>(unit(r, u + 4)));
  }
  // columns 16 t .. 16 t + 15 as lanes, rows of block kb as contraction index
  __device__ __forceinline__ u32x4 across(Lane l, int t, int kb, Order o) const {
    const bf16_t* p[2] = {across_at(l, t, kb, o, 0), across_at(l, t, kb, o, 1)};
    u32x4 x;
    lds_read_tr16_pairs<1>(p, &x);
    return x;
  }
  __device__ __forceinline__ const bf16_t* across_at(Lane l, int t, int kb, Order o, int i) const {
    return unit(32 * kb + l.first(o, i) + (l.n >> 2), 4 * t + (l.n & 3));
  }
};

// 64 values in LDS, one per token: a group's lanes share the tokens 16 t + 4 g + e of their accumulators, lane n holds that of
// t = n / 4, e = n % 4 and the others take it by a data-parallel-primitive move
struct Tokens {
  Slab16::Rows v;
  static __device__ __forceinline__ int own(Lane l) { return 16 * (l.n >> 2) + 4 * l.g + (l.n & 3); }
  __device__ __forceinline__ void load(Lane l, const float* arr) { v.f = arr[own(l)]; }
  __device__ __forceinline__ float get(int t, int e) const { return v.get(t >> 1, 4 * (t & 1) + e); }
};

}  // namespace bl16

template <int DK> struct BwdLocal16Smem {
  // in elements: dV' tiles of four V blocks, later K (per wave the halves of its two tiles that are its columns);
  // R of four V blocks as A operands; v_new tiles [2 stages]; dO rows of a pair of V blocks [2 buffers][64][64];
  // per wave its halves of the S and dS' tiles, later of the Q^T tiles; Tm tiles (0,0), (1,0), (1,1)
  static constexpr int dv = 0, r = dv + 8 * 1024, vn = r + 8 * 1024, raw = vn + 2 * 2048, priv = raw + 2 * 4096,
                       tm = priv + 8 * 1024, elems = tm + 3 * 1024;
  static constexpr int off_row = elems * 2;
  static constexpr int bytes = off_row + (5 * 64 + 2 * 64 + 16) * 4;
  static_assert(bytes <= 80 * 1024, "two workgroups to a CU");
};

// KDA: the kernel ends after its main loop and leaves the sums over V for kda_bwd_finish_kernel (KdaDump); G is not read, bt is
// the transformed beta and there is one value head to a group.  2 x 8192 tokens of 32 heads: 299 us, the four-wave kernel 368.
template <int DK, bool KDA = false>
__global__ __launch_bounds__(512) GDN_WAVES_PER_SIMD(4) void chunk_bwd_local16_kernel(
    const bf16_t* __restrict__ qtf, const bf16_t* __restrict__ kaf, const bf16_t* __restrict__ v, const float* __restrict__ bt,
    int beta_same, const float* __restrict__ G, const bf16_t* __restrict__ Ai, const bf16_t* __restrict__ vf,
    const bf16_t* __restrict__ dvf, const bf16_t* __restrict__ dO, const bf16_t* __restrict__ hf, bf16_t* dhf,
    const float* __restrict__ rstd_q, const float* __restrict__ rstd_k, bf16_t* __restrict__ dq, bf16_t* __restrict__ dk,
    bf16_t* __restrict__ dv_out, void* __restrict__ dbeta, float* __restrict__ dg, const int64_t* __restrict__ cu,
    const int* __restrict__ chunk_offsets, int T_len, int N, int Hqk, int Hv, int V, float scale, TokenStrides ts,
    bf16_t* __restrict__ kda_dump, float* __restrict__ kda_dd) {
  using namespace bl16;
  using T = bf16_t;
  using SM = BwdLocal16Smem<DK>;
  constexpr int NKT = DK / 32;
  T* const base = reinterpret_cast<T*>(gdn_smem);
  float* const Gs = reinterpret_cast<float*>(gdn_smem + SM::off_row);
  float* const egs = Gs + 64;    // e^G
  float* const bs = egs + 64;    // beta
  float* const sgs = bs + 64;    // scale e^G
  float* const egl = sgs + 64;   // e^{G_last - G}
  float* const rv = egl + 64;    // <R_i, v_i>, two parts
  float* const wsum = rv + 128;  // per wave: <S,dS'>, sum_i <k_i, dK_inter_i>
  // in the place of R, once that is consumed:
  float* const rsa = reinterpret_cast<float*>(base + SM::r);   // per wave: <q_i, dQ_i>
  float* const rsb = rsa + 512;                                // per wave: e^G <P_i,k_i> + <E_i,k_i>
  float* const rsc = rsb + 512;                                // per wave: <k_i, dK_i>
  float* const rsd = rsc + 512;                                // per wave: beta (e^G <P_i,k_i> + <E_i,k_i>) - <k_i, dK1_i> - <F_i,k_i>
  float* const rsn = rsd + 512;                                // 1/|q|, 1/|k| of the l2 norm [64 each]

  const SeqInfo s = locate_chunk(blockIdx.x, cu, chunk_offsets, N, T_len);
  if (s.nvalid <= 0) return;
  Lane L = Lane::here();
  const int hq = blockIdx.y, grp = Hv / Hqk, nvalid = s.nvalid;
  const int64_t tok0 = s.bos + (int64_t)s.chunk * kChunk;
  const bool l2 = rstd_q != nullptr;
  const int nblk = V / 32;
  const int64_t chq = (int64_t)blockIdx.x * Hqk + hq;

  // the wave's block of 16 K columns; with K = 64 waves 4 .. 7 repeat what waves 0 .. 3 do, and keep the result to themselves
  auto kw = [](Lane l) { return l.w & (DK / 16 - 1); };

  // copies global -> LDS, 64 x 16 bytes each
  auto issue_dv = [&](int64_t ch, int b0) {   // dV' tiles of V blocks b0 .. b0 + 3 and what a phase of R needs beside them
    if (L.w < 4 || b0 + 2 < nblk) {           // a tile to a wave
      const T* src = dvf + (ch * nblk + b0) * 2048 + L.w * 1024 + L.id * 8;
      load16_to_lds_stream(src, base + SM::dv + L.w * 1024);
      load16_to_lds_stream(src + 512, base + SM::dv + L.w * 1024 + 512);
    }
  };
  auto issue_tm = [&](int64_t ch) {           // tile (0,1) is zero, unused and not stored
    if (L.w < 6) load16_to_lds_stream(Ai + ch * 4096 + (L.w < 2 ? L.w : L.w + 2) * 512 + L.id * 8, base + SM::tm + L.w * 512);
  };
  auto issue_vn = [&](int64_t ch, int vblk) {
    if (L.w < 4) load16_to_lds_stream(vf + (ch * nblk + vblk) * 2048 + L.w * 512 + L.id * 8, base + SM::vn + (vblk & 1) * 2048 + L.w * 512);
  };
  auto issue_priv = [&](int64_t ch, int vblk) {
    const int64_t at = ((ch * nblk + vblk) * NKT + (kw(L) >> 1)) * 1024 + (L.w & 1) * 512 + L.id * 8;
    load16_to_lds_stream(hf + at, base + SM::priv + L.w * 1024);
    load16_to_lds_stream((const T*)dhf + at, base + SM::priv + L.w * 1024 + 512);
  };
  auto issue_raw = [&](int h, int pair) {   // the piece c of row r lies at c ^ (r % 8): eight rows' pieces of one column on all banks
    const int row = 8 * L.w + (L.id >> 3), cc = (L.id & 7) ^ (row & 7);
    const T* from = dO + ((tok0 + imin(row, nvalid - 1)) * Hv + h) * V + 64 * pair + cc * 8;
    load16_to_lds_stream(row < nvalid ? from : reinterpret_cast<const T*>(kZero16), base + SM::raw + (pair & 1) * 4096 + L.w * 512);
  };
  auto issue_k = [&]() {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
      load16_to_lds(kaf + chq * (64 * DK) + ((kw(L) >> 1) * 2 + tb) * 1024 + (L.w & 1) * 512 + L.id * 8,
                    base + SM::dv + L.w * 1024 + tb * 512);
  };
  auto issue_q = [&]() {                    // the 16 rows of the Q^T tiles that are the wave's columns
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
      load16_to_lds(qtf + chq * (64 * DK) + ((kw(L) >> 1) * 2 + tb) * 1024 + (32 * L.g + ((16 * (L.w & 1) + L.n + 4 * L.g) & 31)) * 8,
                    base + SM::priv + L.w * 1024 + tb * 512);
  };
  auto raw_rows = [&](Lane l, int t, int vblk) {   // dO rows 16 t + n, contraction index kRows
    return *reinterpret_cast<const u32x4*>(base + SM::raw + ((vblk >> 1) & 1) * 4096 + (16 * t + l.n) * 64 +
                                           (((4 * (vblk & 1) + l.g) ^ (l.n & 7)) * 8));
  };
  auto r_rows = [&](Lane l, int t, int vblk) { return *reinterpret_cast<const u32x4*>(base + SM::r + (((vblk & 3) * 4 + t) * 64 + l.id) * 8); };
  auto issue_head = [&](int h) {            // the first operands of a head, K and Q's place apart
    const int64_t ch = (int64_t)blockIdx.x * Hv + h;
    issue_tm(ch);
    issue_raw(h, 0);
    issue_vn(ch, 0);
  };

  // The sums over the group's heads travel from one head to the next in the place of its first head's state gradients, which
  // have been read by then (the reverse recurrence rewrites them in every backward pass): two pieces per lane for dq and
  // for dk, read back by the lane that wrote them.  In registers they would be spilled: the kernel is bound by the bytes it
  // moves, and what it spills counts twice.
  auto sums = [&]() { return dhf + ((int64_t)blockIdx.x * Hv + hq * grp) * nblk * NKT * 1024 + (kw(L) * 64 + L.id) * 32; };
  issue_head(hq * grp);
  issue_dv(chq * grp, 0);
  issue_priv(chq * grp, 0);
#pragma clang loop unroll(disable)
  for (int hh = 0; hh < grp; ++hh) {
    const int h = hq * grp + hh;
    const int64_t ch = (int64_t)blockIdx.x * Hv + h;
    const bool last = hh == grp - 1;
    L = Lane::here();
    if (L.w == 0) {
      const int tc = imin(L.id, nvalid - 1);
      const float bv = bt[ch * 64 + L.id];   // beta: 0 past the end
      if constexpr (!KDA) {
        const float gv = G[ch * 64 + tc], gl = G[ch * 64 + nvalid - 1];
        Gs[L.id] = gv;
        egs[L.id] = __expf(gv);
        sgs[L.id] = scale * __expf(gv);
        egl[L.id] = __expf(gl - gv);
      }
      bs[L.id] = bv;
    }

    f32x4 dQ[4], dK[4], P[4], ds[2], rvn[2];   // P without its sign; rvn = R V'^T
#pragma unroll
    for (int t = 0; t < 4; ++t) { dQ[t] = zero4(); dK[t] = zero4(); P[t] = zero4(); }
#pragma unroll
    for (int x = 0; x < 2; ++x) { ds[x] = zero4(); rvn[x] = zero4(); }
    float sds = 0.f;

    const Lane M = Lane::here();   // of the products that every wave forms: their addresses stay in registers
#pragma clang loop unroll(disable)
    for (int vblk = 0; vblk < nblk; ++vblk) {
      L = Lane::here();
      GDN_WAIT_VMEM();       // this wave's share of the block's operands has landed ...
      GDN_LDS_BARRIER();     // ... and so has everybody else's; the other stage and buffer are no longer read
      if ((vblk & 3) == 0) {
        // R^T = dV'^T Tm of four V blocks (lane <-> token), tile t = w % 4 of 16 tokens, blocks w / 4 and w / 4 + 2.  The rows of
        // the two accumulators are V columns 8 g + e and 8 g + 4 + e: packed they are an A operand of order kRows, and a lane
        // stores eight adjacent columns of dv.
        const int t = L.w & 3, jb = t >> 1, row = 16 * t + L.n, nb = imin(4, nblk - vblk);
        const T* from = v + (tok0 + imin(row, nvalid - 1)) * ts.v + (int64_t)h * V + 32 * vblk + 8 * L.g;
        u32x4 vv[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const u32x4* at_v = reinterpret_cast<const u32x4*>(from + 32 * imin((L.w >> 2) + 2 * x, nb - 1));
          // two waves share a line of v.  Kept in the L2 for the second of them: V = 256 5145 -> 5043 us, V = 128 no change, but
          // KDA, which has nothing else to read twice, 300 -> 313.
          if constexpr (KDA) vv[x] = __builtin_nontemporal_load(at_v);
          else vv[x] = *at_v;
        }
        const float bj = bs[row];
        float sv = 0.f;
        u32x4 tm1 = L.turned(base + SM::tm + (1 + jb) * 1024, t & 1, kPiece), tm0 = u32x4{0u, 0u, 0u, 0u};
        if (jb == 0) tm0 = L.turned(base + SM::tm, t & 1, kPiece);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int b = (L.w >> 2) + 2 * x;
          if (b >= nb) break;
          const int64_t col = (int64_t)h * V + 32 * (vblk + b) + 8 * L.g, tok = tok0 + imin(row, nvalid - 1);
          f32x4 r[2] = {zero4(), zero4()};
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int at_row = 8 * (L.n >> 2) + 4 * j + (L.n & 3);
            if (jb == 0) mma(r[j], L.lying(base + SM::dv + 2 * b * 1024, at_row), tm0);
            mma(r[j], L.lying(base + SM::dv + (2 * b + 1) * 1024, at_row), tm1);
          }
          *reinterpret_cast<u32x4*>(base + SM::r + ((b * 4 + t) * 64 + L.id) * 8) = pack2(r[0], r[1]);
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              sv += r[j][e] * at(vv[x], j, e);
              r[j][e] *= bj;
            }
          if (row < nvalid) *reinterpret_cast<u32x4*>(dv_out + tok * ts.dv + col) = pack2(r[0], r[1]);
        }
        sv += __shfl_xor(sv, 16);
        sv += __shfl_xor(sv, 32);
        if (L.g == 0) rv[64 * (L.w >> 2) + row] = vblk == 0 ? sv : rv[64 * (L.w >> 2) + row] + sv;
        GDN_LDS_BARRIER();
      }
      u32x4 St, dSt;
      {
        const T* half = base + SM::priv + M.w * 1024;
        const T* p[4] = {M.turned_at(half, M.w & 1, kRows, 0, true), M.turned_at(half, M.w & 1, kRows, 1, true),
                         M.turned_at(half + 512, M.w & 1, kRows, 0, true), M.turned_at(half + 512, M.w & 1, kRows, 1, true)};
        u32x4 x[2];
        lds_read_tr16_pairs<2>(p, x);
        St = x[0];
        dSt = x[1];
      }
      GDN_KEEP_HERE(St);
      GDN_KEEP_HERE(dSt);
      GDN_WAVE_LDS_SYNC();     // the wave's halves are in registers: the next tenant may be requested
      if (vblk + 1 < nblk) {
        issue_vn(ch, vblk + 1);
        issue_priv(ch, vblk + 1);
        if ((vblk & 1) == 0 && vblk + 2 < nblk) issue_raw(h, (vblk >> 1) + 1);   // its buffer was last read in block vblk - 1
        if ((vblk & 3) == 3) issue_dv(ch, vblk + 1);                             // read at the head of these four blocks
      } else if constexpr (!KDA) {
        issue_k();
        issue_q();
      }
      const T* st = base + SM::vn + (vblk & 1) * 2048;
      {
#pragma unroll
        for (int i = 0; i < 8; ++i) sds += at(St, i >> 2, i & 3) * at(dSt, i >> 2, i & 3);
        // two token tiles at a time: their operands together, then the products
#pragma unroll
        for (int t = 0; t < 4; t += 2) {
          const u32x4 o0 = raw_rows(M, t, vblk), o1 = raw_rows(M, t + 1, vblk), r0 = r_rows(M, t, vblk), r1 = r_rows(M, t + 1, vblk);
          GDN_SCHED_FENCE();
          const T* tile = st + (t >> 1) * 1024;
          const T* p[4] = {M.turned_at(tile, 0, kRows, 0), M.turned_at(tile, 0, kRows, 1), M.turned_at(tile, 1, kRows, 0),
                           M.turned_at(tile, 1, kRows, 1)};
          u32x4 x[2];
          lds_read_tr16_pairs<2>(p, x);
          GDN_SCHED_FENCE();
          mma(dQ[t], o0, St);
          mma(dQ[t + 1], o1, St);
          mma(P[t], r0, St);
          mma(P[t + 1], r1, St);
          mma(dK[t], x[0], dSt);
          mma(dK[t + 1], x[1], dSt);
        }
      }
      GDN_SCHED_FENCE();
      L = Lane::here();
      auto own = [&](int x, int ti, int tj) {
        const u32x4 o = raw_rows(L, ti, vblk), r = r_rows(L, ti, vblk), b = L.turned(st + (tj >> 1) * 1024, tj & 1, kRows);
        GDN_SCHED_FENCE();
        mma(ds[x], o, b);
        mma(rvn[x], r, b);
      };
      own(0, L.ti(0), L.tj(0));
      if (L.tiles() == 2) own(1, L.ti(1), L.tj(1));
    }
    L = Lane::here();
    if constexpr (KDA) {
      using KD = KdaDump<DK>;
      T* const dump = kda_dump + ch * KD::elems;
      if (L.w < DK / 16) {
        // two accumulator tiles of 16 tokens are the piece of a 32x32 tile in fragment order that the lane and the one 32
        // lanes on hold half of each: they trade, and each lane writes 16 bytes
        auto sums_out = [&](const f32x4* acc, T* out) {
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const u32x2 lo = pack1(acc[2 * b]), hi = pack1(acc[2 * b + 1]);
            const auto x = __builtin_amdgcn_permlane32_swap(lo[0], hi[0], false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(lo[1], hi[1], false, false);
            __builtin_nontemporal_store(u32x4{x[0], y[0], x[1], y[1]},
                                        reinterpret_cast<u32x4*>(out + (b * NKT + (L.w >> 1)) * 1024 +
                                                                 frag_slot<T>(L.g >> 1, 16 * (L.w & 1) + L.n + 32 * (L.g & 1)) * 8));
          }
        };
        sums_out(dQ, dump + KD::dq);
        sums_out(dK, dump + KD::dk2);
        sums_out(P, dump + KD::dk1);
        sds += __shfl_xor(sds, 16);
        sds += __shfl_xor(sds, 32);
        if (L.g == 0) kda_dd[ch * DK + 16 * L.w + L.n] = sds;
      }
      auto tile_out = [&](int x, int ti, int tj) {   // a quarter of a 32x32 tile; nobody reads what lies above the diagonal
        const int at = (2 * (ti >> 1) + (tj >> 1)) * 1024 + frag_slot<T>(ti & 1, 16 * (tj & 1) + L.n + 32 * (L.g & 1)) * 8 + 4 * (L.g >> 1);
        *reinterpret_cast<u32x2*>(dump + KD::ds + at) = pack1(ds[x]);
        *reinterpret_cast<u32x2*>(dump + KD::rv + at) = pack1(rvn[x]);
      };
      tile_out(0, L.ti(0), L.tj(0));
      if (L.tiles() == 2) tile_out(1, L.ti(1), L.tj(1));
      if (L.w == 0) reinterpret_cast<float*>(dump + KD::dots)[L.id] = rv[L.id] + rv[64 + L.id];
      return;
    }
    sds = wave_sum(sds);
    if (L.id == 0) wsum[L.w] = sds;
    float norm = 0.f;   // 1/|q|, 1/|k| of the chunk's tokens, two waves' share: they wait in LDS for the last step
    const bool has_norm = l2 && (L.w == 2 || L.w == 3);
    if (has_norm) norm = (L.w == 2 ? rstd_q : rstd_k)[chq * 64 + imin(L.id, nvalid - 1)];   // (written for the tokens there are)
    const Mat64 MS{base + SM::raw}, MD{base + SM::raw + 4096}, MB{base + SM::vn};   // ds^T, dM^T, (beta dM)^T
    GDN_WAIT_VMEM();
    GDN_LDS_BARRIER();   // K and Q have landed; the last block's operands are consumed
    if (has_norm) rsn[64 * (L.w - 2) + L.id] = norm;

    auto tiles_out = [&](int x, int ti, int tj) {
      const float gj = Gs[16 * tj + L.n];
      const f32x4 gi = *reinterpret_cast<const f32x4*>(Gs + 16 * ti + 4 * L.g), bi = *reinterpret_cast<const f32x4*>(bs + 16 * ti + 4 * L.g);
      f32x4 y, m, mb;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float eg = __expf(fminf(gi[e] - gj, 0.f));
        const int i = 16 * ti + 4 * L.g + e, j = 16 * tj + L.n;
        y[e] = i >= j ? scale * ds[x][e] * eg : 0.f;
        m[e] = i > j ? -rvn[x][e] * eg : 0.f;
        mb[e] = m[e] * bi[e];
      }
      MS.put(L, ti, tj, pack1(y));
      MD.put(L, ti, tj, pack1(m));
      MB.put(L, ti, tj, pack1(mb));
    };
    tiles_out(0, L.ti(0), L.tj(0));
    if (L.tiles() == 2) tiles_out(1, L.ti(1), L.tj(1));
    if (L.w < 2) {   // the tiles above the diagonal that a 32-token block of the contraction index covers
      MS.put(L, 2 * L.w, 2 * L.w + 1, u32x2{0u, 0u});
      MD.put(L, 2 * L.w, 2 * L.w + 1, u32x2{0u, 0u});
      MB.put(L, 2 * L.w, 2 * L.w + 1, u32x2{0u, 0u});
    }
    GDN_LDS_BARRIER();

    L = Lane::here();
    // this wave's K and Q columns as B operands over tokens, and row-dot partners of the accumulators; read again for
    // the last step rather than held
    u32x4 KT[2], QT[2];
    auto load_kq = [&]() {
      const T* half = base + SM::dv + L.w * 1024;
      const T* p[4] = {L.turned_at(half, L.w & 1, kAccs, 0, true), L.turned_at(half, L.w & 1, kAccs, 1, true),
                       L.turned_at(half + 512, L.w & 1, kAccs, 0, true), L.turned_at(half + 512, L.w & 1, kAccs, 1, true)};
      lds_read_tr16_pairs<2>(p, KT);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        u32x2 x[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          x[i] = *reinterpret_cast<const u32x2*>(base + SM::priv + L.w * 1024 + b * 512 + ((2 * i + (L.g & 1)) * 16 + L.n) * 8 + 4 * (L.g >> 1));
        QT[b] = join(x[0], x[1]);
      }
    };
    auto rows_sum = [&](const f32x16& p, float* slots) {   // register 4 t + e <-> token 16 t + 4 g + e
      slots[64 * L.w + 16 * (L.n >> 2) + 4 * L.g + (L.n & 3)] = rows16_partial(p);
    };
    {
      f32x16 p;
      float ski = 0.f;
      Tokens f, be;
      load_kq();
      // The inter-chunk parts, which may be far smaller than a chunk's own, are added to the products' sums and are not what the
      // products are added to: a matrix instruction rounds a tie by an addend below the normal range as well, and such an
      // addend does not double where the gradients do.
      f.load(L, sgs);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x4 y = zero4();
#pragma unroll
        for (int b = 0; b <= (t >> 1); ++b) mma(y, MS.across(L, t, b, kAccs), KT[b]);
#pragma unroll
        for (int e = 0; e < 4; ++e) dQ[t][e] = dQ[t][e] * f.get(t, e) + y[e];
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[4 * t + e] = dQ[t][e] * at(QT[t >> 1], t & 1, e);
      rows_sum(p, rsa);
      GDN_SCHED_FENCE();
      f.load(L, egl);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x4 y = zero4();
#pragma unroll
        for (int b = t >> 1; b < 2; ++b) mma(y, MS.along(L, t, b), QT[b]);
#pragma unroll
        for (int b = t >> 1; b < 2; ++b) mma(y, MB.along(L, t, b), KT[b]);   // dM^T (beta K)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = dK[t][e] * f.get(t, e);
          ski += x * at(KT[t >> 1], t & 1, e);           // only the inter-chunk part
          dK[t][e] = x + y[e];
        }
      }
      ski = wave_sum(ski);
      if (L.id == 0) wsum[8 + L.w] = ski;
      GDN_SCHED_FENCE();
      L = Lane::here();
      f.load(L, egs);
      be.load(L, bs);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        // dK += beta e^G P + (beta dM) K, and for dbeta e^G P + dM K.  dG takes <(beta dM) K, k> - <(beta dM)^T K, k> from the
        // one rounded matrix: a pair of tokens then drops out of every sum over a range that holds both, to the last bit.
        f32x4 E = zero4(), Eb = zero4();
#pragma unroll
        for (int b = 0; b <= (t >> 1); ++b) {
          mma(E, MD.across(L, t, b, kAccs), KT[b]);
          mma(Eb, MB.across(L, t, b, kAccs), KT[b]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float k = at(KT[t >> 1], t & 1, e), y = -P[t][e] * f.get(t, e), z = Eb[e] + y * be.get(t, e);
          p[4 * t + e] = (z - dK[t][e]) * k;
          dK[t][e] += z;
          P[t][e] = (y + E[e]) * k;
        }
      }
      rows_sum(p, rsd);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[4 * t + e] = P[t][e];
      rows_sum(p, rsb);
      GDN_SCHED_FENCE();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[4 * t + e] = dK[t][e] * at(KT[t >> 1], t & 1, e);
      rows_sum(p, rsc);
    }
    GDN_LDS_BARRIER();   // the row sums are complete; the matrices are consumed
    L = Lane::here();
    if (!last) issue_head(h + 1);
    auto slots = [&](const float* a, int i) {
      float x = a[i];
#pragma unroll
      for (int k = 1; k < DK / 16; ++k) x += a[64 * k + i];
      return x;
    };
    u32x4 before[4];
    {
      const T* from = hh != 0 ? (const T*)sums() : reinterpret_cast<const T*>(kZero16);   // the choice on the address: no branch to join
#pragma unroll
      for (int b = 0; b < 4; ++b) before[b] = *reinterpret_cast<const u32x4*>(from + (hh != 0 ? 8 * b : 0));
      if (l2) load_kq();
    }
    if (l2) {
      GDN_KEEP_HERE(QT[0]);
      GDN_KEEP_HERE(QT[1]);
    }
    GDN_WAVE_LDS_SYNC();   // K and Q are in registers
    if (!last) {
      issue_dv(ch + 1, 0);
      issue_priv(ch + 1, 0);
    }
    // l2 norm, the sum over the group's heads, and after its last head the rows by way of a [DK][64] matrix in LDS
    const Mat64 MQ{base + SM::raw}, MK{base + SM::dv};
    static_assert(SM::priv - SM::raw == 64 * 128 && SM::r - SM::dv == 64 * 128, "they fit");
    // (the row sums and norms are read where they are used: held over the requests above they are spilled, and the wait
    // for a spilled value is a wait for every request)
    auto finish = [&](f32x4* d, const u32x4* y, const float* row_sums, const float* norms, const u32x4* so_far, T* sum, const Mat64& to) {
      if (l2) {
        const Lane H = Lane::here();
        Tokens dot, r;
        dot.v.f = slots(row_sums, Tokens::own(H));
        r.load(H, norms);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) d[t][e] = (d[t][e] - dot.get(t, e) * at(y[t >> 1], t & 1, e)) * r.get(t, e);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) d[2 * b + i][e] += at(so_far[b], i, e);
        const u32x4 f = pack2(d[2 * b], d[2 * b + 1]);
        if (DK < 128 && L.w >= DK / 16) continue;
        if (last) {
          to.put(L, 2 * b, kw(L), u32x2{f[0], f[1]});
          to.put(L, 2 * b + 1, kw(L), u32x2{f[2], f[3]});
        } else {
          *reinterpret_cast<u32x4*>(sum + 8 * b) = f;
        }
      }
    };
    {
      finish(dQ, QT, rsa, rsn, before, sums(), MQ);
      finish(dK, KT, rsc, rsn + 64, before + 2, sums() + 16, MK);
    }
    if (L.w == 0) {   // d(cumulative G) -> d(g): suffix sum inside the chunk
      // dG_i = <q,dQ> + beta (e^G <P,k> + <E,k>) - <k,dK1> - <F,k>, E = dM K, F = dM^T (beta K)
      const float sbk = slots(rsb, L.id);
      float x = slots(rsa, L.id) + slots(rsd, L.id);
      if (L.id == nvalid - 1) {
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int i = 0; i < DK / 16; ++i) { a += wsum[i]; b += wsum[8 + i]; }
        x += __expf(Gs[63]) * a + b;
      }
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float t = __shfl_down(x, d);
        if (L.id + d < 64) x += t;
      }
      if (L.id < nvalid) {
        dg[(tok0 + L.id) * Hv + h] = x;
        gate_st<T>(dbeta, beta_same, (tok0 + L.id) * Hv + h, sbk + rv[L.id] + rv[64 + L.id]);
      }
    }
    if (last) {
      GDN_LDS_BARRIER();
      // 16 tokens and 64 columns to a wave, 16-byte pieces, 64 adjacent bytes of a token a time
      auto rows_out = [&](const Mat64& m, T* out, int64_t stride) {
        if (64 * (L.w >> 2) < DK) {
          const int row = 16 * (L.w & 3) + L.n;
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const int k0 = 64 * (L.w >> 2) + 32 * x;
            const u32x4 f = m.across(L, L.w & 3, k0 / 32, kRows);
            if (row < nvalid) *reinterpret_cast<u32x4*>(out + (tok0 + row) * stride + hq * DK + k0 + 8 * L.g) = f;
          }
        }
      };
      rows_out(MQ, dq, ts.dq);
      rows_out(MK, dk, ts.dk);
    }
  }
}

}  // namespace gdn
