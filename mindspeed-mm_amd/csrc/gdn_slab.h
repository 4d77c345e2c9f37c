// What one compute wave of the two recurrence kernels owns: a strip of columns of a 32-column slab of the state, and the
// operand fragments its products take.
//
// Slab16 (16-bit types, one slab to a workgroup): 16 columns, v_mfma_f32_16x16x32_bf16, two waves to a slab.  A recurrence is
// a chain of dependent steps and a step lasts as long as its wave has to issue: with 32 columns to a wave a forward step
// was 38 tile products of 32 cycles and twice the vector work on S.  The price is twice the operand reads from LDS.
// Every tile keeps its fragment order in LDS and in memory: a 16x16x32 product adds up over 32 k, lane group g = lane / 16
// holding eight of them, and a stored 16-byte piece (k-group g / 2, half-wave g % 2) is exactly such a set when the rows of the
// accumulator pair that covers a 32-row tile are dealt out as
//     accumulator j (0, 1), row i of 16   <->   tile row 16 (i / 8) + 8 j + i % 8
// so that a lane's eight values (j, e) are the tile rows 16 (g / 2) + 8 j + 4 (g % 2) + e: packed, they are the 16-byte piece
// (g / 2, g % 2) of their column.  Results are those of Slab32, bit for bit.  Forward alone, 4096 tokens, 32 heads of 128:
// 103 -> 84 us; 2 x 8192 tokens 245 -> 210, with the states kept 263 -> 260 (memory), reverse 241 -> 228; segments of 64
// chunks, 8 heads 109 -> 89.
// Slab32: 32 columns, v_mfma_f32_32x32x16_bf16 or 32x32x2_f32, one wave to a slab.  Two slabs to a workgroup: there the LDS
// would be the bound with 16 columns to a wave (four prompts of 66 to 14012 tokens, forward: 372 us, with Slab16 423).
#pragma once
#include "gdn_common.h"

namespace gdn {

// piece i of loader thread lt, of PIECES pieces of 16 bytes dealt to NT threads, the same number to each: indices past the
// end repeat the last piece (the same loads on every path; the duplicate lands on the same LDS address with the same data).
// fp32 keeps the clamp where it does nothing: there a stage's requests and the LDS writes of what they bring stand in one block,
// and without the clamps the compiler mixes them, fewer requests are in flight and a step takes longer (KDA in fp32, 2048
// tokens of 8 heads of 128, reverse recurrence 541 us with, 551 without; forward 407 and 411).
template <int PIECES, int NT> struct Deal { static constexpr int kPer = (PIECES + NT - 1) / NT; };
template <typename T, int PIECES, int NT> __device__ __forceinline__ int dealt(int lt, int i) {
  return sizeof(T) == 2 && PIECES % NT == 0 ? lt + i * NT : imin(lt + i * NT, PIECES - 1);
}

struct Slab16 {
  static constexpr int kCols = 16, kWaves = 2, kVals = 8;
  static constexpr bool kImageT = true;                   // transposing reads want an image of their own (st_t)
  static constexpr int kMma2 = 4;                         // matrix instructions of mma2()
  struct Acc {
    f32x4 t[2];
    __device__ __forceinline__ float get(int r) const { return t[r >> 2][r & 3]; }
    __device__ __forceinline__ void set(int r, float x) { t[r >> 2][r & 3] = x; }
  };
  static __device__ __forceinline__ int group() { return (threadIdx.x & 63) >> 4; }
  static __device__ __forceinline__ int row(int r) { return 16 * (group() >> 1) + 8 * (r >> 2) + 4 * (group() & 1) + (r & 3); }
  static __device__ __forceinline__ int col() { return threadIdx.x & 15; }
  static __device__ __forceinline__ Acc zero() { return Acc{{f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}}; }
  // 64 fp32 values in LDS, one per row of two 32-row tiles.  A group's lanes hold the same eight rows of a tile, two tiles
  // make sixteen: lane n holds the value of row n % 8 of tile n / 8 and the others take it by a data-parallel-primitive
  // move, which the multiplication that follows absorbs.  (One four-byte LDS read per lane instead of four 16-byte ones:
  // a read costs the LDS its 64 lanes' bytes, broadcast or not.)
  struct Rows {
    float f;
    __device__ __forceinline__ void load(const float* arr) {
      const int n = threadIdx.x & 15, g = group();
      f = arr[32 * (n >> 3) + 16 * (g >> 1) + 8 * ((n >> 2) & 1) + 4 * (g & 1) + (n & 3)];
    }
    __device__ __forceinline__ void fetch(int) {}
    __device__ __forceinline__ float get(int tile, int r) const {   // both compile-time constants
      switch (8 * tile + r) {
        case 0: return dpp_mov<0x150>(f);
        case 1: return dpp_mov<0x151>(f);
        case 2: return dpp_mov<0x152>(f);
        case 3: return dpp_mov<0x153>(f);
        case 4: return dpp_mov<0x154>(f);
        case 5: return dpp_mov<0x155>(f);
        case 6: return dpp_mov<0x156>(f);
        case 7: return dpp_mov<0x157>(f);
        case 8: return dpp_mov<0x158>(f);
        case 9: return dpp_mov<0x159>(f);
        case 10: return dpp_mov<0x15A>(f);
        case 11: return dpp_mov<0x15B>(f);
        case 12: return dpp_mov<0x15C>(f);
        case 13: return dpp_mov<0x15D>(f);
        case 14: return dpp_mov<0x15E>(f);
        default: return dpp_mov<0x15F>(f);
      }
    }
  };
  // An image of tiles in LDS that is read transposed only (A::load_t): each tile's pieces cut in halves,
  // [half j][rows / 4][4 slots of 32 bytes][4 rows][8 bytes], the half j of block q = 2 (k-group) + half-wave and row r in slot
  // (q + r / 4) % 4.  A transposing read names one half of the pieces of four rows in four blocks: 128 consecutive bytes here,
  // every bank once.  In fragment order the halves of one kind fill every other 8 bytes and such a read takes twice
  // its cycles (the reverse recurrence counted 512 cycles of bank conflicts a step, 208 with this).
  static __device__ __forceinline__ void st_t(bf16_t* image, int piece, const Vec16<bf16_t>& v) {
    const int p = piece & 127, q = p >> 5, r = (p - 4 * q) & 31;
    bf16_t* to = image + (piece >> 7) * 1024 + (r >> 2) * 64 + ((q + (r >> 2)) & 3) * 16 + (r & 3) * 4;
    *reinterpret_cast<u32x2*>(to) = u32x2{v.raw[0], v.raw[1]};
    *reinterpret_cast<u32x2*>(to + 512) = u32x2{v.raw[2], v.raw[3]};
  }
  // A operand, 32 rows x 32 k of a tile in LDS
  struct A {
    u32x4 f[2];
    // tile rows <-> accumulator rows, k along the pieces
    __device__ __forceinline__ void load(const bf16_t* tile) {
      const int m = threadIdx.x & 15, g = group(), r0 = 16 * (m >> 3) + (m & 7) + 4 * g;
#pragma unroll
      for (int j = 0; j < 2; ++j) f[j] = *reinterpret_cast<const u32x4*>(tile + (32 * g + ((r0 + 8 * j) & 31)) * 8);
    }
    // the transposed tile, from an image written by st_t: tile columns (along the pieces) <-> accumulator rows, k = tile
    // rows.  Lane (e, q) of a group names half j of tile row 16 (g / 2) + 8 i + 4 (g % 2) + e in block q.
    __device__ __forceinline__ void load_t(const bf16_t* tile) {
      const int e = (threadIdx.x & 15) >> 2, q = threadIdx.x & 3, g = group();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r4 = 4 * (g >> 1) + 2 * i + (g & 1);
        const bf16_t* p = tile + r4 * 64 + ((q + r4) & 3) * 16 + e * 4;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x2 x = lds_read_tr16(p + 512 * j);
          f[j][2 * i] = x[0];
          f[j][2 * i + 1] = x[1];
        }
      }
    }
  };
  // B operand, 32 k x 16 columns: the pieces of the wave's half of a fragment-order tile
  struct B {
    u32x4 f;
    __device__ __forceinline__ void pack(const Acc& c) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f[2 * j] = f32x2_to_bf16x2(c.t[j][0], c.t[j][1]);
        f[2 * j + 1] = f32x2_to_bf16x2(c.t[j][2], c.t[j][3]);
      }
    }
    __device__ __forceinline__ Acc unpack() const {
      Acc c;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        c.t[w >> 1][2 * (w & 1)] = __uint_as_float(f[w] << 16);
        c.t[w >> 1][2 * (w & 1) + 1] = __uint_as_float(f[w] & 0xffff0000u);
      }
      return c;
    }
    static __device__ __forceinline__ int place(int strip) { return (32 * group() + ((16 * strip + col() + 4 * group()) & 31)) * 8; }
    __device__ __forceinline__ void store(bf16_t* tile, int strip) const { *reinterpret_cast<u32x4*>(tile + place(strip)) = f; }
    __device__ __forceinline__ void store_stream(bf16_t* tile, int strip) const {
      __builtin_nontemporal_store(f, reinterpret_cast<u32x4*>(tile + place(strip)));
    }
    // from a row-major tile in LDS (x: first row, the wave's first column; rows ld elements apart): k <-> row
    __device__ __forceinline__ void load_cols(const bf16_t* x, int ld) {
      const int e = (threadIdx.x & 15) >> 2, q = threadIdx.x & 3, g = group();
      const bf16_t* p = x + (16 * (g >> 1) + 4 * (g & 1) + e) * ld + 4 * q;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u32x2 y = lds_read_tr16(p + 8 * i * ld);
        f[2 * i] = y[0];
        f[2 * i + 1] = y[1];
      }
    }
  };
  static __device__ __forceinline__ void mma_half(f32x4& c, u32x4 a, u32x4 b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ void mma(Acc& c, const A& a, const B& b) {
    mma_half(c.t[0], a.f[0], b.f);
    mma_half(c.t[1], a.f[1], b.f);
  }
  // two tile products into two accumulators, in turns
  static __device__ __forceinline__ void mma2(Acc& x0, const A& a0, const B& b0, Acc& x1, const A& a1, const B& b1) {
    mma_half(x0.t[0], a0.f[0], b0.f);
    mma_half(x1.t[0], a1.f[0], b1.f);
    mma_half(x0.t[1], a0.f[1], b0.f);
    mma_half(x1.t[1], a1.f[1], b1.f);
  }
};

template <typename T> struct Slab32 {
  static constexpr int kCols = 32, kWaves = 1, kVals = 16;
  static constexpr bool kImageT = false;
  static constexpr int kMma2 = 2 * AccK<T>::kGroups;
  struct Acc {
    f32x16 t;
    __device__ __forceinline__ float get(int r) const { return t[r]; }
    __device__ __forceinline__ void set(int r, float x) { t[r] = x; }
  };
  static __device__ __forceinline__ int row(int r) { return acc_row(r); }
  static __device__ __forceinline__ int col() { return acc_col(); }
  static __device__ __forceinline__ Acc zero() { return Acc{acc_zero()}; }
  struct Rows {   // read tile by tile: sixteen registers each
    const float* p;
    f32x16 v[2];
    __device__ __forceinline__ void load(const float* arr) { p = arr; }
    __device__ __forceinline__ void fetch(int tile) { v[tile] = rows_ld(p, 32 * tile); }
    __device__ __forceinline__ float get(int tile, int r) const { return v[tile][r]; }
  };
  static __device__ __forceinline__ void st_t(T* image, int piece, const Vec16<T>& v) { st16(image + piece * (16 / (int)sizeof(T)), v); }
  typedef AccB<T> A;
  struct B : AccB<T> {
    __device__ __forceinline__ void pack(const Acc& c) { AccB<T>::pack(c.t); }
    __device__ __forceinline__ Acc unpack() const { return Acc{AccB<T>::unpack()}; }
    __device__ __forceinline__ void store(T* tile, int) const { AccB<T>::store(tile); }
    __device__ __forceinline__ void store_stream(T* tile, int) const { AccB<T>::store_stream(tile); }
  };
  static __device__ __forceinline__ void mma(Acc& c, const A& a, const B& b) { mma32_ff<T>(c.t, a, b); }
  // in turns: back to back on one accumulator a matrix instruction costs half as much again (49 cycles against 34, measured)
  static __device__ __forceinline__ void mma2(Acc& x0, const A& a0, const B& b0, Acc& x1, const A& a1, const B& b1) {
#pragma unroll
    for (int kg = 0; kg < AccK<T>::kGroups; ++kg) {
      mfma_kgroup<T>(x0.t, a0.f[kg], b0.f[kg]);
      mfma_kgroup<T>(x1.t, a1.f[kg], b1.f[kg]);
    }
  }
};

// of a workgroup with NW slabs
template <typename T, int NW> struct SlabOf { typedef Slab32<T> type; };
template <> struct SlabOf<bf16_t, 1> { typedef Slab16 type; };
template <typename T> constexpr int slab_waves(int nw) { return sizeof(T) == 2 && nw == 1 ? 2 : 1; }   // compute waves to a slab

}  // namespace gdn
