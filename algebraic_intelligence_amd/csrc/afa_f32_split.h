// fp32 products on the bf16 matrix cores: exact three-plane splits and the LDS tiles of planes.
//
// x = hi + mid + lo with three bf16 values holds an fp32 value exactly (3 x 8 significant bits), and
//   x y = hi hi' + (hi mid' + mid hi') + (mid mid' + hi lo' + lo hi') + terms together below 2^-23 |x y|,
// six products of the bf16 matrix cores, accumulated in fp32.  They run at 16 times the fp32 rate:
// 2.7 times after six passes, and one fp32 rounding serves 16 of the contraction where the fp32
// MFMA's serves two.  Below about 2^-110 the lower planes reach bf16's subnormals (steps of 2^-133) and
// fewer bits of a value are held.
#pragma once

#include "afa_common.h"

namespace afa {

// Planes of a pair, packed.  Rounded to nearest: |mid| < 2^-8 |x| and |lo| < 2^-16 |x|.  An
// infinity, or a value that rounds past the largest bf16, gives a NaN in the lower planes (rows redone in
// fp32, below).
__device__ __forceinline__ void split3_rne(float x0, float x1, unsigned& hi, unsigned& mid, unsigned& lo) {
  hi = pack_bf16(x0, x1);
  const float r0 = x0 - bf16_lo(hi), r1 = x1 - bf16_hi(hi);
  mid = pack_bf16(r0, r1);
  lo = pack_bf16(r0 - bf16_lo(mid), r1 - bf16_hi(mid));
}

// acc += A B over 16 of the contraction, both operands as planes; smallest terms first.
__device__ __forceinline__ f32x16_t mma_planes(const u32x4_t (&a)[3], u32x4_t b0, u32x4_t b1, u32x4_t b2,
                                               f32x16_t acc) {
  const u32x4_t w0 = a[0], w1 = a[1], w2 = a[2];
  const bf16x8_t a0 = __builtin_bit_cast(bf16x8_t, w0), a1 = __builtin_bit_cast(bf16x8_t, w1);
  const bf16x8_t a2 = __builtin_bit_cast(bf16x8_t, w2);
  const bf16x8_t c0 = __builtin_bit_cast(bf16x8_t, b0), c1 = __builtin_bit_cast(bf16x8_t, b1);
  const bf16x8_t c2 = __builtin_bit_cast(bf16x8_t, b2);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, c0, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, c2, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, c1, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, c0, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, c1, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, c0, acc, 0, 0, 0);
}

typedef __attribute__((ext_vector_type(4))) short f32s_s16x4_t;
typedef __attribute__((address_space(3))) f32s_s16x4_t f32s_lds_s16x4_t;

// LDS tile of 32 rows x D features of one plane: rows of RP = 64 or 128 elements whose 16-byte chunks
// are permuted by a key of the row that is conflict-free for reads along the rows (16-byte fragments
// of 32 rows: the 16 rows of a pass take all 16 chunk slots of a bank period) and down the columns
// (ds_read_tr16_b64: the 8 rows of a pass go to different 4-chunk groups).
template <int D>
struct F32Tile {
  static constexpr int RP = D <= 64 ? 64 : 128;
  static constexpr int PLANE = 32 * RP;
  static __device__ __forceinline__ int key(int r) {
    return RP == 128 ? (r & 15) ^ ((r & 3) << 2) : ((r & 2) << 1) | ((r >> 2) & 3);
  }
  // element offset in the plane of features c .. c + 3 (c a multiple of 4) of row r
  static __device__ __forceinline__ int at(int r, int c) { return r * RP + (((c >> 3) ^ key(r)) << 3) + (c & 4); }
  static __device__ __forceinline__ void put(unsigned short* tile, int at, const unsigned (&w)[3][2]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) *(u32x2_t*)(tile + p * PLANE + at) = u32x2_t{w[p][0], w[p][1]};
  }
  // operand rows l32, contraction over the features 16 kk + 8 g .. + 7
  static __device__ __forceinline__ u32x4_t row_frag(const unsigned short* plane, int kk, int lane) {
    const int r = lane & 31, g = lane >> 5;
    return *(const u32x4_t*)(plane + r * RP + (((2 * kk + g) ^ key(r)) << 3));
  }
  // operand rows = features 32 db + l32, contraction over the tile rows
  // 16 kk + 8 (i >> 2) + 4 g + (i & 3), i = 0 .. 7: the row order of an accumulator's elements
  static __device__ __forceinline__ u32x4_t col_frag(const unsigned short* plane, int db, int kk, int lane) {
    const int l16 = lane & 15, m16 = (lane >> 4) & 1, g = lane >> 5;
    u32x4_t f;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int row = 16 * kk + 8 * hh + 4 * g + (l16 >> 2);
      const int col = db * 32 + m16 * 16 + 4 * (l16 & 3);
      const f32s_s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((f32s_lds_s16x4_t*)(plane + at(row, col)));
      const u32x2_t w = __builtin_bit_cast(u32x2_t, v);
      f[2 * hh] = w[0];
      f[2 * hh + 1] = w[1];
    }
    return f;
  }
};

// The 16 elements of an accumulator as B-operand planes of a product that contracts its rows.
__device__ __forceinline__ void split_acc(const float (&x)[16], u32x4_t (&pk)[3][2]) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      unsigned hi, mid, lo;
      split3_rne(x[8 * kk + 2 * u], x[8 * kk + 2 * u + 1], hi, mid, lo);
      pk[0][kk][u] = hi;
      pk[1][kk][u] = mid;
      pk[2][kk][u] = lo;
    }
}

// Planes of 8 consecutive features (two float4), as one 16-feature step's operand.
__device__ __forceinline__ void split8(f32x4_t a, f32x4_t b, u32x4_t& p0, u32x4_t& p1, u32x4_t& p2) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    unsigned hi, mid, lo;
    const f32x4_t x = u < 2 ? a : b;
    split3_rne(x[2 * (u & 1)], x[2 * (u & 1) + 1], hi, mid, lo);
    p0[u] = hi;
    p1[u] = mid;
    p2[u] = lo;
  }
}

// (x0, x1) -> (c x0 - s x1, s x0 + c x1) of two pairs, every operation rounded.
__device__ __forceinline__ f32x4_t f32_rotate4(f32x4_t x, const float* c, const float* s) {
#pragma clang fp contract(off)
  f32x4_t y;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    y[2 * p] = c[p] * x[2 * p] - s[p] * x[2 * p + 1];
    y[2 * p + 1] = s[p] * x[2 * p] + c[p] * x[2 * p + 1];
  }
  return y;
}

// ------------------------------------------------------------------ rows redone in fp32
// An infinite operand, or one that rounds past the largest bf16, leaves NaN in its lower planes and so
// in every product that meets it, where the fp32 product is an infinity or finite.  A wave whose sums hold a NaN
// looks its operands over once its tiles are done and, unless NaN operands account for it, takes its
// rows again in plain fp32: nothing is paid in the tiles, and the second pass reads one row of the other
// side at a time (about ten times the work of the tiles it replaces).

// Any NaN among a wave's sums (an infinite sum counts too: 0 times it is NaN).
template <int N>
__device__ __forceinline__ bool f32_any_nan(const f32x16_t (&acc)[N]) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) t = __builtin_fmaf(acc[i][e], 0.f, t);
  return __ballot(t != t) != 0;
}

// What a wave has seen of its operands: a NaN; a value that planes do not hold.
struct F32Look {
  bool nan = false, big = false;
  __device__ __forceinline__ void add(float x) {
    nan |= x != x;
    big |= __builtin_fabsf(x) > 3.38953138925153547590e38f;  // the largest bf16
  }
  // rows [0, n) of D features, row stride ld, dword aligned
  template <int D>
  __device__ __forceinline__ void rows(const float* p, int64_t ld, int n) {
    typedef f32x4_t f32x4_dword_t __attribute__((aligned(4)));
#pragma unroll 1
    for (int i = threadIdx.x & 63; i < n * (D / 4); i += 64) {
      const f32x4_t x = *(const f32x4_dword_t*)(p + (int64_t)(i / (D / 4)) * ld + 4 * (i % (D / 4)));
#pragma unroll
      for (int u = 0; u < 4; ++u) add(x[u]);
    }
  }
  __device__ __forceinline__ bool redo() const { return __ballot(big) != 0 || __ballot(nan) == 0; }
};

// The features of one row that a lane holds in the accumulators, 8 c + 4 g .. + 3 (rotated when ROT).
template <int D, bool ROT>
__device__ __forceinline__ void f32_half_row(const float* row, const float* rc, const float* rs, int pos,
                                             f32x4_t (&x)[D / 8]) {
  typedef f32x4_t f32x4_dword_t __attribute__((aligned(4)));
  const int g = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    const int m = 8 * c + 4 * g;
    x[c] = *(const f32x4_dword_t*)(row + m);
    if constexpr (ROT) {
      const int64_t t = (int64_t)pos * (D / 2) + m / 2;
      x[c] = f32_rotate4(x[c], rc + t, rs + t);
    }
  }
}

// The dot product of two such rows, both lanes' halves.
template <int N>
__device__ __forceinline__ float f32_half_dot(const f32x4_t (&x)[N], const f32x4_t (&y)[N]) {
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < N; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u) s = __builtin_fmaf(x[c][u], y[c][u], s);
  return s + __shfl_xor(s, 32);
}

// acc += w x for such a row x.
template <int N, int NDB>
__device__ __forceinline__ void f32_half_axpy(float w, const f32x4_t (&x)[N], f32x16_t (&acc)[NDB]) {
#pragma unroll
  for (int c = 0; c < N; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[c >> 2][4 * (c & 3) + u] = __builtin_fmaf(w, x[c][u], acc[c >> 2][4 * (c & 3) + u]);
}

template <int N>
__device__ __forceinline__ void f32_clear(f32x16_t (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
}

}  // namespace afa
