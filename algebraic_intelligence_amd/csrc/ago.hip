// Cayley rotary (AGO) kernels: table construction and pairwise rotation.
//
// Tables (src/attention.py:155-204): with Cayley parameter w_k,
//   c0 = (1 - w^2)/(1 + w^2), s0 = 2w/(1 + w^2);  row 0 = (1, 0);
//   row m+1 = (c0 c - s0 s, s0 c + c0 s) renormalised by rsqrt of its squared norm.
// The recurrence is sequential in position and independent per pair, so one thread owns one
// pair column and walks the positions.  Default w_k = 1/(1 + alpha k)^2 with
// alpha = (sqrt(base) - 1) / max(D/2 - 1, 1), sqrt(base) = base * rsqrt(base) (:180-187).
// Every operation is rounded separately in the table type (no contraction).
//
// Rotation (src/attention.py:142-152): (x0, x1) -> (c x0 - s x1, s x0 + c x1) with c and s
// first cast to the x dtype; computed in fp32 (fp64 for fp64) and rounded once.
#include "afa_common.h"
#include "afa_launch.h"

namespace afa {

template <typename T>
__device__ __forceinline__ T inv_sqrt_ieee(T x) {
  if constexpr (sizeof(T) == 8) {
    return 1.0 / sqrt(x);
  } else {
    return 1.0f / __builtin_sqrtf(x);
  }
}

template <typename T>
__global__ __launch_bounds__(64) void ago_tables_kernel(int pairs, int len, const T* freqs, T base,
                                                        T* c_out, T* s_out) {
#pragma clang fp contract(off)
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= pairs) return;
  T w;
  if (freqs != nullptr) {
    w = freqs[p];
  } else {
    const T sqrt_base = base * inv_sqrt_ieee(base);
    const T denom = pairs - 1 > 1 ? (T)(pairs - 1) : (T)1;
    const T alpha = (sqrt_base - (T)1) / denom;
    const T lin = (T)1 + alpha * (T)p;
    w = (T)1 / (lin * lin);
  }
  const T w2 = w * w;
  const T cb = ((T)1 - w2) / ((T)1 + w2);
  const T sb = ((T)2 * w) / ((T)1 + w2);
  T c = 1, s = 0;
  for (int m = 0; m < len; ++m) {
    c_out[(int64_t)m * pairs + p] = c;
    s_out[(int64_t)m * pairs + p] = s;
    const T cn = cb * c - sb * s;
    const T sn = sb * c + cb * s;
    const T r = inv_sqrt_ieee(cn * cn + sn * sn);
    c = cn * r;
    s = sn * r;
  }
}

hipError_t ago_tables_launch(int table_dtype, int pairs, int len, const void* freqs, double base,
                             void* c_out, void* s_out, hipStream_t st) {
  const int blocks = (pairs + 63) / 64;
  if (table_dtype == AFA_F64) {
    hipLaunchKernelGGL((ago_tables_kernel<double>), dim3(blocks), dim3(64), 0, st, pairs, len,
                       (const double*)freqs, base, (double*)c_out, (double*)s_out);
  } else {
    hipLaunchKernelGGL((ago_tables_kernel<float>), dim3(blocks), dim3(64), 0, st, pairs, len,
                       (const float*)freqs, (float)base, (float*)c_out, (float*)s_out);
  }
  return hipGetLastError();
}

template <int TD>
__device__ __forceinline__ float table_load_f32(const void* t, int64_t i) {
  if constexpr (TD == AFA_F32) return ((const float*)t)[i];
  if constexpr (TD == AFA_F64) return (float)((const double*)t)[i];
  if constexpr (TD == AFA_BF16) return Elem<AFA_BF16>::load(t, i);
  return Elem<AFA_F16>::load(t, i);
}

// One or two tensors of one shape (q and k), any element-aligned layout of the flat arrays: one
// thread per pair.  `sign` is -1 for the transposed rotation.  Kept for fp64, for rows that are no
// whole number of 16-byte chunks and for unaligned arrays.
template <int DT, int TD>
__global__ __launch_bounds__(256) void ago_rotate_kernel(int64_t npairs_total, int64_t seq_len,
                                                         int64_t inner, int pairs, const void* xa, const void* xb,
                                                         void* ya, void* yb, const void* rc, const void* rs,
                                                         float sign) {
#pragma clang fp contract(off)
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= npairs_total) return;
  const void* x = blockIdx.y ? xb : xa;
  void* y = blockIdx.y ? yb : ya;
  const int p = (int)(e % pairs);
  const int64_t row = e / pairs;               // index over (outer, seq, inner)
  const int64_t t = (row / inner) % seq_len;   // sequence position
  const int64_t tix = t * pairs + p;
  if constexpr (DT == AFA_F64) {
    double c, s;
    if constexpr (TD == AFA_F64) {
      c = ((const double*)rc)[tix];
      s = ((const double*)rs)[tix];
    } else {
      c = table_load_f32<TD>(rc, tix);
      s = table_load_f32<TD>(rs, tix);
    }
    s *= (double)sign;
    const double x0 = ((const double*)x)[2 * e], x1 = ((const double*)x)[2 * e + 1];
    ((double*)y)[2 * e] = c * x0 - s * x1;
    ((double*)y)[2 * e + 1] = s * x0 + c * x1;
  } else {
    // cast the table to the x dtype first (c.astype(x.dtype))
    const float c = Elem<DT>::round(table_load_f32<TD>(rc, tix));
    const float s = Elem<DT>::round(table_load_f32<TD>(rs, tix)) * sign;
    const float x0 = Elem<DT>::load(x, 2 * e), x1 = Elem<DT>::load(x, 2 * e + 1);
    const float y0 = c * x0 - s * x1;
    const float y1 = s * x0 + c * x1;
    Elem<DT>::store(y, 2 * e, y0);
    Elem<DT>::store(y, 2 * e + 1, y1);
  }
}

// The same in 16-byte chunks: a thread owns one chunk of a (seq, inner, dim) slice, holds its table
// entries and turns that chunk of ROT_OUTER consecutive slices, their loads in flight together, so
// the table and the index arithmetic (two divisions) are paid once per ROT_OUTER chunks.  HBM
// bound: q and k of (2, 16, 8192, 128) bf16 in one launch 44 us (6.1 TB/s), of (8, 12, 2048, 64) two
// launches of 19 us element by element -> one of 16, the training pass 170 -> 112 us (now the host's time).
constexpr int ROT_OUTER = 4;
template <int DT, int TD>
__global__ __launch_bounds__(256) void ago_rotate_vec_kernel(uint32_t slice, int64_t outer, uint32_t seq_chunks,
                                                             uint32_t row_chunks, uint32_t gx, const void* xa,
                                                             const void* xb, void* ya, void* yb, const void* rc,
                                                             const void* rs, float sign) {
#pragma clang fp contract(off)
  using R = RowChunk<DT>;
  constexpr int NP = R::EPC / 2;  // pairs per chunk
  const uint32_t i = (blockIdx.x % gx) * 256 + threadIdx.x;  // chunk of the slice
  if (i >= slice) return;
  const int64_t o0 = (int64_t)(blockIdx.x / gx) * ROT_OUTER;
  const u32x4_t* x = (const u32x4_t*)(blockIdx.y ? xb : xa) + o0 * slice + i;
  u32x4_t* y = (u32x4_t*)(blockIdx.y ? yb : ya) + o0 * slice + i;
  const int n = (int)(outer - o0 < ROT_OUTER ? outer - o0 : ROT_OUTER);
  u32x4_t w[ROT_OUTER];
#pragma unroll
  for (int u = 0; u < ROT_OUTER; ++u)
    if (u < n) w[u] = x[(int64_t)u * slice];
  // seq_chunks: chunks per sequence position (inner rows of row_chunks)
  const int64_t tix = ((int64_t)(i / seq_chunks) * row_chunks + i % row_chunks) * NP;
  float c[NP], s[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    c[p] = Elem<DT>::round(table_load_f32<TD>(rc, tix + p));
    s[p] = Elem<DT>::round(table_load_f32<TD>(rs, tix + p)) * sign;
  }
#pragma unroll
  for (int u = 0; u < ROT_OUTER; ++u) {
    if (u >= n) break;
    float v[R::EPC], r[R::EPC];
    R::unpack(w[u], v);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      r[2 * p] = c[p] * v[2 * p] - s[p] * v[2 * p + 1];
      r[2 * p + 1] = s[p] * v[2 * p] + c[p] * v[2 * p + 1];
    }
    y[(int64_t)u * slice] = R::pack(r);
  }
}

struct RotateArgs {
  int64_t outer, seq, inner;
  int dim;
  const void *xa, *xb;  // xb nullable
  void *ya, *yb;
  const void *rc, *rs;
  float sign;
};

template <int DT, int TD>
static hipError_t ago_rotate_go(const RotateArgs& a, hipStream_t st) {
  const unsigned tensors = a.xb != nullptr ? 2u : 1u;
  if constexpr (DT != AFA_F64) {
    constexpr int EPC = RowChunk<DT>::EPC;
    const int64_t slice = a.seq * a.inner * (a.dim / EPC), gx = (slice + 255) / 256;
    const int64_t blocks = gx * ((a.outer + ROT_OUTER - 1) / ROT_OUTER);
    const uintptr_t ptrs = (uintptr_t)a.xa | (uintptr_t)a.ya | (uintptr_t)a.xb | (uintptr_t)a.yb;
    if (a.dim % EPC == 0 && (ptrs & 15u) == 0 && slice < (int64_t(1) << 31) && blocks < (int64_t(1) << 24)) {
      hipLaunchKernelGGL((ago_rotate_vec_kernel<DT, TD>), dim3((unsigned)blocks, tensors), dim3(256), 0, st,
                         (uint32_t)slice, a.outer, (uint32_t)(a.inner * (a.dim / EPC)), (uint32_t)(a.dim / EPC),
                         (uint32_t)gx, a.xa, a.xb, a.ya, a.yb, a.rc, a.rs, a.sign);
      return hipGetLastError();
    }
  }
  const int pairs = a.dim / 2;
  const int64_t n = a.outer * a.seq * a.inner * pairs;
  hipLaunchKernelGGL((ago_rotate_kernel<DT, TD>), dim3((unsigned)((n + 255) / 256), tensors), dim3(256), 0, st, n,
                     a.seq, a.inner, pairs, a.xa, a.xb, a.ya, a.yb, a.rc, a.rs, a.sign);
  return hipGetLastError();
}

template <int DT>
static hipError_t ago_rotate_dt(int table_dtype, const RotateArgs& a, hipStream_t st) {
  switch (table_dtype) {
    case AFA_F32: return ago_rotate_go<DT, AFA_F32>(a, st);
    case AFA_F64: return ago_rotate_go<DT, AFA_F64>(a, st);
    case AFA_BF16: return ago_rotate_go<DT, AFA_BF16>(a, st);
    default: return ago_rotate_go<DT, AFA_F16>(a, st);
  }
}

hipError_t ago_rotate_launch(int dtype, int table_dtype, int64_t outer, int64_t seq, int64_t inner, int dim,
                             const void* xa, const void* xb, void* ya, void* yb, const void* rc, const void* rs,
                             bool transpose, hipStream_t st) {
  const RotateArgs a{outer, seq, inner, dim, xa, xb, ya, yb, rc, rs, transpose ? -1.f : 1.f};
  switch (dtype) {
    case AFA_F32: return ago_rotate_dt<AFA_F32>(table_dtype, a, st);
    case AFA_BF16: return ago_rotate_dt<AFA_BF16>(table_dtype, a, st);
    case AFA_F16: return ago_rotate_dt<AFA_F16>(table_dtype, a, st);
    default: return ago_rotate_dt<AFA_F64>(table_dtype, a, st);
  }
}

}  // namespace afa
