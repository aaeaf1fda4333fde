// A-Softmax row kernels and the elementwise octic weight.
//
// algebraic_softmax (src/attention.py:53-91, AVN from src/primitives.py:56-79), per row of n:
//   z = promote(x);  tau = rsqrt(sum(z^2) * (1/n) + eps);  y = tau z
//   k = rho(y)^8, r = rsqrt(1 + y^2);  p = k / (sum k + Omega);  output cast(p, x.dtype)
// VJP (src/attention.py:75-82, src/primitives.py:73-79):
//   ng = 8 r p (g - sum(p g));  dx = tau (ng - (sum(ng y) / n) y)
// Rows are handled by one wave each; values are promoted to fp32 (fp64 stays fp64) and the
// reference's two-branch rho formula is evaluated op for op.  These kernels are HBM bound; rows
// that fit in registers take the single-read kernels further down.
#include "afa_common.h"
#include "afa_launch.h"

namespace afa {

template <int DT>
struct SAcc {
  typedef float T;
};
template <>
struct SAcc<AFA_F64> {
  typedef double T;
};

template <int DT>
__device__ __forceinline__ typename SAcc<DT>::T sload(const void* p, int64_t i) {
  if constexpr (DT == AFA_F64) {
    return ((const double*)p)[i];
  } else {
    return Elem<DT>::load(p, i);
  }
}
template <int DT>
__device__ __forceinline__ void sstore(void* p, int64_t i, typename SAcc<DT>::T x) {
  if constexpr (DT == AFA_F64) {
    ((double*)p)[i] = x;
  } else {
    Elem<DT>::store(p, i, x);
  }
}

template <typename T>
__device__ __forceinline__ T wave_sum(T x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// rho(z)^8 and r = rsqrt(1 + z^2), op for op as src/attention.py:18-26.
template <typename T>
__device__ __forceinline__ T octic_ref(T z, T& r_out) {
  const T one = 1;
  const T zz = z * z;
  T r;
  if constexpr (sizeof(T) == 8) {
    r = 1.0 / sqrt(one + zz);
  } else {
    r = 1.0f / __builtin_sqrtf(one + zz);
  }
  const T u = z * r;
  const T rho = z < 0 ? r / (one - u) : z + (one + zz) * r;
  const T k2 = rho * rho;
  const T k4 = k2 * k2;
  r_out = r;
  return k4 * k4;
}

template <typename T>
__device__ __forceinline__ T inv_sqrt(T x) {
  if constexpr (sizeof(T) == 8) {
    return 1.0 / sqrt(x);
  } else {
    return 1.0f / __builtin_sqrtf(x);
  }
}

template <int DT>
__global__ __launch_bounds__(256) void asoftmax_fwd_kernel(int64_t rows, int64_t n, const void* x,
                                                           void* y, double sink, double eps) {
#pragma clang fp contract(off)
  typedef typename SAcc<DT>::T T;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int64_t base = row * n;
  T ss = 0;
  for (int64_t i = lane; i < n; i += 64) {
    const T z = sload<DT>(x, base + i);
    ss += z * z;
  }
  ss = wave_sum(ss);
  const T tau = inv_sqrt(ss * (T(1) / (T)n) + (T)eps);
  T ks = 0;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    ks += octic_ref(sload<DT>(x, base + i) * tau, r);
  }
  ks = wave_sum(ks);
  const T den = ks + (T)sink;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    const T k = octic_ref(sload<DT>(x, base + i) * tau, r);
    sstore<DT>(y, base + i, k / den);
  }
}

template <int DT>
__global__ __launch_bounds__(256) void asoftmax_bwd_kernel(int64_t rows, int64_t n, const void* x,
                                                           const void* g, void* dx, double sink,
                                                           double eps) {
#pragma clang fp contract(off)
  typedef typename SAcc<DT>::T T;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int64_t base = row * n;
  const T inv_n = T(1) / (T)n;
  T ss = 0;
  for (int64_t i = lane; i < n; i += 64) {
    const T z = sload<DT>(x, base + i);
    ss += z * z;
  }
  ss = wave_sum(ss);
  const T tau = inv_sqrt(ss * inv_n + (T)eps);
  T ks = 0;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    ks += octic_ref(sload<DT>(x, base + i) * tau, r);
  }
  ks = wave_sum(ks);
  const T den = ks + (T)sink;
  // dot = sum(p g)
  T dot = 0;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    const T p = octic_ref(sload<DT>(x, base + i) * tau, r) / den;
    dot += p * sload<DT>(g, base + i);
  }
  dot = wave_sum(dot);
  // radial = sum(ng y) / n
  T rad = 0;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    const T yv = sload<DT>(x, base + i) * tau;
    const T p = octic_ref(yv, r) / den;
    const T ng = T(8) * r * p * (sload<DT>(g, base + i) - dot);
    rad += ng * yv;
  }
  rad = wave_sum(rad) * inv_n;
  for (int64_t i = lane; i < n; i += 64) {
    T r;
    const T yv = sload<DT>(x, base + i) * tau;
    const T p = octic_ref(yv, r) / den;
    const T ng = T(8) * r * p * (sload<DT>(g, base + i) - dot);
    sstore<DT>(dx, base + i, tau * (ng - rad * yv));
  }
}

template <int DT>
__global__ __launch_bounds__(256) void octic_fwd_kernel(int64_t n, const void* x, void* y) {
  typedef typename SAcc<DT>::T T;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T r;
  sstore<DT>(y, i, octic_ref(sload<DT>(x, i), r));
}

// rho(x)^8 and r = rsqrt(1 + x^2), both stored in the accumulation type (fp32, fp64 for fp64
// inputs): src/attention.py:18-26 returns the pair, r being the factor of the VJP 8 r rho^8 g.
template <int DT>
__global__ __launch_bounds__(256) void octic_fwd_r_kernel(int64_t n, const void* x, void* k, void* r) {
  typedef typename SAcc<DT>::T T;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T rr;
  const T kk = octic_ref(sload<DT>(x, i), rr);
  ((T*)k)[i] = kk;
  ((T*)r)[i] = rr;
}

template <int DT>
__global__ __launch_bounds__(256) void octic_bwd_kernel(int64_t n, const void* x, const void* g,
                                                        void* dx) {
#pragma clang fp contract(off)
  typedef typename SAcc<DT>::T T;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T r;
  const T k = octic_ref(sload<DT>(x, i), r);
  sstore<DT>(dx, i, T(8) * r * k * sload<DT>(g, i));
}


// rho(z)^8 and r = rsqrt(1 + z^2) with the hardware reciprocal square root and reciprocal (1 ulp
// each): rho(|z|) = |z| + (1 + z^2) r, which has no cancellation, and rho(-z) = 1 / rho(z).  Used by the
// register-resident kernels.
__device__ __forceinline__ float octic_hw(float z, float& r_out) {
  const float t = __builtin_fmaf(z, z, 1.0f);
  const float r = __builtin_amdgcn_rsqf(t);
  const float pos = __builtin_fmaf(t, r, __builtin_fabsf(z));
  const float rho = z < 0.0f ? __builtin_amdgcn_rcpf(pos) : pos;
  const float k2 = rho * rho;
  const float k4 = k2 * k2;
  r_out = r;
  return k4 * k4;
}

// ---------------------------------------------------------------- register-resident row kernels
// T threads per row (one wave, or 4 to 16 waves for longer rows), the whole row held in registers as its
// aligned 16-byte chunks (RowChunk: any length and any start; thread l owns chunks l, l + T, ...) and,
// where it starts or ends inside a chunk, one element each of the first lanes: one HBM read of x (and
// g), one write; rho^8 and r are evaluated once per element with the hardware rsqrt / reciprocal
// (octic_hw) and the row is normalised with one division and products; the multi-pass kernels above
// keep IEEE 1/sqrt and divisions throughout.  WHOLE, all_whole: every row is whole chunks, none has an edge;
// known when compiled for rows of one chunk a lane (2^20 rows of 8 fp32 218 -> 205 us, VJP 296 -> 279).
// Kernels alone, forward of (18372, 1531) fp32 99 -> 35 us (6.4 TB/s) and its VJP 254 -> 60 us (5.6 TB/s)
// against the multi-pass kernels, which served every row whose length was no multiple of a chunk or
// over 64 x 8 (VJP: 64 x 4) chunks.
template <int T, int K>
__device__ __forceinline__ void row_sum(float (&x)[K], float* sh) {
#pragma unroll
  for (int q = 0; q < K; ++q) x[q] = wave_sum(x[q]);
  if constexpr (T > 64) {
    constexpr int NW = T / 64;
    const int wave = threadIdx.x >> 6;
    __syncthreads();  // the previous sum's values have been read
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int q = 0; q < K; ++q) sh[q * NW + wave] = x[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < K; ++q) {
      x[q] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) x[q] += sh[q * NW + w];
    }
  }
}

template <int DT, int T, int NCH, bool WHOLE>
__global__ __launch_bounds__(T < 256 ? 256 : T) void asoftmax_fwd_reg_kernel(int64_t rows, int n, bool all_whole,
                                                                            const void* x, void* y, float sink,
                                                                            float eps) {
#pragma clang fp contract(off)
  using R = RowChunk<DT>;
  constexpr int RPB = T < 256 ? 256 / T : 1;  // rows per workgroup
  __shared__ float sh[T > 64 ? T / 64 : 1];
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / T;
  if (row >= rows) return;  // whole waves, and only where no barrier follows
  const int tid = threadIdx.x % T;
  const char* xr = (const char*)x + row * n * R::ESZ;
  char* yr = (char*)y + row * n * R::ESZ;
  const bool whole = WHOLE || all_whole;
  const RowSpan sp = whole ? RowSpan{0, n / R::EPC, 0} : R::span(xr, n);
  const int edge = whole ? -1 : R::edge(sp, n, tid);
  u32x4_t raw[NCH];
  float v[NCH][R::EPC];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = tid + T * j;
    raw[j] = u32x4_t{0u, 0u, 0u, 0u};
    if (c < sp.body) raw[j] = *(const u32x4_t*)(xr + (int64_t)(sp.head + c * R::EPC) * R::ESZ);
  }
  float ve = edge >= 0 ? Elem<DT>::load(xr, edge) : 0.f;
  float ss[1] = {ve * ve};
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    R::unpack(raw[j], v[j]);
#pragma unroll
    for (int i = 0; i < R::EPC; ++i) ss[0] += v[j][i] * v[j][i];
  }
  row_sum<T, 1>(ss, sh);
  const float tau = inv_sqrt(ss[0] * (1.f / (float)n) + eps);
  float ks[1] = {0.f};
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (tid + T * j < sp.body) {
#pragma unroll
      for (int i = 0; i < R::EPC; ++i) {
        float r;
        v[j][i] = octic_hw(v[j][i] * tau, r);
        ks[0] += v[j][i];
      }
    }
  }
  if (edge >= 0) {
    float r;
    ve = octic_hw(ve * tau, r);
    ks[0] += ve;
  }
  row_sum<T, 1>(ks, sh);
  const float inv = 1.0f / (ks[0] + sink);
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = tid + T * j;
    if (c < sp.body) {
#pragma unroll
      for (int i = 0; i < R::EPC; ++i) v[j][i] = v[j][i] * inv;
      *(u32x4_t*)(yr + (int64_t)(sp.head + c * R::EPC) * R::ESZ) = R::pack(v[j]);
    }
  }
  if (edge >= 0) Elem<DT>::store(yr, edge, ve * inv);
}

template <int DT, int T, int NCH, bool WHOLE>
__global__ __launch_bounds__(T < 256 ? 256 : T) void asoftmax_bwd_reg_kernel(int64_t rows, int n, bool all_whole,
                                                                            const void* x, const void* g, void* dx,
                                                                            float sink, float eps) {
#pragma clang fp contract(off)
  // The row's x and g stay in registers as their raw 16-byte chunks and are unpacked where used;
  // one float per element, w = 8 r rho^8, carries the octic between passes.  sum(p g) is taken
  // as sum(rho^8 g) / (sum rho^8 + sink) in the pass that forms sum rho^8, so three row
  // reductions serve the row, and the kernel holds few enough registers for several waves per SIMD
  // to keep loads in flight.
  using R = RowChunk<DT>;
  constexpr int RPB = T < 256 ? 256 / T : 1;
  __shared__ float sh[T > 64 ? 2 * (T / 64) : 1];
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / T;
  if (row >= rows) return;
  const int tid = threadIdx.x % T;
  const char* xr = (const char*)x + row * n * R::ESZ;
  const char* gr = (const char*)g + row * n * R::ESZ;
  char* dr = (char*)dx + row * n * R::ESZ;
  const bool whole = WHOLE || all_whole;
  const RowSpan sp = whole ? RowSpan{0, n / R::EPC, 0} : R::span(xr, n);
  const int edge = whole ? -1 : R::edge(sp, n, tid);
  const float inv_n = 1.f / (float)n;
  u32x4_t xw[NCH], gw[NCH];
  float w[NCH][R::EPC];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = tid + T * j;
    xw[j] = gw[j] = u32x4_t{0u, 0u, 0u, 0u};
    if (c < sp.body) {
      const int64_t off = (int64_t)(sp.head + c * R::EPC) * R::ESZ;
      xw[j] = *(const u32x4_t*)(xr + off);
      gw[j] = *(const u32x4_t*)(gr + off);
    }
  }
  const float xe = edge >= 0 ? Elem<DT>::load(xr, edge) : 0.f, ge = edge >= 0 ? Elem<DT>::load(gr, edge) : 0.f;
  float ss[1] = {xe * xe}, we = 0.f;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    float z[R::EPC];
    R::unpack(xw[j], z);
#pragma unroll
    for (int i = 0; i < R::EPC; ++i) ss[0] += z[i] * z[i];
  }
  row_sum<T, 1>(ss, sh);
  const float tau = inv_sqrt(ss[0] * inv_n + eps);
  float kp[2] = {0.f, 0.f};  // sum rho^8, sum rho^8 g
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (tid + T * j < sp.body) {
      float z[R::EPC], gv[R::EPC];
      R::unpack(xw[j], z);
      R::unpack(gw[j], gv);
#pragma unroll
      for (int i = 0; i < R::EPC; ++i) {
        float r;
        const float p = octic_hw(z[i] * tau, r);
        kp[0] += p;
        kp[1] += p * gv[i];
        w[j][i] = 8.f * r * p;
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // one chunk's unpacked values live at a time
  }
  if (edge >= 0) {
    float r;
    const float p = octic_hw(xe * tau, r);
    kp[0] += p;
    kp[1] += p * ge;
    we = 8.f * r * p;
  }
  row_sum<T, 2>(kp, sh);
  const float inv = 1.0f / (kp[0] + sink);
  const float dot = kp[1] * inv;
  float rad[1] = {0.f};
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (tid + T * j < sp.body) {
      float z[R::EPC], gv[R::EPC];
      R::unpack(xw[j], z);
      R::unpack(gw[j], gv);
#pragma unroll
      for (int i = 0; i < R::EPC; ++i) {
        w[j][i] = w[j][i] * inv * (gv[i] - dot);  // ng
        rad[0] += w[j][i] * (z[i] * tau);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  we = we * inv * (ge - dot);  // 0 where the lane has no edge element
  if (edge >= 0) rad[0] += we * (xe * tau);
  row_sum<T, 1>(rad, sh);
  rad[0] *= inv_n;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = tid + T * j;
    if (c < sp.body) {
      float z[R::EPC];
      R::unpack(xw[j], z);
#pragma unroll
      for (int i = 0; i < R::EPC; ++i) w[j][i] = tau * (w[j][i] - rad[0] * (z[i] * tau));
      *(u32x4_t*)(dr + (int64_t)(sp.head + c * R::EPC) * R::ESZ) = R::pack(w[j]);
    }
  }
  if (edge >= 0) Elem<DT>::store(dr, edge, tau * (we - rad[0] * (xe * tau)));
}

// The rows of all tensors start at the same offset from a 16-byte boundary (the chunks of one are the
// chunks of the others).
static bool same_lead(const void* a, const void* b, const void* c) {
  return ((((uintptr_t)a ^ (uintptr_t)b) | (c != nullptr ? (uintptr_t)a ^ (uintptr_t)c : 0)) & 15u) == 0;
}

#define AFA_DISPATCH_DT(dtype, FN, ...)            \
  switch (dtype) {                                 \
    case AFA_F32: FN<AFA_F32>(__VA_ARGS__); break; \
    case AFA_BF16: FN<AFA_BF16>(__VA_ARGS__); break; \
    case AFA_F16: FN<AFA_F16>(__VA_ARGS__); break; \
    default: FN<AFA_F64>(__VA_ARGS__); break;      \
  }

template <int DT>
static void sm_fwd(int64_t rows, int64_t n, const void* x, void* y, double sink, double eps, hipStream_t st) {
  hipLaunchKernelGGL((asoftmax_fwd_kernel<DT>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, rows, n, x, y, sink, eps);
}
template <int DT>
static void sm_bwd(int64_t rows, int64_t n, const void* x, const void* g, void* dx, double sink, double eps, hipStream_t st) {
  hipLaunchKernelGGL((asoftmax_bwd_kernel<DT>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, rows, n, x, g, dx, sink, eps);
}
template <int DT>
static void oc_fwd(int64_t n, const void* x, void* y, hipStream_t st) {
  hipLaunchKernelGGL((octic_fwd_kernel<DT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, x, y);
}
template <int DT>
static void oc_fwd_r(int64_t n, const void* x, void* k, void* r, hipStream_t st) {
  hipLaunchKernelGGL((octic_fwd_r_kernel<DT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, x, k, r);
}
template <int DT>
static void oc_bwd(int64_t n, const void* x, const void* g, void* dx, hipStream_t st) {
  hipLaunchKernelGGL((octic_bwd_kernel<DT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, x, g, dx);
}

// Threads per row and chunks per thread by the row's chunk count: the fewest threads that hold the row
// in at most four chunks each (the VJP's x, g and 8 r rho^8 take 12 or 16 registers a chunk: six
// chunks a lane leave one wave per SIMD, and (18372, 1531) fp32 took 173 us instead of 80).  false: no
// variant holds the row, or a launch would pass 2^32 threads (the multi-pass kernels take 64 per row).
static bool sm_reg_fits(int64_t rows, int nch) { return nch <= 4096 && (nch <= 256 || rows < (1 << 22)); }
#define AFA_SM_GO(KERNEL, T, NCH, WHOLE, ...)                                                                \
  hipLaunchKernelGGL((KERNEL<DT, T, NCH, WHOLE>), dim3((unsigned)((rows * T + (T < 256 ? 255 : T - 1)) /     \
                     (T < 256 ? 256 : T))), dim3(T < 256 ? 256 : T), 0, st, rows, (int)n, whole, __VA_ARGS__)
template <int DT>
static bool sm_fwd_reg(int64_t rows, int64_t n, const void* x, void* y, double sink, double eps, hipStream_t st) {
  if (n > (1 << 20) || !same_lead(x, y, nullptr)) return false;
  const int nch = (int)n / RowChunk<DT>::EPC;  // whole chunks of the best start
  if (!sm_reg_fits(rows, nch)) return false;
  const bool whole = n % RowChunk<DT>::EPC == 0 && ((uintptr_t)x & 15u) == 0;
  // Ragged rows of 2-byte scores that one wave holds with one score to a lane: the multi-pass kernel forms their
  // octics side by side, where a lane here forms a chunk's eight and then its edge element (2^18 rows of
  // 17, 33, 63 bf16 73, 77, 78 against 85 us, fp16 73, 77, 78 against 91).  Below 15 not every row holds a
  // whole chunk (9: 72 against 62), above 64 it takes two turns (2^17 rows of 65: 70 against 44).  fp32
  // chunks hold four (33: 76 against 66), and the VJP's multi-pass kernel reads more (33: 140 against 122).
  if (RowChunk<DT>::EPC == 8 && !whole && n >= 15 && n <= 64) return false;
#define AFA_SM_W(T, NCH, WHOLE) AFA_SM_GO(asoftmax_fwd_reg_kernel, T, NCH, WHOLE, x, y, (float)sink, (float)eps)
#define AFA_SM(T, NCH) AFA_SM_W(T, NCH, false)
  if (nch <= 64 && whole) AFA_SM_W(64, 1, true);  // no edge code where the rows are short
  else if (nch <= 64) AFA_SM(64, 1);
  else if (nch <= 128) AFA_SM(64, 2);
  else if (nch <= 192) AFA_SM(64, 3);
  else if (nch <= 256) AFA_SM(64, 4);
  else if (nch <= 512) AFA_SM(256, 2);
  else if (nch <= 768) AFA_SM(256, 3);
  else if (nch <= 1024) AFA_SM(256, 4);
  else if (nch <= 1536) AFA_SM(512, 3);
  else if (nch <= 2048) AFA_SM(512, 4);
  else AFA_SM(1024, 4);
#undef AFA_SM
#undef AFA_SM_W
  return true;
}
template <int DT>
static bool sm_bwd_reg(int64_t rows, int64_t n, const void* x, const void* g, void* dx, double sink, double eps,
                       hipStream_t st) {
  if (n > (1 << 20) || !same_lead(x, g, dx)) return false;
  const int nch = (int)n / RowChunk<DT>::EPC;  // whole chunks of the best start
  if (!sm_reg_fits(rows, nch)) return false;
  const bool whole = n % RowChunk<DT>::EPC == 0 && ((uintptr_t)x & 15u) == 0;
#define AFA_SM_W(T, NCH, WHOLE) AFA_SM_GO(asoftmax_bwd_reg_kernel, T, NCH, WHOLE, x, g, dx, (float)sink, (float)eps)
#define AFA_SM(T, NCH) AFA_SM_W(T, NCH, false)
  if (nch <= 64 && whole) AFA_SM_W(64, 1, true);
  else if (nch <= 64) AFA_SM(64, 1);
  else if (nch <= 128) AFA_SM(64, 2);
  else if (nch <= 192) AFA_SM(64, 3);
  else if (nch <= 256) AFA_SM(64, 4);
  else if (nch <= 512) AFA_SM(256, 2);
  else if (nch <= 768) AFA_SM(256, 3);
  else if (nch <= 1024) AFA_SM(256, 4);
  else if (nch <= 1536) AFA_SM(512, 3);
  else if (nch <= 2048) AFA_SM(512, 4);
  else AFA_SM(1024, 4);
#undef AFA_SM
#undef AFA_SM_W
  return true;
}
#undef AFA_SM_GO

hipError_t asoftmax_fwd_launch(int dtype, int64_t rows, int64_t n, const void* x, void* y, double sink,
                               double eps, hipStream_t st) {
  const bool done = dtype == AFA_F32    ? sm_fwd_reg<AFA_F32>(rows, n, x, y, sink, eps, st)
                    : dtype == AFA_BF16 ? sm_fwd_reg<AFA_BF16>(rows, n, x, y, sink, eps, st)
                    : dtype == AFA_F16  ? sm_fwd_reg<AFA_F16>(rows, n, x, y, sink, eps, st)
                                        : false;
  if (!done) AFA_DISPATCH_DT(dtype, sm_fwd, rows, n, x, y, sink, eps, st);
  return hipGetLastError();
}
hipError_t asoftmax_bwd_launch(int dtype, int64_t rows, int64_t n, const void* x, const void* g,
                               void* dx, double sink, double eps, hipStream_t st) {
  const bool done = dtype == AFA_F32    ? sm_bwd_reg<AFA_F32>(rows, n, x, g, dx, sink, eps, st)
                    : dtype == AFA_BF16 ? sm_bwd_reg<AFA_BF16>(rows, n, x, g, dx, sink, eps, st)
                    : dtype == AFA_F16  ? sm_bwd_reg<AFA_F16>(rows, n, x, g, dx, sink, eps, st)
                                        : false;
  if (!done) AFA_DISPATCH_DT(dtype, sm_bwd, rows, n, x, g, dx, sink, eps, st);
  return hipGetLastError();
}
hipError_t octic_fwd_launch(int dtype, int64_t n, const void* x, void* y, hipStream_t st) {
  AFA_DISPATCH_DT(dtype, oc_fwd, n, x, y, st);
  return hipGetLastError();
}
hipError_t octic_fwd_r_launch(int dtype, int64_t n, const void* x, void* k, void* r, hipStream_t st) {
  AFA_DISPATCH_DT(dtype, oc_fwd_r, n, x, k, r, st);
  return hipGetLastError();
}
hipError_t octic_bwd_launch(int dtype, int64_t n, const void* x, const void* g, void* dx, hipStream_t st) {
  AFA_DISPATCH_DT(dtype, oc_bwd, n, x, g, dx, st);
  return hipGetLastError();
}

}  // namespace afa
