// OACE loss head: the octic algebraic cross-entropy over an AVN-normalised A-Softmax, either on
// given logits (fused_oace_softmax_loss, src/model.py:180-240) or fused with the vocabulary
// projection z = h W (fused_linear_oace, src/kernels/pallas_oace.py:59-293).
//
// Per row n of logits z (length V), with calc type A (fp32; fp64 for fp64 inputs):
//   tau = rsqrt(sum z^2 / V + eps);  x = tau z;  r = rsqrt(1 + x^2);  rho = x + (1+x^2) r
//   (rho = r / (1 - x r) for x < 0);  k8 = rho^8;  rho7 = rho^7
//   sums  S0 = sum k8, S1 = sum rho7, S2 = sum (r x) k8, S3 = sum (r x) rho7; target rho_t, (r x)_t
//   inv_S = 1/S0, S8 = rsqrt(rsqrt(rsqrt(inv_S))), scale = S8 inv_S, sum_p78 = scale S1,
//   p_c_inv8 = S8 / rho_t, radial = (scale S3 - (r x)_t p_c_inv8 - (sum_p78 - p_c_inv8) inv_S S2) / V,
//   loss = gamma (8 p_c_inv8 + 8/7 sum_p78 - 64/7)                       (pallas_oace.py:166-187)
// and the backward dz = tau c (r bracket - radial x), c = 8 gamma g / N,
//   bracket = scale rho7 - [v = target] p_c_inv8 - (k8 inv_S)(sum_p78 - p_c_inv8)  (:245-256).
//
// This file holds the generic path (any dtype): row kernels over materialised logits, a tiled
// SIMT GEMM for z = h W, dh = dz W^T and dW = h^T dz, and the aligned copy of W used by the
// MFMA path (oace_mfma.hip).
#include <algorithm>

#include "oace_common.h"

namespace afa {

namespace {

template <typename A, typename T>
__device__ __forceinline__ A ld_as(const T* p, int64_t i) {
  if constexpr (std::is_same<T, __bf16>::value) return (A)(float)p[i];
  else if constexpr (std::is_same<T, _Float16>::value) return (A)(float)p[i];
  else return (A)p[i];
}
template <typename T, typename A>
__device__ __forceinline__ void st_as(T* p, int64_t i, A x) {
  if constexpr (std::is_same<T, __bf16>::value) p[i] = (__bf16)(float)x;
  else if constexpr (std::is_same<T, _Float16>::value) p[i] = (_Float16)(float)x;
  else p[i] = (T)x;
}

template <typename A>
__device__ __forceinline__ A wave_sum(A x) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m);
  return x;
}

// Sum over a 256-thread block; every thread gets the result.
template <typename A, int K>
__device__ __forceinline__ void block_sum(A (&x)[K], A* sh /* 4*K */) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < K; ++i) x[i] = wave_sum(x[i]);
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < K; ++i) sh[wave * K + i] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i) x[i] = (sh[i] + sh[K + i]) + (sh[2 * K + i] + sh[3 * K + i]);
}

}  // namespace

// One workgroup per row of z (row stride ldz): both passes, the target capture and the record.
template <typename ZT, typename A>
__global__ __launch_bounds__(256) void oace_rows_fwd_kernel(const ZT* z, int64_t ldz, int64_t V,
                                                            const int64_t* targets, A eps, A gamma, A inv_v,
                                                            A* rows) {
  __shared__ A sh[24];
  const int64_t row = blockIdx.x;
  const ZT* zr = z + row * ldz;
  A ss[1] = {A(0)};
  for (int64_t v = threadIdx.x; v < V; v += 256) {
    const A x = ld_as<A>(zr, v);
    ss[0] += x * x;
  }
  block_sum<A, 1>(ss, sh);
  const A tau = o_rsq<A>(ss[0] * inv_v + eps);
  A s[4] = {A(0), A(0), A(0), A(0)};
  for (int64_t v = threadIdx.x; v < V; v += 256) {
    const A x = ld_as<A>(zr, v) * tau;
    const Oct<A> o = octic(x);
    const A rn = o.r * x;
    s[0] += o.k8;
    s[1] += o.rho7;
    s[2] += rn * o.k8;
    s[3] += rn * o.rho7;
  }
  block_sum<A, 4>(s, sh + 4);
  if (threadIdx.x == 0) {
    const int64_t t = targets[row];
    A rho_t = A(0), rn_t = A(0);  // a target outside [0, V) leaves rho_t = 0 (loss = inf), as the reference
    if (t >= 0 && t < V) {
      const A x = ld_as<A>(zr, t) * tau;
      const Oct<A> o = octic(x);
      rho_t = o.rho;
      rn_t = o.r * x;
    }
    oace_finalize_row<A>(rows + row * OACE_ROW, tau, s[0], s[1], s[2], s[3], rho_t, rn_t, inv_v, gamma);
  }
}

// loss = mean of the per-row losses, in a fixed order.  One workgroup for up to MEAN_ROWS rows; more
// rows are first summed MEAN_ROWS at a time into the last (unused) field of each group's first
// record (one workgroup reads its records at the rate of one compute unit: the forward
// call on (134000, 1000) bf16 took 257 us with one, 114 us with groups).
constexpr int MEAN_ROWS = 4096;
template <typename A>
__global__ __launch_bounds__(256) void oace_mean_kernel(A* rows, int64_t N, int64_t stride, int field, A scale,
                                                        A* loss) {
  __shared__ A sh[4];
  A s[1] = {A(0)};
  const int64_t i0 = (int64_t)blockIdx.x * MEAN_ROWS, i1 = loss == nullptr && i0 + MEAN_ROWS < N ? i0 + MEAN_ROWS : N;
#pragma unroll 4
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) s[0] += rows[i * stride + field];
  block_sum<A, 1>(s, sh);
  if (threadIdx.x == 0) {
    if (loss != nullptr) *loss = s[0] / scale;
    else rows[i0 * OACE_ROW + OACE_ROW - 1] = s[0];
  }
}

// The row records of 16- and 32-bit logits: T threads per row, the row read once into registers as
// its 16-byte chunks (NCH per thread; NCH = 0 streams a longer row twice) and, where it starts or ends
// inside one, one element each of the first lanes.  Bound by the octic terms' VALU issue (about
// 20 instructions and two quarter-rate ones per 16-bit entry) just above its one HBM read:
// (2048, 50257) bf16, forward call with the mean 176 -> 64 us (3.2 TB/s; the two passes of 2-byte
// loads by one 256-thread workgroup per row took 171 of the 176), (1024, 48001) fp32 41 us (4.8 TB/s).
template <int DT, int T, int NCH>
__global__ __launch_bounds__(T < 256 ? 256 : T, 4) void oace_rows_fwd_vec_kernel(const void* z, int64_t ldz, int64_t N,
                                                                             int V, const int64_t* targets, float eps,
                                                                             float gamma, float inv_v, float* rows) {
  using R = RowChunk<DT>;
  constexpr int RPB = T < 256 ? 256 / T : 1;  // rows per workgroup
  constexpr int NW = T / 64;                  // waves per row
  __shared__ float sh[NW > 1 ? 5 * NW : 1];
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / T;
  if (row >= N) return;  // whole waves, and only where no barrier follows (one wave per row)
  const int tid = threadIdx.x % T, lane = threadIdx.x & 63, wave = tid >> 6;
  const char* zr = (const char*)z + row * ldz * R::ESZ;
  const RowSpan sp = R::span(zr, V);
  const int edge = R::edge(sp, V, tid);
  const u32x4_t* body = (const u32x4_t*)(zr + (int64_t)sp.head * R::ESZ);
  constexpr int NR = NCH > 0 ? NCH : 1;
  u32x4_t raw[NR];
  const float ve = edge >= 0 ? Elem<DT>::load(zr, edge) : 0.f;
  float ss = ve * ve;
  auto sq = [&](u32x4_t w) {
    float v[R::EPC];
    R::unpack(w, v);
#pragma unroll
    for (int i = 0; i < R::EPC; ++i) ss = __builtin_fmaf(v[i], v[i], ss);
  };
  if constexpr (NCH > 0) {
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const int c = tid + T * j;
      raw[j] = u32x4_t{0u, 0u, 0u, 0u};
      if (c < sp.body) raw[j] = body[c];
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      sq(raw[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    for (int c = tid; c < sp.body; c += T) sq(body[c]);
  }
  ss = wave_sum(ss);
  if constexpr (NW > 1) {
    if (lane == 0) sh[4 * NW + wave] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) ss += sh[4 * NW + w];
  }
  const float tau = o_rsq<float>(ss * inv_v + eps);
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  auto term = [&](float x) {
    float rho, rho7, r;
    octic7(x, rho, rho7, r);
    s[0] = __builtin_fmaf(rho7, rho, s[0]);
    s[1] += rho7;
    const float m = (r * x) * rho7;
    s[2] = __builtin_fmaf(m, rho, s[2]);
    s[3] += m;
  };
  auto eval = [&](u32x4_t w) {
    float v[R::EPC];
    R::unpack(w, v);
#pragma unroll
    for (int i = 0; i < R::EPC; ++i) term(v[i] * tau);
  };
  if constexpr (NCH > 0) {
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      asm("" : "+v"(raw[j]));  // unpack again here: the first pass's floats would take twice the registers
      if (tid + T * j < sp.body) eval(raw[j]);
      __builtin_amdgcn_sched_barrier(0);  // one chunk's terms live at a time
    }
  } else {
    for (int c = tid; c < sp.body; c += T) eval(body[c]);
  }
  if (edge >= 0) term(ve * tau);
#pragma unroll
  for (int q = 0; q < 4; ++q) s[q] = wave_sum(s[q]);
  if constexpr (NW > 1) {
    if (lane == 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) sh[q * NW + wave] = s[q];
    __syncthreads();
    if (tid != 0) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s[q] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) s[q] += sh[q * NW + w];
    }
  }
  if (tid == 0) {
    const int64_t t = targets[row];
    float rho_t = 0.f, rn_t = 0.f;  // a target outside [0, V) leaves rho_t = 0 (loss = inf), as the reference
    if (t >= 0 && t < V) {
      const float x = Elem<DT>::load(zr, t) * tau;
      const Oct<float> o = octic(x);
      rho_t = o.rho;
      rn_t = o.r * x;
    }
    oace_finalize_row<float>(rows + row * OACE_ROW, tau, s[0], s[1], s[2], s[3], rho_t, rn_t, inv_v, gamma);
  }
}

// dz of 16- and 32-bit logits: one wave per U * 64 whole chunks of a row, U 16-byte loads in flight per
// lane, and a row's first wave takes the elements before and after them, one to a lane.  The terms of
// every entry are formed without the target (the tau, c and sum factors folded into three row scalars);
// the one chunk that holds it is formed again with it.  A factor tau c that an infinite loss cotangent
// makes infinite is not folded, where it would meet itself as NaN, but multiplied on at the end, in code
// of its own: one more multiplication per entry cost 4 us at the size below.  HBM bound: (2048, 50257)
// bf16 157 -> 76 us (5.4 TB/s read and written), against 2-byte loads and stores before.  8 million bf16
// entries in rows of 10: 246 us, of 33: 103, of 65: 57 (350, 112 and 61 with a workgroup per row and
// 2-byte accesses).
template <int DT, int U>
__global__ __launch_bounds__(256) void oace_rows_bwd_vec_kernel(const void* z, int64_t ldz, int64_t N, int V,
                                                                const int64_t* targets, const float* rows,
                                                                const float* g_loss, float c0, void* dz,
                                                                int64_t lddz) {
  using R = RowChunk<DT>;
  const int lane = threadIdx.x & 63;
  const int spans = max(1, (V / R::EPC + 64 * U - 1) / (64 * U));
  const unsigned w = blockIdx.x * 4 + (threadIdx.x >> 6);  // below 2^26
  const int64_t row = w / (unsigned)spans;
  if (row >= N) return;
  const int span = (int)(w % (unsigned)spans);
  const char* zr = (const char*)z + row * ldz * R::ESZ;
  char* dr = (char*)dz + row * lddz * R::ESZ;
  const RowSpan sp = R::span(zr, V);
  const int edge = span == 0 ? R::edge(sp, V, lane) : -1;  // a row's first wave takes its ends
  const u32x4_t* zb = (const u32x4_t*)(zr + (int64_t)sp.head * R::ESZ);
  u32x4_t* db = (u32x4_t*)(dr + (int64_t)sp.head * R::ESZ);
  const int cb = span * (64 * U) + lane;
  u32x4_t raw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = cb + 64 * u;
    raw[u] = u32x4_t{0u, 0u, 0u, 0u};
    if (c < sp.body) raw[u] = zb[c];
  }
  const float ze = edge >= 0 ? Elem<DT>::load(zr, edge) : 0.f;
  const float* rec = rows + row * OACE_ROW;
  const float tau = rec[OACE_TAU], inv_S = rec[OACE_INV_S], pc = rec[OACE_PC_INV8];
  const float tau_c = tau * (c0 * (g_loss ? *g_loss : 1.f));
  const bool inf = __ballot(__builtin_isinf(tau_c)) != 0;  // the same in the whole wave: one row
  const float tc = inf ? 1.f : tau_c;
  const float scale = rec[OACE_S8] * inv_S;
  const float cs = tc * scale, cd = tc * (inv_S * (rec[OACE_SUM_P78] - pc)), cr = tc * rec[OACE_RADIAL];
  const int64_t t = targets[row];
  auto form = [&](auto times_tau_c) {
    auto term = [&](float v, float target) {
      const float x = v * tau;
      float rho, rho7, r;
      octic7(x, rho, rho7, r);
      const float b = rho7 * __builtin_fmaf(-cd, rho, cs) - target;
      const float o = __builtin_fmaf(r, b, -cr * x);
      return times_tau_c.value ? o * tau_c : o;
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = cb + 64 * u;
      if (c < sp.body) {
        const int e0 = sp.head + c * R::EPC;
        float v[R::EPC], o[R::EPC];
        R::unpack(raw[u], v);
#pragma unroll
        for (int i = 0; i < R::EPC; ++i) o[i] = term(v[i], 0.f);
        // the entry of this chunk that is the target (a target outside [0, V) is none)
        if (t >= e0 && t < e0 + R::EPC) {
#pragma unroll
          for (int i = 0; i < R::EPC; ++i)
            if (i == (int)(t - e0)) o[i] = term(v[i], tc * pc);
        }
        db[c] = R::pack(o);
      }
    }
    if (edge >= 0) Elem<DT>::store(dr, edge, term(ze, t == edge ? tc * pc : 0.f));
  };
  if (inf) form(std::true_type());
  else form(std::false_type());
}

// dz = tau c (r bracket - radial x) for every element of rows (grid.y = row), c = c0 * g.
template <typename ZT, typename OT, typename A>
__global__ __launch_bounds__(256) void oace_rows_bwd_kernel(const ZT* z, int64_t ldz, int64_t V,
                                                            const int64_t* targets, const A* rows,
                                                            const A* g_loss, A c0, OT* dz, int64_t lddz) {
  const int64_t row = blockIdx.y;
  const A* rec = rows + row * OACE_ROW;
  const A tau = rec[OACE_TAU], inv_S = rec[OACE_INV_S], S8 = rec[OACE_S8];
  const A pc = rec[OACE_PC_INV8], radial = rec[OACE_RADIAL];
  const A diff = rec[OACE_SUM_P78] - pc;
  const A scale = S8 * inv_S;
  const A c = c0 * (g_loss ? *g_loss : A(1));
  const int64_t t = targets[row];
  const ZT* zr = z + row * ldz;
  OT* dr = dz + row * lddz;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < V; v += (int64_t)gridDim.x * 256) {
    const A x = ld_as<A>(zr, v) * tau;
    const Oct<A> o = octic(x);
    const A bracket = scale * o.rho7 - (v == t ? pc : A(0)) - (o.k8 * inv_S) * diff;
    st_as<OT, A>(dr, v, tau * (c * (o.r * bracket - radial * x)));
  }
}

// C[m][n] (+)= sum_k A[m][k] B[k][n] with arbitrary element strides; 64x64 tiles, 4x4 per thread.
template <typename TA, typename TB, typename TC, typename A>
__global__ __launch_bounds__(256) void oace_gemm_generic_kernel(int64_t M, int64_t Nn, int64_t K, const TA* a,
                                                                int64_t sam, int64_t sak, const TB* b,
                                                                int64_t sbk, int64_t sbn, TC* c, int64_t scm,
                                                                int64_t scn, int accumulate) {
  __shared__ A as[16][65];
  __shared__ A bs[16][65];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t m0 = (int64_t)blockIdx.y * 64, n0 = (int64_t)blockIdx.x * 64;
  A acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = A(0);
  for (int64_t k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = threadIdx.x + 256 * i;  // 1024 = 16 x 64
      const int kk = e >> 6, mm = e & 63;
      const int64_t gm = m0 + mm, gn = n0 + mm, gk = k0 + kk;
      as[kk][mm] = (gm < M && gk < K) ? ld_as<A>(a, gm * sam + gk * sak) : A(0);
      bs[kk][mm] = (gn < Nn && gk < K) ? ld_as<A>(b, gk * sbk + gn * sbn) : A(0);
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      A av[4], bv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        av[i] = as[kk][ty + 16 * i];
        bv[i] = bs[kk][tx + 16 * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += av[i] * bv[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t gm = m0 + ty + 16 * i, gn = n0 + tx + 16 * j;
      if (gm < M && gn < Nn) {
        const int64_t off = gm * scm + gn * scn;
        const A prev = accumulate ? ld_as<A>(c, off) : A(0);
        st_as<TC, A>(c, off, prev + acc[i][j]);
      }
    }
}

// y(k, v) = x[k V + v] for a dense rows x V accumulator, written with strides (sk, sv).
template <typename A, typename E>
__global__ __launch_bounds__(256) void oace_convert_kernel(const A* x, int64_t rows, int64_t V, E* y, int64_t sk,
                                                           int64_t sv) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < rows * V; i += (int64_t)gridDim.x * 256) {
    const int64_t k = i / V, v = i - k * V;
    st_as<E, A>(y, k * sk + v * sv, x[i]);
  }
}

// Rows of 2-byte elements at any alignment copied to 16-byte aligned rows.  A workgroup copies spans of
// 2048 columns of a row, 8 per thread: the two aligned 16-byte chunks that hold them, shifted by the
// row's offset (uniform over the workgroup).  Chunks that would reach outside the matrix go element by
// element.  HBM bound: 768 x 50257 takes 25.6 us, 6.0 TB/s of its 154 MB.
__global__ __launch_bounds__(256) void oace_align_rows16_kernel(const unsigned short* x, int64_t rows, int64_t cols,
                                                                int64_t ldx, unsigned short* y, int64_t ldy,
                                                                int spans) {
  for (int64_t it = blockIdx.x; it < rows * spans; it += gridDim.x) {
    const int64_t r = it / spans;
    const int64_t c = (it % spans) * 2048 + 8 * threadIdx.x;
    if (c >= ldy) continue;
    const unsigned short* src = x + r * ldx + c;
    const int sh = __builtin_amdgcn_readfirstlane((int)(((uintptr_t)(x + r * ldx) & 15u) >> 1));  // elements
    const unsigned short* al = src - sh;
    u32x4_t o = {0u, 0u, 0u, 0u};
    if (c + 8 <= cols && al >= x && al + 16 <= x + (rows - 1) * ldx + cols) {
      const u32x4_t lo = *(const u32x4_t*)al, hi = *(const u32x4_t*)(al + 8);
      const unsigned w[9] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3], 0u};
      auto pick = [&](auto q) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          o[u] = (sh & 1) ? __builtin_amdgcn_alignbit(w[u + q.value + 1], w[u + q.value], 16) : w[u + q.value];
      };
      switch (sh >> 1) {
        case 0: pick(std::integral_constant<int, 0>()); break;
        case 1: pick(std::integral_constant<int, 1>()); break;
        case 2: pick(std::integral_constant<int, 2>()); break;
        default: pick(std::integral_constant<int, 3>()); break;
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c + u < cols) o[u >> 1] |= (unsigned)src[u] << (16 * (u & 1));
    }
    *(u32x4_t*)(y + r * ldy + c) = o;
  }
}

// ------------------------------------------------------------------------------ launchers
namespace {

template <int DT>
struct OTypes;
template <>
struct OTypes<AFA_F32> { typedef float E; typedef float A; };
template <>
struct OTypes<AFA_BF16> { typedef __bf16 E; typedef float A; };
template <>
struct OTypes<AFA_F16> { typedef _Float16 E; typedef float A; };
template <>
struct OTypes<AFA_F64> { typedef double E; typedef double A; };

template <typename TA, typename TB, typename TC, typename A>
void gemm_generic(int64_t M, int64_t N, int64_t K, const TA* a, int64_t sam, int64_t sak, const TB* b, int64_t sbk,
                  int64_t sbn, TC* c, int64_t scm, int64_t scn, bool accumulate, hipStream_t st) {
  const dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
  hipLaunchKernelGGL((oace_gemm_generic_kernel<TA, TB, TC, A>), grid, dim3(256), 0, st, M, N, K, a, sam, sak, b, sbk,
                     sbn, c, scm, scn, accumulate ? 1 : 0);
}

// W element (k, v) strides for a layout.
void w_strides(const OaceArgs& a, int64_t& sk, int64_t& sv) {
  if (a.w_layout == OACE_W_DV) {
    sk = a.ldw;
    sv = 1;
  } else {
    sk = 1;
    sv = a.ldw;
  }
}

// Threads per row and 16-byte chunks per thread by the row's length: the fewest threads that hold
// the row in at most 4 chunks each, then 512 threads with up to 25 (100 registers of a 128-register
// wave, so two workgroups still share a compute unit and one loads while the other evaluates), or half as
// many where 256 or 512 threads hold the row so: a chunk a thread does not have costs its turns all the
// same (calls of 4096 rows of 2100 chunks bf16 69 us in 25s, 50 in 13s; 2048 of 6282 66 and 64, fp32 43 and
// 38).  Longer rows are streamed.
template <int DT>
void rows_fwd_vec(const OaceArgs& a, const void* z, int64_t ldz, void* rows, hipStream_t st) {
  const int nch = (int)a.V / RowChunk<DT>::EPC;  // whole chunks of the best start
  const float inv_v = (float)(1.0 / (double)a.V);
#define OACE_ROWS_VEC(T, NCH)                                                                                       \
  hipLaunchKernelGGL((oace_rows_fwd_vec_kernel<DT, T, NCH>), dim3((unsigned)((a.N * T + (T < 256 ? 255 : T - 1)) /  \
                     (T < 256 ? 256 : T))), dim3(T < 256 ? 256 : T), 0, st, z, ldz, a.N, (int)a.V, a.targets,       \
                     (float)a.eps, (float)a.gamma, inv_v, (float*)rows)
  if (a.N >= (1 << 23)) OACE_ROWS_VEC(64, 0);  // 512 threads per row would pass 2^32 in one launch
  else if (nch <= 64) OACE_ROWS_VEC(64, 1);
  else if (nch <= 128) OACE_ROWS_VEC(64, 2);
  else if (nch <= 256) OACE_ROWS_VEC(64, 4);
  else if (nch <= 512) OACE_ROWS_VEC(256, 2);
  else if (nch <= 1024) OACE_ROWS_VEC(256, 4);
  else if (nch <= 2048) OACE_ROWS_VEC(512, 4);
  else if (nch <= 256 * 13) OACE_ROWS_VEC(256, 13);
  else if (nch <= 512 * 13) OACE_ROWS_VEC(512, 13);
  else if (nch <= 512 * 25) OACE_ROWS_VEC(512, 25);
  else OACE_ROWS_VEC(512, 0);
#undef OACE_ROWS_VEC
}

// z and dz rows must start at the same offset from a 16-byte boundary (the chunks of the one are
// then the chunks of the other); false: the caller takes the element-wise kernel.
template <int DT>
bool rows_bwd_vec(const OaceArgs& a, const void* rows, void* dz, float c0, hipStream_t st) {
  using R = RowChunk<DT>;
  if ((((uintptr_t)a.h ^ (uintptr_t)dz) & 15u) != 0) return false;
  const int nch = std::max(1, (int)a.V / R::EPC);  // whole chunks of the best start
  // four chunks per lane when that still leaves four waves per SIMD, else one
  const bool wide = a.N * ((nch + 255) / 256) >= 4096;
  const int64_t waves = a.N * (int64_t)((nch + (wide ? 255 : 63)) / (wide ? 256 : 64));
  if (waves >= (int64_t(1) << 26)) return false;  // 2^32 threads
  const dim3 grid((unsigned)((waves + 3) / 4));
  if (wide)
    hipLaunchKernelGGL((oace_rows_bwd_vec_kernel<DT, 4>), grid, dim3(256), 0, st, a.h, a.ldh, a.N, (int)a.V, a.targets,
                       (const float*)rows, (const float*)a.g_loss, c0, dz, a.ldh);
  else
    hipLaunchKernelGGL((oace_rows_bwd_vec_kernel<DT, 1>), grid, dim3(256), 0, st, a.h, a.ldh, a.N, (int)a.V, a.targets,
                       (const float*)rows, (const float*)a.g_loss, c0, dz, a.ldh);
  return true;
}

template <int DT>
hipError_t rows_fwd_dt(const OaceArgs& a, const void* z, int64_t ldz, bool z_is_acc, void* rows, hipStream_t st) {
  typedef typename OTypes<DT>::E E;
  typedef typename OTypes<DT>::A A;
  if constexpr (DT == AFA_F64) {
    hipLaunchKernelGGL((oace_rows_fwd_kernel<E, A>), dim3((unsigned)a.N), dim3(256), 0, st, (const E*)z, ldz, a.V,
                       a.targets, a.eps, a.gamma, 1.0 / (double)a.V, (A*)rows);
  } else if (z_is_acc) {
    rows_fwd_vec<AFA_F32>(a, z, ldz, rows, st);
  } else {
    rows_fwd_vec<DT>(a, z, ldz, rows, st);
  }
  return hipGetLastError();
}

unsigned bwd_grid_x(int64_t V) { return (unsigned)std::min<int64_t>((V + 255) / 256, 64); }

}  // namespace

size_t oace_generic_chunk_rows(int dtype, int64_t N, int64_t V) {
  const size_t acc = dtype == AFA_F64 ? 8 : 4;
  const size_t cap = (size_t)256 << 20;
  int64_t r = (int64_t)(cap / ((size_t)V * acc));
  return (size_t)std::max<int64_t>(1, std::min<int64_t>(N, r));
}

size_t oace_generic_workspace(int dtype, int64_t N, int64_t d, int64_t V, bool backward) {
  const size_t acc = dtype == AFA_F64 ? 8 : 4;
  const int64_t R = (int64_t)oace_generic_chunk_rows(dtype, N, V);
  size_t b = (size_t)R * V * acc;  // z / dz chunk
  b = (b + 255) & ~(size_t)255;
  if (backward && R < N) b += (size_t)d * V * acc;  // dW accumulator
  return b;
}

template <int DT>
static hipError_t linear_fwd_generic_dt(const OaceArgs& a, void* rows, void* ws, hipStream_t st) {
  typedef typename OTypes<DT>::E E;
  typedef typename OTypes<DT>::A A;
  const int64_t R = (int64_t)oace_generic_chunk_rows(DT, a.N, a.V);
  A* z = (A*)ws;
  int64_t sk, sv;
  w_strides(a, sk, sv);
  for (int64_t r0 = 0; r0 < a.N; r0 += R) {
    const int64_t rn = std::min(R, a.N - r0);
    gemm_generic<E, E, A, A>(rn, a.V, a.d, (const E*)a.h + r0 * a.ldh, a.ldh, 1, (const E*)a.w, sk, sv, z, a.V, 1,
                             false, st);
    OaceArgs sub = a;
    sub.N = rn;
    sub.targets = a.targets + r0;
    hipError_t e = rows_fwd_dt<DT>(sub, z, a.V, true, (A*)rows + r0 * OACE_ROW, st);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

template <int DT>
static hipError_t linear_bwd_generic_dt(const OaceArgs& a, const void* rows, void* ws, hipStream_t st) {
  typedef typename OTypes<DT>::E E;
  typedef typename OTypes<DT>::A A;
  const int64_t R = (int64_t)oace_generic_chunk_rows(DT, a.N, a.V);
  A* z = (A*)ws;
  const bool chunked = R < a.N;
  A* dwacc = chunked ? (A*)((char*)ws + (((size_t)R * a.V * sizeof(A) + 255) & ~(size_t)255)) : nullptr;
  int64_t sk, sv;
  w_strides(a, sk, sv);
  const A c0 = (A)(8.0 * a.gamma / (double)a.N);
  for (int64_t r0 = 0; r0 < a.N; r0 += R) {
    const int64_t rn = std::min(R, a.N - r0);
    const E* hc = (const E*)a.h + r0 * a.ldh;
    gemm_generic<E, E, A, A>(rn, a.V, a.d, hc, a.ldh, 1, (const E*)a.w, sk, sv, z, a.V, 1, false, st);
    hipLaunchKernelGGL((oace_rows_bwd_kernel<A, A, A>), dim3(bwd_grid_x(a.V), (unsigned)rn), dim3(256), 0, st,
                       (const A*)z, a.V, a.V, a.targets + r0, (const A*)rows + r0 * OACE_ROW, (const A*)a.g_loss, c0,
                       z, a.V);
    // dh (rn x d) = dz (rn x V) W^T: element (n, k) = sum_v dz[n][v] W(k, v)
    gemm_generic<A, E, E, A>(rn, a.d, a.V, z, a.V, 1, (const E*)a.w, sv, sk, (E*)a.dh + r0 * a.d, a.d, 1, false, st);
    // dW(k, v) = sum_n h[n][k] dz[n][v], stored in W's layout
    if (chunked)
      gemm_generic<E, A, A, A>(a.d, a.V, rn, hc, 1, a.ldh, z, a.V, 1, dwacc, a.V, 1, r0 > 0, st);
    else
      gemm_generic<E, A, E, A>(a.d, a.V, rn, hc, 1, a.ldh, z, a.V, 1, (E*)a.dw, sk, sv, false, st);
  }
  if (chunked)  // dW from the accumulator, in the element type and W's layout
    hipLaunchKernelGGL((oace_convert_kernel<A, E>), dim3((unsigned)std::min<int64_t>((a.d * a.V + 255) / 256, 65536)),
                       dim3(256), 0, st, (const A*)dwacc, a.d, a.V, (E*)a.dw, sk, sv);
  return hipGetLastError();
}

hipError_t oace_linear_fwd_generic(int dtype, const OaceArgs& a, void* rows, void* ws, hipStream_t st) {
  hipError_t e;
  switch (dtype) {
    case AFA_F32: e = linear_fwd_generic_dt<AFA_F32>(a, rows, ws, st); break;
    case AFA_BF16: e = linear_fwd_generic_dt<AFA_BF16>(a, rows, ws, st); break;
    case AFA_F16: e = linear_fwd_generic_dt<AFA_F16>(a, rows, ws, st); break;
    default: e = linear_fwd_generic_dt<AFA_F64>(a, rows, ws, st); break;
  }
  if (e != hipSuccess) return e;
  return oace_mean_launch(dtype, rows, a.N, a.loss, st);
}

hipError_t oace_linear_bwd_generic(int dtype, const OaceArgs& a, const void* rows, void* ws, hipStream_t st) {
  switch (dtype) {
    case AFA_F32: return linear_bwd_generic_dt<AFA_F32>(a, rows, ws, st);
    case AFA_BF16: return linear_bwd_generic_dt<AFA_BF16>(a, rows, ws, st);
    case AFA_F16: return linear_bwd_generic_dt<AFA_F16>(a, rows, ws, st);
    default: return linear_bwd_generic_dt<AFA_F64>(a, rows, ws, st);
  }
}

template <typename A>
static hipError_t mean_launch(A* rows, int64_t N, A* loss, hipStream_t st) {
  if (N <= MEAN_ROWS) {
    hipLaunchKernelGGL((oace_mean_kernel<A>), dim3(1), dim3(256), 0, st, rows, N, (int64_t)OACE_ROW, (int)OACE_LOSS,
                       (A)N, loss);
    return hipGetLastError();
  }
  const int64_t groups = (N + MEAN_ROWS - 1) / MEAN_ROWS;
  hipLaunchKernelGGL((oace_mean_kernel<A>), dim3((unsigned)groups), dim3(256), 0, st, rows, N, (int64_t)OACE_ROW,
                     (int)OACE_LOSS, A(1), (A*)nullptr);
  hipLaunchKernelGGL((oace_mean_kernel<A>), dim3(1), dim3(256), 0, st, rows, groups, (int64_t)OACE_ROW * MEAN_ROWS,
                     (int)OACE_ROW - 1, (A)N, loss);
  return hipGetLastError();
}

hipError_t oace_mean_launch(int dtype, void* rows, int64_t N, void* loss, hipStream_t st) {
  if (dtype == AFA_F64) return mean_launch((double*)rows, N, (double*)loss, st);
  return mean_launch((float*)rows, N, (float*)loss, st);
}

hipError_t oace_rows_z(const OaceArgs& a, const float* z, int64_t ldz, void* rows, hipStream_t st) {
  rows_fwd_vec<AFA_F32>(a, z, ldz, rows, st);
  return hipGetLastError();
}

hipError_t oace_softmax_fwd_launch(int dtype, const OaceArgs& a, void* rows, hipStream_t st) {
  hipError_t e;
  switch (dtype) {
    case AFA_F32: e = rows_fwd_dt<AFA_F32>(a, a.h, a.ldh, false, rows, st); break;
    case AFA_BF16: e = rows_fwd_dt<AFA_BF16>(a, a.h, a.ldh, false, rows, st); break;
    case AFA_F16: e = rows_fwd_dt<AFA_F16>(a, a.h, a.ldh, false, rows, st); break;
    default: e = rows_fwd_dt<AFA_F64>(a, a.h, a.ldh, false, rows, st); break;
  }
  if (e != hipSuccess) return e;
  return oace_mean_launch(dtype, rows, a.N, a.loss, st);
}

template <int DT>
static hipError_t softmax_bwd_dt(const OaceArgs& a, const void* rows, void* dz, hipStream_t st) {
  typedef typename OTypes<DT>::E E;
  typedef typename OTypes<DT>::A A;
  const A c0 = (A)(8.0 * a.gamma / (double)a.N);
  if constexpr (DT != AFA_F64)
    if (rows_bwd_vec<DT>(a, rows, dz, c0, st)) return hipGetLastError();
  hipLaunchKernelGGL((oace_rows_bwd_kernel<E, E, A>), dim3(bwd_grid_x(a.V), (unsigned)a.N), dim3(256), 0, st,
                     (const E*)a.h, a.ldh, a.V, a.targets, (const A*)rows, (const A*)a.g_loss, c0, (E*)dz, a.ldh);
  return hipGetLastError();
}

hipError_t oace_softmax_bwd_launch(int dtype, const OaceArgs& a, const void* rows, void* dz, hipStream_t st) {
  switch (dtype) {
    case AFA_F32: return softmax_bwd_dt<AFA_F32>(a, rows, dz, st);
    case AFA_BF16: return softmax_bwd_dt<AFA_BF16>(a, rows, dz, st);
    case AFA_F16: return softmax_bwd_dt<AFA_F16>(a, rows, dz, st);
    default: return softmax_bwd_dt<AFA_F64>(a, rows, dz, st);
  }
}

hipError_t oace_align_rows16(const void* x, int64_t rows, int64_t cols, int64_t ldx, void* y, int64_t ldy,
                             hipStream_t st) {
  if (ldy % 8 != 0 || ldy < cols || ((uintptr_t)y & 15u) != 0) return hipErrorInvalidValue;
  const int64_t spans = (ldy + 2047) / 2048;
  const unsigned blocks = (unsigned)std::min<int64_t>(rows * spans, int64_t(1) << 23);  // below 2^32 threads
  hipLaunchKernelGGL(oace_align_rows16_kernel, dim3(blocks), dim3(256), 0, st,
                     (const unsigned short*)x, rows, cols, ldx, (unsigned short*)y, ldy, (int)spans);
  return hipGetLastError();
}

}  // namespace afa
