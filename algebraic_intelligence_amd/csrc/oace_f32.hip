// Fused Linear + OACE head for fp32 on the bf16 matrix cores (src/kernels/pallas_oace.py:59-293).
//
// Every fp32 operand is split once into three bf16 planes, x = hi + mid + lo exactly (three
// round-to-nearest pieces hold 24 bits), and a product x y is taken as the six terms of at least
// 2^-16 relative weight,
//   lo_x hi_y + hi_x lo_y + mid_x mid_y + mid_x hi_y + hi_x mid_y + hi_x hi_y,
// accumulated in fp32 by v_mfma_f32_32x32x16_bf16: the scheme of a six-pass bf16 product at full
// fp32 precision, which the reference asks of its fp32 dots (Precision.HIGHEST).  The dropped terms
// are together below 2^-23 of the product, one rounding serves 16 of them where an fp32 fma chain rounds
// each, and the bf16 pipes have 16 times the rate of the fp32 ones: 2.7 times after six passes.
// Error against 64 bits (2-norm; SIMT fp32 GEMM it replaces in brackets), 512 x 288 x 50257: dh
// 4.1e-7 (4.0e-6), dW 2.6e-7 (4.1e-7); lower at every size tried from 4 x 32 x 100 to
// 1024 x 1024 x 50257.  Forward + backward of the 512 rows, tied: 12.1 -> 0.434 ms; 1024 x 1024 x 50257 20.4 ->
// 1.84 ms (the two backward GEMMs at 1.3 PFLOP/s of bf16 products, the rate a library bf16 GEMM
// reaches on the device); 4 x 32 x 100 54 -> 51 us, so small problems take this path too.
//
// Pipeline: planes of h and W (contraction-padded with zeros) -> z = h W (fp32, kept while it
// takes at most 256 MB, else in row chunks) -> row records (oace.hip) -> backward: dz of every
// logit, split as it is formed -> dh = dz W^T (contraction split into parts) and dW = h^T dz.
// W stays in its own layout: an operand's planes are read either contraction-contiguous or
// row-contiguous (ds_read_tr16_b64), so no transposed copy is made.
//
// GEMM tile: 64 WM (m) x 64 WN (n), 8 waves of 64 x 64 (2 x 2 blocks of 32x32x16 MFMAs), 32 of the
// contraction per step.  A step loads the three planes of both operands (72 KB) and takes 48 MFMAs
// per wave for them, so the loads of the next step have about 3000 cycles to arrive in the other
// half of the LDS: two stages, one barrier per step.
#include <algorithm>

#include "oace_common.h"

namespace afa {

namespace {

constexpr int XK = 32;  // contraction per step

template <int WM>
struct XCfg {
  static constexpr int WN = 8 / WM;
  static constexpr int TM = 64 * WM, TN = 64 * WN;
  static constexpr int A_PLANE = TM * XK * 2, B_PLANE = TN * XK * 2;
  static constexpr int STAGE = 3 * (A_PLANE + B_PLANE);
  static constexpr int A_LOADS = A_PLANE / (512 * 16), B_LOADS = B_PLANE / (512 * 16);
  static constexpr int LDS = 2 * STAGE;
  static constexpr int PITCH = TM + 4;  // staged output row in floats
  static_assert(TN * PITCH * 4 <= LDS, "the staged output tile must fit the ring");
};

typedef __attribute__((ext_vector_type(4))) short x_s16x4_t;
typedef __attribute__((address_space(3))) x_s16x4_t x_lds_s16x4_t;

struct XArgs {
  const unsigned short* a;  // planes of A, m x K: plane p at a + p * ap
  int64_t lda, ap;
  int am;
  const unsigned short* b;  // planes of B, n x K
  int64_t ldb, bp;
  int bn;
  int K, kpart, parts, mt, nt;  // K and kpart multiples of XK
  float* out;                   // D[n][m] at out[part * part_stride + n * ldo + m]
  int64_t ldo, part_stride;
  int accumulate;  // D is added to what out holds
  const float* g_loss;  // the backward's products: the loss cotangent (nullable) and its factor
  float c0;
};

// Byte offset in a plane's stage of (tile row, logical 16-byte chunk): contraction-contiguous (KC)
// tiles hold 64-byte rows of the operand, row-contiguous (MC) tiles the 32 contraction rows.
template <bool MC, int R>
__device__ __forceinline__ int x_off(int row, int c) {
  if constexpr (MC) return row * (R * 2) + ((c ^ ((row & 3) << 2)) << 4);
  else return row * 64 + ((c ^ ((row >> 2) & 3)) << 4);
}

// Byte offset from the tile's origin in memory of the 16-byte slot s of a stage; operand rows and
// 8-column chunks past the extent read the last valid one (their results are not stored).
template <bool MC, int R>
__device__ __forceinline__ uint32_t x_src(int s, int r0, int rows, int64_t ld) {
  if constexpr (MC) {
    constexpr int CPR = R / 8;
    const int row = s / CPR, c = (s % CPR) ^ ((row & 3) << 2);
    const int col = min(r0 + 8 * c, ((rows + 7) >> 3) * 8 - 8) - r0;
    return (uint32_t)(((int64_t)row * ld + col) * 2);
  } else {
    const int row = s >> 2, c = (s & 3) ^ ((row >> 2) & 3);
    return (uint32_t)(((int64_t)(min(r0 + row, rows - 1) - r0) * ld + 8 * c) * 2);
  }
}

// MFMA operand: 32 operand rows from 32 blk, contraction rows 16 kk + 8 g .. + 7 of a plane.
template <bool MC, int R>
__device__ __forceinline__ bf16x8_t x_frag(const unsigned char* st, int blk, int kk, int lane) {
  const int l32 = lane & 31, g = lane >> 5;
  u32x4_t f;
  if constexpr (MC) {
    const int l16 = lane & 15, m16 = (lane >> 4) & 1;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int row = 16 * kk + 8 * g + 4 * hh + (l16 >> 2);
      const int c = blk * 4 + m16 * 2 + ((l16 & 3) >> 1);
      const unsigned char* p = st + x_off<true, R>(row, c) + (l16 & 1) * 8;
      const x_s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((x_lds_s16x4_t*)p);
      const u32x2_t w = __builtin_bit_cast(u32x2_t, v);
      f[2 * hh] = w[0];
      f[2 * hh + 1] = w[1];
    }
  } else {
    f = *(const u32x4_t*)(st + x_off<false, R>(blk * 32 + l32, 2 * kk + g));
  }
  return __builtin_bit_cast(bf16x8_t, f);
}

// hi, mid, lo of a pair of values, packed; infinities and NaN stay whole in hi (mid = lo = 0), and
// the values between the largest bf16 and the largest fp32 are rounded towards zero in hi.
__device__ __forceinline__ void split3(float x0, float x1, unsigned& hi, unsigned& mid, unsigned& lo) {
  constexpr float kMax = 3.38953138925153547590e38f;  // the largest finite bf16
  const bool f0 = __builtin_fabsf(x0) <= 3.402823466e38f, f1 = __builtin_fabsf(x1) <= 3.402823466e38f;
  const float c0 = f0 ? __builtin_fminf(__builtin_fmaxf(x0, -kMax), kMax) : x0;
  const float c1 = f1 ? __builtin_fminf(__builtin_fmaxf(x1, -kMax), kMax) : x1;
  hi = pack_bf16(c0, c1);
  const float r0 = f0 ? x0 - bf16_lo(hi) : 0.f, r1 = f1 ? x1 - bf16_hi(hi) : 0.f;
  mid = pack_bf16(r0, r1);
  lo = pack_bf16(r0 - bf16_lo(mid), r1 - bf16_hi(mid));
}

}  // namespace

// Planes of x (rows x cols fp32, row stride ld) as (prows x ldp) bf16 each, zeros outside x; a
// second matrix in the same launch (the hidden rows beside the weights).  One thread per 8 columns.
struct SplitJob {
  const float* x;
  int64_t rows, cols, ld, prows, ldp;
  unsigned short* out;
};
__global__ __launch_bounds__(256) void oace_f32_split_kernel(SplitJob j0, SplitJob j1, int64_t n0, int64_t n1) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n0 + n1) return;
  const bool second = i >= n0;
  const SplitJob j = second ? j1 : j0;
  if (second) i -= n0;
  const int64_t cpr = j.ldp / 8, r = i / cpr, c = (i - r * cpr) * 8;
  float v[8];
  const float* src = j.x + r * j.ld + c;
  if (r < j.rows && c + 8 <= j.cols && ((uintptr_t)src & 15u) == 0) {
    const f32x4_t a = *(const f32x4_t*)src, b = *(const f32x4_t*)(src + 4);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v[u] = a[u];
      v[4 + u] = b[u];
    }
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = r < j.rows && c + u < j.cols ? src[u] : 0.f;
  }
  u32x4_t p[3];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    unsigned hi, mid, lo;
    split3(v[2 * u], v[2 * u + 1], hi, mid, lo);
    p[0][u] = hi;
    p[1][u] = mid;
    p[2][u] = lo;
  }
  const int64_t plane = j.prows * j.ldp;
#pragma unroll
  for (int q = 0; q < 3; ++q) *(u32x4_t*)(j.out + q * plane + r * j.ldp + c) = p[q];
}

// dz of the fp32 logits (rows r0 .. of the call), split into planes as it is formed: (prows x ldz)
// each, zeros outside rows x V.  One wave per 512 entries of a row, 8 per lane.  HBM bound: 4 bytes
// read and 6 written per logit.
__global__ __launch_bounds__(256) void oace_f32_dz_kernel(const float* z, int64_t ldz, int64_t N, int64_t prows, int V,
                                                          const int64_t* targets, const float* rows,
                                                          const float* g_loss, float c0, unsigned short* dz) {
  const int lane = threadIdx.x & 63;
  const int spans = (int)((ldz + 511) / 512);
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t row = w / spans;
  const int c = (int)(w % spans) * 512 + 8 * lane;
  if (row >= prows || c >= ldz) return;
  float o[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) o[u] = 0.f;
  if (row < N && c < V) {
    const float* zr = z + row * ldz + c;
    const f32x4_t za = *(const f32x4_t*)zr, zb = *(const f32x4_t*)(zr + 4);
    const float* rec = rows + row * OACE_ROW;
    const float tau = rec[OACE_TAU], inv_S = rec[OACE_INV_S], pc = rec[OACE_PC_INV8];
    // an infinite factor is multiplied on at the end, as in oace_rows_bwd_vec_kernel
    const float tau_c = tau * (c0 * (g_loss ? *g_loss : 1.f));
    const bool inf = __ballot(__builtin_isinf(tau_c)) != 0;
    const float tc = inf ? 1.f : tau_c;
    const float cs = tc * (rec[OACE_S8] * inv_S), cd = tc * (inv_S * (rec[OACE_SUM_P78] - pc));
    const float cr = tc * rec[OACE_RADIAL];
    const int64_t t = targets[row] - c;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float x = (u < 4 ? za[u] : zb[u - 4]) * tau;
      float rho, rho7, r;
      octic7(x, rho, rho7, r);
      const float b = rho7 * __builtin_fmaf(-cd, rho, cs) - (t == u && c + u < V ? tc * pc : 0.f);
      o[u] = c + u < V ? __builtin_fmaf(r, b, -cr * x) : 0.f;
    }
    if (inf) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c + u < V) o[u] *= tau_c;
    }
  }
  u32x4_t p[3];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    unsigned hi, mid, lo;
    split3(o[2 * u], o[2 * u + 1], hi, mid, lo);
    p[0][u] = hi;
    p[1][u] = mid;
    p[2][u] = lo;
  }
  const int64_t plane = prows * ldz;
#pragma unroll
  for (int q = 0; q < 3; ++q) *(u32x4_t*)(dz + q * plane + row * ldz + c) = p[q];
}

template <bool A_MC, bool B_MC, int WM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void oace_f32_gemm_kernel(const XArgs a) {
  using C = XCfg<WM>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int l32 = lane & 31, g = lane >> 5;

  // Work items (part, m tile, n tile) with the n tiles of one m tile side by side, dealt to the
  // XCDs in equal contiguous runs (block b runs on XCD b mod 8): neighbours share an operand slice
  // in that XCD's L2.
  const int items = a.parts * a.mt * a.nt, ipx = (items + 7) / 8;
  const int j = blockIdx.x >> 3, item = (blockIdx.x & 7) * ipx + j;
  if (j >= ipx || item >= items) return;
  const int part = item / (a.mt * a.nt), tile = item % (a.mt * a.nt);
  const int m0 = (tile / a.nt) * C::TM, n0 = (tile % a.nt) * C::TN;
  const int k_lo = part * a.kpart, T = (min(k_lo + a.kpart, a.K) - k_lo) / XK;

  uint32_t aoff[C::A_LOADS], boff[C::B_LOADS];
#pragma unroll
  for (int i = 0; i < C::A_LOADS; ++i) aoff[i] = x_src<A_MC, C::TM>(512 * i + tid, m0, a.am, a.lda);
#pragma unroll
  for (int i = 0; i < C::B_LOADS; ++i) boff[i] = x_src<B_MC, C::TN>(512 * i + tid, n0, a.bn, a.ldb);
  const char* abase = (const char*)(a.a + (A_MC ? (int64_t)k_lo * a.lda + m0 : (int64_t)m0 * a.lda + k_lo));
  const char* bbase = (const char*)(a.b + (B_MC ? (int64_t)k_lo * a.ldb + n0 : (int64_t)n0 * a.ldb + k_lo));
  const int64_t astep = A_MC ? (int64_t)XK * a.lda * 2 : XK * 2;
  const int64_t bstep = B_MC ? (int64_t)XK * a.ldb * 2 : XK * 2;
  // An infinite cotangent leaves no finite dz.  Its zero lower planes, and the signs of the other operand's,
  // would make NaN of every infinite product: all planes are then taken from hi, whose six equal
  // products are infinite, or NaN, as the fp32 product is.
  const bool inf = a.g_loss != nullptr && __builtin_isinf(a.c0 * *a.g_loss);
  const int64_t ap = inf ? 0 : a.ap, bp = inf ? 0 : a.bp;
  auto issue = [&](int t) {
    unsigned char* st = lds + (t & 1) * C::STAGE;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const char* ab = abase + t * astep + p * ap * 2;
#pragma unroll
      for (int i = 0; i < C::A_LOADS; ++i) lds_dma16(ab, aoff[i], st + p * C::A_PLANE + (512 * i + wave * 64) * 16);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const char* bb = bbase + t * bstep + p * bp * 2;
#pragma unroll
      for (int i = 0; i < C::B_LOADS; ++i)
        lds_dma16(bb, boff[i], st + 3 * C::A_PLANE + p * C::B_PLANE + (512 * i + wave * 64) * 16);
    }
  };

  f32x16_t acc[2][2];
#pragma unroll
  for (int vb = 0; vb < 2; ++vb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[vb][nb][e] = 0.f;

  issue(0);
  for (int t = 0; t < T; ++t) {
    // step t's tiles have arrived (every wave's), and the other stage, read in step t-1, is free
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    __syncthreads();
    if (t + 1 < T) issue(t + 1);
    const unsigned char* st = lds + (t & 1) * C::STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t af[3][2], bf[3][2];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int vb = 0; vb < 2; ++vb) af[p][vb] = x_frag<A_MC, C::TM>(st + p * C::A_PLANE, wm * 2 + vb, kk, lane);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          bf[p][nb] = x_frag<B_MC, C::TN>(st + 3 * C::A_PLANE + p * C::B_PLANE, wn * 2 + nb, kk, lane);
      }
      // smallest terms first
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int vb = 0; vb < 2; ++vb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            acc[vb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[PA[q]][vb], bf[PB[q]][nb], acc[vb][nb], 0, 0, 0);
    }
  }
  __syncthreads();

  // ---- epilogue: element e of acc[vb][nb] is m = m0 + 64 wm + 32 vb + 8 (e >> 2) + 4 g + (e & 3),
  // n = n0 + 64 wn + 32 nb + l32; the tile goes through the idle ring, then out in whole rows.
  float* stg = (float*)lds;
#pragma unroll
  for (int vb = 0; vb < 2; ++vb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4_t w;
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = acc[vb][nb][4 * q + u];
        *(f32x4_t*)(stg + (wn * 64 + nb * 32 + l32) * C::PITCH + wm * 64 + vb * 32 + q * 8 + 4 * g) = w;
      }
  __syncthreads();
  float* out = a.out + part * a.part_stride;
  if ((((uintptr_t)out | (uintptr_t)(a.ldo * 4)) & 15u) == 0) {
    for (int idx = tid; idx < C::TN * C::TM / 4; idx += 512) {
      const int r = idx / (C::TM / 4), c = (idx % (C::TM / 4)) * 4;
      if (n0 + r < a.bn && m0 + c < a.am) {
        f32x4_t w = *(const f32x4_t*)(stg + r * C::PITCH + c);
        float* o = out + (int64_t)(n0 + r) * a.ldo + m0 + c;
        if (m0 + c + 4 <= a.am) {
          if (a.accumulate) w += *(const f32x4_t*)o;
          *(f32x4_t*)o = w;
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (m0 + c + u < a.am) o[u] = a.accumulate ? o[u] + w[u] : w[u];
        }
      }
    }
  } else {
    for (int idx = tid; idx < C::TN * C::TM; idx += 512) {
      const int r = idx / C::TM, c = idx % C::TM;
      if (n0 + r < a.bn && m0 + c < a.am) {
        float* o = out + (int64_t)(n0 + r) * a.ldo + m0 + c;
        const float w = stg[r * C::PITCH + c];
        *o = a.accumulate ? *o + w : w;
      }
    }
  }
}

// out (rows x cols, row stride ldo) = the sum over parts, in part order, of partials of row stride
// ldp (a multiple of 4); one thread per 4 columns.
__global__ __launch_bounds__(256) void oace_f32_sum_kernel(const float* part, int parts, int64_t stride, int64_t rows,
                                                           int cols, int64_t ldp, float* out, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t cpr = ldp / 4, r = i / cpr;
  const int c = (int)(i - r * cpr) * 4;
  if (r >= rows) return;
  const float* p = part + r * ldp + c;
  f32x4_t s = *(const f32x4_t*)p;
#pragma unroll 4
  for (int q = 1; q < parts; ++q) s += *(const f32x4_t*)(p + q * stride);
  float* o = out + r * ldo + c;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (c + u < cols) o[u] = s[u];
}

// ------------------------------------------------------------------------------ host side
namespace {

size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }
int64_t up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

// Logits held at a time, 4 bytes each; their dz, 6 bytes each (three planes), come on top, and within it
// when the caller asks for none to be kept (OACE_FLAG_RECOMPUTE_Z).
constexpr size_t Z_MAX_BYTES = (size_t)256 << 20;
constexpr size_t W_MAX_BYTES = (size_t)8 << 30;    // planes of the weights
constexpr int DH_ITEMS = 256;  // workgroups of dh's split contraction: fixed, so the sum order is

struct Plan {
  int64_t dp, Vp, R, Rp;  // padded d_model, vocabulary, rows per chunk (and padded)
  size_t w, h, z, dz, part, total;
  int dh_parts, dh_kpart;
  bool dh_wide;  // dh's tiles are 256 model features x 128 rows instead of 128 x 256
  int64_t wr, wc;  // rows and row length of a weight plane
};

int64_t tiles(int64_t m, int64_t n, int wm) {
  return ((m + 64 * wm - 1) / (64 * wm)) * ((n + 64 * (8 / wm) - 1) / (64 * (8 / wm)));
}
// The tile orientation that covers m x n with fewer tiles (equal areas), 256 x 128 on a tie.
bool wide_m(int64_t m, int64_t n) { return tiles(m, n, 4) <= tiles(m, n, 2); }

bool keeps_z(const OaceArgs& a) { return (a.flags & OACE_FLAG_RECOMPUTE_Z) == 0; }
int64_t rows_that_fit(const OaceArgs& a) { return (int64_t)(Z_MAX_BYTES / ((size_t)up(a.V, 64) * (keeps_z(a) ? 4 : 10))); }

Plan plan_of(const OaceArgs& a) {
  Plan p;
  p.dp = up(a.d, 64);
  p.Vp = up(a.V, 64);
  const int64_t fit = rows_that_fit(a);  // at least XK: oace_f32_supported
  p.R = std::min<int64_t>(a.N, fit >= 256 ? fit / 256 * 256 : fit / XK * XK);
  p.Rp = up(p.R, XK);
  p.wr = a.w_layout == OACE_W_DV ? p.dp : p.Vp;
  p.wc = a.w_layout == OACE_W_DV ? p.Vp : p.dp;
  p.w = al256((size_t)p.wr * p.wc * 6);
  p.h = al256((size_t)up(a.N, XK) * p.dp * 6);
  p.z = al256((size_t)p.R * p.Vp * 4);
  p.dz = al256((size_t)p.Rp * p.Vp * 6);
  p.dh_wide = wide_m(a.d, p.R);
  const int64_t t = tiles(a.d, p.R, p.dh_wide ? 4 : 2), steps = p.Vp / XK;
  const int64_t parts = std::max<int64_t>(1, std::min<int64_t>(DH_ITEMS / t, steps / 8));
  p.dh_kpart = (int)(((steps + parts - 1) / parts) * XK);
  p.dh_parts = (int)((p.Vp + p.dh_kpart - 1) / p.dh_kpart);
  p.part = p.dh_parts > 1 ? al256((size_t)p.dh_parts * p.R * p.dp * 4) : 0;
  p.total = p.w + p.h + p.z + p.dz + p.part;
  return p;
}

template <bool A_MC, bool B_MC>
hipError_t x_gemm(XArgs g, bool wide, hipStream_t st) {
  const int tm = wide ? 256 : 128, tn = wide ? 128 : 256;
  g.mt = (g.am + tm - 1) / tm;
  g.nt = (g.bn + tn - 1) / tn;
  const unsigned grid = 8u * (unsigned)((g.parts * g.mt * g.nt + 7) / 8);
  if (wide) hipLaunchKernelGGL((oace_f32_gemm_kernel<A_MC, B_MC, 4>), dim3(grid), dim3(512), 0, st, g);
  else hipLaunchKernelGGL((oace_f32_gemm_kernel<A_MC, B_MC, 2>), dim3(grid), dim3(512), 0, st, g);
  return hipGetLastError();
}

hipError_t split_launch(SplitJob a, SplitJob b, hipStream_t st) {
  const int64_t n0 = a.prows * a.ldp / 8, n1 = b.prows * b.ldp / 8;
  if (n0 + n1 == 0) return hipSuccess;
  hipLaunchKernelGGL(oace_f32_split_kernel, dim3((unsigned)((n0 + n1 + 255) / 256)), dim3(256), 0, st, a, b, n0, n1);
  return hipGetLastError();
}

SplitJob w_job(const OaceArgs& a, const Plan& p, unsigned short* out) {
  const bool dv = a.w_layout == OACE_W_DV;
  return SplitJob{(const float*)a.w, dv ? a.d : a.V, dv ? a.V : a.d, a.ldw, p.wr, p.wc, out};
}
SplitJob h_job(const OaceArgs& a, const Plan& p, unsigned short* out) {
  return SplitJob{(const float*)a.h, a.N, a.d, a.ldh, up(a.N, XK), p.dp, out};
}

// z (rn x V) of rows r0 .. r0 + rn from the planes, D[n][v].
hipError_t z_gemm(const OaceArgs& a, const Plan& p, const unsigned short* wp, const unsigned short* hp, int64_t r0,
                  int64_t rn, float* z, hipStream_t st) {
  XArgs g = {};
  g.a = wp;
  g.lda = p.wc;
  g.ap = p.wr * p.wc;
  g.am = (int)a.V;
  g.b = hp + r0 * p.dp;
  g.ldb = p.dp;
  g.bp = up(a.N, XK) * p.dp;
  g.bn = (int)rn;
  g.K = g.kpart = (int)p.dp;
  g.parts = 1;
  g.out = z;
  g.ldo = p.Vp;
  return a.w_layout == OACE_W_DV ? x_gemm<true, false>(g, wide_m(a.V, rn), st)
                                 : x_gemm<false, false>(g, wide_m(a.V, rn), st);
}

}  // namespace

bool oace_f32_supported(const OaceArgs& a) {
  // 32-bit lane offsets (256 rows of a plane) and 32-bit extents; a chunk is at least one step of rows
  if (a.N > (1 << 28) || rows_that_fit(a) < XK || a.d >= (1 << 22)) return false;
  return (size_t)up(a.d, 64) * up(a.V, 64) * 6 <= W_MAX_BYTES;
}

size_t oace_f32_workspace(const OaceArgs& a) { return oace_f32_supported(a) ? plan_of(a).total : 0; }

hipError_t oace_linear_fwd_f32(const OaceArgs& a, void* rows, void* ws, hipStream_t st) {
  const Plan p = plan_of(a);
  unsigned short* wp = (unsigned short*)ws;
  unsigned short* hp = (unsigned short*)((char*)ws + p.w);
  float* z = (float*)((char*)ws + p.w + p.h);
  hipError_t e = split_launch(w_job(a, p, wp), h_job(a, p, hp), st);
  for (int64_t r0 = 0; r0 < a.N && e == hipSuccess; r0 += p.R) {
    const int64_t rn = std::min(p.R, a.N - r0);
    if ((e = z_gemm(a, p, wp, hp, r0, rn, z, st)) != hipSuccess) break;
    OaceArgs sub = a;
    sub.N = rn;
    sub.targets = a.targets + r0;
    e = oace_rows_z(sub, z, p.Vp, (float*)rows + r0 * OACE_ROW, st);
  }
  if (e != hipSuccess) return e;
  return oace_mean_launch(AFA_F32, rows, a.N, a.loss, st);
}

hipError_t oace_linear_bwd_f32(const OaceArgs& a, const void* rows, void* ws, hipStream_t st) {
  const Plan p = plan_of(a);
  unsigned short* wp = (unsigned short*)ws;
  unsigned short* hp = (unsigned short*)((char*)ws + p.w);
  float* z = (float*)((char*)ws + p.w + p.h);
  unsigned short* dz = (unsigned short*)((char*)ws + p.w + p.h + p.z);
  float* part = (float*)((char*)ws + p.w + p.h + p.z + p.dz);
  // what the forward left in the workspace: the weights' planes, and, with the hidden rows
  // unchanged too, those of h and (when all rows were one chunk) the logits
  const bool w_ready = (a.flags & (OACE_FLAG_WT_READY | OACE_FLAG_Z_READY)) != 0;
  const bool h_ready = (a.flags & OACE_FLAG_Z_READY) != 0;
  SplitJob wj = w_job(a, p, wp), hj = h_job(a, p, hp);
  if (w_ready) wj.prows = 0;
  if (h_ready) hj.prows = 0;
  hipError_t e = split_launch(wj, hj, st);
  if (e != hipSuccess) return e;
  const bool z_ready = h_ready && p.R == a.N && keeps_z(a);
  const float c0 = (float)(8.0 * a.gamma / (double)a.N);
  const int64_t h_plane = up(a.N, XK) * p.dp;
  for (int64_t r0 = 0; r0 < a.N; r0 += p.R) {
    const int64_t rn = std::min(p.R, a.N - r0), rp = up(rn, XK);
    if (!z_ready && (e = z_gemm(a, p, wp, hp, r0, rn, z, st)) != hipSuccess) return e;
    const int64_t waves = rp * ((p.Vp + 511) / 512);
    hipLaunchKernelGGL(oace_f32_dz_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, (const float*)z, p.Vp,
                       rn, rp, (int)a.V, a.targets + r0, (const float*)rows + r0 * OACE_ROW, (const float*)a.g_loss,
                       c0, dz);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // dh (rn x d) = dz W^T: D[n][k], contraction over the vocabulary
    XArgs g = {};
    g.a = wp;
    g.lda = p.wc;
    g.ap = p.wr * p.wc;
    g.am = (int)a.d;
    g.b = dz;
    g.ldb = p.Vp;
    g.bp = rp * p.Vp;
    g.bn = (int)rn;
    g.K = (int)p.Vp;
    g.kpart = p.dh_kpart;
    g.parts = p.dh_parts;
    float* dh = (float*)a.dh + r0 * a.d;
    g.out = g.parts > 1 ? part : dh;
    g.ldo = g.parts > 1 ? p.dp : a.d;
    g.part_stride = rn * p.dp;
    g.g_loss = (const float*)a.g_loss;
    g.c0 = c0;
    e = a.w_layout == OACE_W_DV ? x_gemm<false, false>(g, p.dh_wide, st) : x_gemm<true, false>(g, p.dh_wide, st);
    if (e != hipSuccess) return e;
    if (g.parts > 1) {
      const int64_t n = rn * p.dp / 4;
      hipLaunchKernelGGL(oace_f32_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const float*)part,
                         g.parts, g.part_stride, rn, (int)a.d, p.dp, dh, a.d);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    // dW over this chunk's rows, in W's layout: D[k][v] = sum_n dz[n][v] h[n][k], or D[v][k]
    XArgs w = {};
    const bool dv = a.w_layout == OACE_W_DV;
    w.a = dv ? dz : hp + r0 * p.dp;
    w.lda = dv ? p.Vp : p.dp;
    w.ap = dv ? rp * p.Vp : h_plane;
    w.am = (int)(dv ? a.V : a.d);
    w.b = dv ? hp + r0 * p.dp : dz;
    w.ldb = dv ? p.dp : p.Vp;
    w.bp = dv ? h_plane : rp * p.Vp;
    w.bn = (int)(dv ? a.d : a.V);
    w.K = w.kpart = (int)rp;
    w.parts = 1;
    w.g_loss = g.g_loss;
    w.c0 = c0;
    w.out = (float*)a.dw;
    w.ldo = a.ldw;
    w.accumulate = r0 > 0;
    if ((e = x_gemm<true, true>(w, wide_m(w.am, w.bn), st)) != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace afa
