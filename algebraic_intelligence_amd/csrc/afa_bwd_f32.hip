// fp32 ("HIGHEST") analytical AFA backward on the bf16 matrix cores, head_dim 32, 48, 64, 96 and 128.
// Contract of tiled_afa_backward (src/kernels/pallas_afa.py:437-522) with fp32 operands, as the
// generic fp32 kernel computes it:
//   E_i = sum_d g_id out_id;  s = (q_i . k_j) * scale;  r = rsqrt(1 + s^2);  w = rho(s)^8 / d_i;
//   ds = 8 scale r w (g_i . v_j - E_i);  dq_i += ds_ij k_j;  dk_j += ds_ij q_i;  dv_j += w_ij g_i,
// with rho^8 by the two-branch form; only the order of the fp32 additions differs.  Every product
// is six bf16 plane products of exactly split operands (afa_f32_split.h), as in the forward.
//
// Three launches, no atomics:
//   * afa_bwd_f32_prep_kernel: E_i and 1/d_i per row into the workspace;
//   * afa_bwd_f32_dq_kernel: one lane per query (32 per wave, 128 per workgroup), the layout of
//     the fp32 forward: the planes of q and g stay in registers; S^T = K Q^T and dP^T = V g^T read
//     K / V rows from LDS; dQ^T += K^T dS^T reads K's columns (ds_read_tr16_b64) and takes the
//     dS^T accumulator, split in registers, as its B operand;
//   * afa_bwd_f32_dkdv_kernel: one lane per key, the mirror image: k and v planes in registers,
//     S = Q K^T and dP = g V^T from Q / g rows in LDS, then dV^T += g^T W and dK^T += Q^T dS.
// Tiles of 32 rows are staged through registers, rotated and split there, into double-buffered LDS
// (one barrier per tile); dq and dk are rotated back through R^T before they are stored.  Waves that met
// an operand the planes do not hold take their rows again in plain fp32 (afa_f32_split.h).
#include "afa_common.h"
#include "afa_f32_split.h"
#include "afa_launch.h"

namespace afa {

namespace {

constexpr int FKT = 32;  // rows per tile

// rho(s)^8 (two-branch: rho(|s|)^8, reciprocal for s < 0) and r = rsqrt(1 + s^2)
__device__ __forceinline__ float frho8r(float s, float& r) {
  const float a = __builtin_fabsf(s);
  const float t = __builtin_fmaf(a, a, 1.0f);
  r = __builtin_amdgcn_rsqf(t);
  const float rho = __builtin_fmaf(t, r, a);
  const float p2 = rho * rho;
  const float p4 = p2 * p2;
  const float p8 = p4 * p4;
  return s < 0.0f ? __builtin_amdgcn_rcpf(p8) : p8;
}

// Rotate the gradients of features m .. m+3 (accumulator elements e0 .. e0+3: two (even, odd)
// pairs) back through R^T with the fp32 tables at row `pos`.
template <int D>
__device__ __forceinline__ void f_unrotate4(f32x16_t& acc, int e0, const float* rc, const float* rs, int pos,
                                            int m) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int64_t t = (int64_t)pos * (D / 2) + m / 2 + p;
    const float c = rc[t], s = rs[t];
    const float x0 = acc[e0 + 2 * p], x1 = acc[e0 + 2 * p + 1];
    acc[e0 + 2 * p] = c * x0 + s * x1;
    acc[e0 + 2 * p + 1] = c * x1 - s * x0;
  }
}

}  // namespace

// E_i = sum_d g_id out_id and 1/d_i: 8 lanes per row, 16-byte chunks.  E at e_ws[row], 1/d at
// e_ws[B H L + row].
__global__ __launch_bounds__(256) void afa_bwd_f32_prep_kernel(const GenArgs a) {
  const int64_t rows = (int64_t)a.B * a.H * a.L;
  const int64_t row = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
  const int sub = threadIdx.x & 7;
  float part = 0.f;
  if (row < rows) {
    const float* gr = (const float*)a.g + row * a.D;
    const float* orow = (const float*)a.out_in + row * a.D;
    for (int c = sub; c < a.D / 4; c += 8) {
      const f32x4_t gw = *(const f32x4_t*)(gr + 4 * c);
      const f32x4_t ow = *(const f32x4_t*)(orow + 4 * c);
      part += gw[0] * ow[0] + gw[1] * ow[1] + gw[2] * ow[2] + gw[3] * ow[3];
    }
  }
  part += __shfl_xor(part, 1);
  part += __shfl_xor(part, 2);
  part += __shfl_xor(part, 4);
  if (row < rows && sub == 0) {
    ((float*)a.e_ws)[row] = part;
    ((float*)a.e_ws)[rows + row] = 1.0f / ((const float*)a.dtot)[row];
  }
}

// ------------------------------------------------------------------------------ dQ
// Bound by the sum of matrix and vector issue, as the forward.  dQ + dK/dV with prep, against
// v_mfma_f32_32x32x2_f32: B=32 H=4 L=1024 D=64 causal rotary 798 -> 472 us, B=1 H=8 L=4096 D=64 1271 ->
// 746 us, B=2 H=8 L=2048 D=128 causal rotary 1323 -> 813 us, B=16 H=6 L=512 D=48 205 -> 130 us; error
// of dq, dk and dv against 64 bits 0.75 to 0.85 of what it was at every size.
// Waves per SIMD by the register planes and accumulators of each kernel (dK/dV at head_dim 64 holds 96
// registers of planes and 64 of accumulators: one wave with 318 of 512).
constexpr int f32_dq_waves(int d) { return d <= 64 ? 2 : 1; }
constexpr int f32_dkdv_waves(int d) { return d <= 32 ? 2 : 1; }

// A 32-row tile of two matrices (x rotated when ROT) in flight from memory to their LDS planes.
template <int D, bool ROT>
struct F32Stage {
  using X = F32Tile<D>;
  static constexpr int JOBS = (FKT * (D / 4) + 255) / 256;  // float4 of each matrix per thread
  static constexpr bool RAGGED = FKT * (D / 4) % 256 != 0;  // head_dim 48: the last job is half a workgroup's
  f32x4_t x[JOBS], y[JOBS];
  float c[JOBS][2], s[JOBS][2];

  static __device__ __forceinline__ int row(int i) { return (int)(threadIdx.x + 256 * i) / (D / 4); }
  static __device__ __forceinline__ int col(int i) { return 4 * ((int)(threadIdx.x + 256 * i) % (D / 4)); }

  // rows from `r0` of two contiguous (L, D) matrices; rows past L load the last one (finite data of
  // masked scores)
  __device__ __forceinline__ void load(const float* xp, const float* yp, const float* rc, const float* rs, int r0,
                                       int L) {
    const int last = L - 1 - r0;
    const char* xt = (const char*)(xp + (int64_t)r0 * D);
    const char* yt = (const char*)(yp + (int64_t)r0 * D);
    const char* ct = (const char*)(rc + (int64_t)r0 * (D / 2));
    const char* st = (const char*)(rs + (int64_t)r0 * (D / 2));
#pragma unroll
    for (int i = 0; i < JOBS; ++i) {
      const uint32_t off = (uint32_t)(min(row(i), last) * D + col(i)) * 4u;
      x[i] = *(const f32x4_t*)(xt + off);
      y[i] = *(const f32x4_t*)(yt + off);
      if constexpr (ROT) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          c[i][p] = ((const float*)(ct + off / 2))[p];
          s[i][p] = ((const float*)(st + off / 2))[p];
        }
      }
    }
  }
  __device__ __forceinline__ void store(unsigned short* xl, unsigned short* yl) const {
#pragma unroll
    for (int i = 0; i < JOBS; ++i) {
      if (RAGGED && row(i) >= FKT) continue;
      const int at = X::at(row(i), col(i));
      unsigned w[3][2];
      const f32x4_t xr = ROT ? f32_rotate4(x[i], c[i], s[i]) : x[i];
      split3_rne(xr[0], xr[1], w[0][0], w[1][0], w[2][0]);
      split3_rne(xr[2], xr[3], w[0][1], w[1][1], w[2][1]);
      X::put(xl, at, w);
      split3_rne(y[i][0], y[i][1], w[0][0], w[1][0], w[2][0]);
      split3_rne(y[i][2], y[i][3], w[0][1], w[1][1], w[2][1]);
      X::put(yl, at, w);
    }
  }
  // zero the padding features of both buffers of both matrices, once (read as operand rows)
  static __device__ __forceinline__ void pad(unsigned short (*xl)[3 * X::PLANE], unsigned short (*yl)[3 * X::PLANE]) {
    if constexpr (D % 32 != 0) {
      for (int e = threadIdx.x; e < 2 * 3 * FKT * 4; e += 256) {
        const int r = (e >> 2) % FKT, pl = (e / (4 * FKT)) % 3, buf = e / (12 * FKT);
        const int at = pl * X::PLANE + X::at(r, D + 4 * (e & 3));
        *(u32x2_t*)&xl[buf][at] = u32x2_t{0u, 0u};
        *(u32x2_t*)&yl[buf][at] = u32x2_t{0u, 0u};
      }
    }
  }
};

// Planes of one row's features 16 kk + 8 g .. + 7 (rotated when ROT), zeros for rows past L.
template <int D, bool ROT>
__device__ __forceinline__ void f32_row_planes(const float* rows, const float* rc, const float* rs, int row, int L,
                                               int g, u32x4_t (&f)[3][D / 16]) {
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const int d0 = 16 * kk + 8 * g;
    f32x4_t x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (row < L) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        x[hh] = *(const f32x4_t*)(rows + (int64_t)row * D + d0 + 4 * hh);
        if constexpr (ROT) {
          const int64_t t = (int64_t)row * (D / 2) + d0 / 2 + 2 * hh;
          x[hh] = f32_rotate4(x[hh], rc + t, rs + t);
        }
      }
    }
    split8(x[0], x[1], f[0][kk], f[1][kk], f[2][kk]);
  }
}

template <int D, bool ROT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_dq_waves(D), f32_dq_waves(D))))
void afa_bwd_f32_dq_kernel(const GenArgs a) {
  using X = F32Tile<D>;
  constexpr int NK = D / 16, NDB = (D + 31) / 32;
  __shared__ __attribute__((aligned(16))) unsigned short ks[2][3 * X::PLANE];
  __shared__ __attribute__((aligned(16))) unsigned short vs[2][3 * X::PLANE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int L = a.L, vlen = a.valid_len, BH = a.B * a.H;
  int bh, qblk;
  block_item(blockIdx.x, BH, (L + 127) / 128, a.causal, bh, qblk);
  const int q0_wg = qblk * 128, q0_w = q0_wg + wave * 32;
  const int qi = q0_w + l32;
  const int kend_wg = a.causal ? min(vlen, min(L, q0_wg + 128)) : vlen;
  const int kend_w = a.causal ? min(vlen, q0_w + 32) : vlen;
  const int ntiles = (kend_wg + FKT - 1) / FKT;
  const int64_t base = (int64_t)bh * L * D;
  const float* kp = (const float*)a.k + base;
  const float* vp = (const float*)a.v + base;
  const float* rc = (const float*)a.rc;
  const float* rs = (const float*)a.rs;
  const float scale = (float)a.scale;
  const float c8 = 8.0f * scale;

  F32Stage<D, ROT> stage;
  if (ntiles > 0) stage.load(kp, vp, rc, rs, 0, L);
  u32x4_t qf[3][NK], gf[3][NK];
  f32_row_planes<D, ROT>((const float*)a.q + base, rc, rs, qi, L, g, qf);
  f32_row_planes<D, false>((const float*)a.g + base, nullptr, nullptr, qi, L, g, gf);
  const int64_t rows = (int64_t)BH * L;
  const float ei = qi < L ? ((const float*)a.e_ws)[(int64_t)bh * L + qi] : 0.f;
  const float invd = qi < L ? ((const float*)a.e_ws)[rows + (int64_t)bh * L + qi] : 0.f;

  f32x16_t dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) dq[db][e] = 0.f;

  F32Stage<D, ROT>::pad(ks, vs);
  if (ntiles > 0) stage.store(ks[0], vs[0]);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) stage.load(kp, vp, rc, rs, (t + 1) * FKT, L);
    const int key0 = t * FKT;
    if (key0 < kend_w && q0_w < L) {
      const unsigned short* kt = ks[t & 1];
      const unsigned short* vt = vs[t & 1];
      f32x16_t st, pt;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        st[e] = 0.f;
        pt[e] = 0.f;
      }
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        u32x4_t kf[3], vf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          kf[p] = X::row_frag(kt + p * X::PLANE, kk, lane);
          vf[p] = X::row_frag(vt + p * X::PLANE, kk, lane);
        }
        st = mma_planes(kf, qf[0][kk], qf[1][kk], qf[2][kk], st);
        pt = mma_planes(vf, gf[0][kk], gf[1][kk], gf[2][kk], pt);
      }
      const bool need_mask = (a.causal && key0 + 31 > q0_w) || key0 + 31 >= vlen || q0_w + 31 >= L;
      float ds[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float rr;
        const float w = frho8r(st[e] * scale, rr) * invd;
        ds[e] = c8 * rr * w * (pt[e] - ei);
      }
      if (need_mask) {
        asm volatile("" ::: "memory");  // kept a branch on the wave-uniform test
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = key0 + 8 * (e >> 2) + 4 * g + (e & 3);
          const bool keep = key < vlen && qi < L && (!a.causal || key <= qi);
          ds[e] = keep ? ds[e] : 0.f;
        }
      }
      u32x4_t pk[3][2];
      split_acc(ds, pk);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4_t kf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) kf[p] = X::col_frag(kt + p * X::PLANE, db, kk, lane);
          dq[db] = mma_planes(kf, pk[0][kk], pk[1][kk], pk[2][kk], dq[db]);
        }
    }
    // the buffer of tile t+1 was last read in tile t-1, before the previous barrier
    if (t + 1 < ntiles) stage.store(ks[(t + 1) & 1], vs[(t + 1) & 1]);
    __syncthreads();
  }

  if (f32_any_nan(dq)) {
    const float* gp = (const float*)a.g + base;
    const float* qp = (const float*)a.q + base;
    F32Look look;
    look.rows<D>(qp + (int64_t)q0_w * D, D, min(32, L - q0_w));
    look.rows<D>(gp + (int64_t)q0_w * D, D, min(32, L - q0_w));
    look.rows<D>(kp, D, kend_w);
    look.rows<D>(vp, D, kend_w);
    look.big |= __builtin_isinf(ei);
    if (look.redo()) {
      f32x4_t qo[D / 8], go[D / 8];
      f32_half_row<D, ROT>(qp + (int64_t)min(qi, L - 1) * D, rc, rs, min(qi, L - 1), qo);
      f32_half_row<D, false>(gp + (int64_t)min(qi, L - 1) * D, nullptr, nullptr, 0, go);
      f32_clear(dq);
#pragma unroll 1
      for (int j = 0; j < kend_w; ++j) {
        f32x4_t kr[D / 8], vr[D / 8];
        f32_half_row<D, ROT>(kp + (int64_t)j * D, rc, rs, j, kr);
        f32_half_row<D, false>(vp + (int64_t)j * D, nullptr, nullptr, 0, vr);
        const float s = f32_half_dot(qo, kr) * scale, p = f32_half_dot(go, vr);
        float rr;
        const float w = frho8r(s, rr) * invd;
        // a masked key's ds is 0, and its infinite entries are NaN, as in the tiles
        f32_half_axpy(!a.causal || j <= qi ? c8 * rr * w * (p - ei) : 0.f, kr, dq);
      }
    }
  }

  if (qi < L) {
    float* op = (float*)a.out + base + (int64_t)qi * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const int m = db * 32 + 8 * e4 + 4 * g;  // features m .. m+3 (two rotation pairs)
        if (D % 32 == 0 || m < D) {
          if constexpr (ROT) f_unrotate4<D>(dq[db], 4 * e4, rc, rs, qi, m);
          f32x4_t w;
#pragma unroll
          for (int u = 0; u < 4; ++u) w[u] = dq[db][4 * e4 + u];
          *(f32x4_t*)(op + m) = w;
        }
      }
  }
}

// ------------------------------------------------------------------------------ dK, dV
template <int D, bool ROT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_dkdv_waves(D), f32_dkdv_waves(D))))
void afa_bwd_f32_dkdv_kernel(const GenArgs a) {
  using X = F32Tile<D>;
  constexpr int NK = D / 16, NDB = (D + 31) / 32;
  __shared__ __attribute__((aligned(16))) unsigned short qs[2][3 * X::PLANE];
  __shared__ __attribute__((aligned(16))) unsigned short gs[2][3 * X::PLANE];
  __shared__ __attribute__((aligned(16))) float es[2][2 * FKT];  // E, then 1/d of the tile's rows

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int L = a.L, vlen = a.valid_len, BH = a.B * a.H;
  int bh, kblk;
  // heaviest first: for causal grids the low key blocks see the most queries
  block_item(blockIdx.x, BH, (L + 127) / 128, 0, bh, kblk);
  const int k0_wg = kblk * 128, k0_w = k0_wg + wave * 32;
  const int kj = k0_w + l32;
  const bool wave_live = k0_w < L && k0_w < vlen;
  const int t0 = a.causal ? k0_wg / FKT : 0;
  const int ntiles = (L + FKT - 1) / FKT;
  const int64_t base = (int64_t)bh * L * D;
  const float* qp = (const float*)a.q + base;
  const float* gp = (const float*)a.g + base;
  const float* rc = (const float*)a.rc;
  const float* rs = (const float*)a.rs;
  const float* ep = (const float*)a.e_ws + (int64_t)bh * L;
  const float* ip = (const float*)a.e_ws + (int64_t)BH * L + (int64_t)bh * L;
  const float scale = (float)a.scale;
  const float c8 = 8.0f * scale;

  F32Stage<D, ROT> stage;
  float ex = 0.f;
  auto load = [&](int t) {
    stage.load(qp, gp, rc, rs, t * FKT, L);
    if (tid < 2 * FKT) {
      const int row = t * FKT + (tid & (FKT - 1));
      ex = row < L ? (tid < FKT ? ep : ip)[row] : 0.f;
    }
  };
  auto store = [&](int buf) {
    stage.store(qs[buf], gs[buf]);
    if (tid < 2 * FKT) es[buf][tid] = ex;
  };
  if (t0 < ntiles) load(t0);
  u32x4_t kf[3][NK], vf[3][NK];
  f32_row_planes<D, ROT>((const float*)a.k + base, rc, rs, kj, L, g, kf);
  f32_row_planes<D, false>((const float*)a.v + base, nullptr, nullptr, kj, L, g, vf);

  f32x16_t dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dk[db][e] = 0.f;
      dv[db][e] = 0.f;
    }

  F32Stage<D, ROT>::pad(qs, gs);
  if (t0 < ntiles) store(t0 & 1);
  __syncthreads();
  for (int t = t0; t < ntiles; ++t) {
    if (t + 1 < ntiles) load(t + 1);
    const int i0 = t * FKT;  // first query of the tile
    const bool live = wave_live && i0 < L && (!a.causal || i0 + 31 >= k0_w);
    if (live) {
      const unsigned short* qt = qs[t & 1];
      const unsigned short* gt = gs[t & 1];
      const float* et = es[t & 1];
      f32x16_t st, pt;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        st[e] = 0.f;
        pt[e] = 0.f;
      }
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        u32x4_t qa[3], ga[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          qa[p] = X::row_frag(qt + p * X::PLANE, kk, lane);
          ga[p] = X::row_frag(gt + p * X::PLANE, kk, lane);
        }
        st = mma_planes(qa, kf[0][kk], kf[1][kk], kf[2][kk], st);
        pt = mma_planes(ga, vf[0][kk], vf[1][kk], vf[2][kk], pt);
      }
      const bool need_mask = (a.causal && i0 < k0_w + 31) || k0_w + 31 >= vlen || i0 + 31 >= L;
      float w[16], ds[16];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        // queries 8 e4 + 4 g .. + 3 of the tile: their E and 1/d
        const f32x4_t ei = *(const f32x4_t*)(et + 8 * e4 + 4 * g), iv = *(const f32x4_t*)(et + FKT + 8 * e4 + 4 * g);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = 4 * e4 + u;
          float rr;
          w[e] = frho8r(st[e] * scale, rr) * iv[u];
          ds[e] = c8 * rr * w[e] * (pt[e] - ei[u]);
        }
      }
      if (need_mask) {
        asm volatile("" ::: "memory");  // kept a branch on the wave-uniform test
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int i = i0 + 8 * (e >> 2) + 4 * g + (e & 3);
          const bool keep = kj < vlen && i < L && (!a.causal || kj <= i);
          w[e] = keep ? w[e] : 0.f;
          ds[e] = keep ? ds[e] : 0.f;
        }
      }
      u32x4_t pk[3][2];
      split_acc(w, pk);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4_t f[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) f[p] = X::col_frag(gt + p * X::PLANE, db, kk, lane);
          dv[db] = mma_planes(f, pk[0][kk], pk[1][kk], pk[2][kk], dv[db]);
        }
      split_acc(ds, pk);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4_t f[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) f[p] = X::col_frag(qt + p * X::PLANE, db, kk, lane);
          dk[db] = mma_planes(f, pk[0][kk], pk[1][kk], pk[2][kk], dk[db]);
        }
    }
    if (t + 1 < ntiles) store((t + 1) & 1);
    __syncthreads();
  }

  if (f32_any_nan(dk) || f32_any_nan(dv)) {
    const float* kp = (const float*)a.k + base;
    const float* vp = (const float*)a.v + base;
    const int i0 = a.causal ? k0_w : 0;  // a NaN: the wave is live, k0_w < L
    F32Look look;
    look.rows<D>(kp + (int64_t)k0_w * D, D, min(32, L - k0_w));
    look.rows<D>(vp + (int64_t)k0_w * D, D, min(32, L - k0_w));
    look.rows<D>(qp + (int64_t)i0 * D, D, L - i0);
    look.rows<D>(gp + (int64_t)i0 * D, D, L - i0);
#pragma unroll 1
    for (int i = i0 + lane; i < L; i += 64) look.big |= __builtin_isinf(ep[i]);
    if (look.redo()) {
      f32x4_t ko[D / 8], vo[D / 8];
      f32_half_row<D, ROT>(kp + (int64_t)min(kj, L - 1) * D, rc, rs, min(kj, L - 1), ko);
      f32_half_row<D, false>(vp + (int64_t)min(kj, L - 1) * D, nullptr, nullptr, 0, vo);
      f32_clear(dk);
      f32_clear(dv);
#pragma unroll 1
      for (int i = i0; i < L; ++i) {
        f32x4_t qr[D / 8], gr[D / 8];
        f32_half_row<D, ROT>(qp + (int64_t)i * D, rc, rs, i, qr);
        f32_half_row<D, false>(gp + (int64_t)i * D, nullptr, nullptr, 0, gr);
        const float s = f32_half_dot(ko, qr) * scale, p = f32_half_dot(vo, gr);
        float rr;
        const float w = frho8r(s, rr) * ip[i];
        const bool keep = kj < vlen && (!a.causal || kj <= i);
        f32_half_axpy(keep ? c8 * rr * w * (p - ep[i]) : 0.f, qr, dk);
        f32_half_axpy(keep ? w : 0.f, gr, dv);
      }
    }
  }

  if (kj < L) {
    float* kout = (float*)a.dk + base + (int64_t)kj * D;
    float* vout = (float*)a.dv + base + (int64_t)kj * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const int m = db * 32 + 8 * e4 + 4 * g;
        if (D % 32 == 0 || m < D) {
          if constexpr (ROT) f_unrotate4<D>(dk[db], 4 * e4, rc, rs, kj, m);
          f32x4_t wk, wv;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            wk[u] = dk[db][4 * e4 + u];
            wv[u] = dv[db][4 * e4 + u];
          }
          *(f32x4_t*)(kout + m) = wk;
          *(f32x4_t*)(vout + m) = wv;
        }
      }
  }
}

bool f32_bwd_supported(int head_dim) {
  return head_dim == 32 || head_dim == 48 || head_dim == 64 || head_dim == 96 || head_dim == 128;
}

template <int D, bool ROT>
static void f32_bwd_launch_d(const GenArgs& a, hipStream_t st) {
  const int nb = a.B * a.H * ((a.L + 127) / 128);
  hipLaunchKernelGGL((afa_bwd_f32_dq_kernel<D, ROT>), dim3(nb), dim3(256), 0, st, a);
  hipLaunchKernelGGL((afa_bwd_f32_dkdv_kernel<D, ROT>), dim3(nb), dim3(256), 0, st, a);
}

template <int D>
static void f32_bwd_launch_r(const GenArgs& a, hipStream_t st) {
  if (a.rc != nullptr) f32_bwd_launch_d<D, true>(a, st);
  else f32_bwd_launch_d<D, false>(a, st);
}

hipError_t f32_bwd_launch(const GenArgs& a, hipStream_t st) {
  const int64_t rows = (int64_t)a.B * a.H * a.L;
  hipLaunchKernelGGL(afa_bwd_f32_prep_kernel, dim3((unsigned)((rows + 31) / 32)), dim3(256), 0, st, a);
  if (a.D == 32) f32_bwd_launch_r<32>(a, st);
  else if (a.D == 48) f32_bwd_launch_r<48>(a, st);
  else if (a.D == 64) f32_bwd_launch_r<64>(a, st);
  else if (a.D == 96) f32_bwd_launch_r<96>(a, st);
  else f32_bwd_launch_r<128>(a, st);
  return hipGetLastError();
}

}  // namespace afa
