// fp32 ("HIGHEST") fused AFA forward on the bf16 matrix cores, for head_dim 32, 48, 64, 96 and 128.
// Same contract as the generic fp32 path (src/kernels/pallas_afa.py:52-151 with fp32 operands): s =
// (q . k) scale in fp32, w = rho(s)^8 by the cancellation-safe two-branch form, out = sum_j w v_j /
// (sum_j w + Omega), d = sum_j w + Omega; only the order of the fp32 additions differs.
//
// Every fp32 operand of the two products is split exactly into three bf16 planes (afa_f32_split.h)
// and a product is the six plane products of at least 2^-16 relative weight, accumulated in fp32: 2.7
// times the rate of v_mfma_f32_32x32x2_f32 for both products.
//
// A wave owns 32 queries; a unit is 32 keys x 32 queries.
//   S^T = K Q^T: 32x32x16 steps over head_dim, the query planes in registers, K planes read as
//   16-byte LDS fragments.
//   O^T += V^T P^T: the S^T accumulator of lane (query c, group g) holds keys 8 (e >> 2) + 4 g +
//   (e & 3); its weights are split in registers and are the B operand as they are, in the key order
//   in which ds_read_tr16_b64 returns the V planes' columns.
// K/V tiles of 32 keys are staged through registers (loads of tile t + 1 in flight during tile t),
// rotated and split there -- a pre-pass that left planes in memory would write and read 6 bytes
// per element where a tile is read by only L / 256 query blocks on average -- into double-buffered
// LDS, one barrier per tile.  Query blocks are dispatched heaviest first (block_item).
// Small grids (fewer workgroups than CUs) split every query block's key tiles over blockIdx.y:
// the numerator and denominator are sums over keys, so each split writes its partial O and row
// sum, and afa_fwd_f32_combine_kernel adds them, adds the sink and divides.
#include <cmath>

#include "afa_common.h"
#include "afa_f32_split.h"
#include "afa_launch.h"

namespace afa {

namespace {

constexpr int KT = 32;  // keys per tile

}  // namespace

// Waves per SIMD: the query planes alone take 24, 48 and 96 registers at head_dim 32, 64 and 128 (at
// head_dim 64 three waves spill 7 to 21 registers and measured 10% slower; at 32 they measured 293 -> 272
// us on B=8 H=16 L=2048).
constexpr int f32_waves(int d) { return d <= 32 ? 3 : d <= 64 ? 2 : 1; }

// Bound by the sum of its matrix and vector issue: at B=1 H=8 L=4096 D=64, 1536 matrix cycles per
// unit and 430 vector instructions of four cycles (rho^8 with its reciprocal 128, the split of the
// weights 88, staging 140) account for 98% of the SIMD cycles, at the 2.0 GHz the device holds.  332
// -> 216 us there, 233 -> 147 us at B=32 H=4 L=1024 D=64 (causal, rotary), 384 -> 267 us at B=2 H=8
// L=2048 D=128, against v_mfma_f32_32x32x2_f32; error against 64 bits 6.3e-7 -> 4.9e-7, 8.3e-7 ->
// 6.5e-7, 9.3e-7 -> 7.6e-7.
template <int D, bool ROT, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f32_waves(D), f32_waves(D))))
void afa_fwd_f32_kernel(const FwdArgs a) {
  using X = F32Tile<D>;
  constexpr int NK = D / 16;               // 16-feature steps of S
  constexpr int NDB = (D + 31) / 32;       // 32-feature output blocks
  constexpr int JOBS = (KT * (D / 4) + 255) / 256;  // float4 of K, and of V, per thread per tile
  constexpr bool RAGGED = KT * (D / 4) % 256 != 0;  // head_dim 48: the last job is half a workgroup's
  __shared__ __attribute__((aligned(16))) unsigned short ks[2][3 * X::PLANE];
  __shared__ __attribute__((aligned(16))) unsigned short vs[2][3 * X::PLANE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  int bh, qblk;
  block_item(blockIdx.x, a.B * a.H, a.nqb, a.causal, bh, qblk);
  const int b = bh / a.H, h = bh % a.H;
  const int L = a.L, vlen = a.valid_len;
  const int q0_wg = qblk * 128, q0_w = q0_wg + wave * 32;
  const int qi = q0_w + l32;
  const int kend_wg = a.causal ? min(vlen, min(L, q0_wg + 128)) : vlen;
  const int kend_w = a.causal ? min(vlen, q0_w + 32) : vlen;
  const int ntiles_wg = (kend_wg + KT - 1) / KT;
  // this workgroup's key tiles [t_beg, ntiles): all of them, or one of gridDim.y even parts
  int t_beg = 0, ntiles = ntiles_wg;
  if constexpr (SPLIT) {
    const int per = (ntiles_wg + (int)gridDim.y - 1) / (int)gridDim.y;
    t_beg = min(ntiles_wg, (int)blockIdx.y * per);
    ntiles = min(ntiles_wg, t_beg + per);
  }
  const float* qp = (const float*)a.q + b * a.q_b + h * a.q_h;
  const float* kp = (const float*)a.k + b * a.k_b + h * a.k_h;
  const float* vp = (const float*)a.v + b * a.v_b + h * a.v_h;
  // rows of q and k may start at any dword (a dwordx4 load needs no more); v and out rows are
  // 16-byte aligned (checked by the caller)
  typedef f32x4_t f32x4_dword_t __attribute__((aligned(4)));
  auto load4 = [](const float* p) -> f32x4_t { return *(const f32x4_dword_t*)p; };
  // the first tile's loads go out before q's
  f32x4_t kx[JOBS], vx[JOBS];
  float kc[JOBS][2], ksn[JOBS][2];
  int jrow[JOBS], jcol[JOBS];
#pragma unroll
  for (int i = 0; i < JOBS; ++i) {
    const int e = tid + 256 * i;
    jrow[i] = e / (D / 4);
    jcol[i] = 4 * (e % (D / 4));
  }
  // Lane offsets within a tile are the same in every tile (32 bits, checked by the caller): a tile
  // moves the uniform base pointers.  In the tile that reaches past the sequence, rows past it load
  // its last row: finite data for masked keys.
  uint32_t koff[JOBS], voff[JOBS], toff[JOBS];
  auto offsets = [&](int last) {
#pragma unroll
    for (int i = 0; i < JOBS; ++i) {
      const int r = min(jrow[i], last);
      koff[i] = (uint32_t)(r * (int)a.k_l + jcol[i]) * 4u;
      voff[i] = (uint32_t)(r * (int)a.v_l + jcol[i]) * 4u;
      toff[i] = (uint32_t)(r * (D / 2) + jcol[i] / 2) * 4u;
    }
  };
  offsets(KT - 1);
  auto load = [&](int t) {
    if (L - t * KT < KT) offsets(L - 1 - t * KT);
    const char* kt = (const char*)(kp + (int64_t)t * KT * a.k_l);
    const char* vt = (const char*)(vp + (int64_t)t * KT * a.v_l);
    const char* ct = (const char*)(a.rc + (int64_t)t * KT * (D / 2));
    const char* st = (const char*)(a.rs + (int64_t)t * KT * (D / 2));
#pragma unroll
    for (int i = 0; i < JOBS; ++i) {
      kx[i] = load4((const float*)(kt + koff[i]));
      vx[i] = load4((const float*)(vt + voff[i]));
      if constexpr (ROT) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          kc[i][p] = ((const float*)(ct + toff[i]))[p];
          ksn[i][p] = ((const float*)(st + toff[i]))[p];
        }
      }
    }
  };
  auto store = [&](int t) {
    const int buf = t & 1;
#pragma unroll
    for (int i = 0; i < JOBS; ++i) {
      const int r = jrow[i], c = jcol[i];
      if (RAGGED && r >= KT) continue;
      const f32x4_t y = ROT ? f32_rotate4(kx[i], kc[i], ksn[i]) : kx[i];
      unsigned w[3][2];
      split3_rne(y[0], y[1], w[0][0], w[1][0], w[2][0]);
      split3_rne(y[2], y[3], w[0][1], w[1][1], w[2][1]);
      X::put(ks[buf], X::at(r, c), w);
      split3_rne(vx[i][0], vx[i][1], w[0][0], w[1][0], w[2][0]);
      split3_rne(vx[i][2], vx[i][3], w[0][1], w[1][1], w[2][1]);
      X::put(vs[buf], X::at(r, c), w);
    }
  };
  if (t_beg < ntiles) load(t_beg);

  // q planes (B operand of S^T): lane (query qi, group g) holds features 16 kc + 8 g .. + 7
  u32x4_t qf[3][NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) {
    const int d0 = 16 * kk + 8 * g;
    f32x4_t x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (qi < L) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        x[hh] = load4(qp + (int64_t)qi * a.q_l + d0 + 4 * hh);
        if constexpr (ROT) {
          const float* c = a.rc + (int64_t)qi * (D / 2) + d0 / 2 + 2 * hh;
          const float* s = a.rs + (int64_t)qi * (D / 2) + d0 / 2 + 2 * hh;
          x[hh] = f32_rotate4(x[hh], c, s);
        }
      }
    }
    split8(x[0] * a.q_scale, x[1] * a.q_scale, qf[0][kk], qf[1][kk], qf[2][kk]);
  }
  if constexpr (D % 32 != 0) {  // the padding features of both V buffers, once
    for (int e = tid; e < 2 * 3 * KT * 4; e += 256) {
      const int r = (e >> 2) % KT, pl = (e / (4 * KT)) % 3, buf = e / (12 * KT);
      *(u32x2_t*)&vs[buf][pl * X::PLANE + X::at(r, D + 4 * (e & 3))] = u32x2_t{0u, 0u};
    }
  }

  f32x16_t o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
  float dsum = 0.f;

  if (t_beg < ntiles) store(t_beg);
  __syncthreads();
  for (int t = t_beg; t < ntiles; ++t) {
    if (t + 1 < ntiles) load(t + 1);  // global loads in flight during this tile's products
    const int key0 = t * KT;
    if (key0 < kend_w && q0_w < L) {
      const unsigned short* kt = ks[t & 1];
      const unsigned short* vt = vs[t & 1];
      f32x16_t st;
#pragma unroll
      for (int e = 0; e < 16; ++e) st[e] = 0.f;
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        u32x4_t kf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) kf[p] = X::row_frag(kt + p * X::PLANE, kk, lane);
        st = mma_planes(kf, qf[0][kk], qf[1][kk], qf[2][kk], st);
      }
      const bool need_mask = (a.causal && key0 + 31 > q0_w) || key0 + 31 >= vlen || q0_w + 31 >= L;
      float w[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) w[e] = rho8_exact(D == 64 ? st[e] : st[e] * a.s_mult);
      if (need_mask) {
        // a side effect the compiler cannot move keeps this a branch on the wave-uniform test
        // instead of a compare and a select per score in every tile
        asm volatile("" ::: "memory");
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = key0 + 8 * (e >> 2) + 4 * g + (e & 3);
          const bool keep = key < vlen && qi < L && (!a.causal || key <= qi);
          w[e] = keep ? w[e] : 0.f;
        }
      }
      float ts = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) ts += w[e];
      // two-level sums: the tile's own (row sum and PV from zero), then added to the running
      // ones, as the reference adds one block's dot(p, v) at a time
      // (src/kernels/pallas_afa.py:131-139); a single chain over L keys would carry a rounding
      // error growing with L (4.8e-6 normwise at L = 4096 against 1.3e-6 for 256-key chains)
      dsum += ts;
      u32x4_t pk[3][2];
      split_acc(w, pk);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        f32x16_t ot;
#pragma unroll
        for (int e = 0; e < 16; ++e) ot[e] = 0.f;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4_t vf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) vf[p] = X::col_frag(vt + p * X::PLANE, db, kk, lane);
          ot = mma_planes(vf, pk[0][kk], pk[1][kk], pk[2][kk], ot);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) o[db][e] += ot[e];
      }
    }
    // the buffer of tile t+1 was last read in tile t-1, before the previous barrier
    if (t + 1 < ntiles) store(t + 1);
    __syncthreads();
  }

  if (f32_any_nan(o)) {  // a NaN: the wave has queries, q0_w < L
    const int key0 = t_beg * KT, key1 = min(kend_w, ntiles * KT);
    F32Look look;
    look.rows<D>(qp + (int64_t)q0_w * a.q_l, a.q_l, min(32, L - q0_w));
    look.rows<D>(kp + (int64_t)key0 * a.k_l, a.k_l, key1 - key0);
    look.rows<D>(vp + (int64_t)key0 * a.v_l, a.v_l, key1 - key0);
    if (look.redo()) {
      f32x4_t qo[D / 8];
      f32_half_row<D, ROT>(qp + (int64_t)min(qi, L - 1) * a.q_l, a.rc, a.rs, min(qi, L - 1), qo);
#pragma unroll
      for (int c = 0; c < D / 8; ++c) qo[c] *= a.q_scale;
      f32_clear(o);
      dsum = 0.f;
#pragma unroll 1
      for (int j = key0; j < key1; ++j) {
        f32x4_t kr[D / 8], vr[D / 8];
        f32_half_row<D, ROT>(kp + (int64_t)j * a.k_l, a.rc, a.rs, j, kr);
        f32_half_row<D, false>(vp + (int64_t)j * a.v_l, nullptr, nullptr, 0, vr);
        const float s = f32_half_dot(qo, kr);
        // a masked key weighs 0, and its infinite values are NaN, as in the tiles
        const float w = !a.causal || j <= qi ? rho8_exact(D == 64 ? s : s * a.s_mult) : 0.f;
        f32_half_axpy(w, vr, o);
        if (g == 0) dsum += w;
      }
    }
  }

  dsum += __shfl_xor(dsum, 32);
  if constexpr (SPLIT) {
    // unnormalised partials of split blockIdx.y: the numerators of all splits (each B, H, L, D),
    // then the row sums of all splits (each B, H, L)
    const int64_t rows = (int64_t)a.B * a.H * L;
    float* po = a.part + (int64_t)blockIdx.y * rows * D;
    float* pd = a.part + (int64_t)gridDim.y * rows * D + (int64_t)blockIdx.y * rows;
    if (qi < L) {
      float* op = po + ((int64_t)bh * L + qi) * D;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          if (D % 32 == 0 || db * 32 + 8 * e4 + 4 * g < D) {
            f32x4_t w;
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] = o[db][4 * e4 + u];
            *(f32x4_t*)(op + db * 32 + 8 * e4 + 4 * g) = w;
          }
        }
      if (g == 0) pd[(int64_t)bh * L + qi] = dsum;
    }
    return;
  }
  if (qi < L) {
    const float tot = dsum + a.omega;
    float* op = (float*)a.out + b * a.o_b + h * a.o_h + (int64_t)qi * a.o_l;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        if (D % 32 == 0 || db * 32 + 8 * e4 + 4 * g < D) {
          f32x4_t* p = (f32x4_t*)(op + db * 32 + 8 * e4 + 4 * g);
          f32x4_t w;
          if (a.acc) {
            // one key shard: the unnormalised sums, stored or added to the caller's arrays
            if (a.acc == ACC_ADD) w = *p;
            else w = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] += o[db][4 * e4 + u];
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] = o[db][4 * e4 + u] / tot;
          }
          *p = w;
        }
      }
    if (a.acc && g == 0) acc_row(a.denom + (int64_t)bh * L + qi, dsum, a.acc);
    else if (a.denom != nullptr && g == 0) a.denom[(int64_t)bh * L + qi] = tot;
  }
}

// out = (sum of the split numerators) / (sum of the split row sums + sink), in split order; one
// thread per 4 features of a row.
template <int D>
__global__ __launch_bounds__(256) void afa_fwd_f32_combine_kernel(const FwdArgs a, int nsplit) {
  const int64_t rows = (int64_t)a.B * a.H * a.L;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * (D / 4)) return;
  const int64_t row = idx / (D / 4);
  const int c4 = (int)(idx % (D / 4));
  float tot = 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int sp = 0; sp < nsplit; ++sp) {
    tot += a.part[(int64_t)nsplit * rows * D + (int64_t)sp * rows + row];
    const f32x4_t v = *(const f32x4_t*)(a.part + (int64_t)sp * rows * D + row * D + 4 * c4);
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] += v[u];
  }
  tot += a.omega;
  const int bh = (int)(row / a.L), l = (int)(row % a.L);
  const int b = bh / a.H, h = bh % a.H;
  float* op = (float*)a.out + b * a.o_b + h * a.o_h + (int64_t)l * a.o_l + 4 * c4;
  if (a.acc) {
    // one key shard: the sums, stored or added to the caller's arrays (the sink is 0)
    f32x4_t w = {0.f, 0.f, 0.f, 0.f};
    if (a.acc == ACC_ADD) w = *(const f32x4_t*)op;
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] += acc[u];
    *(f32x4_t*)op = w;
    if (c4 == 0) acc_row(a.denom + row, tot, a.acc);
    return;
  }
  f32x4_t w;
#pragma unroll
  for (int u = 0; u < 4; ++u) w[u] = acc[u] / tot;
  *(f32x4_t*)op = w;
  if (a.denom != nullptr && c4 == 0) a.denom[row] = tot;
}

bool f32_fwd_supported(int head_dim) {
  return head_dim == 32 || head_dim == 48 || head_dim == 64 || head_dim == 96 || head_dim == 128;
}

size_t f32_fwd_part_floats(const FwdArgs& a, int head_dim, int nsplit) {
  return (size_t)nsplit * a.B * a.H * a.L * (head_dim + 1);
}

template <int D, bool SPLIT>
static void f32_launch_s(const FwdArgs& a, int nsplit, hipStream_t st) {
  const dim3 grid((unsigned)(a.B * a.H * a.nqb), (unsigned)nsplit);
  if (a.rc != nullptr)
    hipLaunchKernelGGL((afa_fwd_f32_kernel<D, true, SPLIT>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((afa_fwd_f32_kernel<D, false, SPLIT>), grid, dim3(256), 0, st, a);
}

template <int D>
static hipError_t f32_launch_d(const FwdArgs& a, int nsplit, hipStream_t st) {
  if (nsplit <= 1) {
    f32_launch_s<D, false>(a, 1, st);
    return hipGetLastError();
  }
  if (a.part == nullptr) return hipErrorInvalidValue;
  f32_launch_s<D, true>(a, nsplit, st);
  const int64_t n = (int64_t)a.B * a.H * a.L * (D / 4);
  hipLaunchKernelGGL((afa_fwd_f32_combine_kernel<D>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a,
                     nsplit);
  return hipGetLastError();
}

hipError_t f32_fwd_launch(int head_dim, FwdArgs a, int nsplit, hipStream_t st) {
  a.nqb = (a.L + 127) / 128;
  // 1/sqrt(D): the power of two below it folded into q exactly, the rest an fp32 factor of the
  // score (1 at D = 64)
  const float scale = (float)(1.0 / std::sqrt((double)head_dim));
  int ex = 0;
  (void)std::frexp(scale, &ex);
  a.q_scale = std::ldexp(1.0f, ex - 1);
  a.s_mult = std::ldexp(scale, 1 - ex);
  if (head_dim == 32) return f32_launch_d<32>(a, nsplit, st);
  if (head_dim == 48) return f32_launch_d<48>(a, nsplit, st);
  if (head_dim == 64) return f32_launch_d<64>(a, nsplit, st);
  if (head_dim == 96) return f32_launch_d<96>(a, nsplit, st);
  return f32_launch_d<128>(a, nsplit, st);
}

}  // namespace afa
