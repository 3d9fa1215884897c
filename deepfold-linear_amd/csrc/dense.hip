// Dense, materialised-cost Sinkhorn on gfx950: the restatement of
// vv137/deepfold-linear src/deepfold/model/sinkhorn.py.
//
//   sinkhorn_solve (:17-112)            K log-domain UOT iterations on a given cost
//                                       C (B,H,N,N): u = kappa (log mu - LSE_j(L + v + cb)),
//                                       v = kappa (log nu - LSE_i(L + u + rb)), L = -C/eps,
//                                       masks as -1e9 biases, early stop on the L-inf change;
//                                       backward = autograd through the executed iterations.
//   compute_transport_output (:115-198) T_norm = exp(ls - max)/(sum + 1e-6), O = T_norm V,
//                                       sigmoid gate, EGNN centroid; backward of those ops.
//
// The solver's passes read C once each and are short (C of a few heads sits in L2 and
// the Infinity Cache), so what bounds them is the number of loads in flight and the
// fixed cost of a launch.  fp32 throughout (the reference's dtype), exponents in base 2.
// Row passes: one wave per row, up to 1024 columns of it in registers at once.
// Column passes: one 1024-thread workgroup per 32 columns; a wave takes several rows of
// the strip at once and the loads of four such steps are in flight together.
// The transport's products run on v_mfma_f32_16x16x4_f32 over 16-row (16-column) tiles.
#include "dense_args.h"
#include "common.h"

#include <algorithm>

namespace dfl {

constexpr int DN_NT = 256;
constexpr int DN_NW = DN_NT / WAVE;
constexpr float MASK_BIAS = -1e9f;  // sinkhorn.py:79-80, 151

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, WAVE));
  return x;
}
__device__ __forceinline__ float mask_bias(const float* mask, int b, int N, int j) {
  return mask ? (1.f - mask[(size_t)b * N + j]) * MASK_BIAS : 0.f;
}
// |x| as ordered bits for an atomic max over non-negative floats (NaN -> +inf bits)
__device__ __forceinline__ unsigned abs_bits(float x) {
  const float a = fabsf(x);
  return a == a ? __float_as_uint(a) : 0x7f800000u;
}

// C is read as float4 where its rows are 16-byte aligned (VEC = 4), else by element.
template <int VEC> struct Vec;
template <> struct Vec<4> {
  __device__ static __forceinline__ void load(float (&x)[4], const float* p) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = t[e];
  }
  __device__ static __forceinline__ void store(float* p, const float (&x)[4]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{x[0], x[1], x[2], x[3]};
  }
};
template <> struct Vec<1> {
  __device__ static __forceinline__ void load(float (&x)[1], const float* p) { x[0] = *p; }
  __device__ static __forceinline__ void store(float* p, const float (&x)[1]) { *p = x[0]; }
};
constexpr float LOWEST = -3.0e38f;  // running maximum before the first element: finite, so that
                                    // exp2(m - m) of a lane without elements is 1 and not NaN
constexpr int RP_LANE = 16;         // columns a lane of a row pass holds at once
constexpr int RP_COLS = RP_LANE * WAVE;

// x2[e] = log2-domain exponent (-C_ij/eps + base + sgn vec_j + cb_j) log2e of this lane's 16 columns
// of a row from c0 on (-inf past the row's end); vec and the sample's mask (or null) span the row.
// Every load is issued, from clamped addresses, before the first use.
template <int VEC>
__device__ __forceinline__ void row_exponents(float (&x2)[RP_LANE], const float* Cr, const float* vec, const float* mask,
                                              float base, float sgn, int c0, int N, int lane, float sc) {
  float t[RP_LANE / VEC][VEC], mk[RP_LANE / VEC][VEC], c[RP_LANE / VEC][VEC];
#pragma unroll
  for (int q = 0; q < RP_LANE / VEC; ++q) {
    const int j = min(c0 + (q * WAVE + lane) * VEC, N - VEC);
    if (c0 + q * WAVE * VEC < N) {  // uniform
      Vec<VEC>::load(c[q], Cr + j);
      Vec<VEC>::load(t[q], vec + j);
      if (mask) Vec<VEC>::load(mk[q], mask + j);
    }
  }
#pragma unroll
  for (int q = 0; q < RP_LANE / VEC; ++q)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      x2[q * VEC + e] = -INFINITY;
      if (c0 + q * WAVE * VEC < N) {
        const float nat = base + sgn * t[q][e] + (mask ? (1.f - mk[q][e]) * MASK_BIAS : 0.f);
        const float x = __builtin_fmaf(c[q][e], sc, nat * LOG2E);
        x2[q * VEC + e] = c0 + (q * WAVE + lane) * VEC < N ? x : -INFINITY;
      }
    }
}

// ---------------------------------------------------------------------------
// Row update of iteration k: r_i = LSE_j(-C_ij/eps + v_j + cb_j), u_i = kappa (log mu_i - r_i).
// One wave per row; 4 rows per workgroup.  v = hist_v[k-1]; writes hist_r[k], hist_u[k].
template <int VEC>
__global__ void __launch_bounds__(DN_NT) dense_row_update_kernel(DenseSinkArgs a, int k) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int N = a.N, nblk = (N + DN_NW - 1) / DN_NW;
  const int bh = blockIdx.x / nblk, i = (blockIdx.x % nblk) * DN_NW + threadIdx.x / WAVE, b = bh / a.H, h = bh % a.H;
  if (i >= N) return;
  const size_t BHN = (size_t)a.B * a.H * N, row = (size_t)bh * N + i;
  const float eps = a.eps[h];
  const float kappa = a.lam / (a.lam + eps);
  const float sc = -LOG2E / eps;
  const float* Cr = a.C + row * N;
  const float* v = a.hist_v + (size_t)(k - 1) * BHN + (size_t)bh * N;
  float m = LOWEST, s = 0.f;
  for (int c0 = 0; c0 < N; c0 += RP_COLS) {
    float x[RP_LANE];
    row_exponents<VEC>(x, Cr, v, a.mask ? a.mask + (size_t)b * N : nullptr, 0.f, 1.f, c0, N, lane, sc);
    float mn = m;
#pragma unroll
    for (int e = 0; e < RP_LANE; ++e) mn = fmaxf(mn, x[e]);
    s *= fast_exp2(m - mn);
#pragma unroll
    for (int e = 0; e < RP_LANE; ++e) s += fast_exp2(x[e] - mn);
    m = mn;
  }
  const float mm = wave_max(m);
  const float ss = wave_sum(s * fast_exp2(m - mm));
  if (lane == 0) {
    const float r = (mm + fast_log2(ss)) * LN2;
    const float u = kappa * (a.log_mu[row] - r);
    a.hist_r[(size_t)k * BHN + row] = r;
    a.hist_u[(size_t)k * BHN + row] = u;
    if (a.delta) atomicMax(a.delta + 2 * k, abs_bits(u - a.hist_u[(size_t)(k - 1) * BHN + row]));
  }
}

// Column passes: workgroup of 16 waves per strip of 32 columns of one (b,h).  A wave reads
// 64 / (32 / VEC) rows of the strip at once; CP_U such steps are loaded together.  At B 2,
// H 8, N 512 the whole strip is in flight at once: 40.9 us (64 columns, 4 waves, one row a
// wave and step in flight) -> 6.1 us.
constexpr int CP_NT = 1024, CP_NW = CP_NT / WAVE, CP_COLS = 32;
template <int VEC> struct ColPass {
  static constexpr int LPR = CP_COLS / VEC;       // lanes per row
  static constexpr int RPW = WAVE / LPR;          // rows per wave and step
  static constexpr int U = VEC == 4 ? 4 : 8;      // steps in flight
};

// Column update of iteration k: c_j = LSE_i(-C_ij/eps + u_i + rb_i), v_j = kappa (log nu_j - c_j).
template <int VEC>
__global__ void __launch_bounds__(CP_NT) dense_col_update_kernel(DenseSinkArgs a, int k) {
  using P = ColPass<VEC>;
  __shared__ float s_m[CP_NW][CP_COLS], s_s[CP_NW][CP_COLS];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int N = a.N;
  const int nblk = (N + CP_COLS - 1) / CP_COLS;
  const int bh = blockIdx.x / nblk, j0 = (blockIdx.x % nblk) * CP_COLS, j = j0 + (lane % P::LPR) * VEC;
  const int b = bh / a.H, h = bh % a.H;
  const size_t BHN = (size_t)a.B * a.H * N;
  const float eps = a.eps[h];
  const float kappa = a.lam / (a.lam + eps);
  const float sc = -LOG2E / eps;
  const float* Cb = a.C + (size_t)bh * N * N;
  const float* u = a.hist_u + (size_t)k * BHN + (size_t)bh * N;
  float m[VEC], s[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) { m[e] = LOWEST; s[e] = 0.f; }
  for (int i0 = wave * P::RPW + lane / P::LPR; i0 < N; i0 += CP_NW * P::RPW * P::U) {
    float c[P::U][VEC], t[P::U];
#pragma unroll
    for (int q = 0; q < P::U; ++q) {
      const int i = i0 + q * CP_NW * P::RPW;
#pragma unroll
      for (int e = 0; e < VEC; ++e) c[q][e] = 0.f;
      t[q] = -INFINITY;
      if (i < N && j < N) {
        Vec<VEC>::load(c[q], Cb + (size_t)i * N + j);
        t[q] = (u[i] + mask_bias(a.mask, b, N, i)) * LOG2E;
      }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      float mn = m[e];
#pragma unroll
      for (int q = 0; q < P::U; ++q) { c[q][e] = __builtin_fmaf(c[q][e], sc, t[q]); mn = fmaxf(mn, c[q][e]); }
      s[e] *= fast_exp2(m[e] - mn);
#pragma unroll
      for (int q = 0; q < P::U; ++q) s[e] += fast_exp2(c[q][e] - mn);
      m[e] = mn;
    }
  }
#pragma unroll
  for (int o = P::LPR; o < WAVE; o <<= 1)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float mo = __shfl_xor(m[e], o, WAVE), so = __shfl_xor(s[e], o, WAVE);
      const float mn = fmaxf(m[e], mo);
      s[e] = s[e] * fast_exp2(m[e] - mn) + so * fast_exp2(mo - mn);
      m[e] = mn;
    }
  if (lane < P::LPR)
#pragma unroll
    for (int e = 0; e < VEC; ++e) { s_m[wave][lane * VEC + e] = m[e]; s_s[wave][lane * VEC + e] = s[e]; }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < CP_COLS && j0 + t < N) {
    float mm = LOWEST, ss = 0.f;
#pragma unroll
    for (int w = 0; w < CP_NW; ++w) mm = fmaxf(mm, s_m[w][t]);
#pragma unroll
    for (int w = 0; w < CP_NW; ++w) ss += s_s[w][t] * fast_exp2(s_m[w][t] - mm);
    const float c = (mm + fast_log2(ss)) * LN2;
    const size_t col = (size_t)bh * N + j0 + t;
    const float vv = kappa * (a.log_nu[col] - c);
    a.hist_c[(size_t)k * BHN + col] = c;
    a.hist_v[(size_t)k * BHN + col] = vv;
    if (a.delta) atomicMax(a.delta + 2 * k + 1, abs_bits(vv - a.hist_v[(size_t)(k - 1) * BHN + col]));
  }
}

// Final potentials (masked) and the iteration-0 entries of the history.
__global__ void dense_init_kernel(DenseSinkArgs a) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t BHN = (size_t)a.B * a.H * a.N;
  if (t < BHN) {
    a.hist_u[t] = a.u_init ? a.u_init[t] : 0.f;
    a.hist_v[t] = a.v_init ? a.v_init[t] : 0.f;
  }
  if (a.delta && t < (size_t)2 * (a.K + 1)) a.delta[t] = 0u;
}
__global__ void dense_finish_kernel(DenseSinkArgs a, int k) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t BHN = (size_t)a.B * a.H * a.N;
  if (t >= BHN) return;
  const int bh = (int)(t / a.N), i = (int)(t % a.N), b = bh / a.H;
  const float mk = a.mask ? a.mask[(size_t)b * a.N + i] : 1.f;
  a.log_u[t] = a.hist_u[(size_t)k * BHN + t] * mk;
  a.log_v[t] = a.hist_v[(size_t)k * BHN + t] * mk;
}

// ---------------------------------------------------------------------------
// Backward of iteration k (autograd through the executed iterations).
// Row pass, one wave per row i, with bvec = -kappa g_v(k) (all j):
//   P_col_ij = exp(L_ij + u_k,i + rb_i - c_k,j),   t_i = sum_j P_col_ij bvec_j
//   g_u(k)_i = [k == K] g_up_u_i + t_i,  avec_i = -kappa g_u(k)_i;   d log mu_i += kappa g_u(k)_i
// The recurrences need only these sums; dL_ij = sum_k P_col_ij bvec_j + P_row_ij avec_i is
// formed by dense_bwd_cost_kernel for a segment of iterations at once, so C is read and dC
// written once a segment and not read and rewritten in every iteration (a row pass at B 2, H 8,
// N 512: 16.7 -> 7.0 us, and 19 us once for 7 iterations' cost gradient).  g_v and avec of a
// segment lie in a ring of slots.
template <int VEC>
__global__ void __launch_bounds__(DN_NT) dense_bwd_row_kernel(DenseSinkBwdArgs a, int k, int slot) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int N = a.N, nblk = (N + DN_NW - 1) / DN_NW;
  const int bh = blockIdx.x / nblk, i = (blockIdx.x % nblk) * DN_NW + threadIdx.x / WAVE, b = bh / a.H, h = bh % a.H;
  if (i >= N) return;
  const size_t BHN = (size_t)a.B * a.H * N, row = (size_t)bh * N + i;
  const float eps = a.eps[h];
  const float kappa = a.lam / (a.lam + eps);
  const float sc = -LOG2E / eps;
  const float* Cr = a.C + row * N;
  const float* ck = a.hist_c + (size_t)k * BHN + (size_t)bh * N;
  const float* gv = a.gv + (size_t)slot * BHN + (size_t)bh * N;
  const float ur = a.hist_u[(size_t)k * BHN + row] + mask_bias(a.mask, b, N, i);
  float t = 0.f;
  for (int c0 = 0; c0 < N; c0 += RP_COLS) {
    float x[RP_LANE];
    float g[RP_LANE / VEC][VEC];
#pragma unroll
    for (int q = 0; q < RP_LANE / VEC; ++q)
      if (c0 + q * WAVE * VEC < N) Vec<VEC>::load(g[q], gv + min(c0 + (q * WAVE + lane) * VEC, N - VEC));
    row_exponents<VEC>(x, Cr, ck, nullptr, ur, -1.f, c0, N, lane, sc);
#pragma unroll
    for (int q = 0; q < RP_LANE / VEC; ++q)
#pragma unroll
      for (int e = 0; e < VEC; ++e)
        if (c0 + q * WAVE * VEC < N) t = __builtin_fmaf(fast_exp2(x[q * VEC + e]), -kappa * g[q][e], t);
  }
  t = wave_sum(t);
  if (lane == 0) {
    const bool first = k == a.K;
    const float gu = (first && a.grad_u ? a.grad_u[row] * (a.mask ? a.mask[(size_t)b * N + i] : 1.f) : 0.f) + t;
    a.avec[(size_t)slot * BHN + row] = -kappa * gu;
    const float dmu = kappa * gu;
    a.dlog_mu[row] = first ? dmu : a.dlog_mu[row] + dmu;
  }
}

// Column pass of iteration k: g_v(k-1)_j = sum_i P_row_ij avec_i with
// P_row_ij = exp(L_ij + v_{k-1},j + cb_j - r_k,i), d log nu_j += kappa g_v(k)_j.
template <int VEC>
__global__ void __launch_bounds__(CP_NT) dense_bwd_col_kernel(DenseSinkBwdArgs a, int k, int slot, int next) {
  using P = ColPass<VEC>;
  __shared__ float s_t[CP_NW][CP_COLS];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int N = a.N;
  const int nblk = (N + CP_COLS - 1) / CP_COLS;
  const int bh = blockIdx.x / nblk, j0 = (blockIdx.x % nblk) * CP_COLS, j = j0 + (lane % P::LPR) * VEC;
  const int b = bh / a.H, h = bh % a.H;
  const size_t BHN = (size_t)a.B * a.H * N;
  const float eps = a.eps[h];
  const float kappa = a.lam / (a.lam + eps);
  const float sc = -LOG2E / eps;
  const float* Cb = a.C + (size_t)bh * N * N;
  const float* rk = a.hist_r + (size_t)k * BHN + (size_t)bh * N;
  const float* av = a.avec + (size_t)slot * BHN + (size_t)bh * N;
  float vj[VEC], t[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    t[e] = 0.f;
    vj[e] = j < N ? a.hist_v[(size_t)(k - 1) * BHN + (size_t)bh * N + j + e] + mask_bias(a.mask, b, N, j + e) : 0.f;
  }
  for (int i0 = wave * P::RPW + lane / P::LPR; i0 < N; i0 += CP_NW * P::RPW * P::U) {
    float c[P::U][VEC], ri[P::U], ai[P::U];
#pragma unroll
    for (int q = 0; q < P::U; ++q) {
      const int i = i0 + q * CP_NW * P::RPW;
#pragma unroll
      for (int e = 0; e < VEC; ++e) c[q][e] = 0.f;
      ri[q] = INFINITY;  // exp2(-inf) = 0
      ai[q] = 0.f;
      if (i < N && j < N) {
        Vec<VEC>::load(c[q], Cb + (size_t)i * N + j);
        ri[q] = rk[i];
        ai[q] = av[i];
      }
    }
#pragma unroll
    for (int q = 0; q < P::U; ++q)
#pragma unroll
      for (int e = 0; e < VEC; ++e)
        t[e] = __builtin_fmaf(fast_exp2(__builtin_fmaf(c[q][e], sc, (vj[e] - ri[q]) * LOG2E)), ai[q], t[e]);
  }
#pragma unroll
  for (int o = P::LPR; o < WAVE; o <<= 1)
#pragma unroll
    for (int e = 0; e < VEC; ++e) t[e] += __shfl_xor(t[e], o, WAVE);
  if (lane < P::LPR)
#pragma unroll
    for (int e = 0; e < VEC; ++e) s_t[wave][lane * VEC + e] = t[e];
  __syncthreads();
  const int c = threadIdx.x;
  if (c < CP_COLS && j0 + c < N) {
    float tt = 0.f;
#pragma unroll
    for (int w = 0; w < CP_NW; ++w) tt += s_t[w][c];
    const size_t col = (size_t)bh * N + j0 + c;
    const float dnu = kappa * a.gv[(size_t)slot * BHN + col];
    a.dlog_nu[col] = k == a.K ? dnu : a.dlog_nu[col] + dnu;
    a.gv[(size_t)next * BHN + col] = tt;  // g_v(k-1)
  }
}

// Cost gradient of the iterations k1 .. k0 (k1 >= k0, at most DENSE_SEG of them, g_v(k) and avec(k)
// in slot (K - k) % (DENSE_SEG + 1)): dL_ij += sum_k P_col_ij (-kappa g_v(k)_j) + P_row_ij avec(k)_i,
// summed from k1 down.  A wave takes 64 VEC columns of 8 rows: the column vectors of an iteration
// are loaded once for the 8 rows.  The segment with k = K starts dC, the one with k = 1 writes
// the final dC = -dL / eps.
constexpr int CG_ROWS = 8;
template <int VEC>
__global__ void __launch_bounds__(DN_NT) dense_bwd_cost_kernel(DenseSinkBwdArgs a, int k1, int k0) {
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int N = a.N;
  const int nc = (N + WAVE * VEC - 1) / (WAVE * VEC), nr = (N + CG_ROWS - 1) / CG_ROWS;
  const int nblk = (nc * nr + DN_NW - 1) / DN_NW, bh = blockIdx.x / nblk, unit = (blockIdx.x % nblk) * DN_NW + wave;
  if (unit >= nc * nr) return;
  const int i0 = unit / nc * CG_ROWS, j = (unit % nc) * WAVE * VEC + lane * VEC;
  const int b = bh / a.H, h = bh % a.H;
  const size_t BHN = (size_t)a.B * a.H * N;
  const float eps = a.eps[h];
  const float kappa = a.lam / (a.lam + eps);
  const float sc = -LOG2E / eps;
  const int jc = min(j, N - VEC), ir = min(i0 + (lane & (CG_ROWS - 1)), N - 1);
  const size_t at = ((size_t)bh * N + i0) * N + jc;
  float L[CG_ROWS][VEC], dl[CG_ROWS][VEC], cb[VEC];
#pragma unroll
  for (int q = 0; q < CG_ROWS; ++q) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) L[q][e] = dl[q][e] = 0.f;
    if (i0 + q < N) {
      Vec<VEC>::load(L[q], a.C + at + (size_t)q * N);
      if (k1 != a.K) Vec<VEC>::load(dl[q], a.dC + at + (size_t)q * N);
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) cb[e] = mask_bias(a.mask, b, N, jc + e);
  const float rb = mask_bias(a.mask, b, N, ir);
  // the vectors of iteration k: columns per lane, rows in lanes 0-7 (read out lane by lane)
  struct It { float ck[VEC], bk[VEC], vp[VEC], u, r, av; };
  auto fetch = [&](It& t, int k) {
    const size_t hk = (size_t)k * BHN + (size_t)bh * N, sl = (size_t)((a.K - k) % (DENSE_SEG + 1)) * BHN + (size_t)bh * N;
    Vec<VEC>::load(t.ck, a.hist_c + hk + jc);
    Vec<VEC>::load(t.bk, a.gv + sl + jc);
    Vec<VEC>::load(t.vp, a.hist_v + hk - BHN + jc);
    t.u = a.hist_u[hk + ir];
    t.r = a.hist_r[hk + ir];
    t.av = a.avec[sl + ir];
  };
  It cur;
  fetch(cur, k1);
#pragma unroll
  for (int q = 0; q < CG_ROWS; ++q)
#pragma unroll
    for (int e = 0; e < VEC; ++e) L[q][e] *= sc;
  for (int k = k1; k >= k0; --k) {
    It nxt = cur;
    if (k > k0) fetch(nxt, k - 1);
    const float ur = cur.u + rb;
#pragma unroll
    for (int q = 0; q < CG_ROWS; ++q) {
      const float uq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ur), q));
      const float rq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cur.r), q));
      const float aq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cur.av), q));
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float pc = fast_exp2(__builtin_fmaf(uq - cur.ck[e], LOG2E, L[q][e]));
        const float pr = fast_exp2(__builtin_fmaf((cur.vp[e] + cb[e]) - rq, LOG2E, L[q][e]));
        dl[q][e] += __builtin_fmaf(pc, -kappa * cur.bk[e], pr * aq);
      }
    }
    cur = nxt;
  }
  const float fin = k0 == 1 ? -1.f / eps : 1.f;
  if (j >= N) return;
#pragma unroll
  for (int q = 0; q < CG_ROWS; ++q)
    if (i0 + q < N) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) dl[q][e] *= fin;
      Vec<VEC>::store(a.dC + at + (size_t)q * N, dl[q]);
    }
}

// g_v(K) = grad_v * mask into the workspace vector.
__global__ void dense_bwd_init_kernel(DenseSinkBwdArgs a) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t BHN = (size_t)a.B * a.H * a.N;
  if (t >= BHN) return;
  const int bh = (int)(t / a.N), i = (int)(t % a.N), b = bh / a.H;
  const float mk = a.mask ? a.mask[(size_t)b * a.N + i] : 1.f;
  a.gv[t] = a.grad_v ? a.grad_v[t] * mk : 0.f;
}
// After the last pass: d log_v_init = g_v(0); d log_u_init = 0 (u_0 feeds nothing for
// K >= 1; for K = 0 the output is the masked initial potential itself).
__global__ void dense_bwd_finish_kernel(DenseSinkBwdArgs a) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t BHN = (size_t)a.B * a.H * a.N;
  if (t >= BHN) return;
  if (a.dlog_v_init) a.dlog_v_init[t] = a.gv[(size_t)(a.K % (DENSE_SEG + 1)) * BHN + t];
  if (a.dlog_u_init) {
    float g = 0.f;
    if (a.K == 0 && a.grad_u) {
      const int bh = (int)(t / a.N), i = (int)(t % a.N), b = bh / a.H;
      g = a.grad_u[t] * (a.mask ? a.mask[(size_t)b * a.N + i] : 1.f);
    }
    a.dlog_u_init[t] = g;
  }
}

__global__ void dense_zero_kernel(float* p, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.f;
}

// ---------------------------------------------------------------------------
// Transport output, forward.  Workgroup of 4 waves per 16 rows of one (b,h):
//   ls_j = u_i - C_ij/eps + v_j + cb_j, T = exp(ls - max), Tn = T / (sum T + 1e-6) * mask_i,
//   O_i = sum_j Tn_j V_j,  x_c = sum_j Tn_j x_j,
//   o = sigma(G) O (permuted to (B,N,H*d)) * mask_i.  Saves O_avg for the backward.
// u_i is left out of the exponents: the row maximum takes it out again, and a smaller sum rounds less
// (T_norm against float64 at B 2, H 8, N 512: 4.4e-7 with it, 2.3e-7 without).
// Each wave takes the statistics of 4 rows, then their Tn chunk by chunk into HBM and LDS; the
// products are 16x16x4 fp32 MFMAs over the chunk, its k-steps dealt to the waves (x_res is one
// more tile of three columns), and the waves' partial tiles meet in LDS.  71 -> 17.5 us at
// B 2, H 8, N 512, d 32 (one row a wave read V once per row).
constexpr int TF_ROWS = 16, TF_CH = 512;
template <int VEC, int NCT, bool KEEP>
__global__ void __launch_bounds__(DN_NT) dense_transport_fwd_kernel(DenseTransportArgs a) {
  constexpr int LD = TF_CH + 4;  // 16 rows x 4 lane groups of an A operand fall in 64 different banks
  __shared__ __attribute__((aligned(16))) float s_T[TF_ROWS * LD];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int N = a.N, d = a.d;
  const int nblk = (N + TF_ROWS - 1) / TF_ROWS;
  const int bh = blockIdx.x / nblk, i0 = (blockIdx.x % nblk) * TF_ROWS, b = bh / a.H, h = bh % a.H;
  const float sc = -LOG2E / a.eps[h];
  const float* v = a.log_v + (size_t)bh * N;
  const float* Vb = a.V + (size_t)bh * N * d;
  const float* xb = a.x_res ? a.x_res + (size_t)b * N * 3 : nullptr;
  constexpr int RW = TF_ROWS / DN_NW;  // rows per wave
  const float* mk = a.mask ? a.mask + (size_t)b * N : nullptr;
  float mrow[RW], scale[RW];
  float ex[KEEP ? RW : 1][RP_LANE];  // KEEP (N <= RP_COLS): the rows' exponentials
#pragma unroll
  for (int q = 0; q < RW; ++q) {
    const int i = min(i0 + wave * RW + q, N - 1);
    const size_t row = (size_t)bh * N + i;
    const float ui = a.log_u[row];
    float m = LOWEST, s = 0.f;
    if (KEEP) {
      row_exponents<VEC>(ex[q], a.C + row * N, v, mk, 0.f, 1.f, 0, N, lane, sc);
      m = ex[q][0];  // (a row without a finite exponent is NaN, as exp(ls - max) is)
#pragma unroll
      for (int e = 1; e < RP_LANE; ++e) m = fmaxf(m, ex[q][e]);
      mrow[q] = wave_max(m);
#pragma unroll
      for (int e = 0; e < RP_LANE; ++e) {
        ex[q][e] = fast_exp2(ex[q][e] - mrow[q]);
        s += ex[q][e];
      }
      s = wave_sum(s);
    } else {
      for (int c0 = 0; c0 < N; c0 += RP_COLS) {
        float x[RP_LANE];
        row_exponents<VEC>(x, a.C + row * N, v, mk, 0.f, 1.f, c0, N, lane, sc);
        float mn = m;
#pragma unroll
        for (int e = 0; e < RP_LANE; ++e) mn = fmaxf(mn, x[e]);
        s *= fast_exp2(m - mn);
#pragma unroll
        for (int e = 0; e < RP_LANE; ++e) s += fast_exp2(x[e] - mn);
        m = mn;
      }
      mrow[q] = wave_max(m);
      s = wave_sum(s * fast_exp2(m - mrow[q]));
      if (mrow[q] == LOWEST) mrow[q] = -INFINITY;
    }
    scale[q] = (mk ? mk[i] : 1.f) / (s + 1e-6f) + (ui - ui);  // (NaN where u is not finite, as exp(ls - max) is)
  }
  f32x4 acc[NCT + 1];  // NCT = ceil(d / 16) rounded up to 1, 2 or 4 column tiles, then x_c
  f32x4 ax[4];         // x_c (its terms nearly cancel) in four shorter chains
#pragma unroll
  for (int c = 0; c <= NCT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; ++q) ax[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int col = lane & 15, grp = lane >> 4;
  // plan entries of the chunk from c0 on into T_norm and LDS; e(q, p): the p-th VEC of row q
  auto put = [&](int c0, auto e) {
#pragma unroll
    for (int q = 0; q < RW; ++q) {
      const int r = wave * RW + q;
      const size_t row = (size_t)bh * N + min(i0 + r, N - 1);
#pragma unroll
      for (int p = 0; p < TF_CH / (WAVE * VEC); ++p) {
        const int jj = (p * WAVE + lane) * VEC, j = c0 + jj;
        float c[VEC];
        e(q, p, row, j, c);
        if (j < N && i0 + r < N) Vec<VEC>::store(a.T_norm + row * N + j, c);
        Vec<VEC>::store(s_T + r * LD + jj, c);
      }
    }
  };
  auto product = [&](int c0) {
    // four k-steps a wave together (the compiler does not unroll a loop with MFMAs and a
    // remainder).  Past the row's end Tn is zero; columns past d (past x_c's three) are not stored
    const int steps = (min(TF_CH, N - c0) + 3) / 4;
    for (int k0 = 0; k0 < steps; k0 += 4 * DN_NW) {
      float t[4], bv[4][NCT], bx[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ks = k0 + q * DN_NW + wave, jc = min(c0 + 4 * ks + grp, N - 1);
        t[q] = s_T[col * LD + 4 * ks + grp];
#pragma unroll
        for (int c = 0; c < NCT; ++c) bv[q][c] = Vb[(size_t)jc * d + min(16 * c + col, d - 1)];
        bx[q] = xb ? xb[3 * jc + min(col, 2)] : 0.f;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int c = 0; c < NCT; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[q], bv[q][c], acc[c], 0, 0, 0);
        ax[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[q], bx[q], ax[q], 0, 0, 0);
      }
    }
  };
  if (KEEP) {
#pragma unroll
    for (int ch = 0; ch < RP_COLS / TF_CH; ++ch)
      if (ch * TF_CH < N) {  // uniform
        if (ch) __syncthreads();
        put(ch * TF_CH, [&](int q, int p, size_t, int, float (&c)[VEC]) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) c[e] = ex[q][ch * (TF_CH / WAVE) + p * VEC + e] * scale[q];
        });
        __syncthreads();
        product(ch * TF_CH);
      }
  } else {
    for (int c0 = 0; c0 < N; c0 += TF_CH) {
      if (c0) __syncthreads();
      put(c0, [&](int q, int, size_t row, int j, float (&c)[VEC]) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) c[e] = 0.f;
        if (j >= N) return;
        Vec<VEC>::load(c, a.C + row * N + j);
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          c[e] = fast_exp2(__builtin_fmaf(c[e], sc, (v[j + e] + mask_bias(a.mask, b, N, j + e)) * LOG2E) -
                           mrow[q]) * scale[q];
      });
      __syncthreads();
      product(c0);
    }
  }
  acc[NCT] = (ax[0] + ax[1]) + (ax[2] + ax[3]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c <= NCT; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) s_T[((c * DN_NW + wave) * 4 + r) * WAVE + lane] = acc[c][r];
  __syncthreads();
  for (int c = wave; c <= NCT; c += DN_NW) {
    if (c == NCT && !xb) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < DN_NW; ++w) t += s_T[((c * DN_NW + w) * 4 + r) * WAVE + lane];
      const int i = i0 + 4 * grp + r, cc = 16 * c + col;
      if (i >= N) continue;
      const size_t row = (size_t)bh * N + i;
      if (c == NCT) {
        if (col < 3) a.x_centroid[row * 3 + col] = t;
      } else if (cc < d) {
        a.o_avg[row * d + cc] = t;
        const float g = a.G ? 1.f / (1.f + __expf(-a.G[row * d + cc])) : 1.f;
        const float mi = a.mask ? a.mask[(size_t)b * N + i] : 1.f;
        a.o[((size_t)b * N + i) * (size_t)(a.H * d) + (size_t)h * d + cc] = g * t * mi;
      }
    }
  }
}

// Transport backward, row pass (workgroup of 8 waves per 16 rows i):
//   gOa_i = sigma(G) gO_i mask_i,  dG_i = sigma (1 - sigma) O_avg_i gO_i mask_i
//   dTn_ij = (gOa_i . V_j + gxc_i . x_j + gT_ij) * mask_i
//   dls_j = (dTn_j - dot) Tn_j with dot = sum_j dTn_j Tn_j and Tn = T / (S + 1e-6) the plan
//   without the row mask, plus, at the first argmax (torch max semantics), the row max's
//   gradient -dot 1e-6 / (S + 1e-6) = -dot 1e-6 max_j Tn_j (T is 1 at the maximum)
//   dC_ij = -dls_ij / eps,  d log_u_i = sum_j dls_ij.  Writes gOa for the column pass.
// Tn comes from the forward's T_norm, so C is not read and no exponential taken.  The products
// gOa V^T are fp32 MFMAs with the streamed j as the A rows: a lane holds four consecutive j of
// its row i = lane % 16.  A wave takes every 8th 16-column tile; with at most BR_KEEP of them
// (N <= 1024) dTn and Tn stay in registers between the sum and the gradients.
// 139 -> 17.3 us at B 2, H 8, N 512, d 32.
constexpr int BR_NT = 512, BR_NW = BR_NT / WAVE, BR_KEEP = 8;
template <int VEC, int DP, bool KEEP>
__global__ void __launch_bounds__(BR_NT) dense_transport_bwd_row_kernel(DenseTransportArgs a) {
  constexpr int RUN = DP / 4;
  __shared__ __attribute__((aligned(16))) float s_g[16][DP + 4];
  __shared__ float s_gx[16][4], s_dot[BR_NW][16], s_max[BR_NW][16], s_du[BR_NW][16];
  __shared__ int s_arg[BR_NW][16];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int N = a.N, d = a.d;
  const int nblk = (N + 15) / 16;
  const int bh = blockIdx.x / nblk, i0 = (blockIdx.x % nblk) * 16, b = bh / a.H, h = bh % a.H;
  const float* gT = a.grad_T;
  // gated output gradients of the 16 rows
  for (int t = threadIdx.x; t < 16 * DP; t += BR_NT) {
    const int r = t / DP, c = t % DP, i = i0 + r;
    float goa = 0.f;
    if (i < N && c < d) {
      const size_t row = (size_t)bh * N + i;
      const float mi = a.mask ? a.mask[(size_t)b * N + i] : 1.f;
      const float go = a.grad_o ? a.grad_o[((size_t)b * N + i) * (size_t)(a.H * d) + (size_t)h * d + c] * mi : 0.f;
      const float sg = a.G ? 1.f / (1.f + __expf(-a.G[row * d + c])) : 1.f;
      goa = sg * go;
      if (a.dG) a.dG[row * d + c] = sg * (1.f - sg) * a.o_avg[row * d + c] * go;
      a.goa[row * d + c] = goa;
    }
    s_g[r][c] = goa;
  }
  if (threadIdx.x < 64) {
    const int r = threadIdx.x / 4, c = threadIdx.x % 4;
    s_gx[r][c] = a.grad_xc && c < 3 && i0 + r < N ? a.grad_xc[((size_t)bh * N + i0 + r) * 3 + c] : 0.f;
  }
  __syncthreads();
  const int col = lane & 15, grp = lane >> 4;
  const int i = i0 + col, ic = min(i, N - 1);
  const size_t row = (size_t)bh * N + ic;
  const float mi = a.mask ? a.mask[(size_t)b * N + ic] : 1.f;
  const float inv_mi = mi != 0.f ? 1.f / mi : 0.f;
  const float* Vb = a.V + (size_t)bh * N * d;
  const float* xb = a.x_res && a.grad_xc ? a.x_res + (size_t)b * N * 3 : nullptr;
  const float* Tr = a.T_norm + row * N;
  float bg[RUN];  // this lane's B operand: its run of gOa of row i
#pragma unroll
  for (int e = 0; e < RUN; ++e) bg[e] = s_g[col][grp * RUN + e];
  const float bx = s_gx[col][grp];
  const bool v_vec = d == DP && ((uintptr_t)a.V & 15) == 0;
  // dTn of columns j .. j + 3 (grad_T and the mask included), and Tn there (zero past the end)
  auto tile = [&](int t, float (&dtn)[4], float (&tn)[4]) {
    const int ja = min(16 * t + col, N - 1);  // A row of the products
    const float* Vj = Vb + (size_t)ja * d + grp * RUN;
    float av[RUN];
    if (v_vec) {
#pragma unroll
      for (int e = 0; e < RUN; e += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(Vj + e);
#pragma unroll
        for (int f = 0; f < 4; ++f) av[e + f] = x[f];
      }
    } else {
#pragma unroll
      for (int e = 0; e < RUN; ++e) av[e] = grp * RUN + e < d ? Vj[e] : 0.f;
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < RUN; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], bg[e], acc, 0, 0, 0);
    if (xb) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(grp < 3 ? xb[3 * ja + grp] : 0.f, bx, acc, 0, 0, 0);
    const int j = 16 * t + 4 * grp;
    float g[4] = {0.f, 0.f, 0.f, 0.f};
    if (VEC == 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) tn[e] = 0.f;
      if (j < N) {
        Vec<4>::load(tn, Tr + j);
        if (gT) Vec<4>::load(g, gT + row * N + j);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        tn[e] = j + e < N ? Tr[j + e] : 0.f;
        if (gT && j + e < N) g[e] = gT[row * N + j + e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) { dtn[e] = (acc[e] + g[e]) * mi; tn[e] *= inv_mi; }
  };
  const int nt = (N + 15) / 16;
  float kd[KEEP ? BR_KEEP : 1][4], kt[KEEP ? BR_KEEP : 1][4];
  // (d log u_i = sum_j dls_ij nearly cancels: what is left is the rounding of dot and of the sum)
  float dot4[4] = {0.f, 0.f, 0.f, 0.f}, mx = -1.f;
  int am = N;
  auto gather = [&](int t, const float (&dtn)[4], const float (&tn)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dot4[e] = __builtin_fmaf(dtn[e], tn[e], dot4[e]);
      if (tn[e] > mx) { mx = tn[e]; am = 16 * t + 4 * grp + e; }
    }
  };
  if (KEEP) {
#pragma unroll
    for (int q = 0; q < BR_KEEP; ++q)
      if (wave + q * BR_NW < nt) {
        tile(wave + q * BR_NW, kd[q], kt[q]);
        gather(wave + q * BR_NW, kd[q], kt[q]);
      }
  } else {
    for (int t = wave; t < nt; t += BR_NW) {
      float dtn[4], tn[4];
      tile(t, dtn, tn);
      gather(t, dtn, tn);
    }
  }
  float dot = sum_groups((dot4[0] + dot4[1]) + (dot4[2] + dot4[3]));
#pragma unroll
  for (int o = 16; o < WAVE; o <<= 1) {
    const float om = __shfl_xor(mx, o, WAVE);
    const int oa = __shfl_xor(am, o, WAVE);
    if (om > mx || (om == mx && oa < am)) { mx = om; am = oa; }
  }
  if (lane < 16) { s_dot[wave][lane] = dot; s_max[wave][lane] = mx; s_arg[wave][lane] = am; }
  __syncthreads();
  dot = 0.f;
#pragma unroll
  for (int w = 0; w < BR_NW; ++w) {
    dot += s_dot[w][col];
    const float om = s_max[w][col];
    const int oa = s_arg[w][col];
    if (om > mx || (om == mx && oa < am)) { mx = om; am = oa; }
  }
  const float dmax = -dot * 1e-6f * mx;
  const float inv_eps = -1.f / a.eps[h];
  float du4[4] = {0.f, 0.f, 0.f, 0.f};
  auto grads = [&](int t, const float (&dtn)[4], const float (&tn)[4]) {
    const int j = 16 * t + 4 * grp;
    float dc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float dls = (dtn[e] - dot) * tn[e];
      if (j + e == am) dls += dmax;
      du4[e] += dls;
      dc[e] = dls * inv_eps;
    }
    if (i >= N) return;
    if (VEC == 4) {
      if (j < N) Vec<4>::store(a.dC + row * N + j, dc);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j + e < N) a.dC[row * N + j + e] = dc[e];
    }
  };
  if (KEEP) {
#pragma unroll
    for (int q = 0; q < BR_KEEP; ++q)
      if (wave + q * BR_NW < nt) grads(wave + q * BR_NW, kd[q], kt[q]);
  } else {
    for (int t = wave; t < nt; t += BR_NW) {
      float dtn[4], tn[4];
      tile(t, dtn, tn);
      grads(t, dtn, tn);
    }
  }
  const float du = sum_groups((du4[0] + du4[1]) + (du4[2] + du4[3]));
  if (lane < 16) s_du[wave][lane] = du;
  __syncthreads();
  if (threadIdx.x < 16 && i0 + threadIdx.x < (unsigned)N) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < BR_NW; ++w) t += s_du[w][threadIdx.x];
    a.dlog_u[(size_t)bh * N + i0 + threadIdx.x] = t;
  }
}

// Transport backward, column pass (workgroup of 8 waves per 32 columns j):
//   dV_j = sum_i Tn_ij gOa_i,  dx_j (this head) = sum_i Tn_ij gxc_i,  d log_v_j = sum_i dls_ij
//   with dls_ij = -eps dC_ij (dC already holds the argmax term).
// fp32 MFMAs with the columns j as the A rows, k = i: a wave takes every 8th group of four rows
// and both 16-column tiles; gxc is one more tile of three columns.  The waves' partial tiles meet
// in LDS.  332 us (a 64-column strip a workgroup, one row a wave in flight) -> 10.9 us at B 2, H 8,
// N 512, d 32.
template <int NCT>
__global__ void __launch_bounds__(BR_NT) dense_transport_bwd_col_kernel(DenseTransportArgs a) {
  __shared__ float s_acc[(NCT + 1) * BR_NW * 4 * WAVE];
  __shared__ float s_lv[BR_NW][32];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int N = a.N, d = a.d;
  const int nblk = (N + 31) / 32;
  const int bh = blockIdx.x / nblk, j0 = (blockIdx.x % nblk) * 32, h = bh % a.H;
  const float* Tb = a.T_norm + (size_t)bh * N * N;
  const float* dCb = a.dC + (size_t)bh * N * N;
  const float* goa = a.goa + (size_t)bh * N * d;
  const float* gxc = a.grad_xc && a.dx_part ? a.grad_xc + (size_t)bh * N * 3 : nullptr;
  const int col = lane & 15, grp = lane >> 4;
  f32x4 acc[2][NCT + 1];
  float lv[2] = {0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int c = 0; c <= NCT; ++c) acc[q][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (N + 3) / 4;
  for (int k0 = 0; k0 < steps; k0 += 4 * BR_NW) {
    float t[4][2], g[4][NCT], gx[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = 4 * (k0 + p * BR_NW + wave) + grp, ic = min(i, N - 1);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int j = j0 + 16 * q + col;
        const bool ok = i < N && j < N;
        const size_t at = (size_t)ic * N + min(j, N - 1);
        const float tv = Tb[at], cv = dCb[at];
        t[p][q] = ok ? tv : 0.f;
        lv[q] += ok ? cv : 0.f;
      }
#pragma unroll
      for (int c = 0; c < NCT; ++c) g[p][c] = goa[(size_t)ic * d + min(16 * c + col, d - 1)];
      gx[p] = gxc ? gxc[3 * ic + min(col, 2)] : 0.f;
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int c = 0; c < NCT; ++c)
          acc[q][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[p][q], g[p][c], acc[q][c], 0, 0, 0);
        acc[q][NCT] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[p][q], gx[p], acc[q][NCT], 0, 0, 0);
      }
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    lv[q] = sum_groups(lv[q]);
    if (lane < 16) s_lv[wave][16 * q + lane] = lv[q];
    if (q) __syncthreads();
#pragma unroll
    for (int c = 0; c <= NCT; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) s_acc[((c * BR_NW + wave) * 4 + r) * WAVE + lane] = acc[q][c][r];
    __syncthreads();
    for (int c = wave; c <= NCT; c += BR_NW) {
      if (c == NCT && !a.dx_part) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < BR_NW; ++w) t += s_acc[((c * BR_NW + w) * 4 + r) * WAVE + lane];
        const int j = j0 + 16 * q + 4 * grp + r, cc = 16 * c + col;
        if (j >= N) continue;
        const size_t at = (size_t)bh * N + j;
        if (c == NCT) {
          if (col < 3) a.dx_part[at * 3 + col] = t;
        } else if (cc < d) {
          a.dV[at * d + cc] = t;
        }
      }
    }
  }
  if (threadIdx.x < 32 && j0 + threadIdx.x < (unsigned)N) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < BR_NW; ++w) t += s_lv[w][threadIdx.x];
    a.dlog_v[(size_t)bh * N + j0 + threadIdx.x] = -a.eps[h] * t;
  }
}

// dx_res[b, j] = sum_h dx_part[b, h, j] (fixed order).
__global__ void dense_transport_dx_kernel(DenseTransportArgs a) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)a.B * a.N * 3) return;
  const int b = (int)(t / ((size_t)a.N * 3));
  const size_t rem = t - (size_t)b * a.N * 3;
  float s = 0.f;
  for (int h = 0; h < a.H; ++h) s += a.dx_part[((size_t)b * a.H + h) * a.N * 3 + rem];
  a.dx_res[t] = s;
}

// ---------------------------------------------------------------------------
static unsigned blocks_for(size_t n, int per) { return (unsigned)((n + per - 1) / per); }

hipError_t dense_sinkhorn_init(const DenseSinkArgs& a, hipStream_t s) {
  const size_t BHN = (size_t)a.B * a.H * a.N;
  const size_t n = std::max(BHN, (size_t)2 * (a.K + 1));
  hipLaunchKernelGGL(dense_init_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}
// rows of these arrays (N floats each, from these bases) can be read as float4
static bool rows16(int N, const void* p, const void* q = nullptr, const void* r = nullptr) {
  return N % 4 == 0 && (((uintptr_t)p | (uintptr_t)q | (uintptr_t)r) & 15) == 0;
}

hipError_t dense_sinkhorn_iteration(const DenseSinkArgs& a, int k, hipStream_t s) {
  const dim3 rows((unsigned)(a.B * a.H) * blocks_for(a.N, DN_NW)), cols((unsigned)(a.B * a.H) * blocks_for(a.N, CP_COLS));
  if (rows16(a.N, a.C, a.hist_v, a.mask)) {
    hipLaunchKernelGGL((dense_row_update_kernel<4>), rows, dim3(DN_NT), 0, s, a, k);
    hipLaunchKernelGGL((dense_col_update_kernel<4>), cols, dim3(CP_NT), 0, s, a, k);
  } else {
    hipLaunchKernelGGL((dense_row_update_kernel<1>), rows, dim3(DN_NT), 0, s, a, k);
    hipLaunchKernelGGL((dense_col_update_kernel<1>), cols, dim3(CP_NT), 0, s, a, k);
  }
  return hipGetLastError();
}
hipError_t dense_sinkhorn_finish(const DenseSinkArgs& a, int k, hipStream_t s) {
  const size_t BHN = (size_t)a.B * a.H * a.N;
  hipLaunchKernelGGL(dense_finish_kernel, dim3(blocks_for(BHN, 256)), dim3(256), 0, s, a, k);
  return hipGetLastError();
}
template <int VEC> static void backward_passes(const DenseSinkBwdArgs& a, hipStream_t s) {
  const dim3 rows((unsigned)(a.B * a.H) * blocks_for(a.N, DN_NW)), cols((unsigned)(a.B * a.H) * blocks_for(a.N, CP_COLS));
  const int per = ((a.N + WAVE * VEC - 1) / (WAVE * VEC)) * ((a.N + CG_ROWS - 1) / CG_ROWS);
  const dim3 cost((unsigned)(a.B * a.H) * blocks_for(per, DN_NW));
  const auto slot = [&](int k) { return (a.K - k) % (DENSE_SEG + 1); };
  for (int k = a.K, k1 = a.K; k >= 1; --k) {
    hipLaunchKernelGGL((dense_bwd_row_kernel<VEC>), rows, dim3(DN_NT), 0, s, a, k, slot(k));
    hipLaunchKernelGGL((dense_bwd_col_kernel<VEC>), cols, dim3(CP_NT), 0, s, a, k, slot(k), slot(k - 1));
    if (k == 1 || k1 - k + 1 == DENSE_SEG) {
      hipLaunchKernelGGL((dense_bwd_cost_kernel<VEC>), cost, dim3(DN_NT), 0, s, a, k1, k);
      k1 = k - 1;
    }
  }
}
hipError_t dense_sinkhorn_backward(const DenseSinkBwdArgs& a, hipStream_t s) {
  const size_t BHN = (size_t)a.B * a.H * a.N;
  hipLaunchKernelGGL(dense_bwd_init_kernel, dim3(blocks_for(BHN, 256)), dim3(256), 0, s, a);
  // the cost pass also reads the history's and the workspace's vectors as float4
  if (rows16(a.N, a.C, a.dC) && rows16(a.N, a.hist_c, a.hist_v, a.gv)) backward_passes<4>(a, s);
  else backward_passes<1>(a, s);
  hipLaunchKernelGGL(dense_bwd_finish_kernel, dim3(blocks_for(BHN, 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t dense_zero(float* p, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(dense_zero_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}
template <int VEC, int NCT> static void transport_fwd(const DenseTransportArgs& a, dim3 grid, hipStream_t s) {
  if (a.N <= RP_COLS) hipLaunchKernelGGL((dense_transport_fwd_kernel<VEC, NCT, true>), grid, dim3(DN_NT), 0, s, a);
  else hipLaunchKernelGGL((dense_transport_fwd_kernel<VEC, NCT, false>), grid, dim3(DN_NT), 0, s, a);
}
hipError_t dense_transport_forward(const DenseTransportArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.H * ((a.N + TF_ROWS - 1) / TF_ROWS)));
  const bool v4 = rows16(a.N, a.C, a.T_norm) && rows16(a.N, a.log_v, a.mask);
  if (v4) {
    if (a.d <= 16) transport_fwd<4, 1>(a, grid, s);
    else if (a.d <= 32) transport_fwd<4, 2>(a, grid, s);
    else transport_fwd<4, 4>(a, grid, s);
  } else {
    if (a.d <= 16) transport_fwd<1, 1>(a, grid, s);
    else if (a.d <= 32) transport_fwd<1, 2>(a, grid, s);
    else transport_fwd<1, 4>(a, grid, s);
  }
  return hipGetLastError();
}
template <int VEC, int DP> static void transport_bwd_rows(const DenseTransportArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.H * ((a.N + 15) / 16)));
  if ((a.N + 15) / 16 <= BR_KEEP * BR_NW)
    hipLaunchKernelGGL((dense_transport_bwd_row_kernel<VEC, DP, true>), grid, dim3(BR_NT), 0, s, a);
  else hipLaunchKernelGGL((dense_transport_bwd_row_kernel<VEC, DP, false>), grid, dim3(BR_NT), 0, s, a);
}
hipError_t dense_transport_backward(const DenseTransportArgs& a, hipStream_t s) {
  const bool v4 = rows16(a.N, a.T_norm, a.grad_T, a.dC);
  const int dp = a.d <= 16 ? 16 : a.d <= 32 ? 32 : 64;
  if (v4) {
    if (dp == 16) transport_bwd_rows<4, 16>(a, s);
    else if (dp == 32) transport_bwd_rows<4, 32>(a, s);
    else transport_bwd_rows<4, 64>(a, s);
  } else {
    if (dp == 16) transport_bwd_rows<1, 16>(a, s);
    else if (dp == 32) transport_bwd_rows<1, 32>(a, s);
    else transport_bwd_rows<1, 64>(a, s);
  }
  const dim3 cols((unsigned)(a.B * a.H * ((a.N + 31) / 32)));
  if (dp == 16) hipLaunchKernelGGL((dense_transport_bwd_col_kernel<1>), cols, dim3(BR_NT), 0, s, a);
  else if (dp == 32) hipLaunchKernelGGL((dense_transport_bwd_col_kernel<2>), cols, dim3(BR_NT), 0, s, a);
  else hipLaunchKernelGGL((dense_transport_bwd_col_kernel<4>), cols, dim3(BR_NT), 0, s, a);
  if (a.dx_res && a.dx_part)
    hipLaunchKernelGGL(dense_transport_dx_kernel, dim3(blocks_for((size_t)a.B * a.N * 3, 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace dfl
