// Backwards with the plan in registers: unrolled (balanced transport and UOT flash-Sinkhorn) and
// implicit (UOT).
//
// The plans of all half-iterations share one matrix: with E_ij = exp(L_ij + alpha_i + beta_j)
// and the last iteration's potentials as alpha, beta (E = P, rows summing to 1),
//   s^{C,k}_ij = E_ij AC_k(i) BC_k(j),   s^{R,k}_ij = E_ij AR_k(i) BR_k(j),
// where the factors are exponentials of differences of recorded potentials:
//   balanced: AC_k = AR_k = exp(u^{k-1}_i - u^{K-1}_i), BR_k = BC_{k-1} = exp(v^{k-1}_j - v^{K-1}_j),
//   UOT:      AC_k = exp(u^k_i - alpha_i),  AR_k = exp(u^k_i/kappa - log mu_i - alpha_i),
//             BR_k = exp(v^{k-1}_j - beta_j), BC_k = exp(v^k_j/kappa - log nu_j - beta_j)
// (u^{-1} = 0 in the balanced transport, v^{-1} = v_init; kappa = 1 in the balanced one).
// The recurrences are then one multiply-add per element and sweep,
//   g^k_i = -kappa AC_k(i) sum_j E_ij y^k_j,   z^k = AR_k g^k,
//   h^{k-1}_j = -kappa BR_k(j) sum_i E_ij z^k_i,   y^{k-1} = BC_{k-1} h^{k-1},
// and the cost gradient of all iterations is eps dC = W0 + kappa E o R with the rank-2K matrix
//   R_ij = sum_k AC_k(i) y^k_j + z^k_i BR_k(j),
// formed once per orientation by fp32 MFMAs; dQ, dK, dV, the coordinate and weight gradients
// follow in that one pass.  The sweeps that recompute the cost and form both terms of every
// iteration (balanced_bwd.hip, unrolled_bwd.hip) took 7-8 us each; these take about 1.5-2 us.
//
// The implicit (IFT) backward is the same with one pair of factors: S_row = E, S_col = E AC BC with
// AC_i = exp(log Z_i), BC_j = exp(-(v_j + col_lse_j)), R_ij = -z_u,i -+ AC_i BC_j z_v,j, and its solve
// (fixed point, or CG on W = AC^1/2 E BC^1/2) takes one multiply-add per element and sweep.
//
// A wave keeps E of its pairs in both orientations, as the register forward (reg_ks, reg_nrm).
// Every factor must lie within 2^+-SB_MAX: E <= 1, so an entry that underflows (below 2^-126)
// then stays below 2^-62 in every plan.  The members of a group agree on that from the recorded
// potentials before they begin; a group outside it runs the general sweeps.
#pragma once
#include "sinkhorn_bwd_kernel.h"
#include "sinkhorn_fwd_kernel.h"

namespace dfl {

constexpr int SB_NT = 512, SB_NW = SB_NT / WAVE;
constexpr float SB_MAX = 32.f;  // log2 units
// most iterations the kept vectors are sized for (the workspace size does not depend on K)
constexpr int SB_KMAX = 64;
// kept exchange words of one (b,h): y^k and z^k of every iteration, then the members' verdicts
__host__ __device__ inline size_t sb_step_words(int N) { return (size_t)(2 * SB_KMAX + 1) * (((size_t)N + 31) / 32 * 32); }

// Clears the words that one call with K iterations uses (the workspace is shared with calls that keep
// other data there): called by every thread of the prep kernel's grid.
__device__ __forceinline__ void sb_clear_steps(uint64_t* steps, int BH, int N, int K) {
  if (K > SB_KMAX) return;
  const size_t Np = ((size_t)N + 31) / 32 * 32, per = sb_step_words(N), used = 2 * (size_t)K * Np;
  const size_t threads = (size_t)gridDim.x * blockDim.x, t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t e = t0; e < (size_t)BH * (used + Np); e += threads) {
    const size_t bh = e / (used + Np), r = e - bh * (used + Np);
    steps[bh * per + (r < used ? r : r - used + 2 * (size_t)SB_KMAX * Np)] = 0;
  }
}

template <typename Args> struct is_bal : std::is_same<Args, BalBwdArgs> {};
template <typename Args> struct is_ift : std::is_same<Args, IftBwdArgs> {};

constexpr int SB_BINS = (BIN_NONE + 4) / 4 * 4;  // (the tables are followed by 16-byte reads)

// floats of the region that holds the stripe's factors and vectors (AC, BR, y, z and, UOT, AR, BC)
// during the sweeps and the waves' output partials afterwards
__host__ __device__ inline int sb_region_floats(int N, int G, int K, bool bal) {
  const int loc = fwd_local_rows(N, G);
  const int f = (bal ? 4 : 6) * K * loc, m = (loc / 16) * SB_NW * 8 * WAVE;
  return f > m ? f : m;
}
inline size_t sb_lds_bytes(int N, int G, int K, bool bal) {
  const size_t Np = ((N + 31) / 32) * 32, cpn = reg_cp_rows(N, (int)Np);
  return ((Np + 15) / 16) * 16 + (7 * Np + 2 * cpn + 2 * SB_BINS + 2 * (size_t)SB_NW * SK_RT * 16 + sb_region_floats(N, G, K, bal)) * 4;
}
// IFT: the CG vectors (5 Np) and three vectors of the stripe take the factors' place
inline size_t ift_lds_bytes(int N, int G) {
  const size_t Np = ((N + 31) / 32) * 32, cpn = reg_cp_rows(N, (int)Np), loc = fwd_local_rows(N, G);
  const size_t f = 5 * Np + 3 * loc, m = (loc / 16) * SB_NW * 8 * WAVE;
  return ((Np + 15) / 16) * 16 + (7 * Np + 2 * cpn + 2 * SB_BINS + 2 * (size_t)SB_NW * SK_RT * 16 + (f > m ? f : m)) * 4;
}
// The unrolled forms: shapes whose workspace holds the kept words, and calls that run them.
inline bool sb_fits_shape(int N, int DP, int G) { return DP == 32 && reg_fits(N, G); }
inline bool sb_fits(int N, int DP, int G, int K, bool bal, size_t limit) {
  return sb_fits_shape(N, DP, G) && K >= 1 && K <= SB_KMAX && sb_lds_bytes(N, G, K, bal) + 2048 <= limit;
}

// The kernel's argument struct (its only parameter) for the general sweeps, read anew from where the
// launch put it: nothing that they read is held in registers through the register form.
template <typename Args> __device__ __forceinline__ const Args& fresh_args() {
  typedef const __attribute__((address_space(4))) Args* Place;
  Place p = (Place)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const Args*)p;
}

// T: input type of Q, K and of the gradients; GEN: the cost may carry bins or geometry (always in
// the balanced mode).  Returns, uniformly over the workgroup, whether the general sweeps have to run: a group
// whose factors are out of range, and a member that owns nothing (they do its part of the zeroing).
// The kernels inline them behind this one test, where nothing of the register form is live.  As a call
// with the arguments by value they read sizes, pointers and branch conditions per lane from its stack.
// Every group out of range, us, in a kernel of their own / as a call / so: implicit, bf16, 16 heads of
// 768 tokens, 20 CG steps 201 / 530 / 207; unrolled, fp32, 16 heads of 300 with bins and geometry
// 1054 / 1645 / 1070; balanced, 16 heads of 256, K 20 309 / 325 / 314.
template <typename T, bool GEN, typename Args>
__device__ __forceinline__ bool scaled_bwd(const Args& a) {
  constexpr bool BAL = is_bal<Args>::value, IFT = is_ift<Args>::value, UNR = !BAL && !IFT;
  constexpr int DP = 32, NC = DP / 16;
  using MQ = Mfma<T, DP>;
  using M = Mfma<float, DP>;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_flagp[2], s_tmp, s_flag, s_local, s_ok, s_cnt;
  __shared__ float sscal[2 * SB_NW], s_red[2 * SB_NW];
  int grp, member;
  if (!group_of(a.B * a.H, a.G, grp, member)) return false;
  const int b = grp / a.H, h = grp % a.H;
  const int N = a.N, d = a.d, BH = a.B * a.H;
  int K = 0;  // (IFT: no recorded iterations)
  if constexpr (!IFT) K = a.K;
  const int Np = ((N + 31) / 32) * 32;
  const size_t bh = (size_t)grp, bhN = bh * N;
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  if (tid == 0) { s_flagp[0] = s_flagp[1] = 0; s_flag = 0; s_local = 1; s_ok = 1; s_cnt = 0; }
  if (blockIdx.x == 0 && tid == 0)
    __hip_atomic_store(a.err.ws + 1, a.salt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // ---- LDS carve-up (must match sb_lds_bytes)
  unsigned char* valid = smem;
  float* xs = reinterpret_cast<float*>(smem + ((Np + 15) / 16) * 16);  // coordinates [Np][3]
  float* gx = xs + 3 * Np;                                             // grad x_c [Np][3]
  float* dcf = gx + 3 * Np;                                            // D
  const int cpn = reg_cp_rows(N, Np), loc = fwd_local_rows(N, a.G);
  float* wY = dcf + Np;   // beta (log2), then y^k of this wave's streamed columns
  float* wZ = wY + cpn;   // alpha (log2), then z^k of this wave's streamed rows
  float* s_posw = wZ + cpn;                        // bin weights in the exponent, and their gradients
  float* s_dpw = s_posw + SB_BINS;
  float* scratch = s_dpw + SB_BINS;                // two slots of wave partials
  float* region = scratch + 2 * SB_NW * SK_RT * 16;
  float* AC = region;                              // [K][loc] each
  float* BR = AC + (size_t)K * loc;
  float* Yo = BR + (size_t)K * loc;
  float* Zo = Yo + (size_t)K * loc;
  float* AR = BAL ? AC : Zo + (size_t)K * loc;
  float* BC = BAL ? nullptr : AR + (size_t)K * loc;
  // IFT: CG vectors [Np] each (region), then z_u, BC z_v and AC of my rows / columns
  float* cy = region;
  float* cr = cy + Np;
  float* cp = cr + Np;
  float* cs = cp + Np;
  float* bch = cs + Np;
  float* zo = bch + Np;
  float* yo = zo + loc;
  float* ao = yo + loc;

  const int n = mask_setup(a.mask ? a.mask + (size_t)b * N : nullptr, N, valid, &s_tmp);
  const int n_tiles = (n + 15) / 16;
  int t0, t1;
  stripe(n_tiles, member, a.G, t0, t1);
  const int nr = t1 - t0, r_lo = t0 * 16;
  if (n == 0 || nr <= 0) return true;
  // ---- factors of my stripe, and whether they are in range
  const float eps = a.eps[h];
  float w_bal = 0.f, kappa = 1.f, wd = 0.f, lm2 = 0.f;
  if constexpr (BAL) {
    int c = 0;
    for (int i = tid; i < n; i += SB_NT) c += valid[i];
    atomicAdd(&s_cnt, c);
    __syncthreads();
    lm2 = -log2f((float)max(s_cnt, 1));
    w_bal = 1.f / (1.f + __expf(-a.alpha[h]));
  } else {
    kappa = a.lam / (a.lam + eps);
    wd = a.w_dist ? a.w_dist[h] : 0.f;
    if (tid <= (int)BIN_NONE) {
      s_posw[tid] = a.pos_w && tid < (int)BIN_NONE ? -LOG2E * a.pos_w[h * 68 + tid] / eps : 0.f;
      s_dpw[tid] = 0.f;
    }
  }
  const float ik = 1.f / kappa;
  const float* hist = nullptr;
  if constexpr (!IFT) hist = a.hist;
  auto Uat = [&](int k) { return hist + ((size_t)(2 * k + 1) * BH + bh) * N; };
  auto Vat = [&](int k) { return hist + ((size_t)(2 * k) * BH + bh) * N; };
  // natural units; alpha without the balanced beta's -lm
  auto alpha_of = [&](int i) -> float {
    if constexpr (BAL) return Uat(K - 1)[i];
    else return a.log_u[bhN + i] - a.log_z[bhN + i];
  };
  auto beta_of = [&](int j) -> float {
    if constexpr (IFT) return a.log_v[bhN + j];
    else return Vat(K - 1)[j];
  };
  auto vprev = [&](int k, int j) -> float {  // v^{k-1}
    if (k >= 1) return Vat(k - 1)[j];
    if constexpr (!UNR) return 0.f;
    else return a.v_init ? a.v_init[bhN + j] : 0.f;
  };
  auto urow = [&](int k, int i) -> float {  // the row potential of AC_k
    if constexpr (BAL) return k >= 1 ? Uat(k - 1)[i] : 0.f;
    else return Uat(k)[i];
  };
  {
    bool in = true;
    for (int e = tid; e < K * nr * 16; e += SB_NT) {
      const int k = e / (nr * 16), q = e % (nr * 16), i = r_lo + q;
      float ac = 0.f, br = 0.f, ar = 0.f, bc = 0.f;
      if (i < n && valid[i]) {
        const float al = alpha_of(i), be = beta_of(i), u = urow(k, i);
        const float ea = (u - al) * LOG2E, eb = (vprev(k, i) - be) * LOG2E;
        in = in && fabsf(ea) <= SB_MAX;
        if (!BAL || k >= 1) in = in && fabsf(eb) <= SB_MAX;
        ac = fast_exp2(ea);
        br = BAL && k == 0 ? 0.f : fast_exp2(eb);
        if constexpr (UNR) {
          const float er = (u * ik - a.log_mu[bhN + i] - al) * LOG2E;
          const float ec = (Vat(k)[i] * ik - a.log_nu[bhN + i] - be) * LOG2E;
          in = in && fabsf(er) <= SB_MAX && fabsf(ec) <= SB_MAX;
          ar = fast_exp2(er);
          bc = fast_exp2(ec);
        }
      }
      AC[(size_t)k * loc + q] = ac;
      BR[(size_t)k * loc + q] = br;
      Yo[(size_t)k * loc + q] = Zo[(size_t)k * loc + q] = 0.f;
      if constexpr (UNR) {
        AR[(size_t)k * loc + q] = ar;
        BC[(size_t)k * loc + q] = bc;
      }
    }
    if constexpr (IFT) {
      for (int q = tid; q < nr * 16; q += SB_NT) {
        const int i = r_lo + q;
        if (i < n && valid[i])
          in = in && fabsf(a.log_z[bhN + i] * LOG2E) <= SB_MAX &&
               fabsf((a.log_v[bhN + i] + a.col_lse[bhN + i]) * LOG2E) <= SB_MAX;
      }
    }
    if (!in) s_ok = 0;  // (the same value from every writer)
  }
  __syncthreads();
  uint64_t* steps;
  uint64_t* verdicts;
  if constexpr (IFT) {
    steps = a.xch + bh * 4 * (size_t)Np;  // three vectors reused by every iteration; the fourth is free
    verdicts = steps + 3 * (size_t)Np;
  } else {
    steps = a.steps + bh * sb_step_words(N);
    verdicts = steps + (size_t)2 * SB_KMAX * Np;
  }
  const uint32_t salt = a.salt << 12;
  if (tid == 0) xch_put(verdicts + member, (s_ok ? 0.f : 2.f) + (xcc_placed() ? 0.f : 1.f), salt | 1u);
  for (int i = tid; i < Np; i += SB_NT) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      xs[3 * i + c] = a.xs[((size_t)b * 3 + c) * Np + i];
      gx[3 * i + c] = a.gxs[(bh * 3 + c) * Np + i];
    }
    dcf[i] = a.dcoef[bh * Np + i];
  }
  for (int i = tid; i < cpn; i += SB_NT) {
    const bool ok = i < n && valid[i];
    wY[i] = ok ? beta_of(i) * LOG2E - lm2 : NEG_BIG;
    wZ[i] = ok ? alpha_of(i) * LOG2E : NEG_BIG;
  }
  {  // the group's verdict: placement (as read_placement) and range
    if (tid < a.G && (long long)n_tiles * (tid + 1) / a.G > (long long)n_tiles * tid / a.G) {
      const int idx[1] = {tid};
      const bool got = poll_words<1>(verdicts, idx, salt | 1u, a.err, [&](int, uint64_t w) {
        const float v = __uint_as_float((uint32_t)(w >> 32));
        if (v >= 2.f) s_ok = 0;
        if (v == 1.f || v == 3.f) s_local = 0;
      });
      if (!got) s_flag = 1;
    }
    __syncthreads();
    if (s_flag) return false;
    if (!s_ok) return true;
  }
  const bool local = s_local != 0;
  // rows past the last valid tile belong to no stripe: zeroed here (row i by member i % G)
  for (int i = n_tiles * 16 + member; i < N; i += a.G) {
    for (int c = tid; c < d; c += SB_NT) {
      reinterpret_cast<T*>(a.dq)[(bhN + i) * d + c] = from_f32<T>(0.f);
      reinterpret_cast<T*>(a.dk)[(bhN + i) * d + c] = from_f32<T>(0.f);
      if (a.dv) reinterpret_cast<T*>(a.dv)[(bhN + i) * d + c] = from_f32<T>(0.f);
    }
    if (tid < 3) a.dx_part[(bhN + i) * 3 + tid] = 0.f;
    if constexpr (!BAL)
      if (tid == 0) a.dlog_mu[bhN + i] = a.dlog_nu[bhN + i] = 0.f;
    if constexpr (UNR)
      if (tid == 0 && a.dv_init) a.dv_init[bhN + i] = 0.f;
  }
  float sc, r0;
  bool geo, use_bins = false, has_h = true;
  Bias bias;
  bias.b8 = bias.b8t = nullptr;
  if constexpr (BAL) {
    sc = LOG2E * (1.f - w_bal) / eps;
    r0 = fmaxf(fabsf(a.r_h[h]), 0.1f);
    bias.geo_scale = -LOG2E * w_bal / eps;
    geo = true;
    has_h = a.has_h != 0;
  } else {
    sc = LOG2E / (sqrtf((float)d) * eps);
    r0 = a.r0;
    bias.geo_scale = -LOG2E * wd / eps;
    // (IFT: d w_dist is non-zero even where w_dist == 0)
    if constexpr (IFT) geo = GEN && a.x != nullptr && a.w_dist != nullptr;
    else geo = GEN && a.has_geo != 0 && wd != 0.f;
    use_bins = GEN && a.bins8 != nullptr && a.pos_w != nullptr;
    if (use_bins) {
      bias.b8 = a.bins8 + (size_t)b * Np * Np;
      bias.b8t = a.bins8t + (size_t)b * Np * Np;
    }
  }
  bias.posw = s_posw;
  bias.xs = geo ? xs : nullptr;
  bias.r0 = r0;
  bias.Np = Np;
  const bool general_cost = GEN && (geo || use_bins);
  const T* qp = reinterpret_cast<const T*>(a.qp) + bh * Np * DP;
  const T* kp = reinterpret_cast<const T*>(a.kp) + bh * Np * DP;
  const T* qt = reinterpret_cast<const T*>(a.qt) + bh * DP * Np;
  const T* kt = reinterpret_cast<const T*>(a.kt) + bh * DP * Np;
  const float* vp = has_h ? a.vp + bh * Np * DP : nullptr;
  const float* gp = has_h ? a.gp + bh * Np * DP : nullptr;
  const float* gt = has_h ? a.gt + bh * DP * Np : nullptr;

  auto run = [&](auto ksc) __attribute__((always_inline)) {
    constexpr int KSL = decltype(ksc)::value;
    constexpr int NRM = reg_nrm(KSL);
    if (nr > NRM) {  // the host's sb_fits rules this out
      if (tid == 0) raise_error(a.err, a.salt, 3u);
      return;
    }
    // ---- E of the wave's pairs: X[r KSL + k], resident tile r against streamed tile wave + 8 k
    f32x4 XR[NRM * KSL], XC[NRM * KSL];
    auto form = [&](auto rowc, f32x4(&X)[NRM * KSL]) __attribute__((always_inline)) {
      constexpr bool ROW = decltype(rowc)::value;
      uint32_t words[GEN ? NRM * KSL : 1];
      if constexpr (GEN && !BAL) {
#pragma unroll
        for (int r = 0; r < NRM; ++r)
#pragma unroll
          for (int k = 0; k < KSL; ++k) {
            const int st = wave + SB_NW * k;
            words[r * KSL + k] = r < nr && st < n_tiles
                                     ? bias.template word<!ROW>((t0 + r) * 16 + (lane & 15), st * 16 + 4 * g) : 0u;
          }
      }
      const float* ps = ROW ? wY : wZ;  // streamed, resident exponent terms
      const float* pr = ROW ? wZ : wY;
#pragma unroll
      for (int r = 0; r < NRM; ++r) {
        if (r < nr) {
          const int ri = (t0 + r) * 16 + (lane & 15);
          typename MQ::Frag fr;
          MQ::load(fr, (ROW ? qp : kp) + (size_t)ri * DP, lane);
          const float ar = pr[ri];
#pragma unroll
          for (int k = 0; k < KSL; ++k) {
            const int sl = r * KSL + k, st = wave + SB_NW * k;
            X[sl] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (st < n_tiles) {
              typename MQ::Frag fs;
              MQ::load(fs, (ROW ? kp : qp) + (size_t)(st * 16 + (lane & 15)) * DP, lane);
              const f32x4 z = {0.f, 0.f, 0.f, 0.f};
              const f32x4 x = MQ::qk(fs, fr, z);
              const f32x4 sv = *reinterpret_cast<const f32x4*>(ps + st * 16 + 4 * g);
              f32x4 bb = z;
              if (general_cost) bb = bias.from_word(words[GEN && !BAL ? sl : 0], ri, st * 16 + 4 * g);
#pragma unroll
              for (int q = 0; q < 4; ++q) X[sl][q] = fast_exp2(__builtin_fmaf(x[q], sc, bb[q]) + (ar + sv[q]));
            }
            if constexpr (GEN) __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };
    form(std::integral_constant<bool, true>{}, XR);
    form(std::integral_constant<bool, false>{}, XC);

    // ---- the centroid's column sums: h^{K-1}_j = sum_i P_ij (dT_ij - D_i)
    uint32_t phase = 1;
    int chunk = 0;
    auto part_slot = [&]() { return scratch + (chunk++ & 1) * (SB_NW * SK_RT * 16); };
    auto vec3 = [&](const float* p, float (&o)[12]) {
      const f32x4* q = reinterpret_cast<const f32x4*>(p);
      const f32x4 x0 = q[0], x1 = q[1], x2 = q[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) { o[e] = x0[e]; o[4 + e] = x1[e]; o[8 + e] = x2[e]; }
    };
    {
      float* part = part_slot();
      float acc[NRM];
      typename M::Frag rf[NRM];
#pragma unroll
      for (int r = 0; r < NRM; ++r) {
        acc[r] = 0.f;
        if (has_h && r < nr) M::load(rf[r], vp + (size_t)((t0 + r) * 16 + (lane & 15)) * DP, lane);
      }
#pragma unroll
      for (int k = 0; k < KSL; ++k) {
        const int st = wave + SB_NW * k;
        if (st < n_tiles) {
          typename M::Frag cf;
          if (has_h) M::load(cf, gp + (size_t)(st * 16 + (lane & 15)) * DP, lane);
          float gv[12];
          vec3(gx + 3 * (st * 16 + 4 * g), gv);
          const f32x4 D = *reinterpret_cast<const f32x4*>(dcf + st * 16 + 4 * g);
#pragma unroll
          for (int r = 0; r < NRM; ++r) {
            if (r < nr) {
              const int rj = (t0 + r) * 16 + (lane & 15);
              const float x0 = xs[3 * rj], x1 = xs[3 * rj + 1], x2 = xs[3 * rj + 2];
              f32x4 t = {0.f, 0.f, 0.f, 0.f};
              if (has_h) t = M::qk(cf, rf[r], t);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float dT = t[e] + (gv[3 * e] * x0 + gv[3 * e + 1] * x1 + gv[3 * e + 2] * x2);
                acc[r] = __builtin_fmaf(XC[r * KSL + k][e], dT - D[e], acc[r]);
              }
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < NRM; ++r)
        if (r < nr) {
          const float ss = sum_groups(acc[r]);
          if (lane < 16) part[(r * 16 + lane) * SB_NW + wave] = ss;
        }
      __syncthreads();  // (also: alpha and beta are read)
    }
    // combining thread of local row / column qc
    const int qc = tid, ic = r_lo + qc;
    const bool has_q = qc < nr * 16, in_c = has_q && ic < n, ok_c = in_c && valid[ic];
    constexpr int NB = (16 * KSL + WAVE - 1) / WAVE;  // words of a lane
    auto words_of = [&](int k, int z) { return steps + (size_t)(2 * k + z) * Np; };
    if constexpr (IFT) {
      uint64_t* xG = steps;
      uint64_t* xZ = steps + Np;
      uint64_t* xY = steps + 2 * (size_t)Np;
      const float lz_c = ok_c ? a.log_z[bhN + ic] * LOG2E : 0.f;
      const float vc_c = ok_c ? (a.log_v[bhN + ic] + a.col_lse[bhN + ic]) * LOG2E : 0.f;
      const float ac_c = ok_c ? fast_exp2(lz_c) : 0.f, bc_c = ok_c ? fast_exp2(-vc_c) : 0.f;
      const float gv_c = has_q ? reg_sum<SB_NW>(scratch, qc) : 0.f;
      float zu_c = 0.f, zv_c = gv_c;
      // No poll writes the entries past the last valid one: zero them in this wave's streamed tiles,
      // where they hold the exponent terms' NEG_BIG (the gradient pass multiplies them by factors of
      // up to 2^SB_MAX, past the float range)
      for (int e = lane; e < 16 * KSL; e += WAVE) {
        const int i = (wave + SB_NW * (e >> 4)) * 16 + (e & 15);
        if (i >= n) wY[i] = wZ[i] = 0.f;
      }
      auto take0 = [&](float* w) {
        return [w](int, int i, float v, bool ok) {
          w[i] = ok ? v : 0.f;
          return 0.f;
        };
      };
      float dm;
      if (a.solver == 0) {
        // Gauss-Seidel (flash_sinkhorn_attn.py:471-542) from z_v = g_v: z_u = kappa S_col z_v,
        // z_v = g_v + kappa S_row^T z_u, with y = BC z_v exchanged
        ++phase;
        if (in_c) xch_put(xY + ic, bc_c * zv_c, salt | phase, local);
        for (int it = 0; it < a.iters; ++it) {
          if (!wave_poll<SB_NW, NB>(xY, n, n_tiles, salt | phase, valid, a.err, dm, take0(wY))) s_flagp[phase & 1] = 1;
          float* part = part_slot();
          reg_scaled<KSL, NRM, SB_NW>(XR, nr, wY, part);
          ++phase;
          lds_barrier();
          if (has_q) {
            zu_c = kappa * ac_c * reg_sum<SB_NW>(part, qc);
            if (in_c) xch_put(xZ + ic, zu_c, salt | phase, local);
          }
          lds_barrier();
          if (s_flagp[(phase - 1) & 1]) return;
          if (!wave_poll<SB_NW, NB>(xZ, n, n_tiles, salt | phase, valid, a.err, dm, take0(wZ))) s_flagp[phase & 1] = 1;
          part = part_slot();
          reg_scaled<KSL, NRM, SB_NW>(XC, nr, wZ, part);
          ++phase;
          lds_barrier();
          if (has_q) {
            zv_c = gv_c + kappa * reg_sum<SB_NW>(part, qc);
            if (in_c) xch_put(xY + ic, bc_c * zv_c, salt | phase, local);
          }
          lds_barrier();
          if (s_flagp[(phase - 1) & 1]) return;
        }
        if (!wave_poll<SB_NW, NB>(xY, n, n_tiles, salt | phase, valid, a.err, dm, take0(wY))) s_flagp[phase & 1] = 1;
        if (a.iters == 0)
          for (int e = lane; e < 16 * KSL; e += WAVE) wZ[min((wave + SB_NW * (e >> 4)) * 16 + (e & 15), cpn - 1)] = 0.f;
        __syncthreads();
        if (s_flagp[phase & 1]) return;
      } else {
        // CG on (I - kappa^2 W^T W) y = BC^1/2 g_v, W = AC^1/2 E BC^1/2; the vectors are kept whole and
        // bit-identical in every member, as in the general backward.  t travels as AC^1/2 t.
        ++phase;
        if (in_c) xch_put(xG + ic, gv_c, salt | phase, local);
        if (!gather_vector(xG, n, Np, salt | phase, cr, valid, a.err, &s_flag)) return;
        for (int i = tid; i < Np; i += SB_NT) {
          const bool ok = i < n && valid[i];
          const float h_ = ok ? fast_exp2(-0.5f * (a.log_v[bhN + i] + a.col_lse[bhN + i]) * LOG2E) : 0.f;
          const float bj = cr[i] * h_;
          bch[i] = h_;
          cy[i] = 0.f;
          cr[i] = bj;
          cp[i] = bj;
        }
        __syncthreads();
        int flip = 0;
        float rr = block_sum(Np, [&](int i) { return cr[i] * cr[i]; }, s_red, flip);
        const bool early_exit = a.cg_rtol > 0.f;
        const float stop2 = a.cg_rtol * a.cg_rtol * rr, k2 = kappa * kappa;
        const float ach_c = ok_c ? fast_exp2(0.5f * lz_c) : 0.f, bch_c = ok_c ? fast_exp2(-0.5f * vc_c) : 0.f;
        float zs[NB], tt[NB], zsum_c = 0.f;
#pragma unroll
        for (int s_ = 0; s_ < NB; ++s_) zs[s_] = tt[s_] = 0.f;
        for (int it = 0; it < a.iters; ++it) {
          if (early_exit && (rr <= stop2 || rr == 0.f)) break;
          // the wave's own streamed columns of BC^1/2 p (it updated them itself)
#pragma unroll
          for (int s_ = 0; s_ < NB; ++s_) {
            const int e = s_ * WAVE + lane, i = (wave + SB_NW * (e >> 4)) * 16 + (e & 15);
            if (e < 16 * KSL && i < n_tiles * 16) wY[i] = bch[i] * cp[i];
          }
          float* part = part_slot();
          reg_scaled<KSL, NRM, SB_NW>(XR, nr, wY, part);
          ++phase;
          lds_barrier();
          float tt_c = 0.f;
          if (has_q) {
            tt_c = ach_c * (ach_c * reg_sum<SB_NW>(part, qc));
            if (in_c) xch_put(xZ + ic, tt_c, salt | phase, local);
          }
          if (!wave_poll<SB_NW, NB>(xZ, n, n_tiles, salt | phase, valid, a.err, dm, [&](int s_, int i, float v, bool ok) {
                wZ[i] = ok ? v : 0.f;
#pragma unroll
                for (int u = 0; u < NB; ++u)
                  if (u == s_) tt[u] = ok ? v : 0.f;
                return 0.f;
              }))
            s_flag = 1;
          part = part_slot();
          reg_scaled<KSL, NRM, SB_NW>(XC, nr, wZ, part);
          ++phase;
          lds_barrier();
          if (has_q && in_c) xch_put(xY + ic, bch_c * reg_sum<SB_NW>(part, qc), salt | phase, local);
          float pAp;
          if (!gather_vector_dot(xY, n, Np, salt | phase, cs, valid, a.err, &s_flag,
                                 [&](int i) { return cp[i] * (cp[i] - k2 * cs[i]); }, s_red, flip, &pAp))
            return;
          if (early_exit && pAp == 0.f) break;
          const float alpha = (pAp != 0.f && rr != 0.f) ? rr / pAp : 0.f;
          const float rr_new = block_sum(Np, [&](int i) {
            cy[i] += alpha * cp[i];
            const float ri = cr[i] - alpha * (cp[i] - k2 * cs[i]);
            cr[i] = ri;
            return ri * ri;
          }, s_red, flip);
          zsum_c += alpha * tt_c;
#pragma unroll
          for (int s_ = 0; s_ < NB; ++s_) zs[s_] += alpha * tt[s_];
          const float beta = rr != 0.f ? rr_new / rr : 0.f;
          rr = rr_new;
          // each wave updates p where its own next row sweep reads it: no barrier
#pragma unroll
          for (int s_ = 0; s_ < NB; ++s_) {
            const int e = s_ * WAVE + lane, i = (wave + SB_NW * (e >> 4)) * 16 + (e & 15);
            if (e < 16 * KSL && i < n_tiles * 16) cp[i] = cr[i] + beta * cp[i];
          }
        }
        zu_c = kappa * zsum_c;
        zv_c = ok_c ? cy[ic] * fast_exp2(0.5f * vc_c) : 0.f;
#pragma unroll
        for (int s_ = 0; s_ < NB; ++s_) {
          const int e = s_ * WAVE + lane, i = (wave + SB_NW * (e >> 4)) * 16 + (e & 15);
          if (e < 16 * KSL && i < n_tiles * 16) {
            wY[i] = bch[i] * cy[i];
            wZ[i] = kappa * zs[s_];
          }
        }
      }
      if (has_q) {
        zo[qc] = ok_c ? zu_c : 0.f;
        yo[qc] = bc_c * zv_c;
        ao[qc] = ac_c;
        if (ic < N) {
          // analytic: d log_mu = kappa lambda_u = -kappa z_u
          a.dlog_mu[bhN + ic] = ok_c ? (a.mode == 1 ? -kappa : kappa) * zu_c : 0.f;
          a.dlog_nu[bhN + ic] = ok_c ? kappa * zv_c : 0.f;
        }
      }
      __syncthreads();
    }
    if constexpr (!IFT) {
    float dmu = 0.f, dnu = 0.f, dv0 = 0.f;
    auto publish_y = [&](int k, float hv) {  // h^k of my column -> y^k
      const float y = BAL ? (k == K - 1 ? hv : BR[(size_t)(k + 1) * loc + qc] * hv) : BC[(size_t)k * loc + qc] * hv;
      Yo[(size_t)k * loc + qc] = ok_c ? y : 0.f;
      if (in_c) xch_put(words_of(k, 0) + ic, y, salt | phase, local);
      dnu += kappa * hv;
    };
    ++phase;
    if (has_q) publish_y(K - 1, reg_sum<SB_NW>(scratch, qc));
    auto take = [&](float* w) {
      return [w](int, int i, float v, bool ok) {
        w[i] = ok ? v : 0.f;
        return 0.f;
      };
    };
    // ---- the recurrences
    constexpr int K_END = BAL ? 1 : 0;
    for (int k = K - 1; k >= K_END; --k) {
      {  // row half: g^k, z^k
        float dm;
        if (!wave_poll<SB_NW, NB>(words_of(k, 0), n, n_tiles, salt | phase, valid, a.err, dm, take(wY)))
          s_flagp[phase & 1] = 1;
        float* part = part_slot();
        reg_scaled<KSL, NRM, SB_NW>(XR, nr, wY, part);
        ++phase;
        lds_barrier();
        if (has_q) {
          const float gk = -kappa * AC[(size_t)k * loc + qc] * reg_sum<SB_NW>(part, qc);
          const float z = AR[(size_t)k * loc + qc] * gk;
          if (in_c) xch_put(words_of(k, 1) + ic, z, salt | phase, local);
          Zo[(size_t)k * loc + qc] = ok_c ? z : 0.f;
          dmu += kappa * gk;
        }
        lds_barrier();
        if (s_flagp[(phase - 1) & 1]) return;
      }
      {  // column half: h^{k-1}, y^{k-1}
        float dm;
        if (!wave_poll<SB_NW, NB>(words_of(k, 1), n, n_tiles, salt | phase, valid, a.err, dm, take(wZ)))
          s_flagp[phase & 1] = 1;
        float* part = part_slot();
        reg_scaled<KSL, NRM, SB_NW>(XC, nr, wZ, part);
        ++phase;
        lds_barrier();
        if (has_q) {
          const float hv = -kappa * BR[(size_t)k * loc + qc] * reg_sum<SB_NW>(part, qc);
          if (k >= 1) publish_y(k - 1, hv);
          else dv0 = hv;
        }
        lds_barrier();
        if (s_flagp[(phase - 1) & 1]) return;
      }
    }
    if constexpr (BAL) {  // y^0 has no row half: the last pass reads its words
      float dm;
      if (!wave_poll<SB_NW, NB>(words_of(0, 0), n, n_tiles, salt | phase, valid, a.err, dm, take(wY)))
        s_flagp[phase & 1] = 1;
      __syncthreads();
      if (s_flagp[phase & 1]) return;
    }
    if constexpr (UNR) {
      if (in_c) {
        a.dlog_mu[bhN + ic] = ok_c ? dmu : 0.f;
        a.dlog_nu[bhN + ic] = ok_c ? dnu : 0.f;
        if (a.dv_init) a.dv_init[bhN + ic] = ok_c ? dv0 : 0.f;
      } else if (has_q && ic < N) {
        a.dlog_mu[bhN + ic] = a.dlog_nu[bhN + ic] = 0.f;
        if (a.dv_init) a.dv_init[bhN + ic] = 0.f;
      }
    }
    __syncthreads();
    }

    // ---- the cost gradient and everything that follows from it, one pass per orientation
    float gb[NRM][3], xt[NRM][3], s_al = 0.f, s_r = 0.f, s_w = 0.f;
    f32x4 dQa[NRM][NC], dKa[NRM][NC], dVa[NRM][NC];
#pragma unroll
    for (int r = 0; r < NRM; ++r) {
#pragma unroll
      for (int c = 0; c < 3; ++c) gb[r][c] = xt[r][c] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) dQa[r][c] = dKa[r][c] = dVa[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto ldf = [](const float* p) { return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto pass = [&](auto rowc, f32x4(&X)[NRM * KSL]) __attribute__((always_inline)) {
      constexpr bool ROW = decltype(rowc)::value;
      const int nst = (K + 1) / 2;
      constexpr int UB = 8;  // factors of a lane in flight together: 16 iterations
      // MFMA slot of this lane: iteration 2 s + (g >> 1), first (AC y) or second (z BR) term
      const bool second = g & 1;
      const bool from_words = ROW ? !second : second;  // the streamed factor: an exchanged vector, else potentials
      constexpr bool shifted = BAL || ROW;  // the potentials of the previous iteration
      const long long pstep = from_words ? 8ll * Np : 4ll * BH * N;
      const float* Bres = ROW ? (second ? Zo : AC) : (second ? BR : Yo);
#pragma unroll
      for (int k = 0; k < KSL; ++k) {
        const int st = wave + SB_NW * k;
        if (st < n_tiles) {
          f32x4 R[NRM];
#pragma unroll
          for (int r = 0; r < NRM; ++r) R[r] = f32x4{0.f, 0.f, 0.f, 0.f};
          const int si = st * 16 + (lane & 15);
          const bool sok = si < n && valid[si];
          float sbase = 0.f;
          if constexpr (!IFT) sbase = sok ? (ROW ? beta_of(si) : alpha_of(si)) : 0.f;
          // the tile's operands, in flight with the first batch of factors
          typename M::Frag cf;
          typename MQ::Frag fs;
          reg_vt<T> op[NC];
          f32x4 go[NC];
          if (has_h) M::load(cf, (ROW ? vp : gp) + (size_t)si * DP, lane);
          if (BAL && ROW) MQ::load(fs, kp + (size_t)si * DP, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const size_t o = (size_t)(c * 16 + (lane & 15)) * Np + st * 16 + 4 * g;
            op[c] = *reinterpret_cast<const reg_vt<T>*>((ROW ? kt : qt) + o);
            if (!ROW && has_h) go[c] = *reinterpret_cast<const f32x4*>(gt + o);
          }
          if constexpr (!IFT) {
          // this lane's streamed factor of iteration kk = 2 s + (g >> 1), one pointer step a slot
          const float* p = from_words ? reinterpret_cast<const float*>(words_of(g >> 1, ROW ? 0 : 1) + si) + 1
                                      : hist + ((long long)(2 * ((g >> 1) - (shifted ? 1 : 0)) + (ROW ? 0 : 1)) * BH + (long long)bh) * N + si;
          const float* bp = Bres + (size_t)(g >> 1) * loc + (lane & 15);
          int kk = g >> 1;
          for (int s0 = 0; s0 < nst; s0 += UB) {
            float av[UB];
            bool live[UB];
#pragma unroll
            for (int u = 0; u < UB; ++u) {
              live[u] = sok && kk < K;
              // (a shifted potential has no entry for iteration 0)
              const bool init = u == 0 && kk == 0 && shifted && !from_words;
              av[u] = ldf(live[u] && !init ? p : hist);
              if (u == 0 && init) av[u] = ROW ? vprev(0, min(si, N - 1)) : 0.f;
              if (BAL && ROW && u == 0 && kk == 0 && second) live[u] = false;  // z^0 is zero
              if (BAL && !ROW && u == 0 && kk == 0 && second) live[u] = false;
              p += pstep;
              kk += 2;
            }
            int kb = kk - 2 * UB;
#pragma unroll
            for (int u = 0; u < UB; ++u) {
              float v = from_words ? av[u] : fast_exp2((av[u] - sbase) * LOG2E);
              v = live[u] ? v : 0.f;
              const float* bq = kb < K ? bp : Bres + (lane & 15);  // past K the streamed factor is zero
#pragma unroll
              for (int r = 0; r < NRM; ++r)
                if (r < nr) R[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, bq[r * 16], R[r], 0, 0, 0);
              bp += 2 * loc;
              kb += 2;
            }
          }
          } else {
            // R_ij = -z_u,i + sgn AC_i y_j (sgn -1, analytic +1)
            const float sgn = a.mode == 1 ? 1.f : -1.f;
            const f32x4 wv = *reinterpret_cast<const f32x4*>((ROW ? wY : wZ) + st * 16 + 4 * g);
            f32x4 as = {0.f, 0.f, 0.f, 0.f};
            if (!ROW) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int i = st * 16 + 4 * g + e;
                if (i < n && valid[i]) as[e] = sgn * fast_exp2(a.log_z[bhN + i] * LOG2E);
              }
            }
#pragma unroll
            for (int r = 0; r < NRM; ++r)
              if (r < nr) {
                const int q = r * 16 + (lane & 15);
                const float m = ROW ? sgn * ao[q] : yo[q], z0 = ROW ? zo[q] : 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) R[r][e] = ROW ? __builtin_fmaf(m, wv[e], -z0) : __builtin_fmaf(as[e], m, -wv[e]);
              }
          }
          float xv[12], gv[12];
          vec3(xs + 3 * (st * 16 + 4 * g), xv);
          f32x4 D = {0.f, 0.f, 0.f, 0.f};
          if (!ROW) {
            vec3(gx + 3 * (st * 16 + 4 * g), gv);
            D = *reinterpret_cast<const f32x4*>(dcf + st * 16 + 4 * g);
          }
#pragma unroll
          for (int r = 0; r < NRM; ++r) {
            if (r < nr) {
              const int ri = (t0 + r) * 16 + (lane & 15);
              const f32x4 z = {0.f, 0.f, 0.f, 0.f};
              f32x4 t = z, x = z;
              if (has_h) {
                typename M::Frag rf;
                M::load(rf, (ROW ? gp : vp) + (size_t)ri * DP, lane);
                t = M::qk(cf, rf, z);
              }
              if (BAL && ROW) {
                typename MQ::Frag fr;
                MQ::load(fr, qp + (size_t)ri * DP, lane);
                x = MQ::qk(fs, fr, z);
              }
              const float xr0 = xs[3 * ri], xr1 = xs[3 * ri + 1], xr2 = xs[3 * ri + 2];
              float gr0 = 0.f, gr1 = 0.f, gr2 = 0.f, Dr = 0.f;
              if (ROW) {
                gr0 = gx[3 * ri];
                gr1 = gx[3 * ri + 1];
                gr2 = gx[3 * ri + 2];
                Dr = dcf[ri];
              }
              uint32_t bw = 0;
              if constexpr (GEN && !BAL && ROW)
                if (use_bins) bw = bias.template word<false>(ri, st * 16 + 4 * g);
              float W[4], P[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float p = X[r * KSL + k][e];
                P[e] = p;
                float dT = t[e];
                if (ROW) dT += gr0 * xv[3 * e] + gr1 * xv[3 * e + 1] + gr2 * xv[3 * e + 2];
                else dT += gv[3 * e] * xr0 + gv[3 * e + 1] * xr1 + gv[3 * e + 2] * xr2;
                const float wv = __builtin_fmaf(kappa * p, R[r][e], -p * (dT - (ROW ? Dr : D[e])));
                W[e] = wv;
                if (!ROW) {
                  xt[r][0] = __builtin_fmaf(p, gv[3 * e], xt[r][0]);
                  xt[r][1] = __builtin_fmaf(p, gv[3 * e + 1], xt[r][1]);
                  xt[r][2] = __builtin_fmaf(p, gv[3 * e + 2], xt[r][2]);
                }
                if (GEN && geo) {
                  const float dx = xr0 - xv[3 * e], dy = xr1 - xv[3 * e + 1], dz = xr2 - xv[3 * e + 2];
                  const float dist = fmaxf(sqrtf(dx * dx + dy * dy + dz * dz), 1e-8f);
                  const float cg = dist / (r0 + dist), om = 1.f - cg;
                  const float f = wv * om * om / dist;
                  gb[r][0] = __builtin_fmaf(f, dx, gb[r][0]);
                  gb[r][1] = __builtin_fmaf(f, dy, gb[r][1]);
                  gb[r][2] = __builtin_fmaf(f, dz, gb[r][2]);
                  if (ROW) {
                    if constexpr (BAL) {
                      s_al = __builtin_fmaf(wv, cg - 1.f + x[e], s_al);
                      s_r = __builtin_fmaf(wv, cg * om, s_r);
                    } else {
                      s_w = __builtin_fmaf(wv, cg, s_w);
                    }
                  }
                }
                if constexpr (GEN && !BAL && ROW)
                  if (use_bins) {
                    const unsigned bin = (bw >> (8 * e)) & 0xffu;
                    if (bin < BIN_NONE && wv != 0.f) atomicAdd(&s_dpw[bin], wv);
                  }
              }
#pragma unroll
              for (int c = 0; c < NC; ++c) {
                if (ROW) dQa[r][c] = reg_pv(W, op[c], dQa[r][c]);
                else dKa[r][c] = reg_pv(W, op[c], dKa[r][c]);
                if (!ROW && has_h) dVa[r][c] = reg_pv(P, go[c], dVa[r][c]);
              }
            }
            __builtin_amdgcn_sched_barrier(0);  // one pair's terms live at a time
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // one tile's operands live at a time
      }
    };
    pass(std::integral_constant<bool, true>{}, XR);
    pass(std::integral_constant<bool, false>{}, XC);
    // ---- outputs of my stripe: the waves' partials meet in the region, dead now
    auto write_rows = [&](f32x4(&acc)[NRM][NC], void* out, float scale) __attribute__((always_inline)) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < NRM; ++r)
        if (r < nr) {
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) region[((size_t)(wave * nr + r) * 8 + 4 * c + e) * WAVE + lane] = acc[r][c][e];
        }
      __syncthreads();
      for (int e = tid; e < nr * 8 * WAVE; e += SB_NT) {
        float v = 0.f;
#pragma unroll
        for (int w_ = 0; w_ < SB_NW; ++w_) v += region[(size_t)w_ * nr * 8 * WAVE + e];
        const int l = e & (WAVE - 1), ce = (e / WAVE) & 7, r = e / (8 * WAVE);
        const int row = (t0 + r) * 16 + 4 * (l >> 4) + (ce & 3), col = (ce >> 2) * 16 + (l & 15);
        if (row < N && col < d)
          reinterpret_cast<T*>(out)[(bhN + row) * d + col] = from_f32<T>((row < n && valid[row]) ? scale * v : 0.f);
      }
    };
    const float fs = BAL ? -(1.f - w_bal) / eps : -1.f / (sqrtf((float)d) * eps);
    write_rows(dQa, a.dq, fs);
    write_rows(dKa, a.dk, fs);
    if (a.dv) write_rows(dVa, a.dv, 1.f);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NRM; ++r)
      if (r < nr) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float s0 = sum_groups(gb[r][c]), s1 = sum_groups(xt[r][c]);
          if (lane < 16) {
            region[((size_t)(wave * nr + r) * 16 + lane) * 6 + c] = s0;
            region[((size_t)(wave * nr + r) * 16 + lane) * 6 + 3 + c] = s1;
          }
        }
      }
    {
      const float s0 = wave_sum(BAL ? s_al : s_w), s1 = wave_sum(s_r);
      if (lane == 0) { sscal[2 * wave] = s0; sscal[2 * wave + 1] = s1; }
    }
    __syncthreads();
    const float gs = BAL ? w_bal / (eps * r0) : (geo ? wd / (eps * r0) : 0.f);
    for (int e = tid; e < nr * 16 * 3; e += SB_NT) {
      const int q = e / 3, c = e % 3, i = r_lo + q;
      float v0 = 0.f, v1 = 0.f;
#pragma unroll
      for (int w_ = 0; w_ < SB_NW; ++w_) {
        v0 += region[((size_t)w_ * nr * 16 + q) * 6 + c];
        v1 += region[((size_t)w_ * nr * 16 + q) * 6 + 3 + c];
      }
      if (i < N) a.dx_part[(bhN + i) * 3 + c] = (i < n && valid[i]) ? gs * v0 + v1 : 0.f;
    }
    if (tid == 0) {
      float s0 = 0.f, s1 = 0.f;
      for (int w_ = 0; w_ < SB_NW; ++w_) { s0 += sscal[2 * w_]; s1 += sscal[2 * w_ + 1]; }
      if constexpr (BAL) {
        const float rh = a.r_h[h];
        const float dsign = fabsf(rh) >= 0.1f ? (rh > 0.f ? 1.f : (rh < 0.f ? -1.f : 0.f)) : 0.f;
        a.ar_part[(bh * a.G + member) * 2 + 0] = w_bal * (1.f - w_bal) / eps * s0;
        a.ar_part[(bh * a.G + member) * 2 + 1] = -(w_bal / (eps * r0)) * s1 * dsign;
      } else {
        a.dw_part[bh * a.G + member] = s0 / eps;
      }
    }
    if constexpr (!BAL)
      if (tid < 68) a.dpw_part[(bh * a.G + member) * 68 + tid] = s_dpw[tid] / eps;
  };
  const int ksg = reg_ks(n_tiles);
  if (ksg == 2) run(std::integral_constant<int, 2>{});
  else if (ksg == 4) run(std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 6>{});
  return false;
}

}  // namespace dfl
