// pst_engine_f32.hpp -- mixed FP32/FP64 simulation engine for gfx950.
//
// Same method as the FP64 kernels (P1_P2.py:54-297, P3.py:29-163,
// gillespie.py:27-149): same epsilon bound, same n_c critical split, same
// SSA fallback burst and sampling rules, same wavefront-uniform loop.
// Precision:
//   FP32: propensities, a0 for the leap decision, mu / sigma^2, the Cao tau
//         bound, Poisson means and the Poisson samplers (inversions; PTRS, for
//         means of 2^16 and above, with its log-density test in a
//         cancellation-free Stirling form), uniforms (24-bit, one Philox word
//         each)
//   FP64: the simulation clock t, and the reaction choice, done as "first j
//         with sum_{r<=j} a_r >= rho2 * a0" accumulated in FP64 so that FP32
//         round-off cannot bias which reaction fires.  Poisson draws whose
//         FP32 root lies next to an integer are decided in FP64, and means of
//         2^22 and above use the FP64 sampler (FP32 cannot resolve the
//         integers).
// Transcendentals use the hardware v_log_f32 / v_exp_f32 / v_rcp_f32.  The
// launch loop, work queue and lane modes are in pst_driver.hpp.
#pragma once
#include "pst_driver.hpp"

namespace pst {

// CalculateG (P1_P2.py:447-486) in FP32
__device__ __forceinline__ float calc_g_f32(int h, int ht, int xi) {
  const float xf = (float)xi;
  if (h == 1) return 1.0f;
  if (h == 2) return (ht == 2) ? 2.0f + fast_rcp(xf - 1.0f) : 2.0f;
  if (h == 3) {
    if (ht == 3) return 3.0f + fast_rcp(xf - 1.0f) + 2.0f * fast_rcp(xf - 2.0f);
    if (ht == 2) return 1.5f * (2.0f + fast_rcp(xf - 1.0f));
    return 3.0f;
  }
  return 0.0f;
}

// log(1 + d) with the rounding of 1 + d corrected (Goldberg's method)
__device__ __forceinline__ float log1p_f32(float d) {
  const float u = 1.0f + d;
  const float m = u - 1.0f;
  return (m == 0.0f) ? d : fast_log(u) * (d * fast_rcp(m));
}

struct PtrsF32 {
  float lam, slam, b, a, vr, twoa;
};

__device__ __forceinline__ PtrsF32 ptrs_setup_f32(float lam) {
  PtrsF32 P;
  P.lam = lam;
  P.slam = __builtin_amdgcn_sqrtf(lam);  // hardware v_sqrt_f32 (1 ulp)
  P.b = 0.931f + 2.53f * P.slam;
  P.a = -0.059f + 0.02483f * P.b;
  P.vr = 0.9277f - 3.6224f * fast_rcp(P.b - 2.0f);
  P.twoa = 2.0f * P.a;
  return P;
}

__device__ __forceinline__ bool ptrs_fast_f32(const PtrsF32& P, float U, float V, float& kf, float& us) {
  us = 0.5f - __builtin_fabsf(U);
  kf = __builtin_floorf((P.twoa * fast_rcp(us) + P.b) * U + P.lam + 0.43f);
  return us >= 0.07f && V <= P.vr;
}

// -lambda + k ln lambda - ln k!, the right-hand side of PTRS's acceptance test.
// For k >= 10, with x = k + 1 and Stirling's series for ln Gamma(x):
//   (x - lambda) - (x - 1/2) log1p((x - lambda)/lambda) - ln(lambda)/2
//   - ln(2 pi)/2 - 1/(12x) + 1/(360x^3)
// which keeps full FP32 accuracy where the direct form cancels.
__device__ __forceinline__ float log_pmf_f32(float kf, float lam) {
  if (kf < 10.0f) {
    const int k = (int)kf;
    const float lf = k < 2 ? 0.0f : (float)logfact_small(k);
    return -lam + kf * fast_log(lam) - lf;
  }
  const float x = kf + 1.0f;
  const float d = x - lam;
  const float r = fast_rcp(x);
  const float ser = r * (1.0f / 12.0f - r * r * (1.0f / 360.0f));
  return d - (x - 0.5f) * log1p_f32(d * fast_rcp(lam)) - 0.5f * fast_log(lam) - 0.91893853320467274f - ser;
}

__device__ __forceinline__ bool ptrs_slow_f32(const PtrsF32& P, float V, float kf, float us) {
  if (kf < 0.0f || (us < 0.013f && V > us)) return false;
  const float invalpha = 1.1239f + 1.1328f * fast_rcp(P.b - 3.4f);
  const float lhs = fast_log(V) + fast_log(invalpha) - fast_log(P.a * fast_rcp(us * us) + P.b);
  return lhs <= log_pmf_f32(kf, P.lam);
}

// PTRS for Poisson means of 2^16 and above (rare: the inversion of
// poisson_asym_f32 covers the means below): iteration i of the draw in word
// slot `slot` of block c uses block (c, 1 + 4 i + slot), U from its word 0
// and V from word 1, so no two draws share a block.  FP32 below 2^22, FP64
// above (FP32 cannot resolve the integers there).  k = -1 at the iteration
// limit.
constexpr float BIG_LAMBDA_F32 = 4194304.0f;  // 2^22

__device__ __noinline__ Draw ptrs_wide(uint32_t k0, uint32_t k1, uint32_t s_lo, uint32_t s_hi, uint64_t c, int slot,
                                       float lamf) {
  Key key;
  key.k0 = k0;
  key.k1 = k1;
  key.s_lo = s_lo;
  key.s_hi = s_hi;
  Draw d = {-1, 0u};
  if (lamf < BIG_LAMBDA_F32) {
    const PtrsF32 P = ptrs_setup_f32(lamf);
    for (int i = 0; i < PTRS_MAX_ITERS; ++i) {
      const Words4 bw = key.block(c, 1u + 4u * (uint32_t)i + (uint32_t)slot);
      d.iters += 1;
      const float U = u24(bw.w0) - 0.5f;
      const float V = u24(bw.w1);
      float kf, us;
      if (ptrs_fast_f32(P, U, V, kf, us) || ptrs_slow_f32(P, V, kf, us)) {
        d.k = (int64_t)kf;
        break;
      }
    }
    return d;
  }
  const double lam = (double)lamf;
  const double loglam = log_f64(lam);
  const double b = 0.931 + 2.53 * __builtin_sqrt(lam);
  const double a = -0.059 + 0.02483 * b;
  const double vr = 0.9277 - 3.6224 / (b - 2.0);
  const double invalpha = 1.1239 + 1.1328 / (b - 3.4);
  for (int i = 0; i < PTRS_MAX_ITERS; ++i) {
    const Words4 bw = key.block(c, 1u + 4u * (uint32_t)i + (uint32_t)slot);
    d.iters += 1;
    const double U = u53(bw.w0, bw.w1) - 0.5;
    const double V = u53(bw.w1, bw.w0);
    const double us = 0.5 - __builtin_fabs(U);
    const double kf = __builtin_floor((2.0 * a / us + b) * U + lam + 0.43);
    if (us >= 0.07 && V <= vr) {
      d.k = (int64_t)kf;
      break;
    }
    if (kf < 0.0 || (us < 0.013 && V > us)) continue;
    const double lhs = log_f64(V) + log_f64(invalpha) - log_f64(a / (us * us) + b);
    const double rhs = -lam + kf * loglam - lgamma_int_f64(kf + 1.0);
    if (lhs <= rhs) {
      d.k = (int64_t)kf;
      break;
    }
  }
  return d;
}

// Per-lane state and steps of one mixed-precision simulation.
template <class Ref>
struct EngineF32 {
  using Real = float;
  static constexpr int NP = Ref::kNP, MP = Ref::kMP;
  static constexpr int NB = (MP + 3) / 4;  // Philox blocks of a leap attempt
  // The larger tables take their draws one after the other through one copy
  // of the sampler: one copy per reaction came to 320 KB of code for 16 x 16.
  static constexpr bool kWorklist = Ref::kTable && MP > 4;
  // blocks generated beside the decision (the one-by-one draws generate theirs)
  static constexpr int NA = kWorklist ? 1 : NB;
  float k[Ref::kKP];  // rates row: per-reaction constants, or hazard parameters
  int32_t x[NP];
  Key key;
  uint64_t bc;
  double t, tnext;
  int F;
  int flag;
  int burst;
  uint32_t nsteps;  // leap decisions + SSA steps so far (step budget)
  int32_t* Ob;

  using Out = SampleOut<Ref::kOutLds>;

  // v[i]: i is a constant in network kernels, wavefront-uniform in table-driven ones
  template <class T>
  static __device__ __forceinline__ T species_of(const T (&v)[NP], int i) {
    if constexpr (Ref::kTable) return at<T, NP>(v, i);
    else return v[i];
  }

  __device__ __forceinline__ void fill_rest(const Ref& tab, bool zero, Counters& cnt) const {
    const auto& P = tab.p();
    cnt.w.samples += (unsigned int)(P.ita - F);
    if (P.layout != LAYOUT_BLOCKS) {
      tab.for_recorded([&](int q) {
        const int32_t val = zero ? 0 : pick_i<NP>(x, tab.Ev(q));
        for (int f = F; f < P.ita; ++f) glb(Ob)[((int64_t)q * P.ita + f) * P.o_stride] = val;
      });
      return;
    }
    for (int f = F; f < P.ita; ++f) {
      tab.for_recorded([&](int q) { Out::put(P, Ob, q, f, zero ? 0 : pick_i<NP>(x, tab.Ev(q))); });
      Out::row_done(P, Ob, P.kappa, f);
    }
  }

  __device__ __forceinline__ int start(const Ref& jr, int64_t sim) {
    const JobParams& P = jr.cold();
    const int64_t set = sim / P.sims_per_set;
#pragma unroll
    for (int j = 0; j < Ref::kKP; ++j) k[j] = (j < P.n_rates) ? (float)glb(P.rates)[set * P.n_rates + j] : 0.0f;
#pragma unroll
    for (int i = 0; i < NP; ++i) x[i] = (i < P.N) ? glb(P.x0)[set * P.N + i] : 0;
    key.init(P.seed, P.sim_offset + (uint64_t)sim);
    bc = 0;
    t = 0.0;
    F = 0;
    tnext = (double)glb(P.I)[0];
    flag = 0;
    burst = 0;
    nsteps = 0;
    Ob = Out::base(P, sim);
    return jr.p().method == 0 ? MODE_DECIDE : MODE_SSA;
  }

  // One direct-method SSA step in its general form -- see EngineF64::ssa_step;
  // the arithmetic is FP32 except the clock and the cumulative sum of the
  // reaction choice.
  __device__ __forceinline__ int ssa_step(const Ref& tab, Counters& cnt, const float (&a)[MP]) {
    const auto& P = tab.p();
    if (P.method == 2 && !(t < P.t_max)) {
      fill_rest(tab, true, cnt);
      return MODE_DONE;
    }
    // step budget, checked before every leap decision and every SSA step
    if (P.max_steps != 0u && nsteps >= P.max_steps) {
      fill_rest(tab, true, cnt);
      flag = FLAG_STEPS;
      return MODE_DONE;
    }
    nsteps += 1;
    float a0 = 0.0f;
#pragma unroll
    for (int j = 0; j < MP; ++j) a0 += a[j];
    if (a0 == 0.0f) {
      fill_rest(tab, false, cnt);
      return MODE_DONE;
    }
    double asum = 0.0;
#pragma unroll
    for (int j = 0; j < MP; ++j) asum += (double)a[j];
    float tau = __builtin_inff();
    uint32_t cw1 = 0;
    if (asum > 0.0) {
      const Words4 bw = key.block(bc, 0);
      bc += 1;
      cnt.w.uniforms += 2;
      cw1 = bw.w1;
      tau = -fast_log(u24(bw.w0)) * fast_rcp((float)asum);
    }
    const int sel = pick_reaction(a, asum, u24(cw1), [](int) { return true; });
    const double t0 = t;
    t = t + (double)tau;
    if (t == t0 && tau > 0.0f) {  // tau == 0 (a draw of u = 1) is a valid event
      fill_rest(tab, true, cnt);
      flag = FLAG_STALL;
      return MODE_DONE;
    }
    // sample-and-hold of the pre-step state
    while (t >= tnext) {
      tab.for_recorded([&](int q) { Out::put(P, Ob, q, F, pick_i<NP>(x, tab.Ev(q))); });
      Out::row_done(P, Ob, P.kappa, F);
      cnt.w.samples += 1;
      F = F + 1;
      if (F == P.ita) return MODE_DONE;
      tnext = (double)glb(P.I)[F];
    }
    bool over = false;
    int32_t d[NP];
    tab.row(sel >= 0 ? sel : 0, d);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      x[i] += sel >= 0 ? d[i] : 0;
      over = over | (x[i] >= COUNT_LIMIT);
    }
    cnt.ssa += 1;
    cnt.events += 1;
    if (over) {
      fill_rest(tab, true, cnt);
      flag = FLAG_OVERFLOW;
      return MODE_DONE;
    }
    if (P.method != 0) return MODE_SSA;
    burst -= 1;
    return burst > 0 ? MODE_SSA : MODE_DECIDE;
  }

  // First j of the mask with sum_{r<=j} a_r >= rho * asum, summed in FP64; the
  // running sum never decreases and the target is positive, so that is the
  // number of positions whose sum is still below it (a masked-out position
  // repeats its predecessor's sum and is never the first to reach it).  A sum
  // that ends below the target takes the last positive masked reaction.
  template <class Mask>
  static __device__ __forceinline__ int pick_reaction(const float (&a)[MP], double asum, float rho, Mask in) {
    const double target = (double)rho * asum;
    double cum = 0.0;
    int below = 0, last = -1;
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      cum += in(j) ? (double)a[j] : 0.0;
      last = (in(j) & (a[j] > 0.0f)) ? j : last;
      below += (cum < target) ? 1 : 0;
    }
    return below < MP ? below : last;
  }

  // One P1_P2 body (P1_P2.py:96-294) of the lanes with `on` -- see
  // EngineF64::decide.
  template <int FORM>
  __device__ __forceinline__ int decide(Ref& tab, Counters& cnt, bool on, const LaneGroup<FORM>& g) {
    const auto& P = tab.p();
    constexpr int ABSORBED = -1;
    int end = 0;  // ABSORBED, or the flag that ends the simulation
    bool live = on;
    if (P.max_steps != 0u) {
      end = (live & (nsteps >= P.max_steps)) ? FLAG_STEPS : 0;
      live = live & (end == 0);
    }
    nsteps += live ? 1u : 0u;
    // Philox blocks bc .. bc + NB - 1, independent of the state: chains beside
    // the decision's.  The first Poisson attempt takes the NB blocks from bc,
    // or those from bc + 1 when the critical draw took block bc.
    const Key uk = key.scalar_seed(P.seed);
    Words4 B[NB];
    B[0] = uk.block(bc, 0);
    if (NA > 1 && !g.grouped()) {
#pragma unroll
      for (int r = 1; r < NA; ++r) B[r] = uk.block(bc + (uint64_t)r, 0);
    }
    float a[MP];
    const float a0 = tab.props_sum(x, k, a);
    // (products already rounded to FP32: not to be contracted into the sums below)
#pragma unroll
    for (int j = 0; j < MP; ++j) asm("" : "+v"(a[j]));
    end = (live & (a0 == 0.0f)) ? ABSORBED : end;
    live = live & !(a0 == 0.0f);
    cnt.w.decisions += live ? 1u : 0u;
    // critical reactions, mu and sigma^2, and the Cao bound (P1_P2.py:314-445)
    unsigned crit, any;
    float mu[NP], s2[NP];
    tab.template sums<float>(x, a, P.n_c, crit, mu, s2, any);
    float tau1 = __builtin_inff();
    const float eta = (float)P.eta;
    tab.for_species([&](int i) {
      if (tab.Irs(i)) {
        const int32_t xi = species_of<int32_t>(x, i);
        const float g_i = calc_g_f32(tab.Hv(i), tab.Htv(i), xi);
        const float num = fmaxf(eta * (float)xi * fast_rcp(g_i), 1.0f);
        const float cand = fminf(num * fast_rcp(fabsf(species_of<float>(mu, i))),
                                 num * num * fast_rcp(species_of<float>(s2, i)));
        tau1 = ((any >> i) & 1u) ? fminf(tau1, cand) : tau1;
      }
    });
    // SSA switch (P1_P2.py:157-173)
    const bool fall = live & (tau1 < 10.0f * fast_rcp(a0));
    burst = fall ? P.ssa_burst : burst;
    live = live & !fall;
    // tau2 and the critical reaction (P1_P2.py:175-220)
    double asum = 0.0;
#pragma unroll
    for (int j = 0; j < MP; ++j) asum += ((crit >> j) & 1u) ? (double)a[j] : 0.0;
    float tau = tau1;
    int sel = -1;
    const bool one = live & (asum > 0.0);
    if (wave_any(one)) {
      const float tauX = -fast_log(u24(B[0].w0)) * fast_rcp((float)asum);
      const bool fire = one & (tau1 > tauX);
      cnt.w.uniforms += (one ? 1u : 0u) + (fire ? 1u : 0u);
      tau = one ? fminf(tau1, tauX) : tau;
      const int c = pick_reaction(a, asum, u24(B[0].w1), [&](int j) { return ((crit >> j) & 1u) != 0u; });
      sel = fire ? c : -1;
      const Words4 e = NA == NB ? uk.block(bc + (uint64_t)NB, 0) : B[0];
#pragma unroll
      for (int r = 0; r < NA; ++r) {
        const Words4 n = r + 1 < NA ? B[r + 1 < NA ? r + 1 : 0] : e;
        B[r].w0 = one ? n.w0 : B[r].w0;
        B[r].w1 = one ? n.w1 : B[r].w1;
        B[r].w2 = one ? n.w2 : B[r].w2;
        B[r].w3 = one ? n.w3 : B[r].w3;
      }
      bc += one ? 1u : 0u;
    }
    end = (live & !(tau < __builtin_inff())) ? FLAG_TAU_INF : end;
    live = live & (tau < __builtin_inff());
    // the leap, with tau halving (P1_P2.py:222-259)
    int32_t xn[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) xn[i] = 0;
    unsigned long long ev = 0;
    bool again = live;
    for (int h = 0;; ++h) {
      const int st = attempt(tab, cnt, again, a, crit, tau, sel, B, xn, ev, uk, g);
      end = (again & (st > 0)) ? st : end;
      again = again & (st < 0);
      if (!wave_any(again)) break;
      cnt.rejected += again ? 1u : 0u;
      tau = again ? tau * 0.5f : tau;
      end = (again & (h + 1 >= MAX_HALVINGS)) ? FLAG_HALVING : end;
      again = again & (h + 1 < MAX_HALVINGS);
#pragma unroll
      for (int r = 0; r < NA; ++r) B[r] = uk.block(bc + (uint64_t)r, 0);
    }
    live = live & (end == 0);
    cnt.events += live ? ev : 0ull;
    cnt.leaps += live ? 1u : 0u;
    // time advance and interpolated samples
    const double t0 = t;
    const double t1 = t + (double)tau;
    t = live ? t1 : t;
    const bool stall = live & (t1 == t0) & (tau > 0.0f);  // tau == 0 is a valid event
    end = stall ? FLAG_STALL : end;
    live = live & !stall;
    bool last = false;
    if (wave_any(live & (t >= tnext))) {
      if (live) {
        const float inv_gap = fast_rcp((float)(t - t0));
        while (t >= tnext) {
          const float frac = (float)(tnext - t0) * inv_gap;
          tab.for_recorded([&](int q) {
            const int s = tab.Ev(q);
            const int32_t xs = pick_i<NP>(x, s);
            const int diff = pick_i<NP>(xn, s) - xs;
            Out::put(P, Ob, q, F, xs + rn_f32_to_int((float)diff * frac));
          });
          Out::row_done(P, Ob, P.kappa, F);
          cnt.w.samples += 1;
          F = F + 1;
          last = F == P.ita;
          if (last) break;
          tnext = (double)glb(P.I)[F];
        }
      }
    }
    if (wave_any(end != 0)) {
      if (end != 0) {
        fill_rest(tab, end != ABSORBED, cnt);
        flag = end != ABSORBED ? end : 0;
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) x[i] = live ? xn[i] : x[i];
    return ((end != 0) | last) ? MODE_DONE : fall ? MODE_SSA : MODE_DECIDE;
  }

  // The random numbers of one SSA step: -ln(rho1) and rho2.
  struct Draw1 {
    float nl, u;
  };
  static __device__ __forceinline__ Draw1 ssa_draw(const Key& uk, uint64_t c) {
    const Words4 w = uk.block(c, 0);
    return {-fast_log(u24(w.w0)), u24(w.w1)};
  }
  static __device__ __forceinline__ Draw1 from_lane(const Draw1& d, int addr) { return {lane_get(d.nl, addr), lane_get(d.u, addr)}; }

  // One SSA step from state (x, t) with draw d: the reaction and the new time;
  // false if the step needs ssa_step (see ssa_run).  ssa_step's arithmetic; a
  // sum of 0 gives an infinite or undefined time, which fails.  A hazard
  // expression may be negative: then the FP32 sum, which ends a simulation where
  // it is 0, can be 0 where this one is not, and ssa_step decides.
  __device__ __forceinline__ bool ssa_try(const Ref& tab, const Draw1& d, double tstop, int& sel, double& t1) const {
    float a[MP];
    tab.template props<float>(x, k, a);
    double cum[MP];
#pragma unroll
    for (int j = 0; j < MP; ++j) cum[j] = (j > 0 ? cum[j > 0 ? j - 1 : 0] : 0.0) + (double)a[j];
    const double asum = cum[MP - 1];
    t1 = t + (double)(d.nl * fast_rcp((float)asum));
    const double target = (double)d.u * asum;  // <= asum: the last sum always reaches it
    sel = 0;
    bool ok = (t1 > t) & (t1 < tstop);
#pragma unroll
    for (int j = 0; j < MP - 1; ++j) sel += (cum[j] < target) ? 1 : 0;
    if constexpr (Ref::kCustom) {
#pragma unroll
      for (int j = 0; j < MP; ++j) ok = ok & (a[j] >= 0.0f);
    }
    return ok;
  }

  // One attempt of the leap for the lanes with `on` -- see EngineF64::attempt
  // for what it returns.  Every draw is an inversion of the Poisson CDF at one
  // 24-bit uniform: reaction j reads word j % 4 of block W[j / 4]; lambda < 10
  // by sequential search, 10 <= lambda < 2^16 by the asymptotic inversion with
  // exact FP64 decisions near integer boundaries (both are inversions, so no
  // draw is rejected and repeated); lambda >= 2^16 by PTRS on blocks of its own
  // (ptrs_wide).
  template <int FORM>
  __device__ __forceinline__ int attempt(Ref& tab, Counters& cnt, bool on, const float (&a)[MP],
                                         unsigned crit, float tau, int sel, const Words4 (&W)[NB],
                                         int32_t (&xn)[NP], unsigned long long& ev, const Key& uk,
                                         const LaneGroup<FORM>& g) {
    const auto& P = tab.p();
    const int M = P.M;
    const uint64_t grp = bc;
    bc += on ? (uint64_t)((M + 3) >> 2) : 0ull;
    float lam[MP];
    int32_t K[MP];
    bool bad = false, fail = false;
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      lam[j] = (on & (j < M) & !((crit >> j) & 1u)) ? a[j] * tau : 0.0f;
      K[j] = (sel == j) ? 1 : 0;
      bad = bad | (lam[j] >= (float)LAMBDA_LIMIT);
    }
    if (kWorklist || g.grouped()) {
      // the lane's own reactions, one after the other
      unsigned todo = 0;
#pragma unroll
      for (int j = 0; j < MP; ++j) todo |= (g.mine(j) & (lam[j] > 0.0f)) ? (1u << j) : 0u;
      todo = bad ? 0u : todo;
      while (wave_any(todo != 0u)) {
        const bool has = todo != 0u;
        const int j = has ? __builtin_ctz(todo) : 0;
        const float l = pick_f<MP>(lam, j);
        const uint64_t c = grp + (uint64_t)(uint32_t)(j >> 2);
        Words4 w;
        if constexpr (NB == 1) w = W[0];
        else w = uk.block(c, 0);
        const int32_t kk = draw(cnt, has, l, u24(word_of(w, j)), c, j & 3, fail);
#pragma unroll
        for (int r = 0; r < MP; ++r) K[r] = (has & (r == j)) ? kk : K[r];
        todo = todo & (todo - 1u);
      }
      if (g.grouped()) {
#pragma unroll
        for (int j = 0; j < MP; ++j) K[j] = g.owners(K[j], j);
        fail = g.any(fail);
      }
    } else {
      float u[MP];
#pragma unroll
      for (int j = 0; j < MP; ++j) u[j] = u24(word_of(W[j >> 2], j));
      draw_all(cnt, bad, lam, u, grp, K, fail);
    }
    bool ok = true, big = false;
    int64_t s[NP];
    tab.advance(x, K, s);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      ok = ok & (s[i] >= 0);
      big = big | (s[i] >= COUNT_LIMIT);
      xn[i] = on ? (int32_t)s[i] : xn[i];
    }
    unsigned long long sum = 0;
#pragma unroll
    for (int j = 0; j < MP; ++j) sum += (unsigned long long)K[j];
    ev = on ? sum : ev;
    return bad ? FLAG_OVERFLOW : fail ? FLAG_PTRS : !ok ? -1 : big ? FLAG_OVERFLOW : 0;
  }

  // word j % 4 of a block
  static __device__ __forceinline__ uint32_t word_of(const Words4& w, int j) {
    const uint32_t odd = 0u - (uint32_t)(j & 1), up = 0u - (uint32_t)((j >> 1) & 1);
    const uint32_t lo = w.w0 ^ ((w.w0 ^ w.w1) & odd), hi = w.w2 ^ ((w.w2 ^ w.w3) & odd);
    return lo ^ ((lo ^ hi) & up);
  }

  // One Poisson draw of mean l at the uniform u for the lanes with `has`.
  __device__ __forceinline__ int32_t draw(Counters& cnt, bool has, float l, float u, uint64_t c, int slot,
                                          bool& fail) const {
    int32_t kk = 0;
    const bool asym = has & (l >= POIS_ASYM_MIN) & (l < POIS_ASYM_MAX);
    if (wave_any(asym)) {
      bool ex = false;
      int32_t m = -1;
      const int32_t ka = poisson_asym_f32(__builtin_fmaxf(l, POIS_ASYM_MIN), u, ex, m);
      kk = asym ? ka : 0;
      cnt.w.asym += asym ? 1u : 0u;
      cnt.w.draws += asym ? 1u : 0u;
      const bool exact = asym & ex;
      if (wave_any(exact)) {
        if (exact) add_stat(ST_EXACT, 1ull);
        if (exact) kk = poisson_exact_f64((double)l, (double)u, m);
      }
    }
    const bool inv = has & (l < POIS_ASYM_MIN);
    if (wave_any(inv)) {
      // the search of draw_all for one reaction
      float p = fast_exp(-l), Fc = p;
      bool live = inv & (u > Fc);
      for (int it = 0; it < INV_MAX_K && wave_any(live); it += 2) {
        const float r1 = fast_rcp((float)(it + 1));
        const float r2 = fast_rcp((float)(it + 2));
        const float q1 = p * l;
        const float p1 = r1 * q1;
        const float F1 = __builtin_fmaf(r1, q1, Fc);
        const float q2 = p1 * l;
        const float F2 = __builtin_fmaf(r2, q2, F1);
        kk = live ? ((u > F1) ? it + 2 : it + 1) : kk;
        live = live & (u > F2) & (F2 > Fc);
        p = r2 * q2;
        Fc = F2;
      }
      cnt.w.draws += inv ? 1u : 0u;
      cnt.w.inv += inv ? (unsigned int)kk : 0u;
    }
    const bool wide = has & (l >= POIS_ASYM_MAX);
    if (wave_any(wide)) {
      if (wide) {
        const Draw dr = ptrs_wide(key.k0, key.k1, key.s_lo, key.s_hi, c, slot, l);
        add_stat(ST_PTRS, dr.iters);
        cnt.w.draws += 2 * dr.iters;
        fail = fail | (dr.k < 0);
        kk = (int32_t)dr.k;
      }
    }
    return kk;
  }

  // Every reaction's draw by the simulation's own lane (G = 1).
  __device__ __forceinline__ void draw_all(Counters& cnt, bool bad, const float (&lam)[MP], const float (&u)[MP],
                                           uint64_t grp, int32_t (&K)[MP], bool& fail) const {
    unsigned inv = 0, exact = 0, wide = 0, nasym = 0;
    int32_t mb[MP];
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      const float l = lam[j];
      const bool asym = !bad & (l >= POIS_ASYM_MIN) & (l < POIS_ASYM_MAX);
      bool ex = false;
      int32_t m = -1;
      int32_t k = 0;
      if (wave_any(asym)) k = poisson_asym_f32(__builtin_fmaxf(l, POIS_ASYM_MIN), u[j], ex, m);
      K[j] = asym ? k : K[j];
      mb[j] = m;
      exact |= (asym & ex) ? (1u << j) : 0u;
      nasym += asym ? 1u : 0u;
      inv |= (!bad & (l > 0.0f) & (l < POIS_ASYM_MIN)) ? (1u << j) : 0u;
      wide |= (!bad & (l >= POIS_ASYM_MAX)) ? (1u << j) : 0u;
    }
    cnt.w.asym += nasym;
    cnt.w.draws += nasym;
    // near an integer boundary, or in a far tail: decide exactly in FP64
    if (wave_any(exact != 0u)) {
      if (exact != 0u) add_stat(ST_EXACT, (unsigned long long)__builtin_popcount(exact));
#pragma unroll
      for (int j = 0; j < MP; ++j)
        if ((exact >> j) & 1u) K[j] = poisson_exact_f64((double)lam[j], (double)u[j], mb[j]);
    }
    // sequential-search inversion (0 < lambda < 10) for all such reactions
    // in lock-step, two search steps per trip: a live search at k = it
    // steps to it + 1 and it + 2 and stops at the first k with u <= F(k);
    // p and F past a search's end are computed but never read
    if (wave_any(inv != 0u)) {
      float p[MP], Fc[MP];
      bool live[MP];
      bool any_live = false;
#pragma unroll
      for (int j = 0; j < MP; ++j) {
        const bool on = (inv >> j) & 1u;
        p[j] = fast_exp(-lam[j]);
        Fc[j] = p[j];
        live[j] = on && u[j] > Fc[j];
        if (on) K[j] = 0;
        any_live = any_live | live[j];
      }
      cnt.w.draws += (unsigned int)__builtin_popcount(inv);
      for (int it = 0; it < INV_MAX_K && wave_any(any_live); it += 2) {
        const float r1 = fast_rcp((float)(it + 1));
        const float r2 = fast_rcp((float)(it + 2));
        any_live = false;
#pragma unroll
        for (int j = 0; j < MP; ++j) {
          const float q1 = p[j] * lam[j];
          const float p1 = r1 * q1;
          const float F1 = __builtin_fmaf(r1, q1, Fc[j]);
          const float q2 = p1 * lam[j];
          const float F2 = __builtin_fmaf(r2, q2, F1);
          K[j] = live[j] ? ((u[j] > F1) ? it + 2 : it + 1) : K[j];
          // a search also ends where the FP32 sum stops growing: past the
          // mode every later term is smaller still, and a u above that sum
          // (u24 can be 1.0, the sum can end a few ulps below it) would
          // otherwise run to INV_MAX_K
          live[j] = live[j] && (u[j] > F2) && (F2 > Fc[j]);
          any_live = any_live | live[j];
          p[j] = r2 * q2;
          Fc[j] = F2;
        }
      }
#pragma unroll
      for (int j = 0; j < MP; ++j)
        if ((inv >> j) & 1u) cnt.w.inv += (unsigned int)K[j];
    }
    // means of 2^16 and above (rare): PTRS, one reaction at a time
    if (wave_any(wide != 0u)) {
#pragma unroll
      for (int j = 0; j < MP; ++j) {
        if ((wide >> j) & 1u) {
          const Draw dr = ptrs_wide(key.k0, key.k1, key.s_lo, key.s_hi, grp + (uint64_t)(j >> 2), j & 3, lam[j]);
          add_stat(ST_PTRS, dr.iters);
          cnt.w.draws += 2 * dr.iters;
          fail = fail | (dr.k < 0);
          K[j] = (int32_t)dr.k;
        }
      }
    }
  }
};

}  // namespace pst
