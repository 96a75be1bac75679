// pst_engine_f64.hpp -- plain FP64 simulation engine for gfx950 (one simulation per lane).
//
// This translation unit is compiled with -ffp-contract=off: every FP64
// operation is a single IEEE-754 rounding, so the integer trajectories are the
// same bits as a plain-double CPU evaluation of the same algorithm on the same
// Philox stream.
//
// Algorithm (per lane, one launch for the whole run):
//   tau-leaping with SSA fallback   P1_P2.py:54-297 + P3.py:29-163, iterated per
//                                   simulation as the host loop
//                                   cuTauLeaping.py:48-76 iterates them
//   forced SSA (gillespie=1)        P1_P2.py:67-74 -> P3 bursts only
//   pure SSA                        gillespie.py:27-149 (stops at t >= t_max)
// The reference's two launches per iteration, the per-iteration gpuarray.sum
// and the host round trip are replaced by a per-lane loop inside one launch:
// simulations never communicate, so each lane runs its simulation to the end.
//
// A simulation alternates between leap decisions (decide) and SSA steps
// (ssa_run in pst_driver.hpp, ssa_step for the rare ones).  Random numbers
// come from fixed positions of the stream (see Key in pst_device.hpp).
// The launch loop, work queue and lane modes are in pst_driver.hpp.
#pragma once
#include "pst_driver.hpp"

namespace pst {

// CalculateG, P1_P2.py:447-486
__device__ __forceinline__ double calc_g_f64(int h, int ht, int xi) {
  if (h == 1) return 1.0;
  if (h == 2) {
    if (ht == 2) return 2.0 + 1.0 / ((double)xi - 1.0);
    return 2.0;
  }
  if (h == 3) {
    if (ht == 3) return 3.0 + 1.0 / ((double)xi - 1.0) + 2.0 / ((double)xi - 2.0);
    if (ht == 2) return 3.0 / 2.0 * (2.0 + 1.0 / ((double)xi - 1.0));
    return 3.0;
  }
  return 0.0;
}

// x[idx] for a run-time idx in [0, NP) (doubles), masked like pick_i (the bits
// are copied, so the value is exact)
template <int NP>
__device__ __forceinline__ double pick(const double (&x)[NP], int idx) {
  uint64_t r = 0;
#pragma unroll
  for (int i = 0; i < NP; ++i) r |= __builtin_bit_cast(uint64_t, x[i]) & (0ull - (uint64_t)(idx == i));
  return __builtin_bit_cast(double, r);
}

// PTRS (Hoermann 1993) constants for one Poisson mean 10 <= lam < 1e9 (every
// argument of log and exp below is then positive, finite and normal)
struct PtrsF64 {
  double lam, loglam, b, a, vr;
};

__device__ __forceinline__ PtrsF64 ptrs_setup_f64(double lam) {
  PtrsF64 P;
  P.lam = lam;
  P.loglam = log_normal_f64(lam);
  const double slam = exp_core_f64(0.5 * P.loglam);
  P.b = 0.931 + 2.53 * slam;
  P.a = -0.059 + 0.02483 * P.b;
  P.vr = 0.9277 - 3.6224 / (P.b - 2.0);
  return P;
}

// The squeeze of one PTRS iteration: kf and whether it is accepted without
// the log-density test.
__device__ __forceinline__ bool ptrs_fast_f64(const PtrsF64& P, double U, double V, double& kf, double& us) {
  us = 0.5 - __builtin_fabs(U);
  kf = __builtin_floor((2.0 * P.a / us + P.b) * U + P.lam + 0.43);
  return (us >= 0.07) & (V <= P.vr);
}

// The log-density test after a failed squeeze (kf >= 0, 0 < V <= 1, us > 0).
// Without a branch: where the lanes of one meet again, hipcc 7.2 has put
// constants back into registers before it switches the other lanes on again.
// Those lanes then draw with what the register held (the table-driven kernel
// for 16 x 16 with its 434 registers; a simulation without end).
__device__ __forceinline__ bool ptrs_slow_f64(const PtrsF64& P, double V, double kf, double us) {
  const double invalpha = 1.1239 + 1.1328 / (P.b - 3.4);
  const double lhs = log_normal_f64(V) + log_normal_f64(invalpha) - log_normal_f64(P.a / (us * us) + P.b);
  const double rhs = -P.lam + kf * P.loglam - lgamma_int_flat_f64(kf + 1.0);
  return lhs <= rhs;
}

// Per-lane state and steps of one FP64 simulation.
template <class Ref>
struct EngineF64 {
  using Real = double;
  static constexpr int NP = Ref::kNP, MP = Ref::kMP;
  double k[Ref::kKP];  // rates row: per-reaction constants, or hazard parameters
  int32_t x[NP];
  Key key;
  uint64_t bc;  // Philox block counter
  double t, tnext;
  int F;
  int flag;
  int burst;    // SSA steps left in the current fallback burst (method 0)
  uint32_t nsteps;  // leap decisions + SSA steps so far (step budget)
  int32_t* Ob;  // the simulation's base in O (SampleOut::base)

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
    for (int j = 0; j < Ref::kKP; ++j) k[j] = (j < P.n_rates) ? glb(P.rates)[set * P.n_rates + j] : 0.0;
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

  // One direct-method SSA step (P3.py:73-149; gillespie.py:70-149 for pure
  // SSA) in its general form, from the propensities of the present state;
  // ordinary steps run in ssa_run (pst_driver.hpp).  Returns the next mode.
  __device__ __forceinline__ int ssa_step(const Ref& tab, Counters& cnt, const double (&a)[MP]) {
    const auto& P = tab.p();
    const int M = P.M;
    if (P.method == 2 && !(t < P.t_max)) {
      // kernel_Gillespie stops at t >= t_max; later samples stay zero (cuGillespie.py:71)
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
    double a0 = 0.0;
#pragma unroll
    for (int j = 0; j < MP; ++j) a0 = a0 + a[j];
    if (a0 == 0.0) {
      fill_rest(tab, false, cnt);
      return MODE_DONE;
    }
    double tau = __builtin_inf();
    uint32_t cw2 = 0, cw3 = 0;
    if (a0 > 0.0) {
      const Words4 bw = key.block(bc, 0);
      bc += 1;
      cnt.w.uniforms += 2;
      cw2 = bw.w2;
      cw3 = bw.w3;
      tau = (1.0 / a0) * log_normal_f64(1.0 / u53(bw.w0, bw.w1));
    }
    // first j with sum_{r<=j} a_r/a0 >= rho (P3.py:179-194); on round-off
    // fall-through the last j with a_j > 0
    const double rho = u53(cw2, cw3);
    const int sel = pick_reaction(M, a, a0, rho, [](int) { return true; });
    const double t_prev = t;
    t = t + tau;
    if (t == t_prev && tau > 0.0) {  // tau == 0 (a draw of u = 1) is a valid event
      fill_rest(tab, true, cnt);
      flag = FLAG_STALL;
      return MODE_DONE;
    }
    // sample-and-hold of the pre-step state (SaveDynamics, P3.py:165-177)
    while (t >= tnext) {
      tab.for_recorded([&](int q) { Out::put(P, Ob, q, F, pick_i<NP>(x, tab.Ev(q))); });
      Out::row_done(P, Ob, P.kappa, F);
      cnt.w.samples += 1;
      F = F + 1;
      if (F == P.ita) return MODE_DONE;  // a step ending the run is not applied
      tnext = (double)glb(P.I)[F];
    }
    // UpdateState (P3.py:196-208)
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

  // SingleCriticalReaction (P1_P2.py:488-507, P3.py:179-194): first j of the
  // mask with sum_{r<=j} a_r/asum >= rho, else the last one with a_j > 0
  template <class Mask>
  static __device__ __forceinline__ int pick_reaction(int M, const double (&a)[MP], double asum, double rho, Mask in) {
    double rc = 0.0;
    int sel = -1, last = -1;
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      const bool m = (j < M) & in(j) & (sel < 0);
      last = (m & (a[j] > 0.0)) ? j : last;
      rc = m ? rc + a[j] / asum : rc;
      sel = (m & (rc >= rho)) ? j : sel;
    }
    return sel < 0 ? last : sel;
  }

  // One P1_P2 body (P1_P2.py:96-294) of the lanes with `on` (all lanes of the
  // wavefront call this together): leap decision, then the leap, or a switch
  // to an SSA burst, whose steps run in ssa_run.  Returns the next mode.
  //
  // Rare outcomes (budget, absorbing state, flags) are collected in `end` and
  // handled once at the end instead of where they arise: each branch on a lane
  // mask costs 50-60 cycles of a step's chain.
  template <int FORM>
  __device__ __forceinline__ int decide(Ref& tab, Counters& cnt, bool on, const LaneGroup<FORM>& g) {
    const auto& P = tab.p();
    const int M = P.M;
    constexpr int ABSORBED = -1;
    int end = 0;  // ABSORBED, or the flag that ends the simulation
    bool live = on;
    if (P.max_steps != 0u) {
      end = (live & (nsteps >= P.max_steps)) ? FLAG_STEPS : 0;
      live = live & (end == 0);
    }
    nsteps += live ? 1u : 0u;
    double a[MP];
    tab.template props<double>(x, k, a);
    double a0 = 0.0;
#pragma unroll
    for (int j = 0; j < MP; ++j) a0 = a0 + a[j];
    end = (live & (a0 == 0.0)) ? ABSORBED : end;
    live = live & !(a0 == 0.0);
    cnt.w.decisions += live ? 1u : 0u;
    // critical reactions, mu and sigma^2 (P1_P2.py:314-383), CalculateTau
    // (P1_P2.py:385-445)
    unsigned crit, any;
    double mu[NP], s2[NP];
    tab.template sums<double>(x, a, P.n_c, crit, mu, s2, any);
    double tau1 = __builtin_inf();
    tab.for_species([&](int i) {
      if (tab.Irs(i)) {
        // one candidate per V entry of this species; all equal, so one suffices
        const int32_t xi = species_of<int32_t>(x, i);
        const double g_i = calc_g_f64(tab.Hv(i), tab.Htv(i), xi);
        const double num = (double)fmaxf((float)(P.eta * (double)xi / g_i), 1.0f);
        const double lhs = num / (double)fabsf((float)species_of<double>(mu, i));
        const double rhs = (num * num) / species_of<double>(s2, i);
        const double tt = (double)fminf((float)lhs, (float)rhs);
        tau1 = (((any >> i) & 1u) & (tt < tau1)) ? tt : tau1;
      }
    });
    // SSA switch (P1_P2.py:157-173)
    const bool fall = live & (tau1 < 10.0 / a0);
    burst = fall ? P.ssa_burst : burst;
    live = live & !fall;
    // tau2 and SingleCriticalReaction (P1_P2.py:175-220)
    double asum = 0.0;
#pragma unroll
    for (int j = 0; j < MP; ++j) asum = ((crit >> j) & 1u) ? asum + a[j] : asum;
    double tau = (double)(float)tau1;
    int sel = -1;
    const bool one = live & (asum > 0.0);
    if (wave_any(one)) {
      const Words4 bw = key.block(bc, 0);
      bc += one ? 1u : 0u;
      const double tauX = (1.0 / asum) * log_normal_f64(1.0 / u53(bw.w0, bw.w1));
      const bool fire = one & (tau1 > tauX);
      cnt.w.uniforms += (one ? 1u : 0u) + (fire ? 1u : 0u);
      tau = one ? (double)fminf((float)tau1, (float)tauX) : tau;
      const int c = pick_reaction(M, a, asum, u53(bw.w2, bw.w3), [&](int j) { return ((crit >> j) & 1u) != 0u; });
      sel = fire ? c : -1;
    }
    end = (live & !(tau < __builtin_inf())) ? FLAG_TAU_INF : end;
    live = live & (tau < __builtin_inf());
    // the leap, with tau halving (P1_P2.py:222-259)
    int32_t xn[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) xn[i] = 0;
    unsigned long long ev = 0;
    bool again = live;
    for (int h = 0;; ++h) {
      const int st = attempt(tab, cnt, again, a, crit, tau, sel, xn, ev, g);
      end = (again & (st > 0)) ? st : end;
      again = again & (st < 0);
      if (!wave_any(again)) break;
      cnt.rejected += again ? 1u : 0u;
      tau = again ? tau / 2.0 : tau;
      end = (again & (h + 1 >= MAX_HALVINGS)) ? FLAG_HALVING : end;
      again = again & (h + 1 < MAX_HALVINGS);
    }
    live = live & (end == 0);
    cnt.events += live ? ev : 0ull;
    cnt.leaps += live ? 1u : 0u;
    // time advance and interpolated samples (SaveInterpolatedDynamics,
    // P1_P2.py:261-286,542-584)
    const double t_prev = t;
    const double t1 = t + tau;
    t = live ? t1 : t;
    const bool stall = live & (t1 == t_prev) & (tau > 0.0);  // tau == 0 is a valid event
    end = stall ? FLAG_STALL : end;
    live = live & !stall;
    bool last = false;
    if (wave_any(live & (t >= tnext))) {
      if (live) {
        while (t >= tnext) {
          const double t0 = t - tau;
          const double gap = t - t0;
          const double frac = (tnext - t0) / gap;
          tab.for_recorded([&](int q) {
            const int s = tab.Ev(q);
            const int32_t xs = pick_i<NP>(x, s);
            const int diff = pick_i<NP>(xn, s) - xs;
            const double inc = (double)diff * frac;
            Out::put(P, Ob, q, F, xs + rn_f32_to_int((float)inc));
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

  // The random numbers of one SSA step: ln(1 / rho1) and rho2.
  struct Draw1 {
    double lr, rho;
  };
  static __device__ __forceinline__ Draw1 ssa_draw(const Key& uk, uint64_t c) {
    const Words4 w = uk.block(c, 0);
    return {log_normal_f64(1.0 / u53(w.w0, w.w1)), u53(w.w2, w.w3)};
  }
  static __device__ __forceinline__ Draw1 from_lane(const Draw1& d, int addr) { return {lane_get(d.lr, addr), lane_get(d.rho, addr)}; }

  // One SSA step from state (x, t) with draw d: the reaction and the new time;
  // false if the step needs ssa_step (see ssa_run).  The waiting time is
  // ssa_step's expression; its reaction choice, the first j with
  // sum_{r<=j} fl(a_r / asum) >= rho, is taken from the running sums against
  // rho * asum instead of M divisions.  Both sums of up to 32 non-negative
  // terms are within 1e-13 of the exact ones relative to asum, so outside a
  // band of 1e-12 asum around a running sum both pick the same reaction; inside
  // it (one step in ~10^11) ssa_step decides, and wherever a propensity is
  // negative.  -0.0, which a dimerisation has at a count of 0, is not (high
  // words of negative numbers are above its 2^31; those that share it are below
  // 2^-1042, nothing next to asum): sent to ssa_step, the
  // steps of a network with two such took 8.10 ms instead of 1.18.
  __device__ __forceinline__ bool ssa_try(const Ref& tab, const Draw1& d, double tstop, int& sel, double& t1) const {
    double a[MP];
    tab.template props<double>(x, k, a);
    double cum[MP];
    uint32_t top = 0u;  // the largest high word: above 2^31 where a propensity is negative
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      cum[j] = (j > 0 ? cum[j > 0 ? j - 1 : 0] : 0.0) + a[j];
      const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, a[j]) >> 32);
      top = hi > top ? hi : top;
    }
    const double asum = cum[MP - 1];
    t1 = t + (1.0 / asum) * d.lr;
    const double target = d.rho * asum;
    const double band = 1e-12 * asum;
    bool ok = (t1 > t) & (t1 < tstop) & (asum > 1e-280) & (asum < 1e280) & (top <= 0x80000000u);
    sel = 0;
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      const double gap = cum[j] - target;
      sel += (gap < 0.0) ? 1 : 0;
      ok = ok & (__builtin_fabs(gap) > band);
    }
    return ok;
  }

  // One attempt of the leap for the lanes with `on`: Poisson draws of the
  // non-critical reactions at `tau` (P1_P2.py:222-243), the critical firing
  // `sel`, x' = x + V K and its check (P1_P2.py:509-540).  Returns 0 (valid),
  // -1 (negative counts: halve tau) or a flag.
  //
  // Reaction j's draw uses blocks (bc + j, it), it = 0, 1, ... for the PTRS
  // iterations.  Every lane works through its own list of draws, one iteration
  // of one draw per trip: a lane whose draw is rejected repeats it while
  // others go on to their next reaction, and the sampler's code exists once.
  // (One inlined sampler per reaction and a retry loop after them came to 58
  // KB of code for Lotka-Volterra, about the instruction cache.)
  template <int FORM>
  __device__ __forceinline__ int attempt(Ref& tab, Counters& cnt, bool on, const double (&a)[MP],
                                         unsigned crit, double tau, int sel, int32_t (&xn)[NP],
                                         unsigned long long& ev, const LaneGroup<FORM>& g) {
    const auto& P = tab.p();
    const int M = P.M;
    const uint64_t grp = bc;
    bc += on ? (uint64_t)M : 0ull;
    double lam[MP];
    int32_t K[MP];
    unsigned todo = 0;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < MP; ++j) {
      const double l = ((j < M) & !((crit >> j) & 1u)) ? a[j] * tau : 0.0;
      lam[j] = l;
      K[j] = (sel == j) ? 1 : 0;
      bad = bad | (l >= LAMBDA_LIMIT);
      todo |= (g.mine(j) & (l > 0.0)) ? (1u << j) : 0u;
    }
    todo = (on & !bad) ? todo : 0u;
    bool fail = false;
    const Key uk = key.scalar_seed(P.seed);
    uint32_t it = 0;
    while (wave_any(todo != 0u)) {
      const int j = todo != 0u ? __builtin_ctz(todo) : 0;
      const double l = pick<MP>(lam, j);
      const Words4 w = uk.block(grp + (uint64_t)(uint32_t)j, it);
      const double u0 = u53(w.w0, w.w1);
      const bool ptrs = (todo != 0u) & (l >= 10.0);
      const bool inv = (todo != 0u) & !(l >= 10.0);
      bool acc = inv;
      int32_t kk = 0;
      if (wave_any(ptrs)) {
        const PtrsF64 Pt = ptrs_setup_f64(ptrs ? l : 10.0);
        const double U = u0 - 0.5;
        const double V = u53(w.w2, w.w3);
        double kf, us;
        bool ok = ptrs_fast_f64(Pt, U, V, kf, us);
        const bool slow = ptrs & !ok & !((kf < 0.0) | ((us < 0.013) & (V > us)));
        if (wave_any(slow)) ok = ok | (slow & ptrs_slow_f64(Pt, V, slow ? kf : 10.0, slow ? us : 0.1));
        cnt.w.draws += ptrs ? 2u : 0u;
        cnt.w.ptrs += ptrs ? 1u : 0u;
        acc = acc | (ptrs & ok);
        kk = (ptrs & ok) ? (int32_t)kf : 0;
      }
      if (wave_any(inv)) {
        // sequential-search inversion; the first eight steps four to a branch
        // (past a search's end p and Fc are computed but not read) and without
        // divisions, each of which was most of a step's chain: Lotka-Volterra,
        // 16,411 simulations, 44.6 -> 42.1 ms, Schloegl, 40,000 to t = 5, 21.7 -> 19.4.
        // (Reciprocals of the later n from a table in memory cost more than the
        // divisions: one simulation per wavefront 0.74 -> 0.78 ms.)
        double p = exp_core_f64(inv ? -l : 0.0);
        double Fc = p;
        bool act = inv & (u0 > Fc);
        const auto step = [&](int n, double pn) {
          p = pn;
          Fc = Fc + p;
          kk = act ? n : kk;
          act = act & (u0 > Fc);
        };
        if (wave_any(act)) {  // (division by a power of two is a product)
          step(1, p * l);
          step(2, p * l * 0.5);
          step(3, div_by<3>(p * l));
          step(4, p * l * 0.25);
          if (wave_any(act)) {
            step(5, div_by<5>(p * l));
            step(6, div_by<6>(p * l));
            step(7, div_by<7>(p * l));
            step(8, p * l * 0.125);
            for (int n = 9; n <= INV_MAX_K && wave_any(act); ++n) step(n, p * l / (double)n);
          }
        }
        cnt.w.draws += inv ? 1u : 0u;
        cnt.w.inv += inv ? (unsigned int)kk : 0u;
      }
#pragma unroll
      for (int r = 0; r < MP; ++r) K[r] = (acc & (r == j)) ? kk : K[r];
      it = acc ? 0u : it + 1u;
      fail = fail | ((todo != 0u) & (it >= (uint32_t)PTRS_MAX_ITERS));
      todo = fail ? 0u : acc ? todo & (todo - 1u) : todo;
    }
    if (g.grouped()) {
#pragma unroll
      for (int j = 0; j < MP; ++j) K[j] = g.owners(K[j], j);
      fail = g.any(fail);
    }
    // TentativeUpdatedState / ValidState (P1_P2.py:509-540)
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
};

}  // namespace pst
