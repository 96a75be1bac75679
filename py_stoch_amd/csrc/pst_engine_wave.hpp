// pst_engine_wave.hpp -- mixed-precision engine for large networks: one
// wavefront per simulation.
//
// Networks up to 64 species and 256 reactions (random mass-action networks
// of 5-50 species and 10-200 reactions, for example) do not fit the
// one-simulation-per-lane kernels: their state, propensities and tables would
// not stay in registers.  Here the 64 lanes of a wavefront share one
// simulation: lane l owns reactions l, l + 64, l + 128, l + 192 and species
// l.  The method is the same as in pst_engine_f32.hpp (P1_P2.py:96-294,
// P3.py:73-149, gillespie.py:70-149) with the sums over reactions and species
// done as wavefront reductions:
//   propensities         per reaction lane, counts read from LDS
//   a0, a0c              wavefront sums (FP32 for the leap decision, FP64 for
//                        the reaction choice)
//   critical reactions   per reaction lane (P1_P2.py:314-327)
//   mu, sigma^2, tau1    per species lane over its column of V (transposed
//                        table, fixed order), then a wavefront minimum
//   reaction choice      FP64 prefix sum over reactions in index order
//   Poisson draws        every reaction lane draws its own K_j from Philox
//                        block (group + j, it) -- all draws of a leap in
//                        parallel
//   x' = x + V K         64-bit integer LDS atomics (order-independent)
// Ordinary SSA steps have a loop of their own (ssa_run).  State of the
// simulation (time, sample cursor, Philox counter, mode) is wavefront-uniform.
// Per wavefront LDS: x, x', propensities of non-critical reactions, the
// critical flags and the net changes of every reaction (about 7 KB).
#pragma once
#include "pst_engine_f32.hpp"

namespace pst {

constexpr int WAVE_MAX_N = 64;
constexpr int WAVE_MAX_M = 256;
constexpr int WAVE_R = WAVE_MAX_M / 64;  // reactions per lane
constexpr int WAVE_MAX_REACT = 4;        // species with a propensity factor, per reaction
constexpr int WAVE_MAX_V = 8;            // non-zero V entries per reaction
constexpr int WAVE_MAX_T = 2048;         // non-zero V entries in total
constexpr int WAVE_MAX_F = 4;            // propensity factors of a reaction in ssa_run

// Network of one job in sparse form (built by the host library).
struct WaveTab {
  int32_t N, M, kappa, nnz;
  uint8_t nr[WAVE_MAX_M];                  // propensity factors of reaction j
  uint8_t rs[WAVE_MAX_M][WAVE_MAX_REACT];  // their species
  uint8_t ro[WAVE_MAX_M][WAVE_MAX_REACT];  // order p (factors of the species)
  uint8_t rst[WAVE_MAX_M][WAVE_MAX_REACT]; // step: 1 falling factorial, 0 power
  uint8_t nv[WAVE_MAX_M];                  // V entries of reaction j
  uint8_t vs[WAVE_MAX_M][WAVE_MAX_V];      // their species
  int8_t vv[WAVE_MAX_M][WAVE_MAX_V];       // their values
  int8_t H[WAVE_MAX_N], Ht[WAVE_MAX_N], irs[WAVE_MAX_N], E[WAVE_MAX_N];
  uint16_t tstart[WAVE_MAX_N + 1];         // column of V of species i: entries tstart[i] .. tstart[i+1]-1
  uint16_t tj[WAVE_MAX_T];                 // reaction of the entry
  int8_t tv[WAVE_MAX_T];                   // value of the entry
  // the same for ssa_run: propensity factors (x_s - sub) one by one, a byte
  // each (species | sub << 6), and how many; net changes as (species, value)
  // byte pairs, species 255 past the last
  uint32_t fw[WAVE_MAX_M];
  uint8_t fn[WAVE_MAX_M];
  uint32_t vrow[WAVE_MAX_M][4];
  int32_t max_f;                           // most factors of a reaction; above WAVE_MAX_F: no ssa_run
};

struct WaveJob {
  JobParams p;
  WaveTab t;
};

struct WaveLds {
  long long xn[WAVE_MAX_N];  // tentative state (x + V K)
  int32_t x[WAVE_MAX_N];     // current state
  float anc[WAVE_MAX_M];     // propensity of non-critical reactions, 0 for critical ones
  int32_t K[WAVE_MAX_M];     // firings of the current leap attempt
  uint8_t crit[WAVE_MAX_M];
  uint32_t vrow[WAVE_MAX_M][4];  // WaveTab::vrow of the current job
};

__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
// v + (v of lane l ^ OFF): one step of a sum over the wavefront in the order of
// a butterfly from 32 down to 1.  Lane exchanges inside the vector unit
// (v_permlane*_swap, DPP) instead of 57-cycle trips through LDS.  A swap of v
// with itself leaves, in every lane, its own value in one result and its
// partner's in the other.  Below 16 the values repeat with the period of the
// step before, so a rotation of the row is the exchange.
template <int OFF>
__device__ __forceinline__ void lane_pair(uint32_t v, uint32_t& x, uint32_t& y) {
  if constexpr (OFF == 32 || OFF == 16) {
    const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false)
                             : __builtin_amdgcn_permlane16_swap(v, v, false, false);
    x = r[0];
    y = r[1];
  } else {
    constexpr int ctrl = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4e : 0xb1;  // row_ror:8, :4, quad_perm
    x = v;
    y = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xf, 0xf, true);
  }
}
template <int OFF>
__device__ __forceinline__ float add_xor(float v) {
  uint32_t x, y;
  lane_pair<OFF>(__builtin_bit_cast(uint32_t, v), x, y);
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
template <int OFF>
__device__ __forceinline__ double add_xor(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  uint32_t xl, yl, xh, yh;
  lane_pair<OFF>((uint32_t)b, xl, yl);
  lane_pair<OFF>((uint32_t)(b >> 32), xh, yh);
  return __builtin_bit_cast(double, ((uint64_t)xh << 32) | xl) + __builtin_bit_cast(double, ((uint64_t)yh << 32) | yl);
}
template <class T>
__device__ __forceinline__ T butterfly_sum(T v) {
  return add_xor<1>(add_xor<2>(add_xor<4>(add_xor<8>(add_xor<16>(add_xor<32>(v))))));
}
__device__ __forceinline__ float wave_sum_f(float v) { return butterfly_sum(v); }
__device__ __forceinline__ double wave_sum_d(double v) { return butterfly_sum(v); }

// inclusive prefix sum over lanes by DPP row shifts and row broadcasts (its
// order of additions is not wave_scan_d's)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double fast_scan_d(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ double read_lane_d(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float wave_min_f(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ long long wave_sum_ll(long long v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
// inclusive prefix sum over lanes
__device__ __forceinline__ double wave_scan_d(double v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// One simulation per wavefront, lanes over reactions and species.  All
// members are wavefront-uniform except the per-lane rate constants.
struct EngineWave {
  float k[WAVE_R];  // rates of the lane's reactions
  uint32_t fw[WAVE_R], fn;  // WaveTab::fw and fn (a byte each) of the lane's reactions

  Key key;
  uint64_t bc;
  double t, tnext;
  int F, flag, burst, mode;
  uint32_t nsteps;  // leap decisions + SSA steps so far (step budget)
  int64_t sim;

  // index of sample f of recorded species q in O (rows or blocks layout,
  // pst_driver.hpp; stored sample by sample by the species lane)
  __device__ __forceinline__ int64_t out_index(const JobParams& P, int q, int f) const {
    if (P.layout != LAYOUT_BLOCKS) return ((int64_t)q * P.ita + f) * P.o_stride + sim;
    return (((int64_t)q * ((P.ita + OUT_BLOCK - 1) / OUT_BLOCK) + f / OUT_BLOCK) * P.o_stride + sim) * OUT_BLOCK +
           (f & (OUT_BLOCK - 1));
  }

  // blocks layout: zeros after the last sample in its block
  __device__ __forceinline__ void pad_last_block(const JobParams& P, int q) const {
    if (P.layout != LAYOUT_BLOCKS) return;
    const int end = (P.ita + OUT_BLOCK - 1) / OUT_BLOCK * OUT_BLOCK;
    for (int f = P.ita; f < end; ++f) glb(P.O)[out_index(P, q, f)] = 0;
  }

  // write samples F..ita-1: x of the recorded species, or zeros
  __device__ __forceinline__ void fill_rest(const WaveJob& J, const WaveLds& L, int lane, bool zero, Counters& cnt) {
    const JobParams& P = J.p;
    if (lane == 0) cnt.w.samples += (unsigned int)(P.ita - F);
    if (lane < P.kappa) {
      const int32_t val = zero ? 0 : L.x[J.t.E[lane]];
      for (int f = F; f < P.ita; ++f) glb(P.O)[out_index(P, lane, f)] = val;
      pad_last_block(P, lane);
    }
  }

  // the parts of a job's table that ssa_run keeps at hand
  __device__ __forceinline__ void load(const WaveJob& J, WaveLds& L, int lane) {
    wave_lds_sync();  // the job before's net changes have been read
    fn = 0;
#pragma unroll
    for (int r = 0; r < WAVE_R; ++r) {
      const int j = lane + 64 * r;
      fw[r] = J.t.fw[j];
      fn |= (uint32_t)J.t.fn[j] << (8 * r);
#pragma unroll
      for (int w = 0; w < 4; ++w) L.vrow[j][w] = J.t.vrow[j][w];
    }
    wave_lds_sync();
  }

  __device__ __forceinline__ void start(const WaveJob& J, WaveLds& L, int lane, int64_t s) {
    const JobParams& P = J.p;
    const int64_t set = s / P.sims_per_set;
    sim = s;
#pragma unroll
    for (int r = 0; r < WAVE_R; ++r) {
      const int j = lane + 64 * r;
      k[r] = (j < P.M) ? (float)glb(P.rates)[set * P.M + j] : 0.0f;
    }
    if (lane < P.N) L.x[lane] = glb(P.x0)[set * P.N + lane];
    wave_lds_sync();
    key.init(P.seed, P.sim_offset + (uint64_t)s);
    bc = 0;
    t = 0.0;
    F = 0;
    tnext = (double)glb(P.I)[0];
    flag = 0;
    burst = 0;
    nsteps = 0;
    mode = P.method == 0 ? MODE_DECIDE : MODE_SSA;
  }

  // propensities of the lane's reactions from the compact factors
  __device__ __forceinline__ void props(const WaveLds& L, int M, int max_f, float (&a)[WAVE_R]) const {
#pragma unroll
    for (int r = 0; r < WAVE_R; ++r) {
      float v = 0.0f;
      if (64 * r < M) {  // whole slots past M are skipped by the wavefront
        v = k[r];
        const int nf = (int)((fn >> (8 * r)) & 0xffu);
#pragma unroll
        for (int e = 0; e < WAVE_MAX_F; ++e) {
          if (e < max_f) {
            const uint32_t b = (fw[r] >> (8 * e)) & 0xffu;
            const int32_t f = L.x[b & 63u] - (int32_t)(b >> 6);
            v = v * (e < nf ? (float)f : 1.0f);
          }
        }
      }
      a[r] = v;
    }
  }

  // The ordinary SSA steps of a burst (or of SSA methods) until one needs
  // step(): the end of the simulation, the last sample, the count limit, a
  // step budget, a stuck clock, or a reaction choice too close to call.  The
  // arithmetic is step()'s except for the prefix sums, whose additions come
  // in another order; both are within 1e-13 of the exact sums relative to
  // asum, so outside a band of 1e-12 asum they choose the same reaction.
  // What the loop needs per reaction is in registers (rates, factors) or LDS
  // (counts, net changes): step() reads the table's bytes from memory, one
  // dependent load after the other, ~19,000 cycles a step at four wavefronts per
  // SIMD.  Lane l draws the numbers of step l of the next 64.  Pure SSA of
  // three networks of 17-40 species, 300 simulations each: 20.5 -> 4.2 ms; 16
  // random networks by tau-leaping (57 M SSA steps, 0.7 M leaps) 162 -> 50 ms.
  __device__ __forceinline__ void ssa_run(const WaveJob& J, WaveLds& L, int lane, Counters& cnt) {
    const JobParams& P = J.p;
    const WaveTab& T = J.t;
    const int M = P.M, N = P.N, max_f = T.max_f;
    const double tstop = (double)glb(P.I)[P.ita - 1];
    const double tend = P.method == 2 ? (P.t_max < tstop ? P.t_max : tstop) : tstop;
    int32_t xl = lane < N ? L.x[lane] : 0;
    float nl = 0.0f, u = 0.0f;
    int left = 0;  // drawn numbers not used yet
    uint32_t n = 0;
    const uint32_t budget = P.max_steps != 0u ? (nsteps < P.max_steps ? P.max_steps - nsteps : 0u) : 0xffffffffu;
    const uint32_t lim = P.method == 0 && (uint32_t)burst < budget ? (uint32_t)burst : budget;
    while (n < lim) {
      if (left == 0) {
        const Words4 w = key.block(bc + (uint64_t)(n + (uint32_t)lane), 0);
        nl = -fast_log(u24(w.w0));
        u = u24(w.w1);
        left = 64;
      }
      const float nl1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, nl), 64 - left));
      const float u1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, u), 64 - left));
      float a[WAVE_R];
      props(L, M, max_f, a);
      double ad = 0.0;
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) ad += (double)a[r];
      const double asum = wave_sum_d(ad);
      const double t1 = t + (double)(nl1 * fast_rcp((float)asum));
      const double target = (double)u1 * asum;
      const double band = 1e-12 * asum;
      bool near = false;
      int sel = -1;
      double carry = 0.0;
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) {
        if (64 * r < M) {
          const double cum = fast_scan_d((double)a[r]) + carry;
          carry = read_lane_d(cum, 63);
          near = near | (__builtin_fabs(cum - target) <= band);
          const unsigned long long hit = __builtin_amdgcn_ballot_w64(cum >= target);
          sel = (sel < 0 && hit != 0ull) ? 64 * r + (int)__builtin_ctzll(hit) : sel;
        }
      }
      // (asum = 0 gives an infinite or undefined time, which fails here)
      const bool ok = (t1 > t) & (t1 < tend) & !near & (sel >= 0);
      if (__builtin_amdgcn_ballot_w64(!ok) != 0ull) break;
      const uint32_t* row = L.vrow[sel];
      int32_t dx = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t e2 = row[w];
        dx += (int)(e2 & 0xffu) == lane ? __builtin_amdgcn_sbfe((int)e2, 8, 8) : 0;
        dx += (int)((e2 >> 16) & 0xffu) == lane ? __builtin_amdgcn_sbfe((int)e2, 24, 8) : 0;
      }
      const int32_t xn = xl + dx;
      if (__builtin_amdgcn_ballot_w64(xn >= COUNT_LIMIT) != 0ull) break;
      while (t1 >= tnext) {  // sample-and-hold: the state before the step
        if (lane < P.kappa) glb(P.O)[out_index(P, lane, F)] = L.x[T.E[lane]];
        if (lane == 0) cnt.w.samples += 1;
        F = F + 1;
        tnext = (double)glb(P.I)[F];
      }
      xl = xn;
      if (lane < N) L.x[lane] = xl;
      wave_lds_sync();
      t = t1;
      n += 1;
      left -= 1;
    }
    bc += (uint64_t)n;
    nsteps += n;
    if (lane == 0) {
      cnt.w.uniforms += 2u * n;
      cnt.ssa += n;
      cnt.events += (unsigned long long)n;
    }
    if (P.method == 0) {
      burst -= (int)n;
      if (burst <= 0) mode = MODE_DECIDE;
    }
  }

  // one step (leap decision + leap, or one SSA step); returns true when the
  // simulation has ended
  __device__ bool step(const WaveJob& J, WaveLds& L, int lane, Counters& cnt) {
    const JobParams& P = J.p;
    const WaveTab& T = J.t;
    const int M = P.M, N = P.N;
    bool ssa = mode == MODE_SSA;
    if (ssa && P.method == 2 && !(t < P.t_max)) {
      fill_rest(J, L, lane, true, cnt);
      return true;
    }
    if (P.max_steps != 0u && nsteps >= P.max_steps) {
      fill_rest(J, L, lane, true, cnt);
      flag = FLAG_STEPS;
      return true;
    }
    nsteps += 1;
    // propensities of the lane's reactions
    float a[WAVE_R];
    if (T.max_f <= WAVE_MAX_F) {
      props(L, M, T.max_f, a);
    } else {
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) {
        const int j = lane + 64 * r;
        float v = 0.0f;
        if (64 * r < M && j < M) {  // whole slots past M are skipped by the wavefront
          v = k[r];
          const int nr = T.nr[j];
          for (int e = 0; e < nr; ++e) {
            const int xi = L.x[T.rs[j][e]];
            const int p = T.ro[j][e], st = T.rst[j][e];
            for (int q = 0; q < p; ++q) v = v * (float)(xi - st * q);
          }
        }
        a[r] = v;
      }
    }
    float a_lane = 0.0f;
    double ad_lane = 0.0;
#pragma unroll
    for (int r = 0; r < WAVE_R; ++r) {
      a_lane += a[r];
      ad_lane += (double)a[r];
    }
    const float a0 = wave_sum_f(a_lane);
    if (a0 == 0.0f) {
      fill_rest(J, L, lane, false, cnt);
      return true;
    }
    bool crit[WAVE_R];
#pragma unroll
    for (int r = 0; r < WAVE_R; ++r) crit[r] = false;
    float tau1 = __builtin_inff();
    if (!ssa) {
      if (lane == 0) cnt.w.decisions += 1;
      // critical reactions on V (P1_P2.py:314-327)
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) {
        const int j = lane + 64 * r;
        bool c = false;
        if (64 * r < M && j < M) {
#pragma unroll
          for (int e = 0; e < WAVE_MAX_V; ++e) {
            const uint32_t b = L.vrow[j][e / 2] >> (16 * (e % 2));
            const int v = __builtin_amdgcn_sbfe((int)b, 8, 8);
            if (v < 0) c = c || ((-v) * P.n_c > L.x[b & 63u]);
          }
          L.anc[j] = c ? 0.0f : a[r];
          L.crit[j] = c ? 1 : 0;
        }
        crit[r] = c;
      }
      wave_lds_sync();
      // mu, sigma^2 and the Cao bound per species (P1_P2.py:330-445)
      float cand = __builtin_inff();
      if (lane < N && T.irs[lane]) {
        float mu = 0.0f, s2 = 0.0f;
        bool any = false;
        const int e1 = T.tstart[lane + 1];
        for (int e = T.tstart[lane]; e < e1; ++e) {
          const int j = T.tj[e];
          const float v = (float)T.tv[e];
          const float aj = L.anc[j];
          mu += v * aj;
          s2 += v * v * aj;
          any = any || (L.crit[j] == 0);
        }
        if (any) {
          const int xi = L.x[lane];
          const float g_i = calc_g_f32(T.H[lane], T.Ht[lane], xi);
          const float num = fmaxf((float)P.eta * (float)xi * fast_rcp(g_i), 1.0f);
          cand = fminf(num * fast_rcp(fabsf(mu)), num * num * fast_rcp(s2));
        }
      }
      tau1 = wave_min_f(cand);
      if (tau1 < 10.0f * fast_rcp(a0)) {
        ssa = true;
        mode = MODE_SSA;
        burst = P.ssa_burst;
        if (T.max_f <= WAVE_MAX_F) return false;  // its steps run in ssa_run
        if (P.max_steps != 0u && nsteps >= P.max_steps) {
          fill_rest(J, L, lane, true, cnt);
          flag = FLAG_STEPS;
          return true;
        }
        nsteps += 1;
      }
    }
    // one-block draw: SSA step, or tau2 and the critical reaction
    double asum;
    if (ssa) {
      asum = wave_sum_d(ad_lane);
    } else {
      double c_lane = 0.0;
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) c_lane += crit[r] ? (double)a[r] : 0.0;
      asum = wave_sum_d(c_lane);
    }
    float tauX = __builtin_inff();
    uint32_t cw1 = 0;
    if (asum > 0.0) {
      const Words4 bw = key.block(bc, 0);
      bc += 1;
      if (lane == 0) cnt.w.uniforms += ssa ? 2 : 1;
      cw1 = bw.w1;
      tauX = -fast_log(u24(bw.w0)) * fast_rcp((float)asum);
    }
    const float tau_f = ssa ? tauX : fminf(tau1, tauX);
    int sel = -1;
    if (ssa || tau1 > tauX) {
      if (!ssa && lane == 0) cnt.w.uniforms += 1;
      // first reaction of the mask with sum_{r<=j} a_r >= rho2 * asum, in index order (FP64)
      const double target = (double)u24(cw1) * asum;
      double carry = 0.0;
      int last = -1;
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) {
        if (64 * r >= M) break;  // wavefront-uniform
        const int j = lane + 64 * r;
        const bool m = (j < M) && (ssa || crit[r]);
        const double v = m ? (double)a[r] : 0.0;
        const double cum = wave_scan_d(v, lane) + carry;
        carry = __shfl(cum, 63, 64);
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(m && cum >= target);
        const unsigned long long pos = __builtin_amdgcn_ballot_w64(m && a[r] > 0.0f);
        if (sel < 0 && hit != 0ull) sel = 64 * r + __builtin_ctzll(hit);
        if (pos != 0ull) last = 64 * r + 63 - __builtin_clzll(pos);
      }
      if (sel < 0) sel = last;
    }
    // tentative state in LDS
    if (lane < N) L.xn[lane] = L.x[lane];
    wave_lds_sync();
    float tau = tau_f;
    if (ssa) {
      if (sel >= 0 && lane < T.nv[sel]) {
        const int s = T.vs[sel][lane];
        L.xn[s] = L.xn[s] + T.vv[sel][lane];  // distinct species per entry
      }
      wave_lds_sync();
    } else {
      if (!(tau < __builtin_inff())) {
        fill_rest(J, L, lane, true, cnt);
        flag = FLAG_TAU_INF;
        return true;
      }
      long long ev = 0;
      const int st = leap(J, L, lane, cnt, sel, tau, ev);
      if (st != 0) {
        fill_rest(J, L, lane, true, cnt);
        flag = st;
        return true;
      }
      if (lane == 0) {
        cnt.events += (unsigned long long)ev;
        cnt.leaps += 1;
      }
    }
    // time advance and samples (sample-and-hold for SSA, interpolation for a leap)
    const double t0 = t;
    t = t + (double)tau;
    if (t == t0 && tau > 0.0f) {  // tau == 0 (a draw of u = 1) is a valid event
      fill_rest(J, L, lane, true, cnt);
      flag = FLAG_STALL;
      return true;
    }
    if (t >= tnext) {
      const float inv_gap = fast_rcp((float)(t - t0));
      while (t >= tnext) {
        const float frac = ssa ? 0.0f : (float)(tnext - t0) * inv_gap;
        if (lane < P.kappa) {
          const int s = T.E[lane];
          const int32_t xs = L.x[s];
          const int diff = (int)(L.xn[s] - (long long)xs);
          glb(P.O)[out_index(P, lane, F)] = xs + rn_f32_to_int((float)diff * frac);
          if (F == P.ita - 1) pad_last_block(P, lane);
        }
        if (lane == 0) cnt.w.samples += 1;
        F = F + 1;
        if (F == P.ita) return true;  // an SSA step ending the run is not applied
        tnext = (double)glb(P.I)[F];
      }
    }
    const bool over = __builtin_amdgcn_ballot_w64(lane < N && L.xn[lane] >= COUNT_LIMIT) != 0ull;
    if (lane < N) L.x[lane] = (int32_t)L.xn[lane];
    wave_lds_sync();
    if (ssa) {
      if (lane == 0) {
        cnt.ssa += 1;
        cnt.events += 1;
      }
      if (over) {
        fill_rest(J, L, lane, true, cnt);
        flag = FLAG_OVERFLOW;
        return true;
      }
      if (P.method == 0) {
        burst -= 1;
        if (burst <= 0) mode = MODE_DECIDE;
      }
    }
    return false;
  }

  // Poisson leap with halving; x' left in L.xn, tau halved in place (the
  // clock advances by the tau of the accepted draw, P1_P2.py:258-261).
  // Returns 0 or a flag.  The
  // lane's reaction slots are walked in a rolled loop with the counts in LDS,
  // so the sampler's code (and its registers) exists once.
  __device__ int leap(const WaveJob& J, WaveLds& L, int lane, Counters& cnt, int sel, float& tau, long long& ev) {
    const JobParams& P = J.p;
    const int M = P.M, N = P.N;
    for (int h = 0; h < MAX_HALVINGS; ++h) {
      const uint64_t grp = bc;
      bc += (uint64_t)M;
      bool bad = false, fail = false;
#pragma unroll 1
      for (int r = 0; r < WAVE_R; ++r) {
        const int j = lane + 64 * r;
        if (j >= M) continue;
        int32_t kk = (j == sel) ? 1 : 0;
        const float l = L.anc[j] * tau;  // 0 for critical reactions
        bad = bad || (l >= (float)LAMBDA_LIMIT);
        if (l > 0.0f && !bad) {
          const Words4 bw = key.block(grp + (uint64_t)j, 0);
          if (l < POIS_ASYM_MIN) {
            // sequential-search inversion
            cnt.w.uniforms += 1;
            const float u = u24(bw.w0);
            float p = fast_exp(-l), Fc = p;
            int n = 0;
            while (u > Fc && n < INV_MAX_K) {
              n += 1;
              p = p * l * fast_rcp((float)n);
              const float Fn = Fc + p;
              if (!(Fn > Fc)) break;  // the FP32 sum stopped growing (far tail; u may be 1.0)
              Fc = Fn;
            }
            cnt.w.inv += (unsigned int)n;
            kk = n;
          } else if (l < POIS_ASYM_MAX) {
            // asymptotic inversion, decided in FP64 near an integer boundary
            cnt.w.asym += 1;
            cnt.w.uniforms += 1;
            const float u = u24(bw.w0);
            bool ex = false;
            int32_t m = -1;
            kk = poisson_asym_f32(l, u, ex, m);
            if (ex) {
              cnt.w.exact += 1;
              kk = poisson_exact_f64((double)l, (double)u, m);
            }
          } else {
            const Draw d = ptrs_wide(key.k0, key.k1, key.s_lo, key.s_hi, grp + (uint64_t)j, 0, l);
            cnt.w.ptrs += d.iters;
            cnt.w.uniforms += 2 * d.iters;
            if (d.k < 0) fail = true;
            else kk = (int32_t)d.k;
          }
        }
        L.K[j] = kk;
      }
      if (__builtin_amdgcn_ballot_w64(bad) != 0ull) return FLAG_OVERFLOW;
      if (__builtin_amdgcn_ballot_w64(fail) != 0ull) return FLAG_PTRS;
      // x' = x + V K (TentativeUpdatedState, P1_P2.py:509-524)
      if (lane < N) L.xn[lane] = L.x[lane];
      wave_lds_sync();
      long long ev_lane = 0;
#pragma unroll
      for (int r = 0; r < WAVE_R; ++r) {
        if (64 * r >= M) break;  // wavefront-uniform
        const int j = lane + 64 * r;
        if (j >= M) continue;
        const int32_t kk = L.K[j];
        if (kk != 0) {
          ev_lane += kk;
          for (int e = 0; e < WAVE_MAX_V; ++e) {
            const uint32_t b = L.vrow[j][e / 2] >> (16 * (e % 2));
            const int v = __builtin_amdgcn_sbfe((int)b, 8, 8);
            if (v == 0) break;  // past the last entry
            atomicAdd((unsigned long long*)&L.xn[b & 63u], (unsigned long long)((long long)kk * v));
          }
        }
      }
      wave_lds_sync();
      // ValidState (P1_P2.py:526-540)
      const bool neg = lane < N && L.xn[lane] < 0;
      if (__builtin_amdgcn_ballot_w64(neg) == 0ull) {
        const bool big = lane < N && L.xn[lane] >= COUNT_LIMIT;
        if (__builtin_amdgcn_ballot_w64(big) != 0ull) return FLAG_OVERFLOW;
        ev = wave_sum_ll(ev_lane);
        return 0;
      }
      if (lane == 0) cnt.rejected += 1;
      tau = tau * 0.5f;
    }
    return FLAG_HALVING;
  }
};

}  // namespace pst
