// pst_args.hpp -- kernel argument blocks shared by the launch code and the kernels.
//
// A network is passed to the table-driven kernels as lists of its non-zero
// entries (NetTab) inside a job descriptor in device memory: every entry is the
// same for all lanes of a wavefront, so every branch on it is a scalar branch.
// Per-simulation data (state, time, sample cursor, Philox counter) lives in
// VGPRs for the whole run.
#pragma once
#ifndef __HIPCC_RTC__
#include <stdint.h>
#include <hip/hip_runtime.h>
#endif

namespace pst {

#ifndef __HIPCC_RTC__  // (the table-driven kernels are built with the library)
// Network table of a size class (capacity NP species x MP reactions) as lists
// of its non-zero entries, species ascending within a reaction.
template <int NP, int MP>
struct NetTab {
  uint16_t fac[NP * MP];   // propensity factors, reaction by reaction: species | step << 5 | last of
                           // its reaction << 6 | order << 8 (order factors of the species, step 1:
                           // x(x-1)(x-2)..., 0: x^order; order 0: a reaction without factors)
  uint16_t vent[NP * MP];  // net changes V = Post - Pre (d_V, P1_P2.py:8): species | (uint8) value << 8
  uint32_t vrange[MP];     // reaction j's net changes: first | end << 16
  uint32_t species[NP];    // H (d_H, P1_P2.py:9) | H_type << 8 (P1_P2.py:10) | 1 << 16 if the species has any
                           // Pre entry (I_rs, P1_P2.py:338-346)
  uint32_t recorded[2];    // recorded species (d_E, P1_P2.py:13), four bits each
  int8_t vrow[MP * NP];    // V once more, dense and reaction-major: the change of every species by reaction j
};

#endif

enum StatIdx {
  ST_EVENTS = 0, ST_LEAPS, ST_REJECTED, ST_SSA, ST_FLAGGED,
  ST_UNIFORMS, ST_PTRS, ST_INV, ST_DECISIONS, ST_SAMPLES, ST_FEVENTS, ST_ASYM, ST_EXACT,
  ST_COUNT = 16
};

// Settings of one job of a launch (uniform across the wavefronts working on it)
struct JobParams {
  int32_t N, M;
  int32_t kappa, ita;
  int32_t n_c;          // critical threshold (tl_parser.py:43)
  int32_t ssa_burst;    // SSA steps per fallback burst (P3.py:71)
  int32_t method;       // 0 tau-leaping, 1 forced SSA, 2 pure SSA
  int32_t n_sims;
  int32_t sims_per_set; // simulations sharing one rates/x0 row
  int32_t ssa_slice;    // SSA steps per pass while other lanes wait to decide (launch tuning)
  int32_t n_rates;      // length of a rates row: M, or the parameter count of compiled hazards
  uint32_t max_steps;   // 0: none; else leap decisions + SSA steps per simulation
  int32_t lanes;        // simulations per wavefront, 1..64 (launch tuning)
  int32_t layout;       // trajectory layout of O: LAYOUT_ROWS or LAYOUT_BLOCKS (pst_driver.hpp)
  double eta;           // tl_parser.py:44
  double t_max;
  uint64_t seed;
  uint64_t sim_offset;
  int64_t o_stride;     // fastest-axis length of O (>= n_sims)
  const double* rates;  // [n_sets][M]
  const int32_t* x0;    // [n_sets][N]
  const float* I;       // [ita] sample times
  int32_t* O;           // rows: [kappa][ita][o_stride]; blocks: [kappa][ceil(ita/8)][o_stride][8]
  int32_t* flags;       // [n_sims] or null
  uint32_t* state;      // [state_words][n_sims] saved simulations between sample ranges, or null
  int32_t state_words;  // words per simulation in state (at least the engine's record)
  int32_t reserved2;
};

// The sample range of a launch (pst_driver.hpp): stop simulations at sample
// f_end (saving their state), and/or resume them from their saved state.
struct Range {
  int32_t f_end;
  int32_t resume;
};
constexpr Range FULL_RUN = {0x7fffffff, 0};

// A job's settings re-read from its descriptor, for the rarely used ones (a
// simulation's start and end, the saved-state record): the pointer is hidden
// from the optimizer, so the scalar loads stay where they are used instead of
// holding a register through the simulation loop.
__device__ __forceinline__ const JobParams& cold_params(const JobParams* jp) {
  uint64_t a = (uint64_t)jp;
  a = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  asm volatile("" : "+s"(a));
  return *(const JobParams*)(__attribute__((address_space(4))) const JobParams*)a;
}

// Copy a job's settings into VGPRs (an empty asm on each 32-bit word hides
// their uniformity).  They are read only by per-lane arithmetic (addresses,
// sample cursor, queue bounds), and held in SGPRs they would exceed the
// scalar register file and be spilled and reloaded lane by lane.
__device__ __forceinline__ void load_params_vgpr(JobParams* dst, const JobParams* src) {
  constexpr int NWORDS = (int)(sizeof(JobParams) / 4);
  uint32_t w[NWORDS];
  __builtin_memcpy(w, src, sizeof(JobParams));
#pragma unroll
  for (int i = 0; i < NWORDS; ++i) asm volatile("" : "+v"(w[i]));
  __builtin_memcpy(dst, w, sizeof(JobParams));
}

// LDS accesses of some lanes of a wavefront before those of others: the
// hardware keeps a wavefront's LDS operations in order, the compiler only where
// it is told that another lane may read or write the same word.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

#ifndef __HIPCC_RTC__
template <int NP, int MP>
struct JobDev {
  NetTab<NP, MP> tab;
  JobParams p;
};

#endif

// v[i] for a wavefront-uniform i: a register picked by index (through a vector
// value, so that the array itself stays in registers)
template <class T, int N>
__device__ __forceinline__ T at(const T (&v)[N], int i) {
  typedef T Vec __attribute__((ext_vector_type(N)));
  Vec w;
#pragma unroll
  for (int q = 0; q < N; ++q) w[q] = v[q];
  return w[i];
}

#ifndef __HIPCC_RTC__
// Kernel-side view of the current job of a table-driven kernel.  The lists are
// held in vector registers, one word per lane, and read one word at a time
// into a scalar register (v_readlane); loops over reactions and their entries
// are rolled, so the code has the size of one entry, whatever the class.  (A
// dense byte table in scalar registers with every loop unrolled came to 84 KB
// of code for 4 x 4 and 300 KB for 16 x 16, beyond the 64 KB instruction
// cache, and walked the zero entries too.)  The net changes of a reaction
// chosen per lane are read from a dense copy in LDS.
// v_readlane reads lanes whether they are on or not, and a copy the register
// allocator makes where some are off leaves theirs undefined: lists are read
// only where the whole wavefront is on.  What branches on a lane mask need (the
// recorded species, net changes) is the same in every lane, or in LDS.
template <int NP, int MP>
struct JobRef {
  static constexpr int kNP = NP, kMP = MP;
  static constexpr int kKP = MP;          // rates per row: one per reaction
  static constexpr bool kCustom = false;  // propensities from the mass-action table
  static constexpr bool kTable = true;    // table entries are run-time values
  static constexpr int kOutLds = NP < 4 ? NP : 4;  // recorded species gathered in LDS (blocked layout)
  using Dev = JobDev<NP, MP>;
  static constexpr int EW = (NP * MP / 2 + 63) / 64;  // registers of an entry list
  uint32_t fac[EW], vent[EW], vrange, species;
  uint64_t recorded;
  JobParams P;
  const JobParams* jp;
  __device__ __forceinline__ const JobParams& cold() const { return cold_params(jp); }

  static __device__ __forceinline__ uint32_t* rows() {
    __shared__ uint32_t buf[4 * NP * MP / 4];
    return buf + (threadIdx.x >> 6) * (NP * MP / 4);
  }
  __device__ __forceinline__ void load(const JobDev<NP, MP>* jd) {
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t* f = reinterpret_cast<const uint32_t*>(jd->tab.fac);
    const uint32_t* v = reinterpret_cast<const uint32_t*>(jd->tab.vent);
#pragma unroll
    for (int r = 0; r < EW; ++r) {
      const int w = r * 64 + lane;
      fac[r] = w < NP * MP / 2 ? f[w] : 0u;
      vent[r] = w < NP * MP / 2 ? v[w] : 0u;
    }
    vrange = lane < MP ? jd->tab.vrange[lane] : 0u;
    species = lane < NP ? jd->tab.species[lane] : 0u;
    recorded = jd->tab.recorded[0] | ((uint64_t)jd->tab.recorded[1] << 32);
    const uint32_t* d = reinterpret_cast<const uint32_t*>(jd->tab.vrow);
    wave_lds_sync();  // the job before's rows have been read
    if (lane < NP * MP / 4) rows()[lane] = d[lane];  // NP * MP / 4 <= 64; read by this wavefront only
    wave_lds_sync();
    jp = &jd->p;
    load_params_vgpr(&P, jp);
  }
  static __device__ __forceinline__ uint32_t word(uint32_t v, int i) { return (uint32_t)__builtin_amdgcn_readlane((int)v, i); }
  static __device__ __forceinline__ uint32_t entry(const uint32_t (&v)[EW], int e) {
    uint32_t w = word(v[0], (e >> 1) & 63);
#pragma unroll
    for (int r = 1; r < EW; ++r) w = (e >> 7) == r ? word(v[r], (e >> 1) & 63) : w;
    return (e & 1) ? w >> 16 : w & 0xffffu;
  }
  __device__ __forceinline__ const JobParams& p() const { return P; }
  __device__ __forceinline__ int n_reactions() const { return __builtin_amdgcn_readfirstlane(P.M); }
  __device__ __forceinline__ int n_species() const { return __builtin_amdgcn_readfirstlane(P.N); }
  __device__ __forceinline__ int n_recorded() const { return __builtin_amdgcn_readfirstlane(P.kappa); }
  __device__ __forceinline__ int method() const { return __builtin_amdgcn_readfirstlane(P.method); }
  __device__ __forceinline__ int Hv(int i) const { return (int)(word(species, i) & 0xffu); }
  __device__ __forceinline__ int Htv(int i) const { return (int)((word(species, i) >> 8) & 0xffu); }
  __device__ __forceinline__ bool Irs(int i) const { return (word(species, i) >> 16) & 1u; }
  __device__ __forceinline__ int Ev(int q) const { return (int)((uint32_t)(recorded >> (4 * q)) & 15u); }

  // body(i) for every species, rolled (i is wavefront-uniform: index arrays with at())
  template <class F>
  __device__ __forceinline__ void for_species(F body) const {
    const int n = n_species();
#pragma unroll 1
    for (int i = 0; i < n; ++i) body(i);
  }
  template <class F>
  __device__ __forceinline__ void for_recorded(F body) const {
    const int n = n_recorded();
#pragma unroll 1
    for (int q = 0; q < n; ++q) body(q);
  }

  // propensities a_j = k_j * product of factors (UpdatePropensities, parser.py:32-55)
  template <class R>
  __device__ __forceinline__ void props(const int32_t (&x)[NP], const R (&k)[MP], R (&a)[MP]) const {
    typedef R RVec __attribute__((ext_vector_type(MP)));
    RVec av;
#pragma unroll
    for (int j = 0; j < MP; ++j) av[j] = (R)0;
    const int n = n_reactions();
    R v = k[0];
    // one trip per listed species, with a branch only for orders above 1 (a
    // uniform branch costs ~50 cycles, a select 9): with branches for order 0 and
    // for the last of a reaction too, 8 reactions, 262,144 simulations, took 34.2
    // ms mixed and 35.7 FP64, now 31.3 and 31.1; Schloegl 39.7 / 40.1, now 38.0 /
    // 38.0.  One entry per factor instead of the inner loop: 47.5 / 45.4.
#pragma unroll 1
    for (int e = 0, j = 0; j < n; ++e) {
      const uint32_t w = entry(fac, e);
      const int order = (int)(w >> 8);
      const int32_t xi = at<int32_t, NP>(x, (int)(w & 31u));
      v = v * (R)(order > 0 ? xi : 1);
      if (order > 1) {
        const int step = (int)((w >> 5) & 1u);
        for (int q = 1; q < order; ++q) v = v * (R)(xi - step * q);
      }
      av[j] = v;
      const bool last = (w & 64u) != 0u;
      j += last ? 1 : 0;
      const R kj = at<R, MP>(k, j & (MP - 1));
      v = last ? kj : v;
    }
#pragma unroll
    for (int j = 0; j < MP; ++j) a[j] = av[j];
  }
  // props and their FP32 sum, of rounded products (they come from a loop)
  __device__ __forceinline__ float props_sum(const int32_t (&x)[NP], const float (&k)[MP], float (&a)[MP]) const {
    props<float>(x, k, a);
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < MP; ++j) sum += a[j];
    return sum;
  }

  // critical reactions (P1_P2.py:314-327, on V) as a bit mask; mu and sigma^2
  // of every species over the non-critical reactions and whether it has any
  // (P1_P2.py:330-383)
  template <class R>
  __device__ __forceinline__ void sums(const int32_t (&x)[NP], const R (&a)[MP], int n_c, unsigned& crit, R (&mu)[NP],
                                       R (&s2)[NP], unsigned& any) const {
    typedef R RVec __attribute__((ext_vector_type(NP)));
    RVec m, s;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      m[i] = (R)0;
      s[i] = (R)0;
    }
    crit = 0u;
    any = 0u;
    const int n = n_reactions();
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      const uint32_t vr = word(vrange, j);
      const int e0 = (int)(vr & 0xffffu), e1 = (int)(vr >> 16);
      bool c = false;
#pragma unroll 1
      for (int e = e0; e < e1; ++e) {
        const uint32_t w = entry(vent, e);
        const int v = (int)(int8_t)(w >> 8);
        if (v < 0) c = c | ((-v) * n_c > at<int32_t, NP>(x, (int)(w & 31u)));
      }
      crit |= c ? (1u << j) : 0u;
      const R aj = at<R, MP>(a, j);
#pragma unroll 1
      for (int e = e0; e < e1; ++e) {
        const uint32_t w = entry(vent, e);
        const int i = (int)(w & 31u), v = (int)(int8_t)(w >> 8);
        m[i] += c ? (R)0 : (R)v * aj;
        s[i] += c ? (R)0 : (R)(v * v) * aj;
        any |= c ? 0u : (1u << i);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      mu[i] = m[i];
      s2[i] = s[i];
    }
  }

  // s = x + V K
  __device__ __forceinline__ void advance(const int32_t (&x)[NP], const int32_t (&K)[MP], int64_t (&s)[NP]) const {
    typedef int64_t LVec __attribute__((ext_vector_type(NP)));
    LVec t;
#pragma unroll
    for (int i = 0; i < NP; ++i) t[i] = x[i];
    const int n = n_reactions();
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      const uint32_t vr = word(vrange, j);
      const int e1 = (int)(vr >> 16);
      const int64_t kj = at<int32_t, MP>(K, j);
#pragma unroll 1
      for (int e = (int)(vr & 0xffffu); e < e1; ++e) {
        const uint32_t w = entry(vent, e);
        t[(int)(w & 31u)] += kj * (int)(int8_t)(w >> 8);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) s[i] = t[i];
  }

  // d = V(., sel) for a per-lane sel in [0, MP)
  __device__ __forceinline__ void row(int sel, int32_t (&d)[NP]) const {
    const uint32_t* r = rows() + sel * (NP / 4);
#pragma unroll
    for (int w = 0; w < NP / 4; ++w) {
      const int32_t b = (int32_t)r[w];
#pragma unroll
      for (int q = 0; q < 4; ++q) d[4 * w + q] = __builtin_amdgcn_sbfe(b, 8 * q, 8);
    }
  }
};

#endif  // !__HIPCC_RTC__

// Kernel-side view of a job whose network is compiled into the kernel (the
// library generates `Net` and compiles it at run time, as the reference
// compiles each model's propensity code, cuTauLeaping.py:34-35): every table
// entry and every network-level setting is a constant, so the loops over
// species and reactions become straight-line code.  Net provides
//   static constexpr int N, M, kappa, n_c, method, ssa_burst;
//   static constexpr double eta;
//   static constexpr int8_t v[N*M], ord[N*M], stp[N*M], H[N], Ht[N], irs[N], E[N];
//   static constexpr bool custom; static constexpr int n_rates;
//   template <class R> static void props(x, c, a)   (used when custom)
// The job descriptor is the JobParams block alone.
template <class Net>
struct FixedParams : JobParams {
  static constexpr int N = Net::N, M = Net::M;
  static constexpr int kappa = Net::kappa, n_c = Net::n_c, method = Net::method, ssa_burst = Net::ssa_burst;
  static constexpr double eta = Net::eta;
};

template <class Net>
struct FixedRef {
  static constexpr int kNP = Net::N, kMP = Net::M;
  static constexpr int kKP = Net::n_rates;   // rates per row
  static constexpr bool kCustom = Net::custom;  // compiled hazard expressions
  static constexpr bool kTable = false;         // table entries are constants
  static constexpr int kOutLds = Net::kappa < 4 ? Net::kappa : 4;  // recorded species gathered in LDS
  using Dev = JobParams;
  FixedParams<Net> P;
  const JobParams* jp;
  __device__ __forceinline__ void load(const JobParams* p) {
    jp = p;
    load_params_vgpr(&P, p);
  }
  __device__ __forceinline__ const JobParams& cold() const { return cold_params(jp); }
  __device__ __forceinline__ const FixedParams<Net>& p() const { return P; }
  __device__ __forceinline__ static constexpr int method() { return Net::method; }
  __device__ __forceinline__ static constexpr int n_reactions() { return kMP; }
  // bytes V(i, 4 r) .. V(i, 4 r + 3) as one word
  static constexpr uint32_t Vword(int i, int r) {
    uint32_t w = 0;
    for (int b = 0; b < 4; ++b)
      if (4 * r + b < kMP) w |= ((uint32_t)Net::v[i * kMP + 4 * r + b] & 0xffu) << (8 * b);
    return w;
  }
  __device__ __forceinline__ static constexpr int V(int i, int j) { return Net::v[i * kMP + j]; }
  __device__ __forceinline__ static constexpr int Hv(int i) { return Net::H[i]; }
  __device__ __forceinline__ static constexpr int Htv(int i) { return Net::Ht[i]; }
  __device__ __forceinline__ static constexpr int Irs(int i) { return Net::irs[i]; }
  __device__ __forceinline__ static constexpr int Ev(int q) { return Net::E[q]; }
  template <class F>
  __device__ __forceinline__ static void for_species(F body) {
#pragma unroll
    for (int i = 0; i < kNP; ++i) body(i);
  }
  template <class F>
  __device__ __forceinline__ static void for_recorded(F body) {
#pragma unroll
    for (int q = 0; q < Net::kappa; ++q) body(q);
  }
  // the same operations as JobRef's, in straight-line code
  template <class R>
  __device__ __forceinline__ static void props(const int32_t (&x)[kNP], const R (&k)[kKP], R (&a)[kMP]) {
    if constexpr (kCustom) {
      Net::template props<R>(x, k, a);  // compiled hazard expressions
    } else {
#pragma unroll
      for (int j = 0; j < kMP; ++j) {
        R v = k[j];
#pragma unroll
        for (int i = 0; i < kNP; ++i)
          for (int q = 0; q < Net::ord[i * kMP + j]; ++q) v = v * (R)(x[i] - Net::stp[i * kMP + j] * q);
        a[j] = v;
      }
    }
  }
  // propensity factors of reaction j, counted with their order
  static constexpr int factors(int j) {
    int n = 0;
    for (int i = 0; i < kNP; ++i) n += Net::ord[i * kMP + j];
    return n;
  }
  // props and their FP32 sum, in which each reaction's last product enters
  // unrounded (one fused operation).  The sum decides between a leap and an SSA
  // burst, so a bit of it can send a simulation another way: it is fused here,
  // not left to the compiler, which fuses only if it keeps sum and products in
  // one basic block (and in decide moved the sum behind a branch wherever two
  // species change: 1 simulation of 8192 took another path).  The sum of hazard
  // expressions is held in their block by the volatile asm.
  __device__ __forceinline__ static float props_sum(const int32_t (&x)[kNP], const float (&k)[kKP], float (&a)[kMP]) {
    float sum = 0.0f;
    if constexpr (kCustom) {
      Net::template props<float>(x, k, a);
#pragma unroll
      for (int j = 0; j < kMP; ++j) sum += a[j];
      asm volatile("" : "+v"(sum));
    } else {
#pragma unroll
      for (int j = 0; j < kMP; ++j) {
        float v = k[j];
        int left = factors(j);
        if (left == 0) sum += v;
#pragma unroll
        for (int i = 0; i < kNP; ++i)
          for (int q = 0; q < Net::ord[i * kMP + j]; ++q) {
            const float f = (float)(x[i] - Net::stp[i * kMP + j] * q);
            if (--left == 0) sum = __builtin_fmaf(v, f, sum);
            v = v * f;
          }
        a[j] = v;
      }
    }
    return sum;
  }
  // s + w aj for a term of mu or sigma^2.  FP32: fused for a reaction that can
  // never be critical, else the product is rounded first (again one form for
  // every build; it matters from net changes of 3 on).
  static constexpr bool never_critical(int j) {
    for (int i = 0; i < kNP; ++i)
      if (V(i, j) < 0) return false;
    return true;
  }
  __device__ __forceinline__ static double add_term(double s, int w, double aj, bool, bool on) {
    return s + (on ? (double)w * aj : 0.0);
  }
  __device__ __forceinline__ static float add_term(float s, int w, float aj, bool never, bool on) {
    return never ? __builtin_fmaf((float)w, aj, s) : s + (on ? (float)w * aj : 0.0f);
  }
  template <class R>
  __device__ __forceinline__ static void sums(const int32_t (&x)[kNP], const R (&a)[kMP], int n_c, unsigned& crit,
                                              R (&mu)[kNP], R (&s2)[kNP], unsigned& any) {
    crit = 0u;
    any = 0u;
    bool cr[kMP];
#pragma unroll
    for (int j = 0; j < kMP; ++j) {
      bool c = false;
#pragma unroll
      for (int i = 0; i < kNP; ++i)
        if (V(i, j) < 0) c = c | (-V(i, j) * n_c > x[i]);
      cr[j] = c;
      crit |= c ? (1u << j) : 0u;
    }
#pragma unroll
    for (int i = 0; i < kNP; ++i) {
      R m = (R)0, s = (R)0;
      bool some = false;
#pragma unroll
      for (int j = 0; j < kMP; ++j) {
        const int v = V(i, j);
        if (v != 0) {
          const bool nc = !cr[j];
          m = add_term(m, v, a[j], never_critical(j), nc);
          s = add_term(s, v * v, a[j], never_critical(j), nc);
          some = some | nc;
        }
      }
      mu[i] = m;
      s2[i] = s;
      any |= some ? (1u << i) : 0u;
    }
  }
  __device__ __forceinline__ static void advance(const int32_t (&x)[kNP], const int32_t (&K)[kMP], int64_t (&s)[kNP]) {
#pragma unroll
    for (int i = 0; i < kNP; ++i) {
      int64_t t = x[i];
#pragma unroll
      for (int j = 0; j < kMP; ++j)
        if (V(i, j) != 0) t += (int64_t)K[j] * V(i, j);
      s[i] = t;
    }
  }
  // bit-field extracts from constants
  __device__ __forceinline__ static void row(int sel, int32_t (&d)[kNP]) {
#pragma unroll
    for (int i = 0; i < kNP; ++i) {
      uint32_t w = Vword(i, 0);
#pragma unroll
      for (int r = 1; r < (kMP + 3) / 4; ++r) w = (sel >> 2) == r ? Vword(i, r) : w;
      d[i] = __builtin_amdgcn_sbfe((int)w, (unsigned)(sel & 3) * 8u, 8u);
    }
  }
};

#ifndef __HIPCC_RTC__
// host-side copy of a network in dense form, built by the C-ABI layer
struct HostNet {
  int N, M, kappa;
  int8_t v[64 * 256];
  int8_t ord[64 * 256];
  int8_t stp[64 * 256];
  int8_t H[64], Ht[64], irs[64];
  int8_t E[64];
};

// size classes compiled into the library
constexpr int NUM_CLASSES = 3;
constexpr int CLASS_NP[NUM_CLASSES] = {4, 8, 16};
constexpr int CLASS_MP[NUM_CLASSES] = {4, 8, 16};

template <int NP, int MP>
inline NetTab<NP, MP> make_tab(const HostNet& h) {
  NetTab<NP, MP> t = {};
  int nf = 0, nv = 0;
  for (int j = 0; j < h.M; ++j) {
    const int v0 = nv;
    int last = -1;
    for (int i = 0; i < h.N; ++i) {
      const int p = h.ord[i * h.M + j], v = h.v[i * h.M + j];
      if (p > 0) t.fac[last = nf++] = (uint16_t)(i | (h.stp[i * h.M + j] ? 1 << 5 : 0) | (p << 8));
      if (v != 0) t.vent[nv++] = (uint16_t)(i | (((unsigned)v & 0xffu) << 8));
      t.vrow[j * NP + i] = (int8_t)v;
    }
    if (last < 0) t.fac[last = nf++] = 0;
    t.fac[last] |= 1 << 6;
    t.vrange[j] = (uint32_t)v0 | ((uint32_t)nv << 16);
  }
  for (int i = 0; i < h.N; ++i)
    t.species[i] = (uint32_t)h.H[i] | ((uint32_t)h.Ht[i] << 8) | ((uint32_t)(h.irs[i] != 0) << 16);
  for (int q = 0; q < h.kappa; ++q) t.recorded[q / 8] |= (uint32_t)h.E[q] << (4 * (q % 8));
  return t;
}

// Launchers, one per translation unit (precision).  `jobs` is a device array
// of JobDev<NP,MP> for the size class `cls`, `queue` n_jobs zeroed counters,
// `waves` the number of wavefronts to launch, `group` whether the jobs have
// fewer than 64 simulations per wavefront (a group of lanes per simulation).
int launch_fp64(int cls, const void* jobs, int n_jobs, unsigned int* queue, unsigned long long* stats,
                int waves, Range range, bool group, hipStream_t stream);
int launch_mixed(int cls, const void* jobs, int n_jobs, unsigned int* queue, unsigned long long* stats,
                 int waves, Range range, bool group, hipStream_t stream);
// the mixed-precision Poisson sampler on given means and words (validation)
int launch_poisson_probe(const float* lam, const uint32_t* words, int64_t n, int32_t* k, int32_t* path,
                         hipStream_t stream);
// resident 256-lane blocks per CU for a class (occupancy)
int blocks_per_cu_fp64(int cls, bool group);
int blocks_per_cu_mixed(int cls, bool group);

// the large-network kernel (one wavefront per simulation, mixed precision):
// `jobs` is a device array of WaveJob
struct WaveTab;
int launch_wave(const void* jobs, int n_jobs, unsigned int* queue, unsigned long long* stats, int waves,
                hipStream_t stream);
int blocks_per_cu_wave();
bool make_wave_tab(const HostNet& h, WaveTab* t, char* why, size_t why_len);

// smallest compiled size class holding (N, M, kappa), or -1
inline int size_class(int N, int M, int kappa) {
  for (int c = 0; c < NUM_CLASSES; ++c)
    if (N <= CLASS_NP[c] && M <= CLASS_MP[c] && kappa <= CLASS_NP[c]) return c;
  return -1;
}

#endif  // !__HIPCC_RTC__

}  // namespace pst
