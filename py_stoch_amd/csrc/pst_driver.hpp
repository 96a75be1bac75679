// pst_driver.hpp -- the persistent, wavefront-uniform simulation driver shared
// by the FP64 and mixed-precision engines.
//
// A launch processes a list of jobs (network + run settings + parameter rows
// + output array).  Each wavefront works on one job at a time, so the network
// table is uniform across its lanes; its first `lanes` lanes (JobParams; 64
// unless the launch has fewer simulations than 64 per SIMD) take simulations
// of that job from a device work queue (one atomic per wavefront per refill)
// and take the next one as soon as theirs ends, so uneven step counts do not
// leave lanes idle until the job's queue is empty.  When the job is exhausted
// and every lane of the wavefront has finished, the wavefront moves to the
// next job.
//
// Per lane the driver keeps a mode -- DECIDE (next step is a leap decision,
// P1_P2.py:96-294), SSA (inside a P3 burst, P3.py:71-151, or pure SSA) or
// DONE.  A pass of its loop decides for the lanes in DECIDE (Engine::decide),
// then takes SSA steps for those in a burst: 1 + ssa_slice, and more the more
// lanes are in a burst than deciding.  A wavefront lasts as long as its
// slowest simulation, and a burst taken one step per pass would add 100
// passes to that simulation's path.
//
// SSA steps that cross no sample time and meet no rare case -- nearly all --
// run in ssa_run: four random blocks at a time, then four steps whose results
// are committed by selects, no branch in between.  The step's chain of
// dependent operations is what bounds it (a dependent operation takes 9
// cycles, a branch on a lane mask 50): Schloegl pure SSA, 100,003
// simulations, mixed 80 -> 40 ms.  Other steps end the run and go through
// Engine::ssa_step, the same arithmetic in general form.
//
// A launch with fewer than 64 simulations per wavefront, and the last
// simulations of a wavefront (LaneForm), replicate each over a group of
// lanes that share its draws.
// Every simulation executes exactly the reference's sequence
// (decision, burst of ssa_burst SSA steps, decision, ...); only the
// interleaving of different simulations within a wavefront changes.
#pragma once
#include "pst_device.hpp"
#include "pst_args.hpp"

namespace pst {

enum Mode { MODE_DECIDE = 0, MODE_SSA = 1, MODE_DONE = 2, MODE_AWAY = 3 /* paired driver: with the burst lane */ };

struct Counters {
  unsigned long long events;
  unsigned long long fevents;  // events of simulations that ended flagged
  unsigned int leaps, rejected, ssa, flagged;
  Work w;
};

// The workgroup's counters, in LDS: wavefronts add theirs (once per job, group
// size and at their end), lanes add the rarely counted events themselves, and
// the last wavefront to leave adds the sums to the launch's.
struct WgStats {
  unsigned long long v[ST_EXACT + 1];
  uint32_t waves;  // still running
};
__device__ __forceinline__ WgStats& wg_stats() {
  __shared__ WgStats s;
  return s;
}
__device__ __forceinline__ void init_stats() {  // every wavefront of the workgroup, then a barrier
  if (threadIdx.x <= ST_EXACT) wg_stats().v[threadIdx.x] = 0ull;
  if (threadIdx.x == 0) wg_stats().waves = blockDim.x / 64u;
}
__device__ __forceinline__ void add_stat(StatIdx i, unsigned long long n) {
  __hip_atomic_fetch_add(&wg_stats().v[i], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0ull; }

// x[idx] for a run-time idx in [0, NP), as an OR of masked elements: a select
// chain is folded back into an indexed load by the compiler, which then moves
// the per-lane array out of registers (into LDS or scratch).
template <int NP>
__device__ __forceinline__ int32_t pick_i(const int32_t (&x)[NP], int idx) {
  int32_t r = 0;
#pragma unroll
  for (int i = 0; i < NP; ++i) r |= x[i] & -(int32_t)(idx == i);
  return r;
}

template <int NP>
__device__ __forceinline__ float pick_f(const float (&x)[NP], int idx) {
  int32_t r = 0;
#pragma unroll
  for (int i = 0; i < NP; ++i) r |= __builtin_bit_cast(int32_t, x[i]) & -(int32_t)(idx == i);
  return __builtin_bit_cast(float, r);
}

// Lane groups: the 64 lanes of a wavefront hold 64 / G simulations, each
// replicated over G adjacent lanes that run in lock-step on the same
// registers; lane r of the group computes what can be split (the random blocks
// of the next SSA steps, the Poisson draws of reactions r, r + G, ...) and the
// results are exchanged.  Forms of a kernel:
//   ONE       G = 1
//   GROUPED   G > 1, fixed per job: launches with fewer than 64 simulations per
//             wavefront (lanes_for in pst_capi.hip)
//   WIDENING  G = 1 while there are simulations for every lane; grows once the
//             queue is empty and most lanes of a wavefront are done (regroup)
enum LaneForm { ONE = 0, GROUPED = 1, WIDENING = 2 };
template <int FORM>
struct LaneGroup {
  int G, r, base;  // size, position in the group, the group's first lane
  __device__ __forceinline__ void set(int lane, int sims_per_wave) {
    // (in one scalar register where branches depend on it)
    G = FORM == ONE ? 1 : 64 / (FORM == WIDENING ? __builtin_amdgcn_readfirstlane(sims_per_wave) : sims_per_wave);
    r = FORM == ONE ? 0 : lane & (G - 1);
    base = FORM == ONE ? lane : lane & ~(G - 1);
  }
  __device__ __forceinline__ bool grouped() const { return FORM == GROUPED || (FORM == WIDENING && G > 1); }
  __device__ __forceinline__ bool lead() const { return FORM == ONE || r == 0; }
  __device__ __forceinline__ bool mine(int j) const { return FORM == ONE || (j & (G - 1)) == r; }
  // p in any lane / in every lane of the group
  __device__ __forceinline__ unsigned long long mask() const { return (G == 64 ? ~0ull : (1ull << G) - 1ull) << base; }
  __device__ __forceinline__ bool any(bool p) const {
    return FORM == ONE ? p : (__builtin_amdgcn_ballot_w64(p) & mask()) != 0ull;
  }
  __device__ __forceinline__ bool all(bool p) const {
    return FORM == ONE ? p : (~__builtin_amdgcn_ballot_w64(p) & mask()) == 0ull;
  }
  // reaction j's value, from the lane that owns it
  __device__ __forceinline__ int32_t owners(int32_t v, int j) const {
    return __builtin_amdgcn_ds_bpermute((base + (j & (G - 1))) * 4, v);
  }
};

// ---------------------------------------------------------------------------
// Trajectory output.  JobParams::layout selects
//   LAYOUT_ROWS    O[q][f][o_stride], the reference's [kappa][ita][U]
//                  (cuTauLeaping.py:126): one 4-byte store per sample.  Lanes
//                  cross sample times at different moments, so every store
//                  dirties a 32-byte sector of its own.
//   LAYOUT_BLOCKS  O[q][f / 8][o_stride][f % 8] (ceil(ita / 8) blocks per
//                  species): the eight consecutive samples of one
//                  simulation fill one 32-byte sector.  A lane gathers its
//                  simulation's samples of the first Ref::kOutLds recorded
//                  species in LDS and writes each block with two 16-byte
//                  stores once its last sample is known, so no sector is
//                  written twice (further species are stored sample by
//                  sample).  The LDS slot is per simulation lane of the
//                  workgroup: the decide and burst lanes of a pair
//                  (run_driver_paired) share it, so a simulation's
//                  partial block travels with it.
// The last block is padded with zeros.
// ---------------------------------------------------------------------------
constexpr int LAYOUT_ROWS = 0, LAYOUT_BLOCKS = 1;
constexpr int OUT_BLOCK = 8;
typedef int32_t I4 __attribute__((ext_vector_type(4)));  // one 16-byte store

template <int KB>
struct SampleOut {
  static constexpr int KS = KB > 0 ? KB : 1;
  static __device__ __forceinline__ int32_t* lds() {
    __shared__ int32_t buf[KS * OUT_BLOCK * 256];
    return buf;
  }
  static __device__ __forceinline__ int slot() { return (int)(((threadIdx.x >> 6) & 3u) * 64u + (threadIdx.x & 63u)); }
  template <class P>
  static __device__ __forceinline__ int64_t block_row(const P& p, int q, int f) {
    return ((int64_t)q * ((p.ita + OUT_BLOCK - 1) / OUT_BLOCK) + (f / OUT_BLOCK)) * p.o_stride * OUT_BLOCK;
  }
  // the simulation's base pointer: O + sim (rows) or O + 8 sim (blocks)
  template <class P>
  static __device__ __forceinline__ int32_t* base(const P& p, int64_t sim) {
    return p.O + (p.layout == LAYOUT_BLOCKS ? sim * OUT_BLOCK : sim);
  }
  // sample f of recorded species q
  template <class P>
  static __device__ __forceinline__ void put(const P& p, int32_t* ob, int q, int f, int32_t v) {
    if (p.layout != LAYOUT_BLOCKS) {
      glb(ob)[((int64_t)q * p.ita + f) * p.o_stride] = v;
    } else if (q < KB) {
      lds()[(q * OUT_BLOCK + (f & (OUT_BLOCK - 1))) * 256 + slot()] = v;
    } else {
      glb(ob)[block_row(p, q, f) + (f & (OUT_BLOCK - 1))] = v;
    }
  }
  // after sample f of every recorded species: write the gathered blocks
  // that sample f completes (the block's last sample, or the run's)
  template <class P>
  static __device__ __forceinline__ void row_done(const P& p, int32_t* ob, int kappa, int f) {
    if (p.layout != LAYOUT_BLOCKS) return;
    const int last = f & (OUT_BLOCK - 1);
    if (last != OUT_BLOCK - 1 && f != p.ita - 1) return;
#pragma unroll
    for (int q = 0; q < KB; ++q) {
      if (q < kappa) {
        int32_t w[OUT_BLOCK];
#pragma unroll
        for (int j = 0; j < OUT_BLOCK; ++j) {
          const int32_t v = lds()[(q * OUT_BLOCK + j) * 256 + slot()];
          w[j] = (j <= last) ? v : 0;
        }
        gptr<I4> dst = (gptr<I4>)glb(ob + block_row(p, q, f));
        dst[0] = I4{w[0], w[1], w[2], w[3]};
        dst[1] = I4{w[4], w[5], w[6], w[7]};
      }
    }
    // species stored sample by sample: zero the padding of the last block
    if (f == p.ita - 1)
      for (int q = KB; q < kappa; ++q)
        for (int j = last + 1; j < OUT_BLOCK; ++j) glb(ob)[block_row(p, q, f) + j] = 0;
  }
};

// ---------------------------------------------------------------------------
// Sample ranges (pst_plan_execute_range, graph-captured chunks).  A launch
// with f_end < ita stops each simulation once it has recorded sample
// f_end - 1 and saves its state to JobParams::state, word-major
// ([word][n_sims]): the engine registers, the mode, the simulation's events
// so far and, for the blocked layout, its gathered samples of the block in
// progress (the step that records sample f_end - 1 may record later samples
// of the same block too); a launch with resume = 1 takes every simulation up
// from there.  A simulation that ends saves MODE_DONE, so later ranges skip it.
// Stopping between two steps and going on from the saved registers changes
// nothing in a simulation's step sequence, so a run split into ranges gives
// the same bits as one launch.  The trajectory base pointer is recomputed on
// resume from the launch's own descriptor.  f_end = INT_MAX,
// resume = 0: one launch runs every simulation to its end.
// ---------------------------------------------------------------------------
// A value the optimizer may not reason about: the word offsets i * n of the
// saved-state records stay inside save/load instead of being hoisted out of
// the simulation loop as ~40 live 64-bit offsets (+68 VGPRs in the pure-SSA
// Schlogl kernel).
__device__ __forceinline__ int32_t opaque_i32(int32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

template <class Engine>
struct StateIO {
  using Out = typename Engine::Out;
  static constexpr int EW = (int)(sizeof(Engine) / 4);
  static constexpr int BW = Out::KS * OUT_BLOCK;  // the lane's LDS sample block words
  static constexpr int WORDS = EW + 3 + BW;
  static_assert(sizeof(Engine) % 4 == 0, "engine state is not whole words");
  template <class P>
  static __device__ __forceinline__ bool fits(const P& p) {
    return p.state != nullptr && p.state_words >= WORDS;
  }
  template <class P>
  static __device__ __forceinline__ void save(const P& p, int64_t sim, const Engine& eng, int mode,
                                              unsigned long long ev) {
    gptr<uint32_t> st = glb(p.state);
    const int64_t n = opaque_i32(p.n_sims);
    uint32_t w[EW];
    __builtin_memcpy(w, &eng, sizeof(Engine));
#pragma unroll
    for (int i = 0; i < EW; ++i) st[(int64_t)i * n + sim] = w[i];
    st[(int64_t)EW * n + sim] = (uint32_t)mode;
    st[(int64_t)(EW + 1) * n + sim] = (uint32_t)ev;
    st[(int64_t)(EW + 2) * n + sim] = (uint32_t)(ev >> 32);
    if (p.layout == LAYOUT_BLOCKS && mode != MODE_DONE) {
#pragma unroll
      for (int i = 0; i < BW; ++i) st[(int64_t)(EW + 3 + i) * n + sim] = (uint32_t)Out::lds()[i * 256 + Out::slot()];
    }
  }
  template <class P>
  static __device__ __forceinline__ int load(const P& p, int64_t sim, Engine& eng, unsigned long long& ev) {
    gptr<uint32_t> st = glb(p.state);
    const int64_t n = opaque_i32(p.n_sims);
    uint32_t w[EW];
#pragma unroll
    for (int i = 0; i < EW; ++i) w[i] = st[(int64_t)i * n + sim];
    __builtin_memcpy(&eng, w, sizeof(Engine));
    ev = ((unsigned long long)st[(int64_t)(EW + 2) * n + sim] << 32) | st[(int64_t)(EW + 1) * n + sim];
    const int mode = (int)st[(int64_t)EW * n + sim];
    if (p.layout == LAYOUT_BLOCKS && mode != MODE_DONE) {
#pragma unroll
      for (int i = 0; i < BW; ++i) Out::lds()[i * 256 + Out::slot()] = (int32_t)st[(int64_t)(EW + 3 + i) * n + sim];
    }
    return mode;
  }
};

// Engine interface (see EngineF64 / EngineF32):
//   int  start(job, sim)            -> initial mode, state loaded
//   int  decide(job, cnt, on, group), int ssa_step(job, cnt, propensities) ->
//     next mode (DONE may set flag)
//   Draw1 ssa_draw(key, c), bool ssa_try(job, draw, tstop, sel, t1): one
//     ordinary SSA step (ssa_run)
//   int  flag
template <class Engine, class Ref>
__device__ __forceinline__ void finish_sim(const Ref& jr, const Engine& eng, int64_t sim, const Counters& cnt,
                                           unsigned long long ev_start, bool lead) {
  int32_t* fl = jr.cold().flags;
  if (fl) glb(fl)[sim] = eng.flag;
  if (eng.flag != 0 && lead) {
    add_stat(ST_FLAGGED, 1ull);
    add_stat(ST_FEVENTS, cnt.events - ev_start);
  }
}

// After a step: record an ended simulation, or stop one that has recorded
// the range's last sample.  Returns the lane's mode.
template <class Engine, class Ref, int FORM>
__device__ __forceinline__ int settle(const Ref& jr, const Engine& eng, int64_t sim, const Counters& cnt,
                                      unsigned long long ev_start, int mode, int f_stop, const LaneGroup<FORM>& g) {
  using SIO = StateIO<Engine>;
  if (mode == MODE_DONE) {
    finish_sim(jr, eng, sim, cnt, ev_start, g.lead());
    if (SIO::fits(jr.cold())) SIO::save(jr.cold(), sim, eng, MODE_DONE, cnt.events - ev_start);
    return MODE_DONE;
  }
  if (eng.F >= f_stop) {
    if (SIO::fits(jr.cold())) {
      SIO::save(jr.cold(), sim, eng, mode, cnt.events - ev_start);
      return MODE_DONE;
    }
  }
  return mode;
}

// A simulation taken from the queue: started, or resumed from its saved
// state.  Returns its mode (MODE_DONE: nothing left to do in this range).
template <class Engine, class Ref>
__device__ __forceinline__ int begin_sim(const Ref& jr, Engine& eng, int64_t sim, Counters& cnt,
                                         unsigned long long& ev_start, bool resume, int f_stop) {
  using SIO = StateIO<Engine>;
  if (resume && SIO::fits(jr.cold())) {
    unsigned long long ev;
    const int mode = SIO::load(jr.cold(), sim, eng, ev);
    ev_start = cnt.events - ev;
    eng.Ob = Engine::Out::base(jr.cold(), sim);
    if (mode == MODE_DONE || eng.F >= f_stop) return MODE_DONE;
    // Without tau-leaping a simulation is only ever in an SSA step (the
    // engines' start and step never return DECIDE then).  Saying so here
    // keeps the mode a compile-time fact in network kernels, whose method is
    // a constant, so their leap code is dropped (the pure-SSA Schlogl
    // kernel shrinks to about a quarter of its machine code).
    return jr.p().method != 0 ? (int)MODE_SSA : mode;
  }
  ev_start = cnt.events;
  return eng.start(jr, sim);
}

template <class Ref>
__device__ __forceinline__ int range_stop(const Ref& jr, int f_end) {
  return f_end < jr.cold().ita ? f_end : jr.cold().ita;
}

// time of the last sample of the range
template <class Ref>
__device__ __forceinline__ double stop_time(const Ref& jr, int f_stop) {
  return (double)glb(jr.cold().I)[f_stop > 0 ? f_stop - 1 : 0];
}

// value of `v` in the lane with byte address `addr` (4 * lane)
__device__ __forceinline__ float lane_get(float v, int addr) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(addr, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_get(double v, int addr) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)(b >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Ordinary SSA steps (P3.py:73-149, gillespie.py:70-149) of the lanes with
// `on`, up to `cap` each, in batches of four steps without a branch.  A
// step is computed from the state and committed by selects only if nothing
// out of the ordinary happens in it.  A lane leaves the loop before a step
// that ends the simulation or its range (absorbing state, last sample,
// count limit, stuck clock, step budget, t_max): `general` is then set and
// Engine::ssa_step takes that step.  A lane whose step crosses a sample time stops
// for the rest of its batch and records the state before that step.
// The batch's Philox blocks and logarithms do not depend on the state; they
// are independent chains beside the steps'.  On gfx950 a dependent vector
// instruction issues every ~9 cycles, a branch on a lane mask costs 50-60: the
// general step, with about ten of them, takes 1,300 cycles for a single lane.
// All lanes of the wavefront call this together.

template <class Engine, class Ref, int FORM>
__device__ __forceinline__ int ssa_run(Ref& jr, Engine& eng, Counters& cnt, int mode, bool on, int cap, double tstop,
                                       bool& general, const LaneGroup<FORM>& g) {
  using Out = typename Engine::Out;
  constexpr int kBatch = 4;
  const auto& P = jr.p();
  int lim = cap;
  if (P.method == 0) lim = eng.burst < lim ? eng.burst : lim;
  if (P.max_steps != 0u) {
    const uint32_t left = eng.nsteps < P.max_steps ? P.max_steps - eng.nsteps : 0u;
    lim = left < (uint32_t)lim ? (int)left : lim;
  }
  if (P.method == 2) tstop = P.t_max < tstop ? P.t_max : tstop;
  // lim steps, each changing a count by 127 at most, cannot reach the count limit
  bool go = on & (lim > 0) & (eng.t < tstop);
  const int safe = COUNT_LIMIT - 127 * lim;
#pragma unroll
  for (int i = 0; i < Engine::NP; ++i) go = go & (eng.x[i] < safe);
  bool stop = on & !go;  // the next step is not for this loop
  const Key uk = eng.key.scalar_seed(P.seed);  // a lane without a simulation may hold any key
  int n = 0;
  while (wave_any(go)) {
    typename Engine::Draw1 d[kBatch];
    // lane r of the group draws for steps r, r + G, ... of the batch
    d[0] = Engine::ssa_draw(uk, eng.bc + (uint64_t)(uint32_t)(n + (FORM == ONE ? 0 : g.r & (kBatch - 1))));
    if (FORM != ONE && g.G >= kBatch) {
#pragma unroll
      for (int s = kBatch - 1; s >= 0; --s) d[s] = Engine::from_lane(d[0], (g.base + s) * 4);
    } else if (g.grouped()) {
      d[2] = Engine::ssa_draw(uk, eng.bc + (uint64_t)(uint32_t)(n + g.r + 2));
      d[3] = Engine::from_lane(d[2], (g.base + 1) * 4);
      d[2] = Engine::from_lane(d[2], g.base * 4);
      d[1] = Engine::from_lane(d[0], (g.base + 1) * 4);
      d[0] = Engine::from_lane(d[0], g.base * 4);
    } else {
#pragma unroll
      for (int s = 1; s < kBatch; ++s) d[s] = Engine::ssa_draw(uk, eng.bc + (uint64_t)(uint32_t)(n + s));
    }
    bool act = go, crossed = false;
    int csel = 0;
#pragma unroll
    for (int s = 0; s < kBatch; ++s) {
      int sel;
      double t1;
      const bool ok = eng.ssa_try(jr, d[s], tstop, sel, t1);
      const bool take = act & (n < lim);
      const bool done = take & ok;
      stop = stop | (take & !ok);
      const bool cross = done & (t1 >= eng.tnext);
      crossed = crossed | cross;
      csel = cross ? sel : csel;
      int32_t dx[Engine::NP];
      jr.row(sel, dx);
#pragma unroll
      for (int i = 0; i < Engine::NP; ++i) eng.x[i] += done ? dx[i] : 0;
      eng.t = done ? t1 : eng.t;
      n += done ? 1 : 0;
      act = done & !cross;
    }
    if (wave_any(crossed)) {
      if (crossed) {
        int32_t before[Engine::NP];  // the state before the crossing step
        jr.row(csel, before);
#pragma unroll
        for (int i = 0; i < Engine::NP; ++i) before[i] = eng.x[i] - before[i];
        do {
          jr.for_recorded([&](int q) { Out::put(P, eng.Ob, q, eng.F, pick_i<Engine::NP>(before, jr.Ev(q))); });
          Out::row_done(P, eng.Ob, P.kappa, eng.F);
          cnt.w.samples += 1;
          eng.F = eng.F + 1;
          eng.tnext = (double)glb(P.I)[eng.F];  // t < tstop: F stays below the range's last sample
        } while (eng.t >= eng.tnext);
      }
    }
    go = go & !stop & (n < lim);
  }
  eng.bc += (uint64_t)(uint32_t)n;
  eng.nsteps += (uint32_t)n;
  cnt.w.uniforms += 2u * (unsigned int)n;
  cnt.ssa += (unsigned int)n;
  cnt.events += (unsigned long long)n;
  general = stop;
  if (P.method == 0) {
    eng.burst -= n;
    if (on && eng.burst <= 0) mode = MODE_DECIDE;
  }
  return mode;
}

// Up to `cap` SSA steps of the lanes with `on`: ordinary ones in ssa_run, and
// the one it leaves over, if any, through ssa_step.
template <class Engine, class Ref, int FORM>
__device__ __forceinline__ int ssa_slice(Ref& jr, Engine& eng, Counters& cnt, int mode, bool on, int cap,
                                         double t_stop, const LaneGroup<FORM>& g) {
  bool general;
  mode = ssa_run(jr, eng, cnt, mode, on, cap, t_stop, general, g);
  if (wave_any(general)) {
    typename Engine::Real a[Engine::MP];
    jr.template props<typename Engine::Real>(eng.x, eng.k, a);  // (with every lane on: JobRef)
    if (general) mode = eng.ssa_step(jr, cnt, a);
  }
  return mode;
}

// Adds a wavefront's counters and clears them.  Lanes of a group count the
// same events: only the first lane's count, except for the Poisson draws,
// which each lane counts for the reactions it drew.
template <int FORM>
__device__ __forceinline__ void add_stats(Counters& cnt, const LaneGroup<FORM>& g) {
  const unsigned long long m = g.lead() ? ~0ull : 0ull;
  // (32-bit per-lane counters: a lane's share of one launch stays far below 2^32)
  add_stat(ST_EVENTS, cnt.events & m);
  add_stat(ST_LEAPS, cnt.leaps & m);
  add_stat(ST_REJECTED, cnt.rejected & m);
  add_stat(ST_SSA, cnt.ssa & m);
  add_stat(ST_UNIFORMS, (cnt.w.uniforms & m) + cnt.w.draws);
  add_stat(ST_PTRS, cnt.w.ptrs);
  add_stat(ST_INV, cnt.w.inv);
  add_stat(ST_DECISIONS, cnt.w.decisions & m);
  add_stat(ST_SAMPLES, cnt.w.samples & m);
  add_stat(ST_ASYM, cnt.w.asym);
  cnt = {};
}
__device__ __forceinline__ void leave_stats(int lane, unsigned long long* __restrict__ stats) {
  uint32_t left = 0;
  wave_lds_sync();  // every lane's share is in
  if (lane == 0)
    left = __hip_atomic_fetch_add(&wg_stats().waves, 0xffffffffu, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
  left = __builtin_amdgcn_readfirstlane(left);
  wave_lds_sync();
  if (left == 1u && lane <= ST_EXACT) atomicAdd(&stats[lane], wg_stats().v[lane]);
}

// A simulation in transit: the engine state, its id, its events so far
// (for the flagged-events counter), the job index and the next mode.
template <class Engine, int STRIDE>
struct SlotIO {
  static constexpr int EW = (int)(sizeof(Engine) / 4);
  static constexpr int WORDS = EW + 6;
  static_assert(sizeof(Engine) % 4 == 0, "engine state is not whole words");
  // word-major [word][slot]: consecutive lanes hit consecutive banks
  static __device__ __forceinline__ void put(uint32_t* data, int slot, const Engine& eng, int64_t sim,
                                             unsigned long long ev, int job, int mode) {
    uint32_t w[EW];
    __builtin_memcpy(w, &eng, sizeof(Engine));
#pragma unroll
    for (int i = 0; i < EW; ++i) data[i * STRIDE + slot] = w[i];
    data[(EW + 0) * STRIDE + slot] = (uint32_t)sim;
    data[(EW + 1) * STRIDE + slot] = (uint32_t)((uint64_t)sim >> 32);
    data[(EW + 2) * STRIDE + slot] = (uint32_t)ev;
    data[(EW + 3) * STRIDE + slot] = (uint32_t)(ev >> 32);
    data[(EW + 4) * STRIDE + slot] = (uint32_t)job;
    data[(EW + 5) * STRIDE + slot] = (uint32_t)mode;
  }
  static __device__ __forceinline__ void get(const uint32_t* data, int slot, Engine& eng, int64_t& sim,
                                             unsigned long long& ev, int& mode) {
    uint32_t w[EW];
#pragma unroll
    for (int i = 0; i < EW; ++i) w[i] = data[i * STRIDE + slot];
    __builtin_memcpy(&eng, w, sizeof(Engine));
    sim = (int64_t)(((uint64_t)data[(EW + 1) * STRIDE + slot] << 32) | data[(EW + 0) * STRIDE + slot]);
    ev = ((unsigned long long)data[(EW + 3) * STRIDE + slot] << 32) | data[(EW + 2) * STRIDE + slot];
    mode = (int)data[(EW + 5) * STRIDE + slot];
  }
  static __device__ __forceinline__ int job(const uint32_t* data, int slot) {
    return (int)data[(EW + 4) * STRIDE + slot];
  }
};

// Once a job's queue is empty, the last simulations of a wavefront take more
// lanes each: with at most 16 of them left they are moved to groups of four
// or more lanes (up to `cap`), so a leap's draws and the random blocks of SSA
// steps no longer run one after the other for the slowest simulations, which
// end the launch.  The states go through LDS (`data`, slots first ..
// first + 15, word-major); the counters so far are added to the launch's,
// because which lanes count changes.
__device__ __forceinline__ int group_cap(int n_reactions) {
  int c = 4;  // the SSA batch
  while (c < n_reactions && c < 32) c *= 2;
  return c;
}
template <int FORM>
__device__ __forceinline__ int wider_group(const LaneGroup<FORM>& g, unsigned long long leads, int cap) {
  const int n = __builtin_popcountll(leads);
  int G = g.G < 4 ? 4 : 2 * g.G;
  if (n == 0 || G > cap || n * G > 64) return 0;
  while (2 * G <= cap && n * 2 * G <= 64) G *= 2;
  return G;
}

template <class Engine, int STRIDE, int FORM>
__device__ __forceinline__ void regroup(uint32_t* data, int first, int G, LaneGroup<FORM>& g, int lane, Engine& eng,
                                        int64_t& sim, unsigned long long& ev_start, Counters& cnt, int& mode,
                                        bool blocks) {
  using IO = SlotIO<Engine, STRIDE>;
  using Out = typename Engine::Out;
  constexpr int BW = Out::KS * OUT_BLOCK;
  const bool moves = g.lead() & (mode != MODE_DONE);
  const unsigned long long leads = __builtin_amdgcn_ballot_w64(moves);
  if (moves) {
    const int to = first + __builtin_popcountll(leads & ((1ull << lane) - 1ull));
    IO::put(data, to, eng, sim, cnt.events - ev_start, lane, mode);
  }
  wave_lds_sync();  // records and sample blocks are read by other lanes
  add_stats(cnt, g);
  g.set(lane, 64 / G);
  const int from = lane / G;
  const bool takes = from < __builtin_popcountll(leads);
  mode = MODE_DONE;
  int32_t w[BW];
  if (takes) {
    unsigned long long ev;
    IO::get(data, first + from, eng, sim, ev, mode);
    ev_start = 0ull - ev;
    if (blocks) {  // the samples of the block in progress
      const int32_t* old = Out::lds() + (Out::slot() & ~63) + IO::job(data, first + from);
#pragma unroll
      for (int i = 0; i < BW; ++i) w[i] = old[i * 256];
    }
  }
  wave_lds_sync();  // ... before the blocks and slots are written again
  if (takes && blocks) {
#pragma unroll
    for (int i = 0; i < BW; ++i) Out::lds()[i * 256 + Out::slot()] = w[i];
  }
}

template <class Engine, class Ref, int FORM>
__device__ __forceinline__ void run_driver(const typename Ref::Dev* __restrict__ jobs, int n_jobs,
                                           unsigned int* __restrict__ queue, unsigned long long* __restrict__ stats,
                                           int f_end, int resume) {
  const int lane = (int)(threadIdx.x & 63u);
  init_stats();
  __syncthreads();  // the only barrier: every lane of the workgroup reaches it
  Counters cnt = {};
  Engine eng;
  int mode = MODE_DONE;
  int64_t sim = -1;
  unsigned long long ev_start = 0;  // cnt.events when this lane's simulation began
  int job = 0;
  bool exhausted = false;

  Ref jr;
  jr.load(jobs);
  int f_stop = range_stop(jr, f_end);
  double t_stop = stop_time(jr, f_stop);
  LaneGroup<FORM> g;
  g.set(lane, jr.cold().lanes);
  constexpr int kSlots = 64;  // sixteen per wavefront
  __shared__ uint32_t s_move[SlotIO<Engine, kSlots>::WORDS * kSlots];

  for (;;) {
    // ---- refill lanes whose simulation ended from the job's queue (the lanes
    // of a group are in lock-step: they end together and take one simulation) ----
    const bool want = (mode == MODE_DONE) && !exhausted && (FORM != ONE || lane < jr.cold().lanes);
    const unsigned long long wmask = __builtin_amdgcn_ballot_w64(want & g.lead());
    if (wmask != 0ull) {
      const int n = __builtin_popcountll(wmask);
      const int leader = __builtin_ctzll(wmask);
      unsigned int base = 0;
      if (lane == leader) base = atomicAdd(&queue[job], (unsigned int)n);
      base = __shfl(base, leader, 64);
      const int n_sims = jr.cold().n_sims;
      if ((int64_t)base + n >= (int64_t)n_sims) exhausted = true;
      if (want) {
        const int rank = __builtin_popcountll(wmask & ((1ull << g.base) - 1ull));
        const int64_t s = (int64_t)base + rank;
        if (s < n_sims) {
          sim = s;
          mode = begin_sim(jr, eng, s, cnt, ev_start, resume != 0, f_stop);
        }
      }
      // in a resumed range a lane may have taken a simulation that had ended: no
      // reason to wait for the others, or to leave the job
      if (resume != 0 && !exhausted && wave_any(want & (mode == MODE_DONE))) continue;
    }
    if (FORM == WIDENING && exhausted) {
      const int G = wider_group(g, __builtin_amdgcn_ballot_w64((mode != MODE_DONE) & g.lead()), group_cap(jr.n_reactions()));
      if (G != 0)
        regroup<Engine, kSlots>(s_move, (int)(threadIdx.x >> 6) * 16, G, g, lane, eng, sim, ev_start, cnt, mode,
                                jr.p().layout == LAYOUT_BLOCKS);
    }
    if (!wave_any(mode != MODE_DONE)) {
      // this wavefront is idle and its job has no work left: next job
      job += 1;
      if (job >= n_jobs) break;
      add_stats(cnt, g);
      jr.load(jobs + job);
      f_stop = range_stop(jr, f_end);
      t_stop = stop_time(jr, f_stop);
      g.set(lane, jr.cold().lanes);
      exhausted = false;
      continue;
    }

    // ---- passes until a simulation ends.  (A loop of its own: in the one
    // above, the engine's registers were copied on its several ways round,
    // 40 moves and a wait for the next sample time per pass.  One call of each
    // function: the code of a step and of the saved-state record exists once.)
    const bool ran = mode != MODE_DONE;
    do {
      // (only tau-leaping decides: a compile-time fact in network kernels)
      if (jr.method() == 0 && wave_any(mode == MODE_DECIDE)) {
        const int next = eng.decide(jr, cnt, mode == MODE_DECIDE, g);
        mode = mode == MODE_DECIDE ? next : mode;
      }
      // SSA steps of the lanes inside a burst: more of them the more lanes are
      // in one than deciding (a burst of 100 steps taken 8 at a time waits
      // through 13 decisions of the others); most if every live lane is inside
      // a burst.  Where no lane ever decides, 512 at the default slice: only a
      // lane whose simulation has ended waits for the others' (64 -> 512:
      // birth-death, 1024 simulations, mixed 0.374 -> 0.360 ms, FP64 0.617 ->
      // 0.604; Schloegl, 200,000, mixed 13.7 -> 13.1, table-driven 33.1 -> 32.1)
      const bool burst = mode == MODE_SSA && eng.F < f_stop;
      const unsigned long long ssa = __builtin_amdgcn_ballot_w64(burst);
      if (ssa != 0ull) {
        const int n_ssa = __builtin_popcountll(ssa);
        const int n_dec = __builtin_popcountll(__builtin_amdgcn_ballot_w64(mode == MODE_DECIDE));
        const int times = jr.method() != 0 ? 64 : n_ssa >= 8 * n_dec ? 8 : n_ssa >= 4 * n_dec ? 4 : n_ssa >= 2 * n_dec ? 2 : 1;
        mode = ssa_slice(jr, eng, cnt, mode, burst, times * (jr.p().ssa_slice + 1), t_stop, g);
      }
    } while (!wave_any(ran & ((mode == MODE_DONE) | (eng.F >= f_stop))));
    if (ran) mode = settle(jr, eng, sim, cnt, ev_start, mode, f_stop, g);
  }

  add_stats(cnt, g);
  leave_stats(lane, stats);
}

// ---------------------------------------------------------------------------
// Paired driver: a workgroup of 512 lanes is four decide wavefronts (0-3) and
// four burst wavefronts (4-7), two wavefronts per SIMD.  A decide wavefront
// runs its simulations like run_driver but takes no SSA-only steps: when a
// leap decision switches a simulation into an SSA fallback burst
// (P1_P2.py:157-173, then P3.py:71-151), the lane writes the simulation's
// state to an LDS slot and lane l of burst wavefront w + 4 takes it, runs the
// burst's remaining SSA steps back to back and hands the state back.  So the
// leap passes of a decide wavefront no longer wait for other lanes' SSA steps,
// a burst no longer waits for leap passes, and each SIMD overlaps the two
// instruction streams (one wavefront per SIMD leaves half its issue slots to
// latency).  Every simulation still executes exactly the reference's
// sequence; only where its steps run changes.
//
// Slot protocol (one slot per decide lane): FREE -> SENT (decide lane, after
// writing the state) -> BACK (burst lane, after writing the state back) ->
// FREE (decide lane, after reading it).  A decide lane with a SENT slot is
// AWAY and skips passes; a decide wavefront moves to its next job only when
// none of its lanes is away, so every simulation a burst wavefront holds
// belongs to its partner's current job.  A burst wavefront never waits for
// its partner except while it has nothing to run, and it leaves once the
// partner has finished every job (DONE flag), when no slot can be SENT.
// ---------------------------------------------------------------------------
enum { SLOT_FREE = 0u, SLOT_SENT = 1u, SLOT_BACK = 2u };
constexpr int PAIR_SLOTS = 256;  // decide lanes per workgroup
constexpr int BURST_SLICE = 8;   // SSA steps of a burst wavefront between two looks at its slots

__device__ __forceinline__ uint32_t lds_load_acquire(uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_store_release(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <class Engine, class Ref, int FORM>
__device__ __forceinline__ void run_driver_paired(const typename Ref::Dev* __restrict__ jobs, int n_jobs,
                                                  unsigned int* __restrict__ queue,
                                                  unsigned long long* __restrict__ stats, int f_end, int resume) {
  using IO = SlotIO<Engine, PAIR_SLOTS>;
  __shared__ uint32_t s_data[IO::WORDS * PAIR_SLOTS];
  __shared__ uint32_t s_state[PAIR_SLOTS];
  __shared__ uint32_t s_done[4];
  __shared__ uint32_t s_lanes[4];  // simulations per wavefront of the pair (64 / G)
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;  // wave-uniform
  const int pair = wave & 3;
  const int slot = pair * 64 + lane;
  if (tid < PAIR_SLOTS) s_state[tid] = SLOT_FREE;
  if (tid < 4) s_done[tid] = 0u;
  init_stats();
  __syncthreads();  // the only barrier: every lane of the workgroup reaches it

  Counters cnt = {};
  Engine eng;
  int64_t sim = -1;
  unsigned long long ev_start = 0;  // cnt.events when this lane's simulation began (here)
  Ref jr;
  LaneGroup<FORM> g;
  g.set(lane, 1);

  if (wave < 4) {
    // ---- decide wavefront ----
    int mode = MODE_DONE;
    int job = 0;
    bool exhausted = false;
    jr.load(jobs);
    int f_stop = range_stop(jr, f_end);
    g.set(lane, jr.cold().lanes);
    if (lane == 0) s_lanes[pair] = (uint32_t)(64 / g.G);
    wave_lds_sync();  // before any lane of this wavefront sends
    for (;;) {
      // a burst handed back (ended simulations were recorded by the burst
      // lane); the lanes of a group take it together
      if (g.all(mode == MODE_AWAY && lds_load_acquire(&s_state[slot]) == SLOT_BACK)) {
        unsigned long long ev;
        IO::get(s_data, slot, eng, sim, ev, mode);
        ev_start = cnt.events - ev;
        s_state[slot] = SLOT_FREE;
      }
      const bool want = (mode == MODE_DONE) && !exhausted && (FORM != ONE || lane < jr.cold().lanes);
      const unsigned long long wmask = __builtin_amdgcn_ballot_w64(want & g.lead());
      if (wmask != 0ull) {
        const int n = __builtin_popcountll(wmask);
        const int leader = __builtin_ctzll(wmask);
        unsigned int base = 0;
        if (lane == leader) base = atomicAdd(&queue[job], (unsigned int)n);
        base = __shfl(base, leader, 64);
        const int n_sims = jr.cold().n_sims;
        if ((int64_t)base + n >= (int64_t)n_sims) exhausted = true;
        if (want) {
          const int rank = __builtin_popcountll(wmask & ((1ull << g.base) - 1ull));
          const int64_t s = (int64_t)base + rank;
          if (s < n_sims) {
            sim = s;
            mode = begin_sim(jr, eng, s, cnt, ev_start, resume != 0, f_stop);
          }
        }
        if (resume != 0 && !exhausted && wave_any(want & (mode == MODE_DONE))) continue;  // as in run_driver
      }
      // regroup when no simulation is away (its slot belongs to its lane): bursts
      // that start meanwhile wait
      bool hold = false;
      if (FORM == WIDENING && exhausted) {
        const int G = wider_group(g, __builtin_amdgcn_ballot_w64((mode != MODE_DONE) & g.lead()), group_cap(jr.n_reactions()));
        hold = G != 0 && wave_any(mode == MODE_AWAY);
        if (G != 0 && !hold) {
          regroup<Engine, PAIR_SLOTS>(s_data, pair * 64, G, g, lane, eng, sim, ev_start, cnt, mode,
                                      jr.p().layout == LAYOUT_BLOCKS);
          if (lane == 0) s_lanes[pair] = (uint32_t)(64 / G);
          wave_lds_sync();
        }
      }
      if (!wave_any(mode != MODE_DONE)) {
        job += 1;
        if (job >= n_jobs) break;
        add_stats(cnt, g);
        jr.load(jobs + job);
        f_stop = range_stop(jr, f_end);
        g.set(lane, jr.cold().lanes);
        if (lane == 0) s_lanes[pair] = (uint32_t)(64 / g.G);
        wave_lds_sync();
        exhausted = false;
        continue;
      }
      const bool ran = (mode == MODE_DECIDE) | (mode == MODE_SSA);
      const bool on = mode == MODE_DECIDE && eng.F < f_stop;
      if (wave_any(on)) {
        const int next = eng.decide(jr, cnt, on, g);
        mode = on ? next : mode;
      } else if (hold || !wave_any(mode == MODE_SSA)) {
        __builtin_amdgcn_s_sleep(2);  // every live lane is away or held: wait for a burst to come back
      }
      if (wave_any(ran & ((mode == MODE_DONE) | (eng.F >= f_stop)))) {
        if (ran) mode = settle(jr, eng, sim, cnt, ev_start, mode, f_stop, g);
      }
      // a burst starts (or a forced-SSA simulation starts): hand it over
      if (mode == MODE_SSA && !hold) {
        IO::put(s_data, slot, eng, sim, cnt.events - ev_start, job, MODE_SSA);
        lds_store_release(&s_state[slot], SLOT_SENT);
        mode = MODE_AWAY;
      }
    }
    lds_store_release(&s_done[pair], 1u);
  } else {
    // ---- burst wavefront ----
    // (Both roles keep the default issue priority: raising the burst
    // wavefront's slowed the Lotka-Volterra workload from 39.9 to 42.3 ms.)
    bool busy = false;
    int bjob = -1;
    int f_stop = 0x7fffffff;
    double t_stop = 0.0;
    for (;;) {
      // (the slots of a group are filled by one store of the partner, but may
      // be read while it is under way)
      const bool sent = !busy && lds_load_acquire(&s_state[slot]) == SLOT_SENT;
      const unsigned long long smask = __builtin_amdgcn_ballot_w64(sent);
      if (smask != 0ull) {
        // all simulations the partner sends belong to its current job
        const int pj = __builtin_amdgcn_readlane(IO::job(s_data, slot), __builtin_ctzll(smask));
        if (pj != bjob) {
          jr.load(jobs + pj);
          bjob = pj;
          f_stop = range_stop(jr, f_end);
          t_stop = stop_time(jr, f_stop);
        }
        // ... and hold its present group size (it changes only while this
        // wavefront has nothing in hand)
        const int sims = (int)s_lanes[pair];
        if (64 / g.G != sims) {
          add_stats(cnt, g);
          g.set(lane, sims);
        }
      }
      const bool pick = g.all(sent);
      const unsigned long long pmask = __builtin_amdgcn_ballot_w64(pick);
      if (pmask != 0ull) {
        if (pick) {
          unsigned long long ev;
          int m;
          IO::get(s_data, slot, eng, sim, ev, m);
          ev_start = cnt.events - ev;
          busy = true;
        }
      }
      if (!wave_any(busy)) {
        if (lds_load_acquire(&s_done[pair]) != 0u) break;
        __builtin_amdgcn_s_sleep(4);
        continue;
      }
      int m = ssa_slice(jr, eng, cnt, (int)MODE_SSA, busy, BURST_SLICE, t_stop, g);
      if (busy) {
        if (m == MODE_DONE) m = settle(jr, eng, sim, cnt, ev_start, m, f_stop, g);
        // back to the decide lane at the burst's end, or at the range's
        // last sample (the decide lane saves it)
        if (m != MODE_SSA || eng.F >= f_stop) {
          IO::put(s_data, slot, eng, sim, cnt.events - ev_start, bjob, m);
          lds_store_release(&s_state[slot], SLOT_BACK);
          busy = false;
        }
      }
    }
  }

  add_stats(cnt, g);
  leave_stats(lane, stats);
}

}  // namespace pst
