// engine_resident.hpp -- many steps in one launch, for slabs few enough that
// every 64-cell tile has a wavefront of its own resident on the chip.
//
// A step of a small engine is not bound by its bytes: launch to launch takes
// 2.4 us on an MI355X, the tables and descriptors come through cold caches
// after every launch, and a tile's 1,750 or so dependent VALU instructions
// take some 4 us on a wavefront that has its SIMD to itself.  Here a tile's
// wavefront keeps the states and stencil weights in registers and runs the
// steps in a loop.  Only Vm crosses between tiles, through the same two boxes
// as in the step kernels, and only with the tiles that hold the 18
// neighbours of its cells:
//
//   each tile publishes how many steps it has done (flags[tile]); before the
//   stencil of step k a tile waits until every neighbouring tile has done k
//   steps.  Then their Vm of step k is in the box read, and none of them still
//   reads the box that this step writes (they read it in step k - 1).
//
// The reaction of a step needs the cell's own Vm only and runs before the
// wait, so the exchange of Vm between the tiles passes under it.
//
// Every tile is resident because the launch is cooperative and the host
// keeps the grid within the kernel's occupancy, so every wait ends.  All the
// same each wait is bounded (ResidentArgs::max_polls): past it the wavefront
// raises `failed`, which the host reports, and nobody waits any longer: a long
// wait looks for it, and so does every wavefront of the launches queued behind,
// before its first step.
//
// Vm and the flags are stored and loaded at agent scope (SC1), where the XCDs'
// caches agree, as relaxed atomics are; a tile's flag is stored after the
// wait for its Vm stores' completion, and a neighbour's Vm is loaded after
// its flag came back.  Agent-scope release and acquire fences in their place
// write back and invalidate a whole XCD's L2 for every wavefront: 22 us a
// step at 821 tiles against 10 without (before the other changes below).
// Everything else a tile touches is its own.
//
// All 18 neighbour loads are in flight at once (left to itself the compiler
// issued them one by one into the same registers: 8.9 against 6.7 us a step
// at 504 cells), and each flag has a cache line of its own (kFlagStride).
//
// Per step on one MI355X, step kernels against this: reference rounding
// 504 cells 10.1 and 6.7 us, 52,500 cells 12.2 and 7.0, 110,592 cells 14.5
// and 9.7, 193,536 cells 18.9 and 12.9; FMA 262,144 cells (4 wavefronts per
// SIMD) 24.5 and 15.1; mixed 52,500 cells 10.6 and 5.9, 262,144 cells 15.4
// and 10.0, 373,248 cells (6 per SIMD) 24.9 and 14.2; exact functions 262,144
// cells by step kernels 26.7, 193,536 cells by this 17.7.  What bounds it: up
// to 1,024 tiles the latency of one wavefront's chain (12,000 of 17,000 cycles
// in the reaction); with a tile to every place VALU issue, 0.6 to 0.7 of the
// SIMDs' cycles by the counters, the rest steps in which all of a SIMD's
// wavefronts wait for their neighbours.  Vm's crossing moves 24 bytes a
// cell-step, 0.4 TB/s at 262,144 cells.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "engine.hpp"
#include "tt06_model.hpp"

namespace cdh {

// Words from one tile's flag to the next: a line each.  With 32 flags to a
// line, the stores of 32 tiles and the polls of their neighbours all met
// there: at 2,940 tiles (mixed) a wait took 17,400 cycles of a step, with a
// line each 4,000.
constexpr int kFlagStride = 32;
// Polls between two looks at the bound and at `failed`: 10 us.  A look at every poll
// delays the next one (500 steps of 504 cells 1,504 us, this 1,461).
constexpr uint32_t kResidentPolls = 64;

struct ResidentArgs {
   // both by the tile's place in the list of live tiles
   uint32_t *flags;             // steps done, counted on from launch to launch, one flag
                                // to a cache line (kFlagStride)
   const uint32_t *links;       // 3 ranges {first, last + 1} of neighbouring tiles
   uint32_t base;               // every tile's flag at the launch
   int nsteps;
   double *box[2];              // box[k & 1] is read in step k of this launch
   uint32_t *failed;            // 1 once a wait has passed its bound; on the device
   uint32_t *failed_host;       // the same in host memory
   uint32_t max_polls;          // that bound
   int tile_ranges;             // the tiles' range records in EngineArgs::ranges (resident_range)
};

typedef const SlabDev CDH_CONSTANT ConstSlab;

struct ModelTables {
   ModelConst *K;
   ExactConst *E;
   CoefPtr coef;
};

// what a wavefront knows of its tile
struct ResidentTile {
   ConstSlab *S;
   int j, blk, sl, lane;        // its place in the list of live tiles, the tile, its slab
   uint32_t meta;
   bool live;
   uint32_t b8;                 // this lane's box offset in bytes
   uint32_t lc, rw;             // its place in the run of cells its states are in, the run's width
   int64_t run_cell;            // the run's first cell in the arena
   // false: nothing to do for the whole workgroup
   __device__ __forceinline__ bool find(const EngineArgs &a)
   {
      j = engine_tile_group(a);
      if (j >= a.ntile) return false;
      lane = threadIdx.x & (kBlk - 1);
      blk = __builtin_amdgcn_readfirstlane(a.tiles ? (int)a.tiles[j] : a.tile_base + j);
      sl = __builtin_amdgcn_readfirstlane((int)a.blk_slab[blk]);
      if (sl == kNoSlab) return false;
      S = (ConstSlab *)(a.slabs + sl);
      if (!S->active) return false;
      const int64_t i = (int64_t)blk * kBlk + lane;
      meta = a.meta[i];
      live = !(meta & kMetaPad);
      b8 = a.bi[i] * 8u;
      const int64_t k0 = (int64_t)(blk - S->first_blk) * kBlk;
      const int64_t r0 = k0 & ~(kRun - 1);
      rw = (uint32_t)run_width(k0, (int64_t)S->ntile * kBlk);
      run_cell = (int64_t)S->first_blk * kBlk + r0;
      lc = (uint32_t)(k0 - r0 + lane);
      return true;
   }
   // node k's Vm from the box behind R, past the caches that other XCDs'
   // stores do not reach
   __device__ __forceinline__ double neighbour(__amdgpu_buffer_rsrc_t R, int k) const
   {
      return box_load_agent(R, b8, S->soff[k]);
   }
   __device__ __forceinline__ const ParamSet *params(const EngineArgs &a) const
   {
      return a.params + S->param_base + (int)(meta & 0xFFu);
   }
   // The cell's number, made anew: the addresses that only a sensor event or
   // an out-of-range cell needs are then made there, not held over the loop.
   __device__ __forceinline__ uint32_t cell() const
   {
      uint32_t c = (uint32_t)blk * kBlk + lane;
      asm volatile("" : "+v"(c));
      return c;
   }
};

// The tables' addresses made anew in every step: otherwise their loads move
// out of the loop, hundreds of scalars that no wavefront can hold.
__device__ __forceinline__ void renew(ModelTables &T)
{
   asm volatile("" : "+s"(T.K), "+s"(T.E), "+s"(T.coef));
}

__device__ __forceinline__ bool resident_failed(const ResidentArgs &r)
{
   return __builtin_amdgcn_readfirstlane(
       __hip_atomic_load(r.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The look of a wait that has polled for a while; whether it is to end, for its
// own bound or for another wavefront's.  The bound counts polls and no time: a
// wavefront that is held off the chip, as all of a process's are while another
// process has its turn, does not poll, and whom it waits for is held off too.
__device__ __forceinline__ bool resident_give_up(const ResidentArgs &r, int lane, uint32_t polls)
{
   if (resident_failed(r)) return true;
   if (polls <= r.max_polls) return false;
   if (lane == 0) {
      __hip_atomic_store(r.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(r.failed_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
   }
   return true;
}

// Waits until every tile of the three ranges has done `target` - base steps.
__device__ __forceinline__ void resident_wait(const ResidentArgs &r, const uint32_t *lk, int lane,
                                              uint32_t target, bool &bail)
{
   const int n0 = (int)(lk[1] - lk[0]), n1 = (int)(lk[3] - lk[2]), n2 = (int)(lk[5] - lk[4]);
   const int n = n0 + n1 + n2;
   for (int q = lane; !bail && __ballot(q < n); q += kBlk) {
      const bool mine = q < n;
      const uint32_t t = !mine ? 0u
                         : q < n0 ? lk[0] + q
                         : q < n0 + n1 ? lk[2] + (q - n0) : lk[4] + (q - n0 - n1);
      for (uint32_t polls = 1;; polls++) {
         const uint32_t f = mine ? __hip_atomic_load(r.flags + kFlagStride * t, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                                 : target;
         if (!__ballot((int32_t)(f - target) < 0)) break;
         if (polls % kResidentPolls) continue;
         bail = __builtin_amdgcn_readfirstlane(resident_give_up(r, lane, polls));
         if (bail) break;
      }
   }
}

// The neighbours of a tile and the steps they have done.
struct ResidentLinks {
   uint32_t lk[6];
   bool bail = false;
   __device__ __forceinline__ void load(const ResidentArgs &r, int j)
   {
#pragma unroll
      for (int q = 0; q < 6; q++) lk[q] = __builtin_amdgcn_readfirstlane(r.links[6 * j + q]);
      bail = resident_failed(r);
   }
   // before the stencil of step k of the launch
   __device__ __forceinline__ void wait(const ResidentArgs &r, const ResidentTile &t, int k)
   {
      if (k > 0) {
         resident_wait(r, lk, t.lane, r.base + (uint32_t)k, bail);
         asm volatile("" ::: "memory");
      }
   }
   // after the tile's Vm stores of step k
   __device__ __forceinline__ void done(const ResidentArgs &r, const ResidentTile &t, int k)
   {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (t.lane == 0)
         __hip_atomic_store(r.flags + kFlagStride * t.j, r.base + (uint32_t)k + 1u,
                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
   }
};

// The slab's clock and stimuli over the launch's steps, as slab_advance and
// slab_stim keep them from step to step.
struct ResidentClock {
   double time;
   int loop;
   uint32_t stim;               // the stimuli that reach any cell of the tile
   __device__ __forceinline__ void load(const EngineArgs &a, const ResidentTile &t)
   {
      time = t.S->time[a.parity];
      loop = t.S->loop[a.parity];
      stim = 0;
      for (int q = 0; q < kSlabStim; q++)
         if (__ballot((t.meta >> (16 + q)) & 1u)) stim |= 1u << q;
   }
   __device__ __forceinline__ double iStim(const ResidentTile &t) const
   {
      double s = 0.0;
      for (uint32_t m = stim; m; m &= m - 1) {
         const int q = __builtin_ctz(m);
         const PulseDev p{t.S->stim[q].t0, t.S->stim[q].tf, t.S->stim[q].period,
                          t.S->stim[q].phase, t.S->stim[q].duration, t.S->stim[q].amplitude};
         const double val = pulse_value(p, time);
         // later stimuli overwrite earlier ones where they are on
         if (((t.meta >> (16 + q)) & 1u) && val != 0.0) s = val;
      }
      return s;
   }
   __device__ __forceinline__ void advance(double dt)
   {
      time = time + dt;
      ++loop;
   }
};

// The sensors of a step (engine_sensors), with APD90's phase and largest Vm
// in registers between the steps.
struct ResidentSensors {
   int phase = 0;
   double vmax = 0.0, vrest = 0.0;
   __device__ __forceinline__ void load(const EngineArgs &a, const ResidentTile &t)
   {
      if (a.sensors & 2) {
         const uint32_t i = t.cell();
         phase = a.apd_phase[i];
         vmax = a.vmax[i];
         vrest = t.params(a)->Vm0;
      }
   }
   // Vm before and after the step that begins at clock c
   __device__ __forceinline__ void eval(const EngineArgs &a, const ResidentTile &t,
                                        const ResidentClock &c, double V, double Vn)
   {
      SlabView v{};
      v.time1 = c.time + a.dt;
      v.first_eval = c.loop == t.S->sensor_start;
      v.threshold = t.S->threshold;
      const uint32_t i = t.cell();
      EngineArgs as = a;
      as.sensors = a.sensors & 1;
      uint32_t ev = 0;
      if (t.live && a.sensors) ev = engine_sensors(as, v, i, V, Vn, 0.0);
      if (a.sensors & 2) {
         // apd_eval on the registers
         if (phase == 0) {
            if (ev & kEvTactPacked) {
               phase = 1;
               vmax = Vn;
            }
         } else if (phase == 1) {
            if (Vn > vmax) {
               vmax = Vn;
            } else if (Vn < vrest + 0.1 * (vmax - vrest)) {
               if (t.live) a.t90[i] = v.time1;
               phase = 2;
            }
         }
      }
      if (a.sensors & 1) sensor_count(a.counts + 4 * t.sl, ev);
   }
   __device__ __forceinline__ void store(const EngineArgs &a, const ResidentTile &t) const
   {
      if ((a.sensors & 2) && t.live) {
         const uint32_t i = t.cell();
         a.apd_phase[i] = (uint8_t)phase;
         a.vmax[i] = vmax;
      }
   }
};

// The range check of a step (engine_range).  The tiles are at different steps,
// so the slab's record cannot be the first one that comes: each tile keeps
// the first of its own in this launch (count 1, taken the launch's base)
// behind the slabs' records, and k_slab_clock gives the slab the one of the
// earliest step.
__device__ __forceinline__ void resident_range(const EngineArgs &a, const ResidentArgs &r,
                                               const ResidentTile &t, const ResidentClock &c,
                                               double V, double dVR, double dVD)
{
   if (!t.S->check_range) return;
   const bool out = t.live && (V > t.S->vm_max || V < t.S->vm_min);
   const uint64_t m = __ballot(out);
   if (__builtin_expect(m != 0, 0) && t.lane == __builtin_ctzll(m)) {
      atomicAdd(&a.ranges[t.sl].count, (unsigned long long)__builtin_popcountll(m));
      RangeRec &f = a.ranges[r.tile_ranges + t.j];
      if (!f.count || f.taken != (int32_t)r.base)
         f = RangeRec{1ull, (int32_t)r.base, c.loop, (int64_t)t.cell(), V, dVR, dVD};
   }
}

// f(g) for the 12 gates, g a constant
template <class F, int... G>
__device__ __forceinline__ void each_gate(F &&f, std::integer_sequence<int, G...>)
{
   (f(std::integral_constant<int, G>{}), ...);
}
template <class F>
__device__ __forceinline__ void each_gate(F &&f)
{
   each_gate(f, std::make_integer_sequence<int, N_STATE - S_M>{});
}

// The launch's steps of one tile by one wavefront.  C holds the cell's states
// and weights and gives the reaction, the stencil sum and what follows Vm's
// update, each as the step kernel of its precision has it.
template <class C>
__device__ __forceinline__ void resident_run(const EngineArgs &a, const ResidentArgs &r,
                                             typename C::Shared *sh)
{
   ResidentTile t;
   if (!t.find(a)) return;
   C c;
   c.load(a, t, sh);
   double V = r.box[0][t.b8 / 8u];
   const ParamSet *const params = t.params(a);
   ResidentLinks links;
   links.load(r, t.j);
   ResidentClock clock;
   clock.load(a, t);
   ResidentSensors sensors;
   sensors.load(a, t);
   ModelTables T{constant_ptr(a.K), constant_ptr(a.E), constant_ptr(a.coef)};
   for (int k = 0; k < r.nsteps; k++) {
      renew(T);
      const ParamSet &P = *params;
      const double dVR = c.react(a, T, P, t, V);
      links.wait(r, t, k);
      const double dVD = c.diffuse(t, box_rsrc(r.box[k & 1]), V, t.S->scale);
      resident_range(a, r, t, clock, V, dVR, dVD);
      const double iStim = clock.iStim(t);
      const double Vn = V + a.dt * (dVR + dVD + iStim);
      c.finish(a, T, dVD, iStim);
      if (t.live) box_store_agent(Vn, box_rsrc(r.box[(k & 1) ^ 1]), t.b8, t.S->soff[0]);
      links.done(r, t, k);
      sensors.eval(a, t, clock, V, Vn);
      V = Vn;
      clock.advance(a.dt);
   }
   c.store(t);
   sensors.store(a, t);
}

// ---- six wavefronts to a tile
//
// With at most four tiles to a CU (1,024 in all) a step is still one
// wavefront's chain of dependent instructions, at some 7 cycles each.  The
// gates depend on Vm and themselves alone, and the non-gate update falls into
// a calcium and a sodium and potassium part that meet in two currents, so the
// chain is dealt to six wavefronts of a workgroup:
//   0     sodium and potassium currents; the sums, the stimulus, Vm
//   1     calcium part
//   2     Vm's exchange with the neighbouring tiles and the stencil
//   3..5  four gates each; 4 evaluates the sensors too
// Each keeps its states in registers.  What others read of them crosses in
// LDS: gates, Na_i and Ca_i in two copies by step parity, so that the next
// values are written while the present ones are read.  Two barriers to a
// step: before the sums, when every part is there, and after Vm.
//
// Per step on one MI355X, step kernels, one wavefront to a tile, and this:
// reference rounding 504 cells 10.1, 6.6 and 2.5 us, 52,500 cells 12.1, 7.0
// and 4.9 (821 tiles: the kernel of 64 registers), 46,656 cells 11.6 and 4.0;
// FMA 52,500 cells 11.7 and 4.2; mixed 504 cells 9.1, 5.8 and 2.5, 52,500
// cells 10.5, 5.8 and 3.4; exact functions 504 cells 11.9, 9.7 and 3.1.
// Bounded by the exchange of Vm between tiles (a store to its acknowledgement,
// a flag, a load: some 3,000 cycles) and by the longest part's chain.
constexpr int kSplitWaves = 6;

// all wavefronts of the workgroup: LDS writes before it are there after it
// (a full __syncthreads would wait for the global stores as well)
__device__ __forceinline__ void lds_barrier()
{
   asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
   __builtin_amdgcn_s_barrier();
   asm volatile("" ::: "memory");
}

// G: the gates' type, WT the weights' (words of them per cell: NW).  C: see
// SplitF64 (engine_f64.hip).
template <class G, class WT, int NW>
struct SplitShared {
   WT w[NW][kBlk];
   G gate[2][12][kBlk];
   double ca[2][kBlk], na[2][kBlk];
   double I_sum[kBlk], I_CaL[kBlk], dVD[kBlk], V[kBlk];
};

template <class C, int W>
__device__ __forceinline__ void split_gate_wave(const EngineArgs &a, const ResidentArgs &r,
                                                const ResidentTile &t, ModelTables T,
                                                typename C::Shared *sh)
{
   C c;
   c.template load_gates<kSplitGates[W]>(a, t);
   c.template share_gates<kSplitGates[W]>(sh, 0, t.lane);
   const int s_switch = t.params(a)->s_switch;
   ResidentClock clock;
   ResidentSensors sensors;
   if constexpr (W == 1) {
      clock.load(a, t);
      sensors.load(a, t);
   }
   lds_barrier();
   for (int k = 0; k < r.nsteps; k++) {
      renew(T);
      const double V = sh->V[t.lane];
      c.gates(a, T, s_switch, t.meta, V, a.gate_mask & kSplitGates[W]);
      c.template share_gates<kSplitGates[W]>(sh, (k & 1) ^ 1, t.lane);
      lds_barrier();
      lds_barrier();
      if constexpr (W == 1) {
         sensors.eval(a, t, clock, V, sh->V[t.lane]);
         clock.advance(a.dt);
      }
   }
   c.template store_gates<kSplitGates[W]>(t);
   if constexpr (W == 1) sensors.store(a, t);
}

template <class C>
__device__ __forceinline__ void resident_split_run(const EngineArgs &a, const ResidentArgs &r,
                                                   typename C::Shared *sh)
{
   ResidentTile t;
   if (!t.find(a)) return;      // the whole workgroup: the tile is its tile
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kBlk);
   ModelTables T{constant_ptr(a.K), constant_ptr(a.E), constant_ptr(a.coef)};
   // every branch passes the same barriers: one at the start, two to a step
   if (wave == 0) {
      C c;
      c.load_na_k(a, t);
      double V = r.box[0][t.b8 / 8u];
      sh->V[t.lane] = V;
      c.share_na(sh, 0, t.lane);
      const ParamSet *const params = t.params(a);
      ResidentClock clock;
      clock.load(a, t);
      lds_barrier();
      for (int k = 0; k < r.nsteps; k++) {
         renew(T);
         c.na_k(a, T, *params, V, sh, k & 1, t.lane);
         lds_barrier();
         const double dVD = sh->dVD[t.lane];
         const double dVR = c.sum(a, T, sh, t.lane);
         resident_range(a, r, t, clock, V, dVR, dVD);
         const double iStim = clock.iStim(t);
         V = V + a.dt * (dVR + dVD + iStim);
         c.finish(a, T, dVD, iStim);
         sh->V[t.lane] = V;
         c.share_na(sh, (k & 1) ^ 1, t.lane);
         lds_barrier();
         clock.advance(a.dt);
      }
      c.store_na_k(t);
   } else if (wave == 1) {
      C c;
      c.load_ca(a, t);
      c.share_ca(sh, 0, t.lane);
      const ParamSet *const params = t.params(a);
      lds_barrier();
      for (int k = 0; k < r.nsteps; k++) {
         renew(T);
         c.calcium(a, T, *params, sh->V[t.lane], sh, k & 1, t.lane);
         c.share_ca(sh, (k & 1) ^ 1, t.lane);
         lds_barrier();
         lds_barrier();
      }
      c.store_ca(t);
   } else if (wave == 2) {
      C c;
      c.load_weights(a, t, sh);
      ResidentLinks links;
      links.load(r, t.j);
      lds_barrier();
      for (int k = 0; k < r.nsteps; k++) {
         const double V = sh->V[t.lane];
         links.wait(r, t, k);
         sh->dVD[t.lane] = c.diffuse(t, box_rsrc(r.box[k & 1]), V, t.S->scale, sh);
         lds_barrier();
         lds_barrier();
         const double Vn = sh->V[t.lane];
         if (t.live) box_store_agent(Vn, box_rsrc(r.box[(k & 1) ^ 1]), t.b8, t.S->soff[0]);
         links.done(r, t, k);
      }
   } else if (wave == 3) {
      split_gate_wave<C, 0>(a, r, t, T, sh);
   } else if (wave == 4) {
      split_gate_wave<C, 1>(a, r, t, T, sh);
   } else {
      split_gate_wave<C, 2>(a, r, t, T, sh);
   }
}

}  // namespace cdh
