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
// same each wait is bounded (kResidentWaitTicks): past it the wavefront
// raises `failed`, which the host reports, and nobody waits any longer.
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
// SIMD) 24.5 and 16.5; mixed 52,500 cells 10.6 and 5.9, 262,144 cells 15.4
// and 10.4; exact functions 52,500 cells 13.5 and 9.7.  What bounds it: up
// to 1,024 tiles the latency of one wavefront's chain (12,000 of 17,000 cycles
// in the reaction), with more tiles VALU issue.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "engine.hpp"
#include "tt06_model.hpp"

namespace cdh {

// Words from one tile's flag to the next: a line each.  With 32 flags to a
// line, the stores of 32 tiles and the polls of their neighbours all met
// there: at 2,940 tiles (mixed) a wait took 17,400 cycles of a step, with a
// line each 4,000.
constexpr int kFlagStride = 32;
constexpr uint64_t kResidentWaitTicks = 2000000000ull;   // 20 s of the 100 MHz clock

struct ResidentArgs {
   // both by the tile's place in the list of live tiles
   uint32_t *flags;             // steps done, counted on from launch to launch, one flag
                                // to a cache line (kFlagStride)
   const uint32_t *links;       // 3 ranges {first, last + 1} of neighbouring tiles
   uint32_t base;               // every tile's flag at the launch
   int nsteps;
   double *box[2];              // box[k & 1] is read in step k of this launch
   uint32_t *failed;            // host memory; 1 once a wait has passed its bound
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
   int blk, lane;
   uint32_t b8;                 // this lane's box offset in bytes
   uint32_t lc, rw;             // its place in the run of cells its states are in, the run's width
   int64_t run_cell;            // the run's first cell in the arena
   // node k's Vm from the box behind R, past the caches that other XCDs'
   // stores do not reach
   __device__ __forceinline__ double neighbour(__amdgpu_buffer_rsrc_t R, int k) const
   {
      return box_load_agent(R, b8, S->soff[k]);
   }
};

// Waits until every tile of the three ranges has done `target` - base steps.
__device__ __forceinline__ void resident_wait(const ResidentArgs &r, const uint32_t *lk, int lane,
                                              uint32_t target, bool &bail)
{
   const int n0 = (int)(lk[1] - lk[0]), n1 = (int)(lk[3] - lk[2]), n2 = (int)(lk[5] - lk[4]);
   const int n = n0 + n1 + n2;
   for (int q = lane; __ballot(q < n); q += kBlk) {
      const bool mine = q < n;
      const uint32_t t = !mine ? 0u
                         : q < n0 ? lk[0] + q
                         : q < n0 + n1 ? lk[2] + (q - n0) : lk[4] + (q - n0 - n1);
      uint64_t since = 0;
      while (!bail) {
         const uint32_t f = mine ? __hip_atomic_load(r.flags + kFlagStride * t, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                                 : target;
         if (!__ballot((int32_t)(f - target) < 0)) break;
         const uint64_t now = __builtin_amdgcn_s_memrealtime();
         if (since == 0) since = now;
         if (now - since > kResidentWaitTicks) {
            if (lane == 0) __hip_atomic_store(r.failed, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_SYSTEM);
            bail = true;
         }
      }
   }
}

// The launch's steps of one tile.  C holds the cell's states and weights and
// gives the reaction, the stencil sum and what follows Vm's update, each as
// the step kernel of its precision has it.
template <class C>
__device__ __forceinline__ void resident_run(const EngineArgs &a, const ResidentArgs &r,
                                             typename C::Shared *sh)
{
   const int lane = threadIdx.x;
   const int j = engine_tile_group(a);
   if (j >= a.ntile) return;
   ResidentTile t;
   t.lane = lane;
   t.blk = __builtin_amdgcn_readfirstlane(a.tiles ? (int)a.tiles[j] : a.tile_base + j);
   const int sl = __builtin_amdgcn_readfirstlane((int)a.blk_slab[t.blk]);
   if (sl == kNoSlab) return;
   t.S = (ConstSlab *)(a.slabs + sl);
   if (!t.S->active) return;
   const int64_t i = (int64_t)t.blk * kBlk + lane;
   const uint32_t meta = a.meta[i];
   const bool live = !(meta & kMetaPad);
   const uint32_t b = a.bi[i];
   t.b8 = b * 8u;
   const int64_t k0 = (int64_t)(t.blk - t.S->first_blk) * kBlk;
   const int64_t r0 = k0 & ~(kRun - 1);
   t.rw = (uint32_t)run_width(k0, (int64_t)t.S->ntile * kBlk);
   t.run_cell = (int64_t)t.S->first_blk * kBlk + r0;
   t.lc = (uint32_t)(k0 - r0 + lane);
   C c;
   c.load(a, t, sh);
   double V = r.box[0][b];
   const ParamSet *const params = a.params + t.S->param_base + (int)(meta & 0xFFu);
   uint32_t lk[6];
#pragma unroll
   for (int q = 0; q < 6; q++) lk[q] = __builtin_amdgcn_readfirstlane(r.links[6 * j + q]);
   // the stimuli that reach any cell of the tile
   uint32_t tile_stim = 0;
   for (int q = 0; q < kSlabStim; q++)
      if (__ballot((meta >> (16 + q)) & 1u)) tile_stim |= 1u << q;
   SlabView v;
   v.scale = t.S->scale;
   v.threshold = t.S->threshold;
   v.check_range = t.S->check_range;
   v.vm_min = t.S->vm_min;
   v.vm_max = t.S->vm_max;
   double time = t.S->time[a.parity];
   int loop = t.S->loop[a.parity];
   const int sensor_start = t.S->sensor_start;
   // APD90's phase and largest Vm stay in registers between the steps
   int apd_phase = 0;
   double apd_vmax = 0.0, vrest = 0.0;
   if (a.sensors & 2) {
      apd_phase = a.apd_phase[i];
      apd_vmax = a.vmax[i];
      vrest = params->Vm0;
   }
   EngineArgs as = a;           // the sensors' arguments without APD90
   as.sensors = a.sensors & 1;
   bool bail = false;
   ModelTables T{constant_ptr(a.K), constant_ptr(a.E), constant_ptr(a.coef)};
   for (int k = 0; k < r.nsteps; k++) {
      // the tables' addresses made anew in every step: otherwise their loads
      // move out of the loop, hundreds of scalars that no wavefront can hold
      asm volatile("" : "+s"(T.K), "+s"(T.E), "+s"(T.coef));
      // likewise the cell's place, so that the addresses that only a sensor
      // event or an out-of-range cell needs are made there, not held
      uint32_t cell = (uint32_t)t.blk * kBlk + lane;
      asm volatile("" : "+v"(cell));
      const ParamSet &P = *params;
      const double dVR = c.react(a, T, P, meta, V);
      if (k > 0) {
         resident_wait(r, lk, lane, r.base + (uint32_t)k, bail);
         asm volatile("" ::: "memory");
      }
      const __amdgpu_buffer_rsrc_t from = box_rsrc(r.box[k & 1]);
      const __amdgpu_buffer_rsrc_t to = box_rsrc(r.box[(k & 1) ^ 1]);
      const double dVD = c.diffuse(t, from, V, v.scale);
      if (v.check_range) {
         const bool out = live && (V > v.vm_max || V < v.vm_min);
         const uint64_t m = __ballot(out);
         if (m) range_report(a.ranges + sl, m, lane, loop, cell, V, dVR, dVD);
      }
      double iStim = 0.0;
      for (uint32_t m = tile_stim; m; m &= m - 1) {
         const int q = __builtin_ctz(m);
         const PulseDev p{t.S->stim[q].t0, t.S->stim[q].tf, t.S->stim[q].period,
                          t.S->stim[q].phase, t.S->stim[q].duration, t.S->stim[q].amplitude};
         const double val = pulse_value(p, time);
         // later stimuli overwrite earlier ones where they are on
         if (((meta >> (16 + q)) & 1u) && val != 0.0) iStim = val;
      }
      const double Vn = V + a.dt * (dVR + dVD + iStim);
      c.finish(a, T, dVD, iStim);
      v.time1 = time + a.dt;
      v.first_eval = loop == sensor_start;
      if (live) box_store_agent(Vn, to, t.b8, t.S->soff[0]);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0)
         __hip_atomic_store(r.flags + kFlagStride * j, r.base + (uint32_t)k + 1u, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
      uint32_t ev = 0;
      if (live && a.sensors) ev = engine_sensors(as, v, cell, V, Vn, 0.0);
      if (a.sensors & 2) {
         // apd_eval on the registers
         if (apd_phase == 0) {
            if (ev & (kEvTactPacked)) {
               apd_phase = 1;
               apd_vmax = Vn;
            }
         } else if (apd_phase == 1) {
            if (Vn > apd_vmax) {
               apd_vmax = Vn;
            } else if (Vn < vrest + 0.1 * (apd_vmax - vrest)) {
               if (live) a.t90[cell] = v.time1;
               apd_phase = 2;
            }
         }
      }
      if (a.sensors & 1) sensor_count(a.counts + 4 * sl, ev);
      V = Vn;
      time = v.time1;
      ++loop;
   }
   c.store();
   if ((a.sensors & 2) && live) {
      a.apd_phase[i] = (uint8_t)apd_phase;
      a.vmax[i] = apd_vmax;
   }
}

}  // namespace cdh
