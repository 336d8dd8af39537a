// engine_f64.hip -- the fused FP64 step over the engine's slabs (gfx950).
//
// Compiled with -ffp-contract=off: with FMA = false the reaction, the
// stencil and the Vm update round as the reference CPU path does, operation
// by operation (TT06Dev_Reaction::calc, elec/TT06Dev_Reaction.cc:393-407;
// FGRDiffusionOMP::calc, elec/FGRDiffusionOMP.cc:109-131; the integrator,
// elec/simulationLoop.cc:221-227).  KIND selects the reaction's arithmetic:
// kFits, the 33 rational fits as the reference rounds them; kFitsFma, the
// fit polynomials with fused multiply-adds (half the instructions of the
// multiply-add pairs) and everything else as it is; kExact, configuration A
// (TT06Dev tolerance 0, the factory's default deck): the exact voltage
// functions with the device's exp, log, sqrt and pow and the generic gate
// update (elec/TT06Func.cc:64-161), rounded as the drop-in reaction object
// rounds them, so that the fused step equals the unfused loop bit for bit.
#pragma clang fp contract(off)

#include "engine.hpp"
#include "engine_resident.hpp"
#include "tt06_exact.hpp"

namespace cdh {

namespace {

template <int KIND>
__device__ __forceinline__ void cell_f64(const EngineArgs &a, const SlabDev &S, int sl,
                                         const SlabView &v, int blk, int lane)
{
   const int64_t i = (int64_t)blk * kBlk + lane;
   // padding cells of a slab's last tile compute on a copy of a tissue
   // cell's box point and store only their own states, so the tile runs
   // without a divergent exit
   const uint32_t meta = a.meta[i];
   const bool live = !(meta & kMetaPad);
   const uint32_t b = a.bi[i];
   const uint32_t b8 = b * 8u;
   const __amdgpu_buffer_rsrc_t R = box_rsrc(a.box_cur);
   const double V = box_load(R, b8, S.soff[0]);

   // the stencil first (FGRDiffusionOMP::calc order: A0*phi0, then
   // A_k*phi_k for k = 1..18): its neighbour and weight loads are issued with
   // the state loads at the start, so the reaction's arithmetic covers them.
   // The centre weight is minus the double sum of the 18 float weights in
   // order (FGRDiffusionOMP.cc:214-219), recomputed here bit for bit rather
   // than streamed from memory.
   // (one load per weight: the drop-in stencil's grouped loads, grp_index18,
   // measured no faster here, 1.516 against 1.513 ms per FMA step)
   const float *wp = a.Aw + (int64_t)blk * (18 * kBlk) + lane;
   float w[18];
   double A0 = 0.0;
#pragma unroll
   for (int k = 0; k < 18; k++) {
      w[k] = __builtin_nontemporal_load(wp + kBlk * k);
      A0 -= w[k];
   }
   double tmp = A0 * V;
#pragma unroll
   for (int k = 1; k < 19; k++) tmp += (double)w[k - 1] * box_load(R, b8, S.soff[k]);
   const double dVD = tmp * v.scale;

   // states stream once per step (non-temporal), in the slab's runs of kRun
   // cells with the fields in pairs (run_pair_index): a buffer over the
   // run's base, the pair's offset in an SGPR, the lane's cell in a VGPR
   const int first = __builtin_amdgcn_readfirstlane(S.first_blk);
   const int64_t k0 = (int64_t)(blk - first) * kBlk;
   const int64_t r0 = k0 & ~(kRun - 1);
   const uint32_t rw =
       (uint32_t)run_width(k0, (int64_t)__builtin_amdgcn_readfirstlane(S.ntile) * kBlk);
   const __amdgpu_buffer_rsrc_t RS = stream_rsrc(a.state + ((int64_t)first * kBlk + r0) * N_STATE);
   const uint32_t lc = (uint32_t)(k0 - r0 + lane);
   static_assert(N_STATE % 2 == 1, "the last state field stands alone after the pairs");
   double st[N_STATE];
#pragma unroll
   for (int s = 0; s + 1 < N_STATE; s += 2)
      stream_load_f64x2(RS, 16u * lc, 8u * rw * s, st[s], st[s + 1]);
   st[N_STATE - 1] = stream_load_f64(RS, 8u * lc, 8u * rw * (N_STATE - 1));
   const ParamSet P = a.params[v.param_base + (int)(meta & 0xFFu)];
   // the non-gate update in a basic block of its own (gate_mask bit 12,
   // always set): otherwise the compiler hoists its scalar coefficient loads
   // to the kernel entry and spills them
   double dVR = 0.0;
   if constexpr (KIND == kExact) {
      if (a.gate_mask & (1u << 12))
         dVR = nongate_core64(*a.K, P, exact_voltage_fns(a.E, a.K), a.dt, V, st);
      if (!((meta >> 8) & kFlagGatesFixed))
         gates_exact64(*a.E, P.s_switch, a.dt, V, st, a.gate_mask);
   } else {
      constexpr bool FMA = KIND == kFitsFma;
      if (a.gate_mask & (1u << 12)) dVR = nongate64<FMA>(*a.K, P, a.coef, a.dt, V, st);
      gates64<FMA>(a.coef, a.K->exp_coef, P.s_switch, (uint8_t)(meta >> 8), V, st, a.gate_mask);
   }
   // Reads of the slab's descriptor after a vector store become vector loads
   // that wait for it, so the range check's limits come from the view read
   // at the start.  Since then the stores' place makes no difference: on one
   // MI355X, both instances within 0.2 % with the stores before or after the
   // range check and the stimulus (the FMA step 0.5 % faster than when the
   // limits were read here).
   if constexpr (KIND == kFitsFma) {
#pragma unroll
      for (int s = 0; s + 1 < N_STATE; s += 2)
         stream_store_f64x2(st[s], st[s + 1], RS, 16u * lc, 8u * rw * s);
      stream_store_f64(st[N_STATE - 1], RS, 8u * lc, 8u * rw * (N_STATE - 1));
   }
   engine_range(a, S, v, sl, a.parity, live, lane, i, V, dVR, dVD);
   const double iStim = slab_stim(S, v, a.parity, meta);
   const double Vn = V + a.dt * (dVR + dVD + iStim);
   if constexpr (KIND != kFitsFma) {
#pragma unroll
      for (int s = 0; s + 1 < N_STATE; s += 2)
         stream_store_f64x2(st[s], st[s + 1], RS, 16u * lc, 8u * rw * s);
      stream_store_f64(st[N_STATE - 1], RS, 8u * lc, 8u * rw * (N_STATE - 1));
   }
   uint32_t ev = 0;
   if (live) {
      a.box_next[b] = Vn;
      if (a.sensors) ev = engine_sensors(a, v, i, V, Vn, P.Vm0);
   }
   // every lane of the tile is here (padding lanes with no events)
   if (a.sensors & 1) sensor_count(a.counts + 4 * sl, ev);
}

}  // namespace

// Workgroups map to tiles in the XCD-aware order of engine_tile_group.  The
// grid covers the live slabs' tiles only: tiles of removed slabs cost nothing.
// When the live tiles are one range (one anatomy, a batch without holes)
// the tile is the index plus a base, with no list to read first.
template <int WAVES, int KIND>
__global__ __launch_bounds__(256, WAVES) void k_engine_f64(EngineArgs a)
{
   const int wpg = blockDim.x >> 6;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int lane = threadIdx.x & 63;
   const int j = engine_tile_group(a) * wpg + wave;
   if (j >= a.ntile) return;
   const int blk = a.tiles ? (int)a.tiles[j] : a.tile_base + j;
   const int sl = a.blk_slab[blk];
   if (sl == kNoSlab) return;
   SlabDev &S = a.slabs[sl];
   if (!S.active) return;
   SlabView v;
   slab_view(S, a.parity, a.dt, v);
   cell_f64<KIND>(a, S, sl, v, blk, lane);
   if (blk == S.first_blk && lane == 0) slab_advance(S, a.parity, v);
}

template __global__ void k_engine_f64<2, kFits>(EngineArgs);
template __global__ void k_engine_f64<3, kFits>(EngineArgs);
template __global__ void k_engine_f64<2, kFitsFma>(EngineArgs);
template __global__ void k_engine_f64<3, kFitsFma>(EngineArgs);
template __global__ void k_engine_f64<2, kExact>(EngineArgs);
template __global__ void k_engine_f64<3, kExact>(EngineArgs);

// ---- resident form (engine_resident.hpp)

namespace {

// The 18 weights wait in LDS between the steps' stencils, the states in
// registers.  At four wavefronts per SIMD (128 VGPRs) the first kParked gates
// wait in LDS too, from one use to the next: 9.5 KB to a tile, so that 16
// tiles take the CU's 160 KB.  With all states in registers that kernel
// spilled 9 of them to scratch: 64^3 cells FMA 16.1 us a step, reference
// rounding 18.3; now 15.1 and 17.3.
constexpr int kParked = 10;

template <int KIND, int NPARK>
struct ResidentF64 {
   struct Shared {
      float w[18][kBlk];
      double park[NPARK > 0 ? NPARK : 1][kBlk];
   };
   double st[N_STATE];
   template <class G>
   __device__ __forceinline__ void fetch(G, int lane)
   {
      if constexpr (G::value < NPARK) st[S_M + G::value] = sh->park[G::value][lane];
   }
   template <class G>
   __device__ __forceinline__ void park(G, int lane)
   {
      if constexpr (G::value < NPARK) sh->park[G::value][lane] = st[S_M + G::value];
   }
   Shared *sh;
   __amdgpu_buffer_rsrc_t RS;
   uint32_t lc, rw;

   __device__ __forceinline__ void load(const EngineArgs &a, const ResidentTile &t, Shared *shared)
   {
      sh = shared;
      const float *wp = a.Aw + (int64_t)t.blk * (18 * kBlk) + t.lane;
#pragma unroll
      for (int k = 0; k < 18; k++) sh->w[k][t.lane] = wp[kBlk * k];
      rw = t.rw;
      lc = t.lc;
      RS = stream_rsrc(a.state + t.run_cell * N_STATE);
#pragma unroll
      for (int s = 0; s + 1 < N_STATE; s += 2)
         stream_load_f64x2(RS, 16u * lc, 8u * rw * s, st[s], st[s + 1]);
      st[N_STATE - 1] = stream_load_f64(RS, 8u * lc, 8u * rw * (N_STATE - 1));
      each_gate([&](auto g) { park(g, t.lane); });
   }
   __device__ __forceinline__ void store(const ResidentTile &t)
   {
      each_gate([&](auto g) { fetch(g, t.lane); });
#pragma unroll
      for (int s = 0; s + 1 < N_STATE; s += 2)
         stream_store_f64x2(st[s], st[s + 1], RS, 16u * lc, 8u * rw * s);
      stream_store_f64(st[N_STATE - 1], RS, 8u * lc, 8u * rw * (N_STATE - 1));
   }
   __device__ __forceinline__ double react(const EngineArgs &a, const ModelTables &T,
                                           const ParamSet &P, const ResidentTile &t, double V)
   {
      const uint32_t meta = t.meta;
      double dVR = 0.0;
      each_gate([&](auto g) { fetch(g, t.lane); });
      if (a.gate_mask & (1u << 12)) {
         if constexpr (KIND == kExact)
            dVR = nongate_core64<true>(*T.K, P, exact_voltage_fns(T.E, T.K), a.dt, V, st);
         else
            dVR = nongate64<KIND == kFitsFma, true>(*T.K, P, T.coef, a.dt, V, st);
      }
      auto gates = [&](uint32_t mask) {
         if constexpr (KIND == kExact) {
            if (!((meta >> 8) & kFlagGatesFixed))
               gates_exact64(*T.E, P.s_switch, a.dt, V, st, mask);
         } else {
            gates64<KIND == kFitsFma>(T.coef, T.K->exp_coef, P.s_switch, (uint8_t)(meta >> 8), V,
                                      st, mask);
         }
      };
      if constexpr (NPARK == 0) {
         gates(a.gate_mask);
      } else {
         each_gate([&](auto g) {
            asm volatile("" ::: "memory");   // fetched here, not before
            fetch(g, t.lane);
            gates(a.gate_mask & (1u << g.value));
            park(g, t.lane);
         });
      }
      return dVR;
   }
   // the sums of cell_f64, in its order
   __device__ __forceinline__ double diffuse(const ResidentTile &t, __amdgpu_buffer_rsrc_t R, double V,
                                             double scale)
   {
      double nb[18];
#pragma unroll
      for (int k = 0; k < 18; k++) nb[k] = t.neighbour(R, k + 1);
      __builtin_amdgcn_sched_barrier(0);   // all loads in flight before the first sum
      double A0 = 0.0;
#pragma unroll
      for (int k = 0; k < 18; k++) A0 -= sh->w[k][t.lane];
      double tmp = A0 * V;
#pragma unroll
      for (int k = 1; k < 19; k++) tmp += (double)sh->w[k - 1][t.lane] * nb[k - 1];
      return tmp * scale;
   }
   __device__ __forceinline__ void finish(const EngineArgs &, const ModelTables &, double, double)
   {
   }
};

// One wavefront's part of a cell for resident_split_run; each uses the states
// it owns, and the others' from LDS.
template <int KIND>
struct SplitF64 {
   using Shared = SplitShared<double, float, 18>;
   double st[N_STATE];
   SodiumPotassiumCurrents nk;
   double I_NaCa, A0;

   // one field of the pair layout (run_pair_index)
   __device__ __forceinline__ static uint32_t lane_off(const ResidentTile &t, int q)
   {
      return q < N_STATE - 1 ? 16u * t.lc + 8u * (q & 1) : 8u * t.lc;
   }
   __device__ __forceinline__ static uint32_t field_off(const ResidentTile &t, int q)
   {
      return 8u * t.rw * (q < N_STATE - 1 ? (q & ~1) : q);
   }
   __amdgpu_buffer_rsrc_t RS;
   __device__ __forceinline__ void load(const ResidentTile &t, int q)
   {
      st[q] = box_load(RS, lane_off(t, q), field_off(t, q));
   }
   __device__ __forceinline__ void store(const ResidentTile &t, int q)
   {
      stream_store_f64(st[q], RS, lane_off(t, q), field_off(t, q));
   }
   __device__ __forceinline__ void states(const EngineArgs &a, const ResidentTile &t)
   {
      RS = stream_rsrc(a.state + t.run_cell * N_STATE);
   }

   __device__ __forceinline__ void load_na_k(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
      load(t, S_DVK_I);
      load(t, S_NA_I);
   }
   __device__ __forceinline__ void store_na_k(const ResidentTile &t)
   {
      store(t, S_DVK_I);
      store(t, S_NA_I);
   }
   __device__ __forceinline__ void share_na(Shared *sh, int p, int lane)
   {
      sh->na[p][lane] = st[S_NA_I];
   }
   __device__ __forceinline__ void load_ca(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
      for (int q : {S_CA_I, S_CA_SS, S_CA_SR, S_R_PRIME, S_FCASS}) load(t, q);
   }
   __device__ __forceinline__ void store_ca(const ResidentTile &t)
   {
      for (int q : {S_CA_I, S_CA_SS, S_CA_SR, S_R_PRIME, S_FCASS}) store(t, q);
   }
   __device__ __forceinline__ void share_ca(Shared *sh, int p, int lane)
   {
      sh->ca[p][lane] = st[S_CA_I];
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void load_gates(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
#pragma unroll
      for (int q = S_M; q < N_STATE; q++)
         if ((GATES >> (q - S_M)) & 1) load(t, q);
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void store_gates(const ResidentTile &t)
   {
#pragma unroll
      for (int q = S_M; q < N_STATE; q++)
         if ((GATES >> (q - S_M)) & 1) store(t, q);
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void share_gates(Shared *sh, int p, int lane)
   {
#pragma unroll
      for (int q = S_M; q < N_STATE; q++)
         if ((GATES >> (q - S_M)) & 1) sh->gate[p][q - S_M][lane] = st[q];
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void take_gates(const Shared *sh, int p, int lane)
   {
#pragma unroll
      for (int q = S_M; q < N_STATE; q++)
         if ((GATES >> (q - S_M)) & 1) st[q] = sh->gate[p][q - S_M][lane];
   }
   template <class F>
   __device__ __forceinline__ static void voltage_fns(const ModelTables &T, F &&f)
   {
      if constexpr (KIND == kExact) f(exact_voltage_fns(T.E, T.K));
      else f(fit_voltage_fns<KIND == kFitsFma>(T.coef));
   }
   __device__ __forceinline__ void na_k(const EngineArgs &, const ModelTables &T, const ParamSet &P,
                                        double V, const Shared *sh, int p, int lane)
   {
      take_gates<kGatesNaK>(sh, p, lane);
      voltage_fns(T, [&](const auto &fvs) {
         double fv[6];
         fvs.fv05(V, fv);
         I_NaCa = exchanger64(st[S_NA_I], sh->ca[p][lane], fv[1], fv[2]);
         nk = nongate_na_k64(*T.K, P, fvs, V, fv[0], fv[5], I_NaCa, st);
      });
   }
   __device__ __forceinline__ void calcium(const EngineArgs &a, const ModelTables &T,
                                           const ParamSet &P, double V, Shared *sh, int p, int lane)
   {
      take_gates<kGatesCa>(sh, p, lane);
      voltage_fns(T, [&](const auto &fvs) {
         double fv[6];
         fvs.fv05(V, fv);
         const double I = exchanger64(sh->na[p][lane], st[S_CA_I], fv[1], fv[2]);
         const CalciumCurrents ca = nongate_calcium64(*T.K, P, a.dt, V, fv[3], fv[4], I, st);
         sh->I_sum[lane] = ca.I_sum;
         sh->I_CaL[lane] = ca.I_CaL;
      });
   }
   __device__ __forceinline__ double sum(const EngineArgs &a, const ModelTables &T,
                                         const Shared *sh, int lane)
   {
      return nongate_sum64(*T.K, a.dt, I_NaCa, CalciumCurrents{sh->I_sum[lane], sh->I_CaL[lane]},
                           nk, st);
   }
   __device__ __forceinline__ void finish(const EngineArgs &, const ModelTables &, double, double)
   {
   }
   __device__ __forceinline__ void gates(const EngineArgs &a, const ModelTables &T, int s_switch,
                                         uint32_t meta, double V, uint32_t mask)
   {
      if constexpr (KIND == kExact) {
         if (!((meta >> 8) & kFlagGatesFixed))
            gates_exact64(*T.E, s_switch, a.dt, V, st, mask);
      } else {
         gates64<KIND == kFitsFma>(T.coef, T.K->exp_coef, s_switch, (uint8_t)(meta >> 8), V, st,
                                   mask);
      }
   }
   __device__ __forceinline__ void load_weights(const EngineArgs &a, const ResidentTile &t,
                                                Shared *sh)
   {
      const float *wp = a.Aw + (int64_t)t.blk * (18 * kBlk) + t.lane;
#pragma unroll
      for (int k = 0; k < 18; k++) sh->w[k][t.lane] = wp[kBlk * k];
      A0 = 0.0;
#pragma unroll
      for (int k = 0; k < 18; k++) A0 -= sh->w[k][t.lane];
   }
   __device__ __forceinline__ double diffuse(const ResidentTile &t, __amdgpu_buffer_rsrc_t R,
                                             double V, double scale, const Shared *sh)
   {
      double nb[18];
#pragma unroll
      for (int k = 0; k < 18; k++) nb[k] = t.neighbour(R, k + 1);
      __builtin_amdgcn_sched_barrier(0);
      double tmp = A0 * V;
#pragma unroll
      for (int k = 1; k < 19; k++) tmp += (double)sh->w[k - 1][t.lane] * nb[k - 1];
      return tmp * scale;
   }
};

}  // namespace

template <int KIND, int WAVES>
__global__ __launch_bounds__(64, WAVES) void k_resident_f64(EngineArgs a, ResidentArgs r)
{
   using C = ResidentF64<KIND, WAVES == 4 ? kParked : 0>;
   __shared__ typename C::Shared sh;
   resident_run<C>(a, r, &sh);
}

template <int KIND, int WAVES>
__global__ __launch_bounds__(kSplitWaves * 64, WAVES) void k_resident_split_f64(EngineArgs a,
                                                                                ResidentArgs r)
{
   __shared__ typename SplitF64<KIND>::Shared sh;
   resident_split_run<SplitF64<KIND>>(a, r, &sh);
}

template __global__ void k_resident_split_f64<kFits, 6>(EngineArgs, ResidentArgs);
template __global__ void k_resident_split_f64<kFits, 8>(EngineArgs, ResidentArgs);
template __global__ void k_resident_split_f64<kFitsFma, 6>(EngineArgs, ResidentArgs);
template __global__ void k_resident_split_f64<kFitsFma, 8>(EngineArgs, ResidentArgs);
template __global__ void k_resident_split_f64<kExact, 6>(EngineArgs, ResidentArgs);
template __global__ void k_resident_split_f64<kExact, 8>(EngineArgs, ResidentArgs);
template __global__ void k_resident_f64<kFits, 3>(EngineArgs, ResidentArgs);
template __global__ void k_resident_f64<kFits, 4>(EngineArgs, ResidentArgs);
template __global__ void k_resident_f64<kFitsFma, 3>(EngineArgs, ResidentArgs);
template __global__ void k_resident_f64<kFitsFma, 4>(EngineArgs, ResidentArgs);
template __global__ void k_resident_f64<kExact, 3>(EngineArgs, ResidentArgs);

}  // namespace cdh
