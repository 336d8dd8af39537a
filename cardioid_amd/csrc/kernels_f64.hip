// kernels_f64.hip -- FP64 kernels of the drop-in path (gfx950).
//
// Compiled with -ffp-contract=off: every kernel here reproduces the
// reference CPU path's rounding, operation by operation.
//
//   k_tt06_calc_f64, k_tt06_calc_split_f64  TT06Dev_Reaction::calc
//                       elec/TT06Dev_Reaction.cc:393-407; configuration A
//                       (exact functions, generic gates) elec/TT06Func.cc:64-161
//   k_scatter_f64       FGRDiffusionOMP::updateLocalVoltage  elec/FGRDiffusionOMP.cc:75-89
//   k_fgr_calc_f64      FGRDiffusionOMP::calc           elec/FGRDiffusionOMP.cc:109-131
//   k_integrate_f64     Vm += dt*(dVmR+dVmD+iStim)      elec/simulationLoop.cc:221-227
//   k_fill_f64 / k_set_list_f64   iStim = 0; BoxStimulus  elec/simulationLoop.cc:186-193,
//                                                   elec/BoxStimulus.cc:53-64
//   k_sensor_f64        ActivationTimeSensor / ActivationAndRecoverySensor eval
#pragma clang fp contract(off)

#include "kernels.hpp"
#include "row_shift.hpp"
#include "tt06_exact.hpp"
#include "tt06_f64.hpp"

namespace cdh {

// The drop-in objects keep their states and weights in 64-cell tiles:
// field q of cell i at blk_index(q, i, nq), a wavefront's fields one
// contiguous run.
//
// TT06Dev_Reaction::calc, one tile to a wavefront, a wavefront to a
// workgroup.  A call reads its states first and computes after, and what
// fills the one phase with the other is wavefronts that are not in step: four
// to a SIMD (at most 128 VGPRs), each its own workgroup, so that the next tile
// begins when one ends and not when four have.  Workgroups of four wavefronts
// and a persistent grid of 3 wavefronts per SIMD, each with its next tile's
// loads in flight, kept them in step; us a call on one MI355X, persistent and
// this: fits 131,072 cells 14.3 and 12.8, 300,007 cells 26.6 and 24.4,
// 600,000 cells 50.0 and 44.1, 6.7 million cells 491 and 450 (4.8 TB/s);
// exact functions, in workgroups of four and this: 300,007 cells 40.3 and
// 37.3, 600,000 cells 71 and 67, 6.7 million cells 694 and 676.  3 and 5
// wavefronts per SIMD are within 1 % of 4; streaming (nontemporal) states
// beat cached ones by 3 % and more.  Bounded by VALU issue with the states'
// bytes close behind.
//
// EXACT: configuration A, the non-gate update with the exact fv0..fv6, then
// the generic gate update with the exact steady states and rates, at the
// step's Vm.  Gate flags bit 0 holds every gate of a cell; the generic loop has
// no v2 loop bounds, so otherwise every cell's gates advance.
//
// Without kMaskGates (the pdr loop's updateNonGate) the gates are read and not
// stored: 208 bytes a cell instead of 304.  Exact functions, us a call, in
// workgroups of four with the gates stored, as this with them stored, and this:
// 500,000 cells 27.7, 27.7 and 21.3, 1 million 49.5, 53.2 and 38.5, 1.3 million
// 63, 69 and 49; the fits, persistent, as this with them stored, and this: 1
// million 59.5, 53.2 and 37.4.
//
// The body takes its arrays as restrict-qualified arguments: the stores then
// provably leave the constants and fit coefficients alone, and their reads
// stay scalar loads.  One parameter set per object (pid is not used).
namespace {

template <bool EXACT>
__device__ __forceinline__ void calc_tile(const TT06Const *__restrict__ K,
                                          const TT06ExactConst *__restrict__ E,
                                          const double *__restrict__ coef,
                                          const ParamSet *__restrict__ params,
                                          const uint8_t *__restrict__ flags,
                                          double *__restrict__ state, const int *__restrict__ index,
                                          const double *__restrict__ Vm, double *__restrict__ dVm,
                                          int n, double dt, uint32_t gate_mask)
{
   // states and flags are padded to a whole tile; lanes past n take Vm[0] and
   // store nothing
   const int i = blockIdx.x * kBlk + threadIdx.x;
   const bool live = i < n;
   const int e = live ? (index ? index[i] : i) : 0;
   const double V = Vm[e];
   const uint8_t fl = flags[i];
   double *sp = state + blk_base(i, N_STATE);
   double st[N_STATE];
#pragma unroll
   for (int s = 0; s < N_STATE; s++) st[s] = __builtin_nontemporal_load(sp + kBlk * s);
   const ParamSet P = params[0];
   double dVR = 0.0;
   if constexpr (EXACT) {
      if (gate_mask & kMaskNonGate)
         dVR = nongate_core64(*K, P, exact_voltage_fns(E, K), dt, V, st);
      if (!(fl & kFlagGatesFixed)) gates_exact64(*E, P.s_switch, dt, V, st, gate_mask);
   } else {
      if (gate_mask & kMaskNonGate) dVR = nongate64(*K, P, coef, dt, V, st);
      gates64(coef, K->exp_coef, P.s_switch, fl, V, st, gate_mask);
   }
   if (!live) return;
#pragma unroll
   for (int s = 0; s < S_M; s++) __builtin_nontemporal_store(st[s], sp + kBlk * s);
   if (gate_mask & kMaskGates) {
#pragma unroll
      for (int s = S_M; s < N_STATE; s++) __builtin_nontemporal_store(st[s], sp + kBlk * s);
   }
   dVm[e] = dVR;
}

}  // namespace

template <bool EXACT>
__global__ __launch_bounds__(kBlk, 4) void k_tt06_calc_f64(ReactionArgs a)
{
   calc_tile<EXACT>(a.K, a.E, a.coef, a.params, a.flags, a.state, a.index, a.Vm, a.dVm, a.n, a.dt,
                    a.gate_mask);
}

template __global__ void k_tt06_calc_f64<false>(ReactionArgs);
template __global__ void k_tt06_calc_f64<true>(ReactionArgs);

// TT06Dev_Reaction::calc with a tile's work dealt to five wavefronts of a
// workgroup, for objects of few tiles.  There a call is bound by one
// wavefront's dependent chain, some 1,700 VALU instructions (3,300 with the
// exact functions) at about 7 cycles each; here the longest of the five has
// about 400:
//   wave 0     sodium and potassium currents, the sums, dVm
//   wave 1     calcium part
//   wave 2..4  gates (kSplitGates)
// Waves 0 and 1 read gates that the others advance: every wavefront stores
// after the one barrier, behind which all have read what they need.  The
// expressions are those of the other kernels, the results the same bit for
// bit.  With more tiles the five wavefronts of each only take each other's
// place: see kSplitTiles (plugins.hip) for where that begins.
namespace {

template <bool EXACT, uint32_t GATES>
__device__ __forceinline__ void calc_split_gates(const ReactionArgs &a, int i, bool live, double V,
                                                 double *sp)
{
   double st[N_STATE];
#pragma unroll
   for (int q = S_M; q < N_STATE; q++)
      if ((GATES >> (q - S_M)) & 1) st[q] = sp[kBlk * q];
   const int s_switch = a.params[0].s_switch;
   const uint8_t fl = a.flags[i];
   const uint32_t mask = a.gate_mask & GATES;
   if constexpr (EXACT) {
      if (!(fl & kFlagGatesFixed))
         gates_exact64(*constant_ptr(a.E), s_switch, a.dt, V, st, mask);
   } else {
      gates64(constant_ptr(a.coef), constant_ptr(a.K)->exp_coef, s_switch, fl, V, st, mask);
   }
   __syncthreads();
   if (!live || !mask) return;
#pragma unroll
   for (int q = S_M; q < N_STATE; q++)
      if ((GATES >> (q - S_M)) & 1) sp[kBlk * q] = st[q];
}

}  // namespace

template <bool EXACT>
__global__ __launch_bounds__(kCalcSplitWaves * 64) void k_tt06_calc_split_f64(ReactionArgs a)
{
   __shared__ double xc[2][kBlk];     // I_sum, I_CaL
   const int lane = threadIdx.x & (kBlk - 1);
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kBlk);
   // states and flags are padded to a whole tile; lanes past n take the first
   // cell's Vm and store nothing
   const int i = blockIdx.x * kBlk + lane;
   const bool live = i < a.n;
   const int e = live ? (a.index ? a.index[i] : i) : 0;
   const double V = live ? a.Vm[e] : a.Vm[a.index ? a.index[0] : 0];
   double *sp = a.state + blk_base(i, N_STATE);
   ModelConst *K = constant_ptr(a.K);
   const ParamSet &P = a.params[0];
   double st[N_STATE];
   auto voltage_fns = [&](auto &&f) {
      if constexpr (EXACT) f(exact_voltage_fns(constant_ptr(a.E), K));
      else f(fit_voltage_fns<false>(constant_ptr(a.coef)));
   };
   if (wave == 0) {
#pragma unroll
      for (int q = 0; q < N_STATE; q++)
         if (q == S_DVK_I || q == S_NA_I || q == S_CA_I ||
             (q >= S_M && ((kGatesNaK >> (q - S_M)) & 1)))
            st[q] = sp[kBlk * q];
      double fv[6], I_NaCa = 0.0;
      SodiumPotassiumCurrents nk{};
      voltage_fns([&](const auto &fvs) {
         fvs.fv05(V, fv);
         I_NaCa = exchanger64(st[S_NA_I], st[S_CA_I], fv[1], fv[2]);
         nk = nongate_na_k64(*K, P, fvs, V, fv[0], fv[5], I_NaCa, st);
      });
      __syncthreads();
      const double dVR =
          nongate_sum64(*K, a.dt, I_NaCa, CalciumCurrents{xc[0][lane], xc[1][lane]}, nk, st);
      if (live) {
         sp[kBlk * S_DVK_I] = st[S_DVK_I];
         sp[kBlk * S_NA_I] = st[S_NA_I];
         a.dVm[e] = dVR;
      }
   } else if (wave == 1) {
#pragma unroll
      for (int q = 0; q < N_STATE; q++)
         if (q == S_NA_I || (q < S_M && q != S_DVK_I) ||
             (q >= S_M && ((kGatesCa >> (q - S_M)) & 1)))
            st[q] = sp[kBlk * q];
      voltage_fns([&](const auto &fvs) {
         double fv[6];
         fvs.fv05(V, fv);
         const double I_NaCa = exchanger64(st[S_NA_I], st[S_CA_I], fv[1], fv[2]);
         const CalciumCurrents ca = nongate_calcium64(*K, P, a.dt, V, fv[3], fv[4], I_NaCa, st);
         xc[0][lane] = ca.I_sum;
         xc[1][lane] = ca.I_CaL;
      });
      __syncthreads();
      if (live) {
#pragma unroll
         for (int q = 0; q < S_M; q++)
            if (q != S_DVK_I && q != S_NA_I) sp[kBlk * q] = st[q];
      }
   } else if (wave == 2) {
      calc_split_gates<EXACT, kSplitGates[0]>(a, i, live, V, sp);
   } else if (wave == 3) {
      calc_split_gates<EXACT, kSplitGates[1]>(a, i, live, V, sp);
   } else {
      calc_split_gates<EXACT, kSplitGates[2]>(a, i, live, V, sp);
   }
}

template __global__ void k_tt06_calc_split_f64<false>(ReactionArgs);
template __global__ void k_tt06_calc_split_f64<true>(ReactionArgs);

// Gate update only (Reaction::updateGate of the pdr loop): the 12 gates at Vm.
__global__ __launch_bounds__(256) void k_tt06_gate_f64(ReactionArgs a)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= a.n) return;
   const int e = a.index ? a.index[i] : i;
   const double V = a.Vm[e];
   double st[N_STATE];
#pragma unroll
   for (int s = S_M; s < N_STATE; s++) st[s] = a.state[blk_index(s, i, N_STATE)];
   const ParamSet P = a.params[a.pid ? a.pid[i] : 0];
   gates64(a.coef, a.K->exp_coef, P.s_switch, a.flags[i], V, st, a.gate_mask);
#pragma unroll
   for (int s = S_M; s < N_STATE; s++) a.state[blk_index(s, i, N_STATE)] = st[s];
}

// Configuration A gate update only (Reaction::updateGate of the pdr loop).
__global__ __launch_bounds__(256) void k_tt06_gate_exact_f64(ReactionArgs a)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= a.n) return;
   const int e = a.index ? a.index[i] : i;
   const double V = a.Vm[e];
   double st[N_STATE];
#pragma unroll
   for (int s = S_M; s < N_STATE; s++) st[s] = a.state[blk_index(s, i, N_STATE)];
   gates_exact64(*a.E, a.params[0].s_switch, a.dt, V, st, a.gate_mask);
#pragma unroll
   for (int s = S_M; s < N_STATE; s++) a.state[blk_index(s, i, N_STATE)] = st[s];
}

__global__ __launch_bounds__(256) void k_scatter_f64(int n, const uint32_t *__restrict__ bi,
                                                     const double *__restrict__ src,
                                                     double *__restrict__ box)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) box[bi[i]] = src[i];
}

// The same, four cells per thread: one 16-byte load of box indices and two
// of values per thread (bi and src 16-byte aligned; the host checks).
__global__ __launch_bounds__(256) void k_scatter4_f64(int n, const uint32_t *__restrict__ bi,
                                                      const double *__restrict__ src,
                                                      double *__restrict__ box)
{
   const int64_t i = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
   if (i + 3 < n) {
      const uint4 b = *reinterpret_cast<const uint4 *>(bi + i);
      const double2 s0 = *reinterpret_cast<const double2 *>(src + i);
      const double2 s1 = *reinterpret_cast<const double2 *>(src + i + 2);
      box[b.x] = s0.x;
      box[b.y] = s0.y;
      box[b.z] = s1.x;
      box[b.w] = s1.y;
   } else {
      for (int64_t k = i; k < n; k++) box[bi[k]] = src[k];
   }
}

// the drop-in box's neighbour loads, for gather_rows
struct DropInBox {
   const double *box;
   const int *off;
   __device__ __forceinline__ double at(uint32_t b, int k) const { return box[(int64_t)b + off[k]]; }
   __device__ __forceinline__ uint32_t rel(int k) const { return (uint32_t)off[k]; }
   __device__ __forceinline__ double at_rel(uint32_t b, uint32_t r) const
   {
      return box[(int64_t)b + (int32_t)r];
   }
};

// Blocks are dealt round-robin to the 8 XCDs; each XCD takes a contiguous
// range of cells, so that its L2 holds the box rows and planes they read.
__global__ __launch_bounds__(256) void k_fgr_calc_f64(StencilArgs a)
{
   const int xcd = blockIdx.x & 7;
   const int64_t i =
       ((int64_t)xcd * a.groups_per_xcd + (blockIdx.x >> 3)) * blockDim.x + threadIdx.x;
   // a wavefront past the last cell has nothing to do; in the last one,
   // lanes past it work on the last cell and store nothing, so that every
   // lane takes part in the lane exchanges of the neighbour loads
   if ((i & ~(int64_t)(kBlk - 1)) >= a.n) return;
   const bool act = i < a.n;
   const int64_t ic = act ? i : a.n - 1;
   // Every load is issued before any arithmetic: the box index, then the
   // weights (they stream while the index arrives), then the neighbours.
   // Left to itself the compiler interleaves the neighbour loads with waits
   // on the weights for the centre-weight sum, which costs a third round
   // trip to memory per wave (4 % of the kernel's time).
   const uint32_t b = a.bi[ic];
   // the 18 weights in five loads (grp_index18): four of 16 bytes and one
   // of 8 bytes per lane.  The kernel's texture units are busy for 95 % of
   // its time (rocprof TA_TA_BUSY, TD_TD_BUSY), so fewer load instructions
   // help: 365 against 373 us per call on the 20.1 M-cell shell with one
   // load per weight, bit for bit the same
   const float *tw = a.Aw + (ic >> 6) * (18 * kBlk);
   const int lane = (int)(i & (kBlk - 1));
   float w[18];
#pragma unroll
   for (int g = 0; g < 4; g++) {
      const f32x4 q = __builtin_nontemporal_load((const f32x4 *)(tw + g * 4 * kBlk) + lane);
      w[4 * g] = q.x;
      w[4 * g + 1] = q.y;
      w[4 * g + 2] = q.z;
      w[4 * g + 3] = q.w;
   }
   {
      const f32x2 q = __builtin_nontemporal_load((const f32x2 *)(tw + 16 * kBlk) + lane);
      w[16] = q.x;
      w[17] = q.y;
   }
   __builtin_amdgcn_sched_barrier(0);
   // the 19 neighbours: nine loads, the ten x-1 / x+1 values from the
   // neighbouring lanes where they hold them (row_shift.hpp)
   double v[19];
   gather_rows<kRowsX>(DropInBox{a.box, a.off}, b, act, lane, v);
   __builtin_amdgcn_sched_barrier(0);
   // the weights stream once per step; the centre weight is minus their sum
   // in order, in double (FGRDiffusionOMP.cc:214-219), recomputed bit for bit
   double A0 = 0.0;
#pragma unroll
   for (int k = 0; k < 18; k++) A0 -= w[k];
   double tmp = A0 * v[0];
#pragma unroll
   for (int k = 1; k < 19; k++) tmp += (double)w[k - 1] * v[k];
   if (act) __builtin_nontemporal_store(tmp * a.scale, a.dVm + i);
}

__global__ __launch_bounds__(256) void k_integrate_f64(int n, double dt, double *__restrict__ Vm,
                                                       const double *__restrict__ dVmR,
                                                       const double *__restrict__ dVmD,
                                                       const double *__restrict__ iStim)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) Vm[i] += dt * (dVmR[i] + dVmD[i] + iStim[i]);
}

__global__ __launch_bounds__(256) void k_fill_f64(int n, double v, double *__restrict__ x)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) x[i] = v;
}

__global__ __launch_bounds__(256) void k_set_list_f64(int n, const int *__restrict__ list, double v,
                                                      double *__restrict__ x)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) x[list[i]] = v;
}

// Sensor evaluation at (time, loop) after the step; Vm in cell order.
__global__ __launch_bounds__(256) void k_sensor_f64(SensorArgs a, const double *__restrict__ Vm,
                                                    const double *__restrict__ vrest)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   const uint32_t ev = i < a.n ? sensor_events_packed(sensor_eval(a, i, Vm[i], a.apd ? vrest[i] : 0.0)) : 0u;
   sensor_count(a.counts, ev);
}

// The same, four cells per thread: the flags of the four as one 4-byte
// load each, Vm as two 16-byte loads (Vm 16-byte aligned; the host checks).
__global__ __launch_bounds__(256) void k_sensor4_f64(SensorArgs a, const double *__restrict__ Vm,
                                                     const double *__restrict__ vrest)
{
   const int64_t i = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
   uint32_t ev = 0;
   if (i + 3 < a.n) {
      const uint32_t acd = *reinterpret_cast<const uint32_t *>(a.activated + i);
      const uint32_t act = *reinterpret_cast<const uint32_t *>(a.active + i);
      const double2 v01 = *reinterpret_cast<const double2 *>(Vm + i);
      const double2 v23 = *reinterpret_cast<const double2 *>(Vm + i + 2);
      const double v[4] = {v01.x, v01.y, v23.x, v23.y};
#pragma unroll
      for (int k = 0; k < 4; k++)
         ev += sensor_events_packed(sensor_eval_flags(a, (int)i + k, v[k],
                                                      a.apd ? vrest[i + k] : 0.0,
                                                      (uint8_t)(acd >> (8 * k)),
                                                      (uint8_t)(act >> (8 * k))));
   } else {
      for (int k = (int)i; k < a.n; k++)
         ev += sensor_events_packed(sensor_eval(a, k, Vm[k], a.apd ? vrest[k] : 0.0));
   }
   sensor_count(a.counts, ev);
}

// The end of a step of the host's loop in one pass: Simulate::checkRanges on
// Vm before the integrator (elec/simulationLoop.cc:214-217; CHECK), and the
// integrator (:221-227).  Bound by its 40 bytes a cell; passes of their own
// read 16 bytes a cell more and launched once more.  With iStim's zeroing only
// after a step that had a stimulus on, 1.06 million cells take 157 -> 151 us a
// step of the loop.
template <bool CHECK>
__global__ __launch_bounds__(256) void k_step_end_f64(int n, double dt, double *__restrict__ Vm,
                                                      const double *__restrict__ dVmR,
                                                      const double *__restrict__ dVmD,
                                                      const double *__restrict__ iStim,
                                                      double vmin, double vmax, int loop,
                                                      RangeRec *r)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   const bool in = i < n;
   double v = 0.0, dR = 0.0, dD = 0.0;
   if (in) {
      v = Vm[i];
      dR = dVmR[i];
      dD = dVmD[i];
      Vm[i] = v + dt * (dR + dD + iStim[i]);
   }
   if constexpr (CHECK) {
      const uint64_t m = __ballot(in && (v > vmax || v < vmin));
      if (m) range_report(r, m, threadIdx.x & 63, loop, i, v, dR, dD);
   }
}

template __global__ void k_step_end_f64<false>(int, double, double *, const double *,
                                               const double *, const double *, double, double, int,
                                               RangeRec *);
template __global__ void k_step_end_f64<true>(int, double, double *, const double *,
                                              const double *, const double *, double, double, int,
                                              RangeRec *);

}  // namespace cdh
