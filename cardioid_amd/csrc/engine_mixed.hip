// engine_mixed.hip -- the mixed-precision fused step over the engine's slabs
// (gfx950).
//
// Same step as engine_f64.hip with the storage and arithmetic of
// tt06_mixed.hpp and an FP32 stencil on voltage differences,
//    dVm_D = scale * sum_{k=1..18} A_k * (phi_k - phi_0),
// which is the FGR operator itself (its centre weight is minus the sum of
// the others, elec/FGRDiffusionOMP.cc:214-219) without the centre weight.
// The weights A_k are held compactly: a float per tile and neighbour plus
// an FP16 difference per cell (slab.cpp::compact_weights).
#pragma clang fp contract(fast)

#include <hip/hip_fp16.h>

#include "engine.hpp"
#include "engine_resident.hpp"
#include "tt06_mixed.hpp"

namespace cdh {

using namespace mixed;

namespace {

// ref + the low (or high) FP16 half of a word, in one v_fma_mix_f32 with the
// inline constant 1.0: exact sum, rounded once, so ref + (-ref) is exactly 0
__device__ __forceinline__ float half_lo_plus(uint32_t packed, float ref)
{
   float r;
   asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(packed), "s"(ref));
   return r;
}
__device__ __forceinline__ float half_hi_plus(uint32_t packed, float ref)
{
   float r;
   asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
       : "=v"(r)
       : "v"(packed), "s"(ref));
   return r;
}

__device__ __forceinline__ void cell_mixed(const EngineArgs &a, const SlabDev &S, int sl,
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
   // the cell's parameter set first: every later wait for it would also
   // wait for whatever was issued before it
   const ParamSet P = a.params[v.param_base + (int)(meta & 0xFFu)];
   __builtin_amdgcn_sched_barrier(0);
   const double V = box_load(R, b8, S.soff[0]);

   // states stream once per step (non-temporal), in the slab's runs of kRun
   // cells (run_index): the base addresses and the run width are wave-uniform
   // (buffer resources over the run's base, field s at SGPR offset
   // s * run width * field size, the lane's cell at VGPR offset)
   const int first = __builtin_amdgcn_readfirstlane(S.first_blk);
   const int64_t k0 = (int64_t)(blk - first) * kBlk;
   const int64_t r0 = k0 & ~(kRun - 1);
   const uint32_t rw =
       (uint32_t)run_width(k0, (int64_t)__builtin_amdgcn_readfirstlane(S.ntile) * kBlk);
   const int64_t c0 = (int64_t)first * kBlk + r0;
   const __amdgpu_buffer_rsrc_t R32 = stream_rsrc(a.st32 + c0 * N_STATE32);
   const __amdgpu_buffer_rsrc_t R64 = stream_rsrc(a.st64 + c0 * N_STATE64);
   const uint32_t lc = (uint32_t)(k0 - r0 + lane);
   float s32[N_STATE32];
#pragma unroll
   for (int s = 0; s < N_STATE32; s++) s32[s] = stream_load_f32(R32, 4u * lc, 4u * rw * s);
   double s64[N_STATE64];
#pragma unroll
   for (int s = 0; s < N_STATE64; s++) s64[s] = stream_load_f64(R64, 8u * lc, 8u * rw * s);
   __builtin_amdgcn_sched_barrier(0);
   // then the stencil's weights and neighbours: loads return in issue order,
   // so the reaction waits for the states only and the stencil's loads land
   // under its arithmetic; the sum comes after the reaction
   // the weight words in three loads (grp_index9): two of 16 and one of 4
   // bytes per lane (0.932 against 0.941 ms per step on the 20.1 M-cell
   // shell with one load per word, bit for bit the same)
   const uint32_t *wp = a.Aw16 + (int64_t)blk * (9 * kBlk);
   uint32_t hw[9];
   double nb[18];
#pragma unroll
   for (int g = 0; g < 2; g++) {
      const u32x4 q = __builtin_nontemporal_load((const u32x4 *)(wp + g * 4 * kBlk) + lane);
      hw[4 * g] = q.x;
      hw[4 * g + 1] = q.y;
      hw[4 * g + 2] = q.z;
      hw[4 * g + 3] = q.w;
   }
   hw[8] = __builtin_nontemporal_load(wp + 8 * kBlk + lane);
#pragma unroll
   for (int k = 0; k < 18; k++) nb[k] = box_load(R, b8, S.soff[k + 1]);
   __builtin_amdgcn_sched_barrier(0);

   const double K_i = P.K0 + (double)s32[M_DK_I];
   double iK;
   double dVR = 0.0;
   iK = 0.0;
   if (a.gate_mask & (1u << 12)) dVR = nongateM(*a.K, P, a.coef, a.dt, V, K_i, s32, s64, &iK);
   gatesM(a.coef, a.K->exp_coef, P.s_switch, (uint8_t)(meta >> 8), V, s32, a.gate_mask);

   // the stencil: weight (in units of 2^-wexp) = the tile's reference
   // (wave-uniform, scalar loads) plus the cell's FP16 difference, exact zero
   // for a zero weight; the unit goes into the diffusion scale
   const float *ref = a.Aref + (int64_t)blk * 18;
   float acc = 0.0f;
#pragma unroll
   for (int p = 0; p < 9; p++) {
      const float w0 = half_lo_plus(hw[p], ref[2 * p]);
      const float w1 = half_hi_plus(hw[p], ref[2 * p + 1]);
      acc = __builtin_fmaf(w0, (float)(nb[2 * p] - V), acc);
      acc = __builtin_fmaf(w1, (float)(nb[2 * p + 1] - V), acc);
   }
   const double dVD = (double)acc * (v.scale * (double)S.wdelta_scale);

   engine_range(a, S, v, sl, a.parity, live, lane, i, V, dVR, dVD);
   const double iStim = slab_stim(S, v, a.parity, meta);
   const double Vn = V + a.dt * (dVR + dVD + iStim);
   // K_i follows dVK_i = K_i/c9 + Vm of the reference: dK_i = c9*dt*(iK - dVm_D - iStim)
   s32[M_DK_I] = (float)((double)s32[M_DK_I] + (a.dt * a.K->c9) * (iK - dVD - iStim));
#pragma unroll
   for (int s = 0; s < N_STATE32; s++) stream_store_f32(s32[s], R32, 4u * lc, 4u * rw * s);
#pragma unroll
   for (int s = 0; s < N_STATE64; s++) stream_store_f64(s64[s], R64, 8u * lc, 8u * rw * s);
   uint32_t ev = 0;
   if (live) {
      a.box_next[b] = Vn;
      if (a.sensors) ev = engine_sensors(a, v, i, V, Vn, P.Vm0);
   }
   // every lane of the tile is here (padding lanes with no events)
   if (a.sensors & 1) sensor_count(a.counts + 4 * sl, ev);
}

}  // namespace

// Tile-to-XCD mapping as k_engine_f64.
template <int WAVES>
__global__ __launch_bounds__(256, WAVES) void k_engine_mixed(EngineArgs a)
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
   cell_mixed(a, S, sl, v, blk, lane);
   if (blk == S.first_blk && lane == 0) slab_advance(S, a.parity, v);
}

template __global__ void k_engine_mixed<3>(EngineArgs);
template __global__ void k_engine_mixed<4>(EngineArgs);

// ---- resident form (engine_resident.hpp)

namespace {

// PARK: the weights and the gates wait in LDS from one use to the next, 5.25 KB
// to a tile (6.25 as it is allocated, so that 24 of 25 that a CU has room for
// are used), for six wavefronts per SIMD (80 VGPRs); else all is in registers,
// for four.  Up to 6,144 tiles instead of 4,096: us a step by step kernels and
// this, 287,496 cells 21.2 and 12.0, 373,248 cells 24.9 and 14.2, 389,017 cells
// 26.3 and 14.1.
template <bool PARK>
struct ResidentMixed {
   struct Shared {
      uint32_t w[9][kBlk];
      float gate[12][kBlk];
   };
   float s32[N_STATE32];
   double s64[N_STATE64];
   uint32_t hw[9];
   Shared *sh;
   template <class G>
   __device__ __forceinline__ void fetch(G, int lane)
   {
      if constexpr (PARK) s32[M_M + G::value] = sh->gate[G::value][lane];
   }
   template <class G>
   __device__ __forceinline__ void park(G, int lane)
   {
      if constexpr (PARK) sh->gate[G::value][lane] = s32[M_M + G::value];
   }
   __amdgpu_buffer_rsrc_t R32, R64;
   const float CDH_CONSTANT *ref;
   float wscale;
   uint32_t lc, rw;
   double iK;

   __device__ __forceinline__ void load(const EngineArgs &a, const ResidentTile &t, Shared *shared)
   {
      sh = shared;
      rw = t.rw;
      lc = t.lc;
      R32 = stream_rsrc(a.st32 + t.run_cell * N_STATE32);
      R64 = stream_rsrc(a.st64 + t.run_cell * N_STATE64);
#pragma unroll
      for (int s = 0; s < N_STATE32; s++) s32[s] = stream_load_f32(R32, 4u * lc, 4u * rw * s);
#pragma unroll
      for (int s = 0; s < N_STATE64; s++) s64[s] = stream_load_f64(R64, 8u * lc, 8u * rw * s);
      const uint32_t *wp = a.Aw16 + (int64_t)t.blk * (9 * kBlk);
#pragma unroll
      for (int g = 0; g < 2; g++) {
         const u32x4 q = *((const u32x4 *)(wp + g * 4 * kBlk) + t.lane);
         hw[4 * g] = q.x;
         hw[4 * g + 1] = q.y;
         hw[4 * g + 2] = q.z;
         hw[4 * g + 3] = q.w;
      }
      hw[8] = wp[8 * kBlk + t.lane];
      if constexpr (PARK) {
#pragma unroll
         for (int g = 0; g < 9; g++) sh->w[g][t.lane] = hw[g];
      }
      each_gate([&](auto g) { park(g, t.lane); });
      ref = (const float CDH_CONSTANT *)(a.Aref + (int64_t)t.blk * 18);
      wscale = t.S->wdelta_scale;
   }
   __device__ __forceinline__ void store(const ResidentTile &t)
   {
      each_gate([&](auto g) { fetch(g, t.lane); });
#pragma unroll
      for (int s = 0; s < N_STATE32; s++) stream_store_f32(s32[s], R32, 4u * lc, 4u * rw * s);
#pragma unroll
      for (int s = 0; s < N_STATE64; s++) stream_store_f64(s64[s], R64, 8u * lc, 8u * rw * s);
   }
   __device__ __forceinline__ double react(const EngineArgs &a, const ModelTables &T,
                                           const ParamSet &P, const ResidentTile &t, double V)
   {
      const double K_i = P.K0 + (double)s32[M_DK_I];
      double dVR = 0.0;
      iK = 0.0;
      each_gate([&](auto g) { fetch(g, t.lane); });
      if (a.gate_mask & (1u << 12)) dVR = nongateM(*T.K, P, T.coef, a.dt, V, K_i, s32, s64, &iK);
      auto gates = [&](uint32_t mask) {
         gatesM(T.coef, T.K->exp_coef, P.s_switch, (uint8_t)(t.meta >> 8), V, s32, mask);
      };
      if constexpr (!PARK) {
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
   // the sums of cell_mixed, in its order
   __device__ __forceinline__ double diffuse(const ResidentTile &t, __amdgpu_buffer_rsrc_t R, double V,
                                             double scale)
   {
      double nb[18];
#pragma unroll
      for (int k = 0; k < 18; k++) nb[k] = t.neighbour(R, k + 1);
      __builtin_amdgcn_sched_barrier(0);   // all loads in flight before the first sum
      float acc = 0.0f;
#pragma unroll
      for (int p = 0; p < 9; p++) {
         const uint32_t h = PARK ? sh->w[p][t.lane] : hw[p];
         const float w0 = half_lo_plus(h, ref[2 * p]);
         const float w1 = half_hi_plus(h, ref[2 * p + 1]);
         acc = __builtin_fmaf(w0, (float)(nb[2 * p] - V), acc);
         acc = __builtin_fmaf(w1, (float)(nb[2 * p + 1] - V), acc);
      }
      return (double)acc * (scale * (double)wscale);
   }
   __device__ __forceinline__ void finish(const EngineArgs &a, const ModelTables &T, double dVD,
                                          double iStim)
   {
      s32[M_DK_I] = (float)((double)s32[M_DK_I] + (a.dt * T.K->c9) * (iK - dVD - iStim));
   }
};

// One wavefront's part of a cell for resident_split_run (SplitF64 in
// engine_f64.hip).
struct SplitMixed {
   struct Shared : SplitShared<float, uint32_t, 9> {
      double CaL_b[kBlk];      // I_CaL's second factor (its first is in I_CaL)
   };
   float s32[N_STATE32];
   double s64[N_STATE64];
   __amdgpu_buffer_rsrc_t R32, R64;
   const float CDH_CONSTANT *ref;
   SodiumPotassiumCurrents nk;
   double I_NaCa;

   __device__ __forceinline__ void states(const EngineArgs &a, const ResidentTile &t)
   {
      R32 = stream_rsrc(a.st32 + t.run_cell * N_STATE32);
      R64 = stream_rsrc(a.st64 + t.run_cell * N_STATE64);
   }
   __device__ __forceinline__ void load32(const ResidentTile &t, int q)
   {
      s32[q] = stream_load_f32(R32, 4u * t.lc, 4u * t.rw * q);
   }
   __device__ __forceinline__ void store32(const ResidentTile &t, int q)
   {
      stream_store_f32(s32[q], R32, 4u * t.lc, 4u * t.rw * q);
   }
   __device__ __forceinline__ void load64(const ResidentTile &t, int q)
   {
      s64[q] = stream_load_f64(R64, 8u * t.lc, 8u * t.rw * q);
   }
   __device__ __forceinline__ void store64(const ResidentTile &t, int q)
   {
      stream_store_f64(s64[q], R64, 8u * t.lc, 8u * t.rw * q);
   }

   __device__ __forceinline__ void load_na_k(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
      load32(t, M_DK_I);
      load64(t, M_NA_I);
   }
   __device__ __forceinline__ void store_na_k(const ResidentTile &t)
   {
      store32(t, M_DK_I);
      store64(t, M_NA_I);
   }
   __device__ __forceinline__ void share_na(Shared *sh, int p, int lane)
   {
      sh->na[p][lane] = s64[M_NA_I];
   }
   __device__ __forceinline__ void load_ca(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
      for (int q : {M_CA_SS, M_CA_SR, M_R_PRIME, M_FCASS}) load32(t, q);
      load64(t, M_CA_I);
   }
   __device__ __forceinline__ void store_ca(const ResidentTile &t)
   {
      for (int q : {M_CA_SS, M_CA_SR, M_R_PRIME, M_FCASS}) store32(t, q);
      store64(t, M_CA_I);
   }
   __device__ __forceinline__ void share_ca(Shared *sh, int p, int lane)
   {
      sh->ca[p][lane] = s64[M_CA_I];
   }
   // gate g (from 0, the order of S_M .. S_S) is slot M_M + g
   template <uint32_t GATES>
   __device__ __forceinline__ void load_gates(const EngineArgs &a, const ResidentTile &t)
   {
      states(a, t);
#pragma unroll
      for (int g = 0; g < 12; g++)
         if ((GATES >> g) & 1) load32(t, M_M + g);
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void store_gates(const ResidentTile &t)
   {
#pragma unroll
      for (int g = 0; g < 12; g++)
         if ((GATES >> g) & 1) store32(t, M_M + g);
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void share_gates(Shared *sh, int p, int lane)
   {
#pragma unroll
      for (int g = 0; g < 12; g++)
         if ((GATES >> g) & 1) sh->gate[p][g][lane] = s32[M_M + g];
   }
   template <uint32_t GATES>
   __device__ __forceinline__ void take_gates(const Shared *sh, int p, int lane)
   {
#pragma unroll
      for (int g = 0; g < 12; g++)
         if ((GATES >> g) & 1) s32[M_M + g] = sh->gate[p][g][lane];
   }
   __device__ __forceinline__ void na_k(const EngineArgs &, const ModelTables &T, const ParamSet &P,
                                        double V, const Shared *sh, int p, int lane)
   {
      take_gates<kGatesNaK>(sh, p, lane);
      const double fv0 = fitM<0>(T.coef, V), fv1 = fitM<1>(T.coef, V), fv2 = fitM<2>(T.coef, V);
      const double fv5 = fitM<5>(T.coef, V);
      I_NaCa = exchangerM(s64[M_NA_I], sh->ca[p][lane], fv1, fv2);
      nk = na_kM(*T.K, P, T.coef, V, P.K0 + (double)s32[M_DK_I], fv0, fv5, I_NaCa, s32, s64);
   }
   __device__ __forceinline__ void calcium(const EngineArgs &a, const ModelTables &T,
                                           const ParamSet &P, double V, Shared *sh, int p, int lane)
   {
      take_gates<kGatesCa>(sh, p, lane);
      const double fv1 = fitM<1>(T.coef, V), fv2 = fitM<2>(T.coef, V);
      const double fv3 = fitM<3>(T.coef, V), fv4 = fitM<4>(T.coef, V);
      const double I = exchangerM(sh->na[p][lane], s64[M_CA_I], fv1, fv2);
      const CalciumCurrentsM ca = calciumM(*T.K, P, a.dt, V, fv3, fv4, I, s32, s64);
      sh->I_sum[lane] = ca.I_sum;
      sh->I_CaL[lane] = ca.CaL_a;
      sh->CaL_b[lane] = ca.CaL_b;
   }
   __device__ __forceinline__ double sum(const EngineArgs &a, const ModelTables &T,
                                         const Shared *sh, int lane)
   {
      return sumM(*T.K, a.dt, I_NaCa,
                  CalciumCurrentsM{sh->I_sum[lane], sh->I_CaL[lane], sh->CaL_b[lane]}, nk, s64);
   }
   __device__ __forceinline__ void finish(const EngineArgs &a, const ModelTables &T, double dVD,
                                          double iStim)
   {
      s32[M_DK_I] = (float)((double)s32[M_DK_I] + (a.dt * T.K->c9) * (nk.iK - dVD - iStim));
   }
   __device__ __forceinline__ void gates(const EngineArgs &, const ModelTables &T, int s_switch,
                                         uint32_t meta, double V, uint32_t mask)
   {
      gatesM(T.coef, T.K->exp_coef, s_switch, (uint8_t)(meta >> 8), V, s32, mask);
   }
   __device__ __forceinline__ void load_weights(const EngineArgs &a, const ResidentTile &t,
                                                Shared *sh)
   {
      const uint32_t *wp = a.Aw16 + (int64_t)t.blk * (9 * kBlk);
#pragma unroll
      for (int g = 0; g < 2; g++) {
         const u32x4 q = *((const u32x4 *)(wp + g * 4 * kBlk) + t.lane);
         sh->w[4 * g][t.lane] = q.x;
         sh->w[4 * g + 1][t.lane] = q.y;
         sh->w[4 * g + 2][t.lane] = q.z;
         sh->w[4 * g + 3][t.lane] = q.w;
      }
      sh->w[8][t.lane] = wp[8 * kBlk + t.lane];
      ref = (const float CDH_CONSTANT *)(a.Aref + (int64_t)t.blk * 18);
   }
   __device__ __forceinline__ double diffuse(const ResidentTile &t, __amdgpu_buffer_rsrc_t R,
                                             double V, double scale, const Shared *sh)
   {
      double nb[18];
#pragma unroll
      for (int k = 0; k < 18; k++) nb[k] = t.neighbour(R, k + 1);
      __builtin_amdgcn_sched_barrier(0);
      float acc = 0.0f;
#pragma unroll
      for (int p = 0; p < 9; p++) {
         const uint32_t hw = sh->w[p][t.lane];
         const float w0 = half_lo_plus(hw, ref[2 * p]);
         const float w1 = half_hi_plus(hw, ref[2 * p + 1]);
         acc = __builtin_fmaf(w0, (float)(nb[2 * p] - V), acc);
         acc = __builtin_fmaf(w1, (float)(nb[2 * p + 1] - V), acc);
      }
      return (double)acc * (scale * (double)t.S->wdelta_scale);
   }
};

}  // namespace

template <int WAVES>
__global__ __launch_bounds__(64, WAVES) void k_resident_mixed(EngineArgs a, ResidentArgs r)
{
   using C = ResidentMixed<(WAVES > 4)>;
   if constexpr (WAVES > 4) {
      __shared__ typename C::Shared sh;
      resident_run<C>(a, r, &sh);
   } else {
      resident_run<C>(a, r, nullptr);
   }
}

template __global__ void k_resident_mixed<4>(EngineArgs, ResidentArgs);
template __global__ void k_resident_mixed<6>(EngineArgs, ResidentArgs);

__global__ __launch_bounds__(kSplitWaves * 64, 8) void k_resident_split_mixed(EngineArgs a,
                                                                              ResidentArgs r)
{
   __shared__ SplitMixed::Shared sh;
   resident_split_run<SplitMixed>(a, r, &sh);
}

}  // namespace cdh
