// shim.hip -- the library's C++ parts that no C entry point shows, for the
// tests (native.py).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <vector>

#include "engine_host.hpp"
#include "engine_resident.hpp"
#include "host/simulate.hpp"
#include "resident_rules.hpp"

using namespace cdh;

namespace cdh {
struct EngineProbe {
   static void set_wait(Engine &e, uint32_t polls) { e.max_polls_ = polls; }
   // Has the first tile wait for one that the engine does not have, whose flag
   // nobody advances; the kernels' bounded wait then passes its bound.
   static void wait_for_nobody(Engine &e)
   {
      e.sync();
      CDH_REQUIRE(!e.links_dirty_ && e.nlist_ + 1 < e.resident_tiles_, "no resident run yet");
      const uint32_t far = (uint32_t)e.resident_tiles_ - 1;
      const uint32_t link[2] = {far, far + 1};
      e.flags_.upload(&e.epoch_, 1, kFlagStride * (size_t)far);
      e.flags_.upload(link, 2, kFlagStride * (size_t)e.resident_tiles_ + 4);
      CDH_HIP(hipDeviceSynchronize());
   }
};
}  // namespace cdh

namespace {

// a row of n cells along x with one cell type and no conduction to speak of,
// stimulated in its first `nstim` cells; the exact functions, so no fits
std::unique_ptr<host::Simulate> row_simulation(int n, int nstim, const cdh_box_stim &pulse)
{
   auto sim = std::make_unique<host::Simulate>(nullptr);
   sim->dt = 0.02;
   sim->nLocal = n;
   for (DevBuf<double> *b : {&sim->Vm, &sim->iStim, &sim->dVmReaction, &sim->dVmDiffusion}) {
      b->alloc(n);
      b->zero();
   }
   sim->range.alloc(1);
   sim->range.zero();
   cdh_tt06_params tp{};
   tp.dt = sim->dt;
   tp.mod = 1;
   if (cdh_celltype_standard("endoCellML", &tp.celltype) != CDH_OK) throw std::runtime_error("cell type");
   tp.s_kr = tp.s_cal = tp.s_na = 1.0;
   std::vector<int> cells(n), tissue(n, 1);
   std::vector<int64_t> gid(n);
   std::vector<double> sigma(6 * (size_t)n, 0.0);
   for (int k = 0; k < n; k++) {
      cells[k] = k;
      gid[k] = k;
      sigma[6 * k] = sigma[6 * k + 3] = sigma[6 * k + 5] = 1e-4;
   }
   sim->reaction = std::make_unique<host::ReactionManager>();
   sim->reaction->addReaction(host::reactionFactory("TT06Dev", tp, n, nullptr), cells);
   sim->reaction->initializeMembraneVoltage(sim->Vm.p);
   cdh_fgr_params fp{};
   fp.nx = n;
   fp.ny = fp.nz = 1;
   fp.dx = fp.dy = fp.dz = 0.2;
   fp.diffusionScale = 1.0;
   fp.nLocal = n;
   fp.gid = gid.data();
   fp.cellType = tissue.data();
   fp.sigma = sigma.data();
   sim->diffusion = host::diffusionFactory("FGR", fp, nullptr);
   cells.resize(nstim);
   sim->stimulus.push_back(std::make_unique<host::BoxStimulus>(pulse, cells, nullptr));
   return sim;
}

}  // namespace

extern "C" {

// iStim after each of `ncall` calls of simulationLoop of steps[k] steps, in
// out[ncall][n]; before each call every cell of it is set to `before`.
int shim_loop_istim(int n, int nstim, double t0, double duration, double amplitude, int ncall,
                    const int *steps, double before, double *out)
{
   try {
      cdh_box_stim pulse{};
      pulse.t0 = -1.0;
      pulse.tf = 1e9;
      pulse.period = 1000.0;
      pulse.phase = t0;
      pulse.duration = duration;
      pulse.amplitude = amplitude;
      auto sim = row_simulation(n, nstim, pulse);
      const std::vector<double> set(n, before);
      for (int k = 0; k < ncall; k++) {
         sim->iStim.upload(set.data(), n);
         host::simulationLoop(*sim, steps[k]);
         CDH_HIP(hipDeviceSynchronize());
         sim->iStim.download(out + (size_t)k * n, n);
      }
   } catch (const std::exception &e) {
      set_last_error(e.what());
      return 1;
   }
   return 0;
}

// the batch's resident runs time out after `polls`, in a wait that nothing ends
int shim_resident_stuck(cdh_batch *b, unsigned polls)
{
   return guard([&] {
      EngineProbe::set_wait(batch_engine(b), polls);
      EngineProbe::wait_for_nobody(batch_engine(b));
   });
}

// the three ranges of each tile of a slab with cells at box points bi[ncell],
// out[tiles][3][2]
void shim_tile_ranges(int64_t ncell, const int64_t *bi, int64_t plane, int64_t row, int *out)
{
   const int ntile = (int)((ncell + kBlk - 1) / kBlk);
   for (int64_t t = 0; t < ntile; t++)
      for (int part = 0; part < 3; part++) {
         const TileRange r =
             tile_range(part, bi[kBlk * t], bi[std::min<int64_t>(kBlk * t + kBlk, ncell) - 1], plane,
                        row, ntile, [&](int m) { return bi[(int64_t)kBlk * m]; });
         out[6 * t + 2 * part] = r.begin;
         out[6 * t + 2 * part + 1] = r.end;
      }
}

int shim_resident_refused(int error) { return resident_refused((hipError_t)error); }

}  // extern "C"
