// dpm_launch.h -- launchers of the kernels compiled per (interaction, potential): each instance is
// an explicit specialisation in a translation unit of its own (dpm_step.hip, dpm_fire.hip), so
// that the instances compile side by side.
#pragma once

#include "dpm_internal.h"

namespace dpm {

static inline int grid_v(long n) { return (int)((n + 255) / 256); }
static inline int grid_w(int ntiles) { return (ntiles + 3) / 4; }

// Waves per tile of the loops where the caller set none: 8 while two workgroups a CU, all that registers
// leave room for, hold the set (32 to 1,024 rings: 2 to 5% faster than 4 where a step waits for a rebuild or
// the tile's longest wave; without rebuilds the same, 459 tiles 7.2 us a vertex-vertex step with either), 4
// beyond (590 tiles 7.1 us against 11.1 with 8; vertex-segment 8.1 against 12.3).
static inline int loop_waves(const dpm_set_s* S) { return S->splitSet ? S->split : (S->V.ntiles <= 512 ? 8 : 4); }

// the step kernel of MODE bits `mode` on every tile of the set
template <int INTER, int POT>
hipError_t step_launch(dpm_set_s* S, int mode, const StepArgs& A);

// `chunk` iterations of the persistent FIRE kernel on every system, `threads` per workgroup
template <int INTER, int POT>
hipError_t fire_launch(dpm_set_s* S, int chunk, int threads);

#define DPM_FOR_POTENTIALS(DECL, INTER) \
  DECL(INTER, POT_HARMONIC) DECL(INTER, POT_LJ) DECL(INTER, POT_ADHESIVE) DECL(INTER, POT_WCA)
#define DPM_DECLARE_LAUNCH(INTER, POT)                                             \
  template <>                                                                      \
  hipError_t step_launch<INTER, POT>(dpm_set_s * S, int mode, const StepArgs& A);  \
  template <>                                                                      \
  hipError_t fire_launch<INTER, POT>(dpm_set_s * S, int chunk, int threads);
DPM_FOR_POTENTIALS(DPM_DECLARE_LAUNCH, INT_VV)
DPM_FOR_POTENTIALS(DPM_DECLARE_LAUNCH, INT_SMOOTH)
DPM_FOR_POTENTIALS(DPM_DECLARE_LAUNCH, INT_ALL)

}  // namespace dpm
