// Launches of the mixed form's kernels (FP32 flux evaluation, FP64 RK
// registers), defined in mixed.hip (single domain) and mixed_ensemble.hip
// (ensembles).  Those translation units alone instantiate the FP32 kernels:
// they allow contraction into FMA within an expression, under one pragma,
// while the FP64 kernels keep the reference's operation order, so a
// mixed-form ensemble member still advances bit-for-bit as it would alone.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_ensemble.hpp"

namespace mhd {

// Resident blocks of a variant (stream_resident; MHD or hydro, with rotation).
int mixed_stream_resident(bool mag, int waves, int sched);

// One stage (launch_stream_stage<float, ...>).
void mixed_stage(bool mag, bool rot, int stage, const StageArgs& a, hipStream_t s, int waves,
                 int sched, int target_blocks, int walls, const StepEnds& e);

// Wall planes of one stage (stage_wall_kernel<float, ...>; full: every flux, see wall_point).
void mixed_wall(bool mag, bool rot, int stage, bool full, const StageArgs& a, const StepEnds& e, dim3 grid,
                dim3 block, hipStream_t s);

// Host stub of the ensemble's interior stage-2 kernel of the given variant.
const void* mixed_ens_stage_fn(int waves, int sched);

// One ensemble stage: the persistent interior launch over `items` (grid_int
// blocks) and the persistent wall launch over `walls` (grid_wall blocks); an
// empty list launches nothing.
void mixed_ens_stage(int stage, int waves, int sched, const StageArgs* args, const WorkItem* items,
                     int nitems, int grid_int, const WallItem* walls, int nwalls, int grid_wall,
                     bool full_walls, hipStream_t s);

}  // namespace mhd
