#pragma once

// Host side of the wave engine (kernels/coulomb_wave.h, CoulombPacked.hip): plans from configurations,
// and the launch.

#include "CoulombPackedPlan.h"
#include "CoulombRuntime.h"

namespace ktt
{

/** The plan of one shape; throws KttException for a shape the kernel does not take or that does
 *  not fit the LDS. */
PackedPlan MakePackedPlan(int px, int rows, int waves, int blocks, int atomCount, long rowLength, long rowsTotal, bool compensated);

/** The plan a configuration names: WAVE_SPLIT (waves), POINTS_X, ROWS_PER_THREAD and ATOM_BLOCKS, each
 *  optional but WAVE_SPLIT. */
PackedPlan PackedPlanOf(const CoulombConfig& config, int atomCount, long rowLength, long rowsTotal, bool compensated);

/** The compiled kernel of a plan (compiles at its first use). slice as for LaunchPacked. */
std::shared_ptr<HipKernel> GetPackedKernel(const PackedPlan& plan, bool compensated, bool slice);

/** energyGrid += V on rows of rowLength points. slice: rows = y and the atoms' z holds dz^2; else
 *  rows = z * rowLength + y of a cube. */
void LaunchPacked(const PackedPlan& plan, const float* atoms, int atomCount, float spacing, int rowLength, int rowsTotal,
    float* energyGrid, bool compensated, bool slice, hipStream_t stream, float* kernelMs);

} // namespace ktt
