#pragma once

// Host side of the wave engine (kernels/coulomb_wave.h, CoulombPacked.hip): the launch it makes for a
// grid and an atom count, and the choice among its shapes. Needs no device except to launch.

#include "CoulombRuntime.h"

namespace ktt
{

/** Launch of the wave engine: points per lane (px x rows), row groups a wave may touch, and the
 *  waves of a workgroup, which own the same 64 lanes and share the atoms. */
struct PackedPlan
{
    int px = 0;
    int rows = 0;
    int touched = 0;    // row groups a wave touches at most, and that rounded up to a power of two
    int cap = 0;
    int waves = 0;
    int blocks = 1;     // atom blocks (plain form; more than one add with FP32 atomics)
    int lanesX = 0;     // lanes per row group
    int rowGroups = 0;
    int share = 0;      // atoms per wave
    unsigned int workgroups = 0;
    unsigned int ldsBytes = 0;
};

/** The plan of one shape; throws KttException for a shape the kernel does not take or that does
 *  not fit the LDS. */
PackedPlan MakePackedPlan(int px, int rows, int waves, int blocks, int atomCount, long rowLength, long rowsTotal, bool compensated);

/** The shape with the smallest estimated time. */
PackedPlan ChoosePackedPlan(int atomCount, long rowLength, long rowsTotal, bool compensated);

/** The plan a configuration names: WAVE_SPLIT (waves), POINTS_X, ROWS_PER_THREAD and ATOM_BLOCKS, each
 *  optional but WAVE_SPLIT. */
PackedPlan PackedPlanOf(const CoulombConfig& config, int atomCount, long rowLength, long rowsTotal, bool compensated);

/** energyGrid += V on rows of rowLength points. slice: rows = y and the atoms' z holds dz^2; else
 *  rows = z * rowLength + y of a cube. */
void LaunchPacked(const PackedPlan& plan, const float* atoms, int atomCount, float spacing, int rowLength, int rowsTotal,
    float* energyGrid, bool compensated, bool slice, hipStream_t stream, float* kernelMs);

} // namespace ktt
