// CoulombSum3d and CoulombSum2d for gfx950 on the wave engine (coulomb_wave.h): any row length fills
// the lanes, and the waves of a workgroup split the atoms. Semantics as CoulombSum3d.hip and
// CoulombSum2d.hip: index z*G*G + y*G + x, coordinates h * index, "+=" store
// (Examples/CoulombSum3d/CoulombSum3d.cu:10-15, :46; Examples/CoulombSum2d/CoulombSum2d.cl:126, :945).
//
//   POINTS_X, ROWS_PER_THREAD  points per lane (x run, rows)
//   ROW_GROUP_CAP              row groups a wave may touch (RowGroupCap in CoulombPackedPlan.h)
//   COMPENSATED                sums of 64 atoms added in 0: FP32, 1: FP64
//   WAVE_LANES                 lanes a wave takes (LanesPerWave in CoulombPackedPlan.h)
//   ROW_MODE                   0: a volume (rows = z * G + y), 1: one slice (rows = y, .z holds dz^2)
//
// Launch: kc::packedSum. Several atom blocks (plain form only) add to the grid with FP32 atomics.
#include "coulomb_wave.h"

#ifndef ROW_GROUP_CAP
#define ROW_GROUP_CAP 2
#endif
#ifndef COMPENSATED
#define COMPENSATED 0
#endif
#ifndef WAVE_LANES
#define WAVE_LANES 64
#endif
#ifndef ROW_MODE
#define ROW_MODE 0
#endif

using W = kc::WaveEngine<POINTS_X, ROWS_PER_THREAD, ROW_GROUP_CAP, ROW_MODE, COMPENSATED != 0>;

// 5 waves per SIMD: the compensated 2 x 8 block takes exactly the 96 VGPRs that they allow.
extern "C" __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5))) void coulombPacked(const float4* atoms, int numberOfAtoms, int share, float gridSpacing,
    int lanesX, int rowGroups, int rowLength, int rowsTotal, float* energyGrid)
{
    extern __shared__ __attribute__((aligned(16))) float shared[];
    kc::packedSum<W, WAVE_LANES>(shared, atoms, numberOfAtoms, share, gridSpacing, lanesX, rowGroups, rowLength, rowsTotal, energyGrid);
}
