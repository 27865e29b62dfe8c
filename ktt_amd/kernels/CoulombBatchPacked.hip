// Batched direct Coulomb summation on the wave engine (coulomb_wave.h): one workgroup per 64 packed
// lanes of one system, in the compensated form. The default of ktt_coulomb_batch_run; CoulombBatched.hip
// keeps the tile-shape buckets that a configuration or the autotuner sets.
//
// Work items (system, 64-lane block) are listed by the host, systems with the most atoms first, and
// workgroups start in that order, so that the long items do not end last. The waves of a workgroup
// split the system's atoms. Lanes are packed within each system, so a side of any size wastes at most its
// last wave, and one block serves all sides of a class: 2 x 8 points per lane from 64 points up, 1 x 8 from
// 32, 1 x 4 below, which keeps a wave to 3 or 4 row groups and its brackets to 8 KiB of LDS.
//
//   CAP_WIDE, CAP_NARROW, CAP_SMALL  most row groups a wave touches in each class (0: no such system)
//
// Bound by FP32 VALU issue as the other kernels. Measured on MI355X against the buckets' default shapes,
// which were tuned for the first batch: 1,024 systems of sides 32, 48, 64, 96 and 128 252.6 -> 246.5 ms (122
// TFLOP/s at 11 per interaction), 100 of 128^3 92.4 -> 74.0, 78 of 52, 53 and 110 18.6 -> 14.7, 64 of
// 113 17.1 -> 12.4, 40 of 24 1.34 -> 0.31.
#include "coulomb_wave.h"

#ifndef CAP_WIDE
#define CAP_WIDE 3
#endif
#ifndef CAP_NARROW
#define CAP_NARROW 4
#endif
#ifndef CAP_SMALL
#define CAP_SMALL 4
#endif

// One system of the batch (32 bytes; the host writes the same layout).
struct BatchSystem
{
    int atomOffset;
    int atomCount;
    int gridSize;
    int bucket;
    float spacing;
    int reserved;
    long long gridOffset;
};

namespace
{

template <int PX, int ROWS, int CAP>
__device__ __forceinline__ void sumBlock(float* shared, const float4* atoms, const BatchSystem& system, const int block, float* grids)
{
    if constexpr (CAP > 0)
    {
        using W = kc::WaveEngine<PX, ROWS, CAP, kc::Volume, true>;
        const int G = system.gridSize;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int waves = blockDim.x >> 6;
        // Whole unrolled steps of 8 atoms per wave.
        const unsigned int share = (static_cast<unsigned int>(system.atomCount) + 8u * waves - 1u) / (8u * waves) * 8u;
        const unsigned int count = static_cast<unsigned int>(system.atomCount);
        const unsigned long long first = static_cast<unsigned long long>(wave) * share;
        const unsigned int a0 = first < count ? static_cast<unsigned int>(first) : count;
        const unsigned int a1 = share < count - a0 ? a0 + share : count;
        W engine;
        engine.place(block, (G + PX - 1) / PX, (G * G + ROWS - 1) / ROWS);
        engine.accumulate(shared + wave * W::WaveFloats, atoms + system.atomOffset, a0, a1, system.spacing, G);
        engine.store(shared, waves, wave, grids + system.gridOffset, G, G * G, false);
    }
}

} // namespace

// items: int4 (system, 64-lane block, 0, 0).
extern "C" __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5))) void coulombBatchPacked(const float4* atoms,
    const BatchSystem* systems, const int4* items, float* grids)
{
    extern __shared__ __attribute__((aligned(16))) float shared[];
    const int4 work = items[blockIdx.x];
    const BatchSystem system = systems[work.x];
    if (system.gridSize >= 64)
    {
        sumBlock<2, 8, CAP_WIDE>(shared, atoms, system, work.y, grids);
    }
    else if (system.gridSize >= 32)
    {
        sumBlock<1, 8, CAP_NARROW>(shared, atoms, system, work.y, grids);
    }
    else
    {
        sumBlock<1, 4, CAP_SMALL>(shared, atoms, system, work.y, grids);
    }
}
