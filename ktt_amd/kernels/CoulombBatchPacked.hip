// Batched direct Coulomb summation on the wave engine (coulomb_wave.h): one workgroup per 64 packed
// lanes of one system (32 at sides 6 and 7), in the compensated form. The default of ktt_coulomb_batch_run; CoulombBatched.hip
// keeps the tile-shape buckets that a configuration or the autotuner sets.
//
// Work items (system, block of lanes) are listed by the host, systems with the most atoms first, and
// workgroups start in that order, so that the items of large systems do not end last. (By atoms alone: an item of a
// small grid holds fewer points per lane. Ordering by atoms times points per lane takes the same time on twelve
// mixed batches, 27.96 against 27.97 ms on the one with 7s below.) The waves of a workgroup
// split the system's atoms. Lanes are packed within each system, so a side of any size wastes at most its
// last wave, and one block serves all sides of a class: 2 x 8 points per lane from 64 points up, 1 x 8 from
// 32, 1 x 4 below. From side 21 up that keeps a wave to 3 or 4 row groups and its LDS to 8 KiB; smaller sides
// touch up to 8 groups of 4 rows, 10 KiB. One LDS size holds for the whole launch, so one small system sets
// how many waves every system has: at 10 KiB 16 per CU instead of 19 or 20, which costs under 1% (128
// systems of sides 48 to 128 and 5, 16 or 32: 27.9, 28.0 and 28.3 ms). 64 lanes at sides 6 and 7 would touch 9
// and 10 groups, 18 KiB, 8 waves per CU: with 7s that batch took 33.1 ms, on 32 lanes 28.0 (buckets 28.2).
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
__device__ __forceinline__ void sumBlock(float* shared, const float4* atoms, const BatchSystem& system, const int block, const int lanes, float* grids)
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
        engine.place(block, (G + PX - 1) / PX, (G * G + ROWS - 1) / ROWS, lanes);
        engine.accumulate(shared + wave * W::WaveFloats, atoms + system.atomOffset, a0, a1, system.spacing, G);
        engine.store(shared, waves, wave, grids + system.gridOffset, G, G * G, false);
    }
}

} // namespace

// items: int4 (system, block, lanes per block, 0).
extern "C" __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5))) void coulombBatchPacked(const float4* atoms,
    const BatchSystem* systems, const int4* items, float* grids)
{
    extern __shared__ __attribute__((aligned(16))) float shared[];
    const int4 work = items[blockIdx.x];
    const BatchSystem system = systems[work.x];
    if (system.gridSize >= 64)
    {
        sumBlock<2, 8, CAP_WIDE>(shared, atoms, system, work.y, 64, grids);
    }
    else if (system.gridSize >= 32)
    {
        sumBlock<1, 8, CAP_NARROW>(shared, atoms, system, work.y, 64, grids);
    }
    else
    {
        sumBlock<1, 4, CAP_SMALL>(shared, atoms, system, work.y, work.z, grids);
    }
}
