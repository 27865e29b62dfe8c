#pragma once

// The launch the wave engine (kernels/coulomb_wave.h) makes for a grid and an atom count, and the
// choice among its shapes, for the hipRTC launches (CoulombPacked.cpp) and the precompiled ones
// (noalloc/CoulombNoAlloc.hip). Needs no device.

#include <algorithm>
#include <cmath>
#include <limits>

namespace ktt
{

/** Launch of the wave engine: points per lane (px x rows), row groups a wave may touch, and the
 *  waves of a workgroup, which own the same 64 lanes and share the atoms. */
struct PackedPlan
{
    int px = 0;
    int rows = 0;
    int lanes = 64;     // lanes a wave takes
    int touched = 0;    // row groups a wave touches at most, and what the kernel is compiled for
    int cap = 0;
    int waves = 0;
    int blocks = 1;     // atom blocks (plain form; more than one add with FP32 atomics)
    int lanesX = 0;     // lanes per row group
    int rowGroups = 0;
    int share = 0;      // atoms per wave
    unsigned int workgroups = 0;
    unsigned int ldsBytes = 0;
};

// LDS of a workgroup on gfx950.
constexpr long kPackedLdsBytes = 160 * 1024;

// Row groups a wave of `lanes` lanes touches at most when a row group has lanesX lanes, of those there are.
inline int RowGroupsPerWave(const int lanesX, const int rowGroups, const int lanes = 64)
{
    return std::min(rowGroups, lanesX % lanes == 0 ? 1 : (lanes % lanesX == 0 ? lanes / lanesX : (lanes - 2) / lanesX + 2));
}

// Lanes a wave takes by default: 64, fewer while they touch more than 8 row groups (of volumes, 32 at sides 6 and
// 7 in groups of 4 rows). 9 or 10 groups need brackets for 16 (RowGroupCap), 18 KiB of LDS per wave, and
// leave 8 waves per CU where 8 groups leave 16: 7^3 x 200,000 compensated takes 2,342 us on 64 lanes and
// 1,656 on 32, a batch of 128 systems up to 128^3 with some of side 7 33.1 and 28.0 ms.
inline int LanesPerWave(const int lanesX, const int rowGroups)
{
    int lanes = 64;
    while (lanes > 1 && RowGroupsPerWave(lanesX, rowGroups, lanes) > 8)
    {
        lanes /= 2;
    }
    return lanes;
}

// Row groups a kernel is compiled for when its waves touch up to `touched` of them: the next power of two,
// and 3 for groups of 8 rows, whose brackets then leave room for 19 waves per CU instead of 16 (3
// groups of 4 rows would put the lanes' 16-byte bracket stores on the same LDS banks).
inline int RowGroupCap(const int touched, const int rows)
{
    if (touched == 3 && rows == 8)
    {
        return 3;
    }
    int cap = 1;
    while (cap < touched)
    {
        cap *= 2;
    }
    return cap;
}

// The plan of a shape, or one with no workgroups when the shape does not fit the LDS or a launch.
inline PackedPlan PlanShape(const int px, const int rows, const int waves, const int blocks, const int atomCount, const long rowLength,
    const long rowsTotal, const bool compensated, const int lanes = 64)
{
    PackedPlan plan;
    plan.px = px;
    plan.rows = rows;
    plan.waves = waves;
    plan.blocks = blocks;
    const long lanesX = (rowLength + px - 1) / px;
    const long rowGroups = (rowsTotal + rows - 1) / rows;
    const long workgroups = (lanesX * rowGroups + lanes - 1) / lanes;
    plan.lanes = lanes;
    plan.lanesX = static_cast<int>(lanesX);
    plan.rowGroups = static_cast<int>(rowGroups);
    plan.touched = RowGroupsPerWave(plan.lanesX, plan.rowGroups, lanes);
    plan.cap = RowGroupCap(plan.touched, rows);
    // Whole unrolled steps of 8 atoms per wave.
    const long shares = static_cast<long>(waves) * blocks;
    const long perWave = (atomCount + shares - 1) / shares;
    plan.share = static_cast<int>(std::min<long>((perWave + 7) / 8 * 8, std::numeric_limits<int>::max()));
    const long ldsBytes = waves * 64L * ((compensated ? 4 : 2) + static_cast<long>(plan.cap) * rows + 4) * 4;
    // Lane numbers are 32-bit, and a launch holds fewer than 2^32 threads.
    if (ldsBytes <= kPackedLdsBytes && workgroups * 64 * shares <= 0x7fffffffL)
    {
        plan.ldsBytes = static_cast<unsigned int>(ldsBytes);
        plan.workgroups = static_cast<unsigned int>(workgroups);
    }
    return plan;
}

// The shapes tried, with what the estimate below needs of each.
struct PackedShape
{
    int px;
    int rows;
    double atom;      // us a SIMD takes per wave and atom with enough waves to hide latency
    double compensated; // what the compensated form's offsets and sums multiply it by
    double alone;     // share of that rate that one wave per SIMD reaches
    int wavesPerSimd; // at the kernel's registers (78, 50, 46 and 96, 67, 51 VGPRs), plain and compensated
    int wavesPerSimdCompensated;
};
constexpr PackedShape kPackedShapes[] = {{2, 8, 0.071, 1.035, 0.49, 6, 5}, {1, 8, 0.0376, 1.0, 0.36, 8, 7},
    {1, 4, 0.0192, 1.124, 0.41, 8, 8}};

// Workgroups a CU holds at once, by registers and LDS.
inline int PackedGroupsPerUnit(const PackedPlan& plan, const PackedShape& shape, const bool compensated)
{
    const int slots = compensated ? shape.wavesPerSimdCompensated : shape.wavesPerSimd;
    return std::max(1, std::min(slots * 4 / plan.waves, static_cast<int>(kPackedLdsBytes / plan.ldsBytes)));
}

// Estimated time of a plan in us beyond the launch itself. The constants are a fit to 27 grids of 24^3 to
// 320^3 points with 64 to 20,000 atoms, both forms, each timed on MI355X at every shape and 4, 8 and 16
// waves (1 too for 64 atoms): the shape it picks is within 1.0% of the fastest of these on average (at worst
// 7%), while any one shape for all is several times slower somewhere. It knows nothing of the store of rows
// that a lane's run does not divide: with up to 64 atoms on full spans it is 5 to 9% off (127^3 x 64 plain 21.4
// us, 19.7 in 2 x 8 blocks).
inline double EstimatePacked(const PackedPlan& plan, const PackedShape& shape, const bool compensated)
{
    constexpr double kComputeUnits = 256.0;
    const double size = plan.px * plan.rows / 16.0;
    const double tiles = (plan.share + 63) / 64;
    // One wave: its atoms, the brackets of its rows per 64 atoms, the start and the store, and, if
    // the waves of a workgroup split the atoms, their meeting in LDS.
    double wave = plan.share * shape.atom * (compensated ? shape.compensated : 1.0);
    wave += tiles * plan.touched * plan.rows * (compensated ? 0.0054 : 0.0085);
    wave += 0.07 + size * (compensated ? 0.51 : 0.24);
    wave += plan.waves > 1 ? size * (compensated ? 0.044 : 0.012) : 0.0;
    // Waves per SIMD of the 256 CUs: whole workgroups per CU while they all fit at once; more than
    // that are handed out as others end, with a partial last round.
    const double perGroup = plan.waves / 4.0;
    const double resident = PackedGroupsPerUnit(plan, shape, compensated) * perGroup;
    double load = plan.waves < 4 ? std::ceil(plan.workgroups * perGroup / kComputeUnits)
                                 : std::ceil(plan.workgroups / kComputeUnits) * perGroup;
    double busy = load;
    if (load > resident)
    {
        busy = resident;
        load = plan.workgroups * perGroup / kComputeUnits + 0.62 * std::max(1.0, perGroup);
    }
    const double rate = 1.0 - (1.0 - shape.alone) * std::pow(std::max(busy, 1.0), -0.735);
    return load * wave / rate;
}

/** Whether a volume of side^3 points runs the wave engine without a configuration (but for a few atoms on some
 *  sides, below): not at multiples of 256, whose lanes and chip the workgroup shapes fill, and not above 1,024, where
 *  their idle lanes are under an eighth (the figures stand at PackedPlanFor in CoulombApi.cpp). */
inline bool WaveEngineByDefault(const int side)
{
    return side % 256 != 0 && side <= 1024;
}

// The wave engine's launch for a slice: 1 x 4 points per lane, 8 waves per workgroup, at most 32 atoms a wave.
constexpr int kSlicePx = 1;
constexpr int kSliceRows = 4;
constexpr int kSliceWaves = 8;
inline int SliceAtomBlocks(const int atomCount)
{
    return atomCount > 256 ? (atomCount - 1) / 256 + 1 : 1;
}

/** Whether a slice runs the wave engine without a configuration. A small slice is over in a few microseconds,
 *  most of them one workgroup's start: tile, barriers, brackets, adds, which the wave engine does faster. It
 *  then costs more per workgroup and per atom than the workgroup shapes of CoulombSum2d.hip. MI355X, workgroup
 *  shapes / wave engine, over 19 grids of 64^2 to 2,048^2 points and 1 to 30,000 atoms:
 *   - up to 512^2 points the wave engine up to 75 million interactions: 256^2 x 64 5.97 / 4.14 us, 64 x 1,024 x 512
 *     7.20 / 6.17, 64^2 x 16,384 12.77 / 9.91, 512^2 x 128 7.04 / 6.77. Near the limit it is between 6% slower and
 *     level (384^2 x 256 7.49 / 8.01, 192^2 x 1,024 7.49 / 7.96, 256^2 x 1,024 9.64 / 9.70), for an error that is a
 *     quarter smaller (1.1e-7 against 1.5e-7 of the slice at 384^2 x 256: 32 atoms a partial sum, not 64);
 *   - above, only with at most 16 atoms, 8 above 2^20 points: 768^2 x 16 8.07 / 6.50, 1,024^2 x 16 10.06 / 9.72,
 *     2,048^2 x 8 31.0 / 29.3. The wave engine's workgroups no longer start at once there and each costs its start: 64
 *     x 8,192 x 64 6.6 / 8.2, 1,024^2 x 32 10.0 / 10.8 and x 64 10.0 / 14.3, 2,048^2 x 16 31.0 / 32.4, 4,096^2 x 1
 *     105 / 116. */
inline bool SliceOnWaveEngine(const long gridX, const long gridY, const int atomCount)
{
    const long points = gridX * gridY;
    if (points <= 1L << 18)
    {
        return points * atomCount <= 75000000L;
    }
    return points <= 1L << 22 && atomCount <= (points <= 1L << 20 ? 16 : 8);
}

/** Whether a volume of few atoms in the plain form runs faster on the workgroup shapes although its side takes the wave
 *  engine by default. Up to 64 atoms are one tile of either kernel, and clearing, reading and writing the grid count
 *  as much as the sum. The workgroup shapes win where they compute no padding to speak of: atoms that fill their 16-,
 *  32- or 64-atom tile to the wave engine's step of 8, and rows that nearly fill the 128-point spans (MI355X, workgroup
 *  shapes / wave engine):
 *   - below a side of 128, where 2 x 8 blocks are two waves per SIMD and the chooser's narrower ones pay for their
 *     start: 117^3 x 16 0.86, 125^3 x 32 0.83, 127^3 x 64 0.90, but 113^3 x 64 1.07;
 *   - at odd sides, whose rows the wave engine stores point by point: 9 to 16 atoms at 251^3 0.90, at 511^3 0.85, at
 *     1,023^3 0.87 (32 atoms 0.96, 0.94, 0.98; even sides 1.0 to 1.5), and 1 to 8 atoms above a side of 448: 511^3
 *     0.93, 1,023^3 0.94 (383^3 1.10).
 *  The plain sums are as exact either way (one tile, added in order: 1.1e-7 of the map at 117^3 x 16). The compensated
 *  form stays on the wave engine, 0.77 to 1.1 below a side of 128 and level above: its x offsets carry one rounding, the
 *  workgroup shapes' two (127^3 x 64 at a spacing of 0.49: 1.8e-7 against 4.3e-7, 117^3 x 16 1.2e-7 against 1.1e-6). */
inline bool FewAtomsOnWorkgroupShapes(const int side, const int atomCount, const bool compensated)
{
    const int spans = (side + 127) / 128;
    const int tile = atomCount <= 16 ? 16 : (atomCount <= 32 ? 32 : 64);
    if (compensated || atomCount < 1 || atomCount > tile)
    {
        return false;
    }
    const bool full = (atomCount + 7) / 8 * 8 == tile;
    if (side < 128)
    {
        return full && side * 10 >= 128 * 9;
    }
    return side % 2 != 0 && side * 20 >= spans * 128 * 17 && atomCount <= 16 && (full || side > 448);
}

/** The shape with the smallest estimated time. */
inline PackedPlan ChoosePackedPlan(const int atomCount, const long rowLength, const long rowsTotal, const bool compensated)
{
    PackedPlan best;
    double bestTime = std::numeric_limits<double>::max();
    for (const PackedShape& shape : kPackedShapes)
    {
        for (const int waves : {1, 4, 8, 16})
        {
            const int lanes = LanesPerWave(static_cast<int>((rowLength + shape.px - 1) / shape.px),
                static_cast<int>((rowsTotal + shape.rows - 1) / shape.rows));
            const PackedPlan plan = PlanShape(shape.px, shape.rows, waves, 1, atomCount, rowLength, rowsTotal, compensated, lanes);
            // One-wave workgroups win while a wave's atoms are a tile or two (256^3 x 64: 102 us against
            // 118 with 4 waves) and lose 5 to 10% beyond (180^3 x 500: 303 against 280).
            if (waves == 1 && atomCount > 128)
            {
                continue;
            }
            // A short row wraps a wave over many row groups, whose brackets then cost more LDS and
            // instructions than a narrower block saves.
            if (plan.workgroups == 0 || (shape.px > 1 && plan.touched > 4))
            {
                continue;
            }
            // Four-wave workgroups that all start at once stay where the first round put them, unevenly;
            // eight-wave ones leave a part for CUs that finish early (100^3 x 30,000: 2,882 us against 3,051).
            if (waves == 4 && atomCount >= 256 && plan.workgroups > 256u
                && (plan.workgroups + 255u) / 256u <= static_cast<unsigned int>(PackedGroupsPerUnit(plan, shape, compensated)))
            {
                continue;
            }
            const double time = EstimatePacked(plan, shape, compensated);
            if (time < bestTime)
            {
                bestTime = time;
                best = plan;
            }
        }
    }
    return best;
}

// The compensated kernels that ChoosePackedPlan picks among for the volumes WaveEngineByDefault takes: all of them, each
// for some volume. The no-allocation library holds these.
struct PackedVariant
{
    int px;
    int rows;
    int cap;
    int lanes;
};
constexpr PackedVariant kPackedVariants[] = {{2, 8, 1, 64}, {2, 8, 2, 64}, {2, 8, 3, 64}, {2, 8, 4, 64}, {1, 8, 1, 64}, {1, 8, 2, 64},
    {1, 8, 3, 64}, {1, 4, 1, 64}, {1, 4, 2, 64}, {1, 4, 4, 64}, {1, 4, 8, 64}, {1, 4, 8, 32}};
constexpr int kPackedVariantCount = static_cast<int>(sizeof(kPackedVariants) / sizeof(kPackedVariants[0]));

// Index of a plan's kernel in kPackedVariants, or -1.
inline int PackedVariantOf(const PackedPlan& plan)
{
    for (int v = 0; v < kPackedVariantCount; ++v)
    {
        const PackedVariant& variant = kPackedVariants[v];
        if (variant.px == plan.px && variant.rows == plan.rows && variant.cap == plan.cap && variant.lanes == plan.lanes)
        {
            return v;
        }
    }
    return -1;
}

} // namespace ktt
