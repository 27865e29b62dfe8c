#include "CoulombPacked.h"

#include <KttException.h>

namespace ktt
{

PackedPlan MakePackedPlan(const int px, const int rows, const int waves, const int blocks, const int atomCount,
    const long rowLength, const long rowsTotal, const bool compensated)
{
    if (px < 1 || px > 4 || (rows != 4 && rows != 8) || waves < 1 || waves > 16)
    {
        throw KttException("the wave engine takes WAVE_SPLIT 1 to 16, POINTS_X 1 to 4 and ROWS_PER_THREAD 4 or 8");
    }
    if (blocks < 1 || blocks > 65535 || (compensated && blocks > 1))
    {
        throw KttException("WAVE_SPLIT takes ATOM_BLOCKS from 1 to 65,535 in the plain form and 1 in the compensated form");
    }
    const PackedPlan plan = PlanShape(px, rows, waves, blocks, atomCount, rowLength, rowsTotal, compensated);
    if (plan.workgroups == 0)
    {
        throw KttException("WAVE_SPLIT=" + std::to_string(waves) + " with " + std::to_string(px) + " x " + std::to_string(rows)
            + " points per thread exceeds the device limits on rows of " + std::to_string(rowLength) + " points",
            ExceptionReason::DeviceLimitsExceeded);
    }
    return plan;
}

PackedPlan PackedPlanOf(const CoulombConfig& config, const int atomCount, const long rowLength, const long rowsTotal,
    const bool compensated)
{
    const auto value = [&config](const char* name, const long fallback)
    {
        return static_cast<int>(std::min<long>(std::max<long>(config.Get(name, fallback), -1), 1 << 20));
    };
    return MakePackedPlan(value("POINTS_X", 2), value("ROWS_PER_THREAD", 8), value("WAVE_SPLIT", 1), value("ATOM_BLOCKS", 1), atomCount,
        rowLength, rowsTotal, compensated);
}

std::shared_ptr<HipKernel> GetPackedKernel(const PackedPlan& plan, const bool compensated, const bool slice)
{
    std::vector<std::string> defines = {"-DPOINTS_X=" + std::to_string(plan.px), "-DROWS_PER_THREAD=" + std::to_string(plan.rows),
        "-DROW_GROUP_CAP=" + std::to_string(plan.cap), std::string("-DCOMPENSATED=") + (compensated ? "1" : "0"),
        std::string("-DROW_MODE=") + (slice ? "1" : "0")};
    if (plan.lanes != 64)
    {
        defines.push_back("-DWAVE_LANES=" + std::to_string(plan.lanes));
    }
    return CoulombRuntime::Get().GetKernel("CoulombPacked.hip", "coulombPacked", defines);
}

void LaunchPacked(const PackedPlan& plan, const float* atoms, int atomCount, float spacing, int rowLength, int rowsTotal,
    float* energyGrid, const bool compensated, const bool slice, hipStream_t stream, float* kernelMs)
{
    const auto kernel = GetPackedKernel(plan, compensated, slice);
    const unsigned int grid[3] = {plan.workgroups, static_cast<unsigned int>(plan.blocks), 1};
    const unsigned int block[3] = {static_cast<unsigned int>(plan.waves) * 64, 1, 1};
    int share = plan.share;
    int lanesX = plan.lanesX;
    int rowGroups = plan.rowGroups;
    void* arguments[] = {&atoms, &atomCount, &share, &spacing, &lanesX, &rowGroups, &rowLength, &rowsTotal, &energyGrid};
    CoulombRuntime::Launch(*kernel, grid, block, arguments, stream, kernelMs, plan.ldsBytes);
}

} // namespace ktt
