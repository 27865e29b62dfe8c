// Wave engine of the direct Coulomb sum for gfx950: one wave owns a packed run of points and works
// alone, without workgroup barriers, so that any grid side fills its lanes and the atoms of one run
// can be split over the waves of a workgroup.
//
// Points. A row is the set of x points that share one (y, z) (coulomb_core.h). Rows are taken ROWS at
// a time (a row group) and a row's points PX at a time, which makes lanesX = ceil(rowLength / PX)
// lanes per row group. Lanes are numbered row group * lanesX + x lane over the whole grid, and wave b
// takes lanes [64 b, 64 b + 64): they wrap from one row group into the next, so that only the grid's
// last wave and a row length that PX does not divide leave lanes idle. (A workgroup of coulomb_core.h
// spans a fixed number of x points instead: at a side of 150 its 128-point spans leave 41% of the
// lanes idle, at 64 half of them.) A wave touches at most CAP row groups; the host derives CAP from
// lanesX (RowGroupsPerWave in CoulombPackedPlan.h). Rows of 6 and 7 points would make 64 lanes touch 9
// and 10 groups, whose brackets leave room for 8 waves per CU: such waves take 32 lanes (LanesPerWave).
//
// Atoms are staged by the wave 64 at a time, one per lane, into LDS that only this wave uses: the
// atom's x and charge, and the brackets B = (y - Y)^2 + (z - Z)^2 of every row of the wave's groups.
// A wave's LDS operations complete in order, so the tile needs no barrier. B costs 3 to 4 instructions
// per (row, atom), formed row after row with the row's y and z in scalars; the atom of the next tile
// is read from memory while this one is summed. The inner loop is the issue-phased loop of
// coulomb_core.h. The plain form keeps the last atom's r^-1 in flight over the tile's end; the compensated
// form, whose brackets in FP64 need its registers, lands it there.
//
// Split. The WAVE_SPLIT waves of a workgroup own the same 64 lanes and a contiguous share of the atoms
// each. They meet in LDS once, in wave order (plain FP32; compensated FP64), so results do not depend on
// timing. A grid with few points fills the chip this way: 64^3 points are 256 waves of 2 x 8 points, a
// quarter of the 1,024 SIMDs, and 256 workgroups of 16 waves when the atoms are split.
//
// Bound by FP32 VALU issue as the workgroup engine is (per interaction 2 FMAs that pair with another
// wave's and a v_rsq_f32 of two quad-cycles); small grids by the launch. Measured on MI355X with the
// fill before it, workgroup shapes -> wave engine: 150^3 x 20,011 compensated 12,990 -> 6,194 us (120
// TFLOP/s at 11 per interaction), 99^3 x 3,001 plain 636 -> 292, 64^3 x 5,000 compensated 363 -> 138,
// 32^3 x 200 plain 59 -> 7 to 8. On 256^3 x 8,192, which the workgroup shapes fill, 11,660 -> 11,740 us
// plain and 11,770 -> 12,010 compensated: every wave forms its own row brackets, and the compensated
// dx takes one FMA more per atom.
#pragma once

#include "coulomb_core.h"

namespace kc
{

template <bool CONDITION, class A, class B>
struct Select
{
    using Type = A;
};
template <class A, class B>
struct Select<false, A, B>
{
    using Type = B;
};

// Orders this wave's LDS accesses for the compiler; the hardware keeps them in order.
__device__ __forceinline__ void waveFence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int PX, int ROWS, int CAP, int MODE, bool COMP>
struct WaveEngine
{
    using Sum = typename Select<COMP, double, float>::Type;
    static constexpr int Tile = 64;
    static constexpr int Unroll = 8;
    static constexpr int Points = PX * ROWS;
    // Atoms per issue phase. A change of phase costs a few cycles, which the plain 1 x 4 block's four
    // v_rsq_f32 feel: two atoms at a time take 128^3 x 4,000 from 797 to 779 us and 32^3 x 5,000 from 41.0
    // to 39.0. The larger blocks, and the compensated ones with their per-tile landing, lose as much
    // to the registers of the second atom as they gain (1 x 8 758 -> 758, compensated 1 x 4 833 -> 860).
    static constexpr int Phase = !COMP && Points <= 4 ? 2 : 1;
    static_assert(Unroll % Phase == 0, "whole phases per unrolled step");
    static constexpr int AtomFloats = COMP ? 4 : 2;
    // Row brackets of one atom, padded so that the 16-byte stores of 8 lanes hit all 64 banks once.
    static constexpr int RowStride = CAP * ROWS + 4;
    static constexpr int WaveFloats = Tile * (AtomFloats + RowStride);
    // Rows of a lane's points that fit a wave's LDS when the waves of a split meet.
    static constexpr int MeetWhole = WaveFloats * 4 / (64 * PX * static_cast<int>(sizeof(Sum)));
    static constexpr int MeetRows = MeetWhole < ROWS ? MeetWhole : ROWS;

    static_assert(MeetRows >= 1, "the waves meet at least one row at a time");
    static_assert(ROWS % 4 == 0, "row brackets are stored four at a time");

    // Position of this lane's points: x0 = xLane * PX, rows row0 .. row0 + ROWS - 1.
    int lane;
    int xLane;
    int rowGroup;
    int firstGroup;  // the wave's first row group and the number it touches (uniform)
    int groups;
    bool valid;
    bool whole;  // every lane of the wave has points (uniform)

    float part[ROWS][PX];
    Sum sum[ROWS][PX];

    // lanes: lanes that a wave takes, 64 or a power of two below it (the others idle).
    __device__ __forceinline__ void place(const unsigned int waveBlock, const int lanesX, const int rowGroups, const int lanes)
    {
        lane = threadIdx.x & 63;
        const unsigned int total = static_cast<unsigned int>(lanesX) * static_cast<unsigned int>(rowGroups);
        const unsigned int first = waveBlock * static_cast<unsigned int>(lanes);
        const unsigned int end = total - first < static_cast<unsigned int>(lanes) ? total : first + static_cast<unsigned int>(lanes);
        const unsigned int mine = first + lane;
        valid = mine < end;
        whole = end - first == 64u;
        const unsigned int index = valid ? mine : end - 1u;
        rowGroup = static_cast<int>(index / static_cast<unsigned int>(lanesX));
        xLane = static_cast<int>(index - static_cast<unsigned int>(rowGroup) * lanesX);
        firstGroup = __builtin_amdgcn_readfirstlane(rowGroup);
        groups = __builtin_amdgcn_readlane(rowGroup, 63) - firstGroup + 1;
#pragma unroll
        for (int k = 0; k < ROWS; ++k)
        {
#pragma unroll
            for (int i = 0; i < PX; ++i)
            {
                part[k][i] = 0.0f;
                sum[k][i] = 0;
            }
        }
    }

    static __device__ __forceinline__ float4 loadAtom(const float4* atoms, const unsigned int index, const unsigned int end)
    {
        return index < end ? atoms[index] : make_float4(kPadCoord, kPadCoord, kPadCoord, 0.0f);
    }

    // h * i - X with the grid coordinate rounded first, as the reference kernel and its generator round
    // it (Examples/CoulombSum3d/CoulombSum3d.cu:13-15): an atom at float(h * i) is then at distance 0.
    template <class Real>
    static __device__ __forceinline__ Real offset(const Real h, const int i, const Real X)
    {
#pragma clang fp contract(off)
        const Real coordinate = h * static_cast<Real>(i);
        return coordinate - X;
    }

    template <class Real>
    static __device__ __forceinline__ Real square(const Real v)
    {
        return v * v;
    }

    // One atom per lane into the wave's LDS, with the brackets of the wave's rows.
    // Compensated x: X = h n + d with n a near grid index and d formed in FP64, so that
    // x - X = h (i - n) - d carries one rounding whatever the coordinate's size. n is clamped to
    // 2^23, where i - n is still exact in FP32; beyond it (or with h = 0) d holds the rest.
    __device__ __forceinline__ void stage(float* lds, const float4 at, const float h, const int rowsPerPlane) const
    {
        float* sB = lds + Tile * AtomFloats + lane * RowStride;
        if constexpr (COMP)
        {
            const double X = static_cast<double>(at.x);
            const double n = __builtin_rint(__builtin_fmin(__builtin_fmax(X * (1.0 / static_cast<double>(h)), -8388608.0), 8388608.0));
            const double d = X - static_cast<double>(h) * n;
            *reinterpret_cast<float4*>(lds + lane * 4) = make_float4(static_cast<float>(n), static_cast<float>(-d), at.w, 0.0f);
        }
        else
        {
            *reinterpret_cast<float2*>(lds + lane * 2) = make_float2(at.x, at.w);
        }
        using Real = typename Select<COMP, double, float>::Type;
        const Real Y = static_cast<Real>(at.y);
        const Real Z = static_cast<Real>(at.z);
        const Real step = static_cast<Real>(h);
        int row = firstGroup * ROWS;
        int y = (MODE == Volume) ? row % rowsPerPlane : row;
        int z = (MODE == Volume) ? row / rowsPerPlane : 0;
        Real dz2 = (MODE == Volume) ? square(offset(step, z, Z)) : Z;
        Real dy = offset(step, y, Y);
        const int quads = groups * (ROWS / 4);
#pragma unroll 1
        for (int g = 0; g < quads; ++g)
        {
            float b[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                b[k] = static_cast<float>(dy * dy + dz2);
                ++y;
                if constexpr (COMP)
                {
                    dy += step;  // FP64: a step's rounding is far below B's own to FP32
                }
                if (MODE == Volume && y == rowsPerPlane)
                {
                    y = 0;
                    ++z;
                    dz2 = square(offset(step, z, Z));
                    dy = -Y;
                }
                if constexpr (!COMP)
                {
                    dy = offset(step, y, Y);
                }
            }
            *reinterpret_cast<float4*>(sB + g * 4) = make_float4(b[0], b[1], b[2], b[3]);
        }
    }

    // Adds atoms [a0, a1) into this lane's points.
    __device__ __forceinline__ void accumulate(float* lds, const float4* atoms, const unsigned int a0, const unsigned int a1, const float h,
        const int rowsPerPlane)
    {
        const float* sB = lds + Tile * AtomFloats + (rowGroup - firstGroup) * ROWS;
        float x[PX];
#pragma unroll
        for (int i = 0; i < PX; ++i)
        {
            x[i] = COMP ? static_cast<float>(xLane * PX + i) : h * static_cast<float>(xLane * PX + i);
        }
        float hV = h;  // in a VGPR: an SGPR operand would keep the FMA from pairing
        asm volatile("" : "+v"(hV));
        float rr[Phase][ROWS][PX];  // r^2 of the atoms in flight, then their r^-1
        float qPrev[Phase];
#pragma unroll
        for (int p = 0; p < Phase; ++p)
        {
            qPrev[p] = 0.0f;
#pragma unroll
            for (int k = 0; k < ROWS; ++k)
            {
#pragma unroll
                for (int i = 0; i < PX; ++i)
                {
                    rr[p][k][i] = 0.0f;
                }
            }
        }
        float4 next;
        if constexpr (!COMP)
        {
            next = loadAtom(atoms, a0 + lane, a1);
        }
        for (unsigned int t = a0; t < a1; t += Tile)
        {
            waveFence();  // the previous tile has been read
            if constexpr (COMP)
            {
                // Not read ahead: four registers more would cost a wave per SIMD.
                next = loadAtom(atoms, t + lane, a1);
            }
            stage(lds, next, h, rowsPerPlane);
            if constexpr (!COMP)
            {
                next = loadAtom(atoms, t + Tile + lane, a1);
            }
            waveFence();
            const int count = a1 - t < Tile ? static_cast<int>(a1 - t) : Tile;
            int a = 0;
            if constexpr (COMP)
            {
                addAtoms<true>(lds, sB, 0, x, hV, qPrev, rr);
                a = Unroll;
            }
            for (; a < count; a += Unroll)
            {
                addAtoms<false>(lds, sB, a, x, hV, qPrev, rr);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
            if constexpr (COMP)
            {
                // Land the atom in flight: its 16 registers are free while the next tile is staged,
                // which keeps the kernel at 5 waves per SIMD.
                land(qPrev, rr);
            }
            fold();
        }
        if constexpr (!COMP)
        {
            land(qPrev, rr);
            fold();
        }
    }

    // Adds Unroll atoms of the staged tile from atom a on, in issue phases. FIRST (one atom per phase): the
    // tile's first atoms, before which no atom is in flight and no sum begun. Clearing both per tile and
    // adding a charge of zero takes three instructions per point and tile, 1.5% of the compensated loop: without
    // them 150^3 x 20,011 takes 6,194 us instead of 6,303, 64^3 x 5,000 138.5 instead of 141.3. The plain form
    // carries its atom over the tiles and has only the sums to clear.
    template <bool FIRST>
    __device__ __forceinline__ void addAtoms(const float* lds, const float* sB, const int a, const float (&x)[PX], const float hV,
        float (&qPrev)[Phase], float (&rr)[Phase][ROWS][PX])
    {
#pragma unroll
        for (int u = 0; u < Unroll; u += Phase)
        {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int p = 0; p < Phase; ++p)
            {
                float dx[PX];
                float q;
                if constexpr (COMP)
                {
                    const float4 v = *reinterpret_cast<const float4*>(lds + (a + u + p) * 4);
                    dx[0] = fmaf(hV, x[0] - v.x, v.y);
#pragma unroll
                    for (int i = 1; i < PX; ++i)
                    {
                        dx[i] = dx[i - 1] + hV;
                    }
                    q = v.z;
                }
                else
                {
                    const float2 v = *reinterpret_cast<const float2*>(lds + (a + u + p) * 2);
#pragma unroll
                    for (int i = 0; i < PX; ++i)
                    {
                        dx[i] = x[i] - v.x;
                    }
                    q = v.y;
                }
                float b[ROWS];
#pragma unroll
                for (int k = 0; k < ROWS; k += 4)
                {
                    const float4 v = *reinterpret_cast<const float4*>(sB + (a + u + p) * RowStride + k);
                    b[k] = v.x;
                    b[k + 1] = v.y;
                    b[k + 2] = v.z;
                    b[k + 3] = v.w;
                }
#pragma unroll
                for (int k = 0; k < ROWS; ++k)
                {
#pragma unroll
                    for (int i = 0; i < PX; ++i)
                    {
                        if constexpr (FIRST)
                        {
                            // The tile's first atom finds none in flight, and its second starts the sums.
                            if (u == 1)
                            {
                                part[k][i] = qPrev[p] * rr[p][k][i];
                            }
                            else if (u > 1)
                            {
                                part[k][i] = fmaf(qPrev[p], rr[p][k][i], part[k][i]);
                            }
                        }
                        else
                        {
                            part[k][i] = fmaf(qPrev[p], rr[p][k][i], part[k][i]);
                        }
                        rr[p][k][i] = fmaf(dx[i], dx[i], b[k]);
                    }
                }
                qPrev[p] = q;
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(3);
#pragma unroll
            for (int p = 0; p < Phase; ++p)
            {
#pragma unroll
                for (int k = 0; k < ROWS; ++k)
                {
#pragma unroll
                    for (int i = 0; i < PX; ++i)
                    {
                        rr[p][k][i] = __builtin_amdgcn_rsqf(rr[p][k][i]);
                    }
                }
            }
        }
    }

    // part += q r^-1 of the atoms in flight.
    __device__ __forceinline__ void land(const float (&q)[Phase], const float (&rr)[Phase][ROWS][PX])
    {
#pragma unroll
        for (int p = 0; p < Phase; ++p)
        {
#pragma unroll
            for (int k = 0; k < ROWS; ++k)
            {
#pragma unroll
                for (int i = 0; i < PX; ++i)
                {
                    part[k][i] = fmaf(q[p], rr[p][k][i], part[k][i]);
                }
            }
        }
    }

    // Moves the 64-atom partial sums into the running sums. Plain: FP32, which takes the rounding of a
    // long FP32 sum off for 0.7% of the time and 16 registers (6 waves per SIMD, not 8): at 128^3 x 8,192
    // the error against 64 bits is 3.1e-7 of the map, 8.5e-7 without. Compensated: FP64, two
    // instructions in the two registers that a (sum, compensation) pair would take seven for, and an
    // infinite term (an atom on a grid point) stays infinite.
    __device__ __forceinline__ void fold()
    {
#pragma unroll
        for (int k = 0; k < ROWS; ++k)
        {
#pragma unroll
            for (int i = 0; i < PX; ++i)
            {
                sum[k][i] += static_cast<Sum>(part[k][i]);
                if constexpr (!COMP)
                {
                    part[k][i] = 0.0f;
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // one row at a time: few registers
        }
    }

    // grid += v over row k of this lane's points. inside: the wave's points are all in the grid (uniform),
    // pairs: and two x points may be read and written at once. atomic: other workgroups add to the same points.
    __device__ __forceinline__ void addRow(float* out, const int k, const Sum (&v)[PX], const int rowLength, const int rowsTotal,
        const bool inside, const bool pairs, const bool atomic) const
    {
        float* row = out + static_cast<size_t>(k) * rowLength;
        if (!COMP && atomic)
        {
#pragma unroll
            for (int i = 0; i < PX; ++i)
            {
                if (inside || (valid && xLane * PX + i < rowLength && rowGroup * ROWS + k < rowsTotal))
                {
                    unsafeAtomicAdd(row + i, static_cast<float>(v[i]));
                }
            }
            return;
        }
        if constexpr (PX == 2)
        {
            if (pairs)
            {
                float2 o = *reinterpret_cast<float2*>(row);
                o.x = static_cast<float>(static_cast<Sum>(o.x) + v[0]);
                o.y = static_cast<float>(static_cast<Sum>(o.y) + v[1]);
                *reinterpret_cast<float2*>(row) = o;
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < PX; ++i)
        {
            if (inside || (valid && xLane * PX + i < rowLength && rowGroup * ROWS + k < rowsTotal))
            {
                row[i] = static_cast<float>(static_cast<Sum>(row[i]) + v[i]);
            }
        }
    }

    // grid += the sum over the workgroup's waves, each of which holds the same points' sums over its
    // own atoms. shared: waves * WaveFloats floats. A wave whose points are all inside the grid stores
    // without a check per point, which a launch of few atoms feels (256^3 x 64: 16 read-modify-writes of
    // some 20 instructions each beside 64 atoms of 67).
    __device__ __forceinline__ void store(float* shared, const int waves, const int wave, float* grid, const int rowLength,
        const int rowsTotal, const bool atomic) const
    {
        float* out = grid + static_cast<size_t>(rowGroup) * ROWS * rowLength + xLane * PX;
        const bool inside = whole && rowLength % PX == 0 && (firstGroup + groups) * ROWS <= rowsTotal;
        const bool pairs = inside && rowLength % 2 == 0 && (reinterpret_cast<size_t>(grid) & 7u) == 0;
        if (waves == 1)
        {
            if constexpr (PX == 2)
            {
                if (pairs && !atomic)
                {
                    float2 o[ROWS];
#pragma unroll
                    for (int k = 0; k < ROWS; ++k)
                    {
                        o[k] = *reinterpret_cast<float2*>(out + static_cast<size_t>(k) * rowLength);
                    }
#pragma unroll
                    for (int k = 0; k < ROWS; ++k)
                    {
                        o[k].x = static_cast<float>(static_cast<Sum>(o[k].x) + sum[k][0]);
                        o[k].y = static_cast<float>(static_cast<Sum>(o[k].y) + sum[k][1]);
                        *reinterpret_cast<float2*>(out + static_cast<size_t>(k) * rowLength) = o[k];
                    }
                    return;
                }
            }
#pragma unroll
            for (int k = 0; k < ROWS; ++k)
            {
                addRow(out, k, sum[k], rowLength, rowsTotal, inside, pairs, atomic);
            }
            return;
        }
        Sum* meet = reinterpret_cast<Sum*>(shared);
#pragma unroll
        for (int first = 0; first < ROWS; first += MeetRows)
        {
            __syncthreads();
#pragma unroll
            for (int k = first; k < first + MeetRows && k < ROWS; ++k)
            {
#pragma unroll
                for (int i = 0; i < PX; ++i)
                {
                    meet[((wave * MeetRows + k - first) * PX + i) * 64 + lane] = sum[k][i];
                }
            }
            __syncthreads();
            for (int k = first + wave; k < first + MeetRows && k < ROWS; k += waves)
            {
                Sum total[PX];
#pragma unroll
                for (int i = 0; i < PX; ++i)
                {
                    total[i] = meet[((k - first) * PX + i) * 64 + lane];
                }
                for (int w = 1; w < waves; ++w)
                {
#pragma unroll
                    for (int i = 0; i < PX; ++i)
                    {
                        total[i] += meet[((w * MeetRows + k - first) * PX + i) * 64 + lane];
                    }
                }
                addRow(out, k, total, rowLength, rowsTotal, inside, pairs, atomic);
            }
        }
    }
};

// The body of a wave-engine kernel: block 64 x waves threads, grid (blocks of LANES lanes, atom blocks), dynamic
// LDS of waves * WaveFloats floats. Wave w of atom block b sums atoms [(b * waves + w) * share, + share).
template <class W, int LANES>
__device__ __forceinline__ void packedSum(float* shared, const float4* atoms, const int numberOfAtoms, const int share,
    const float gridSpacing, const int lanesX, const int rowGroups, const int rowLength, const int rowsTotal, float* energyGrid)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const long long first = static_cast<long long>(blockIdx.y * waves + wave) * share;
    const int a0 = first < numberOfAtoms ? static_cast<int>(first) : numberOfAtoms;
    const int a1 = share < numberOfAtoms - a0 ? a0 + share : numberOfAtoms;
    W engine;
    engine.place(blockIdx.x, lanesX, rowGroups, LANES);
    engine.accumulate(shared + wave * W::WaveFloats, atoms, a0, a1, gridSpacing, rowLength);
    engine.store(shared, waves, wave, energyGrid, rowLength, rowsTotal, gridDim.y > 1);
}

} // namespace kc
