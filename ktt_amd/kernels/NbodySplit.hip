// N-body integration step for gfx950 at any number of bodies that is a multiple of 1,024: the default
// of ktt_nbody_step. Same formula, arguments and issue phases as Nbody.hip (its kernel keeps the tuning
// space's shapes):
//   a_i  = sum_j m_j (p_j - p_i) / (|p_j - p_i|^2 + eps^2)^(3/2)
//   p_i' = p_i + dt v_i + damping dt^2 a_i,   v_i' = v_i + dt a_i
//
// Decomposition. A workgroup of 1,024 threads owns BODY_LANES * BODIES_PER_THREAD target bodies. Its
// lanes are 1,024 / BODY_LANES source groups of BODY_LANES lanes; group g sums every source j with
// j % groups == g of each LDS tile, BODIES_PER_THREAD targets at a time, so that a tile of sources is
// read as one broadcast per group, of adjacent addresses within a wave (no bank conflict). The groups'
// partial accelerations are added in a fixed order: by lane exchange within a wave, then wave by wave
// through LDS.
//
// Fewer BODY_LANES make more workgroups of the same 16 waves, which is what few bodies need: 16,384
// bodies are 64 workgroups of 64 lanes x 4 bodies, a quarter of the 256 CUs, and 512 of 8 x 4.
//
// Bound by FP32 VALU issue: 12 plain instructions (6 quad-cycles when they pair) and a v_rsq_f32 (2)
// per interaction, 62.5% of the FP32 peak at 20 operations. Measured on MI355X against 64 x 16 threads
// of nbody_kernel: 16,384 bodies 263 -> 71 us (76 TFLOP/s), 98,304 3,006 -> 2,270 us, 131,072 4,001 ->
// 3,973 us (86 TFLOP/s). 8 waves per SIMD (64 VGPRs) let two workgroups share a CU.
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#endif

#ifndef BODY_LANES
#define BODY_LANES 64
#endif
#ifndef BODIES_PER_THREAD
#define BODIES_PER_THREAD 4
#endif

namespace
{

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kTile = 1024;                       // sources per LDS tile, one per thread
constexpr int kGroups = kThreads / BODY_LANES;    // source groups
constexpr int kSteps = kTile / kGroups;           // sources per group and tile
constexpr int kUnroll = kSteps >= 32 ? 16 : (kSteps > 1 ? kSteps / 2 : 1);
constexpr int kBodies = BODY_LANES * BODIES_PER_THREAD;

static_assert(64 % BODY_LANES == 0, "a wave holds whole source groups");
static_assert(kBodies <= kThreads, "one thread per body finishes the step");

// Ends an issue phase: the values are computed before it. The scheduling barriers bind only the scheduler;
// some compilers move the FMAs past the change of priority before it runs.
__device__ __forceinline__ void holdPhase(float (&v)[BODIES_PER_THREAD])
{
#pragma unroll
    for (int b = 0; b < BODIES_PER_THREAD; ++b)
    {
        asm volatile("" : "+v"(v[b]));
    }
}

__device__ __forceinline__ void holdPhase(float (&x)[BODIES_PER_THREAD], float (&y)[BODIES_PER_THREAD], float (&z)[BODIES_PER_THREAD],
    float (&r)[BODIES_PER_THREAD])
{
    holdPhase(x);
    holdPhase(y);
    holdPhase(z);
    holdPhase(r);
}

} // namespace

extern "C" __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) void nbody_split(float timeDelta, const float4* __restrict__ oldBodyInfo,
    float4* __restrict__ newBodyInfo, const float4* __restrict__ oldVel, float4* __restrict__ newVel, float damping,
    float softeningSqr, int n)
{
    // The source tiles and, after the last one, the waves' partial accelerations.
    constexpr int kTileBytes = 2 * kTile * 16;
    constexpr int kPartialBytes = kWaves * 3 * kBodies * 4;
    __shared__ __attribute__((aligned(16))) unsigned char lds[kTileBytes > kPartialBytes ? kTileBytes : kPartialBytes];
    float4 (*tile)[kTile] = reinterpret_cast<float4 (*)[kTile]>(lds);
    float (*partial)[3][kBodies] = reinterpret_cast<float (*)[3][kBodies]>(lds);

    const int tid = threadIdx.x;
    const int lane = tid % BODY_LANES;
    const int group = tid / BODY_LANES;
    const int base = blockIdx.x * kBodies;

    float px[BODIES_PER_THREAD], py[BODIES_PER_THREAD], pz[BODIES_PER_THREAD];
    float ax[BODIES_PER_THREAD], ay[BODIES_PER_THREAD], az[BODIES_PER_THREAD];
    // The source in flight: its displacements from every target, r^2 and then r^-1, its mass.
    float dxp[BODIES_PER_THREAD], dyp[BODIES_PER_THREAD], dzp[BODIES_PER_THREAD], rr[BODIES_PER_THREAD];
#pragma unroll
    for (int b = 0; b < BODIES_PER_THREAD; ++b)
    {
        const float4 p = oldBodyInfo[base + b * BODY_LANES + lane];
        px[b] = p.x;
        py[b] = p.y;
        pz[b] = p.z;
        ax[b] = 0.0f;
        ay[b] = 0.0f;
        az[b] = 0.0f;
        dxp[b] = 0.0f;
        dyp[b] = 0.0f;
        dzp[b] = 0.0f;
        rr[b] = 0.0f;
    }
    float mPrev = 0.0f;
    float epsV;  // in a VGPR: an SGPR operand would keep the FMA from pairing
    asm volatile("v_mov_b32 %0, %1" : "=v"(epsV) : "s"(softeningSqr));

    tile[0][tid] = oldBodyInfo[tid];
    __syncthreads();
    for (int first = 0; first < n; first += kTile)
    {
        const int current = (first / kTile) & 1;
        const bool more = first + kTile < n;
        const float4 next = oldBodyInfo[(more ? first + kTile : 0) + tid];
        const float4* source = tile[current] + group;
#pragma unroll kUnroll
        for (int j = 0; j < kSteps; ++j, source += kGroups)
        {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
            const float4 q = *source;
#pragma unroll
            for (int b = 0; b < BODIES_PER_THREAD; ++b)
            {
                const float s = mPrev * rr[b] * (rr[b] * rr[b]);
                ax[b] = fmaf(s, dxp[b], ax[b]);
                ay[b] = fmaf(s, dyp[b], ay[b]);
                az[b] = fmaf(s, dzp[b], az[b]);
                dxp[b] = q.x - px[b];
                dyp[b] = q.y - py[b];
                dzp[b] = q.z - pz[b];
                rr[b] = fmaf(dxp[b], dxp[b], fmaf(dyp[b], dyp[b], fmaf(dzp[b], dzp[b], epsV)));
            }
            mPrev = q.w;
            holdPhase(ax, ay, az, rr);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(3);
#pragma unroll
            for (int b = 0; b < BODIES_PER_THREAD; ++b)
            {
                rr[b] = __builtin_amdgcn_rsqf(rr[b]);
            }
            holdPhase(rr);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
        if (more)
        {
            // The other buffer was read before the last barrier.
            tile[current ^ 1][tid] = next;
            __syncthreads();
        }
    }

    __syncthreads();  // the last tile has been read
#pragma unroll
    for (int b = 0; b < BODIES_PER_THREAD; ++b)
    {
        const float s = mPrev * rr[b] * (rr[b] * rr[b]);
        ax[b] = fmaf(s, dxp[b], ax[b]);
        ay[b] = fmaf(s, dyp[b], ay[b]);
        az[b] = fmaf(s, dzp[b], az[b]);
#pragma unroll
        for (int width = BODY_LANES; width < 64; width *= 2)
        {
            ax[b] += __shfl_xor(ax[b], width);
            ay[b] += __shfl_xor(ay[b], width);
            az[b] += __shfl_xor(az[b], width);
        }
        if (tid % 64 < BODY_LANES)
        {
            partial[tid / 64][0][b * BODY_LANES + lane] = ax[b];
            partial[tid / 64][1][b * BODY_LANES + lane] = ay[b];
            partial[tid / 64][2][b * BODY_LANES + lane] = az[b];
        }
    }
    __syncthreads();
    if (tid >= kBodies)
    {
        return;
    }
    float x = 0.0f, y = 0.0f, z = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
    {
        x += partial[w][0][tid];
        y += partial[w][1][tid];
        z += partial[w][2][tid];
    }
    const float dtdt = damping * timeDelta * timeDelta;
    const int i = base + tid;
    const float4 p = oldBodyInfo[i];
    const float4 v = oldVel[i];
    newBodyInfo[i] = make_float4(p.x + (timeDelta * v.x + dtdt * x), p.y + (timeDelta * v.y + dtdt * y),
        p.z + (timeDelta * v.z + dtdt * z), p.w);
    newVel[i] = make_float4(v.x + timeDelta * x, v.y + timeDelta * y, v.z + timeDelta * z, 0.0f);
}
