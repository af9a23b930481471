// Shared definitions for the gfx950 TTI kernels: FD coefficients, grid indexing, launch-status plumbing.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Return codes of every C entry point (0 = success).
#define TTI_OK 0
#define TTI_EINVAL (-1)    // inconsistent sizes / ranges / null pointers
#define TTI_EORDER (-2)    // unsupported FD order
#define TTI_EHIP_BASE (-1000) // -1000 - hipError_t

namespace tti {

// 8th-order least-squares coefficients, FP32 as in the reference tables (kernels/fd_coef.h:467-470 first-order
// staggered c1..c4; kernels/fd_coef.h:517-521 second-order central e0..e4). The staggered set equals the Taylor set
// 1225/1024, -245/3072, 49/5120, -5/7168 to FP32 rounding.
constexpr float C1 = 1.19628906250000e+00f;
constexpr float C2 = -7.97526041666667e-02f;
constexpr float C3 = 9.57031250000000e-03f;
constexpr float C4 = -6.97544642857143e-04f;
constexpr float E0 = -0.2903117E+1f;
constexpr float E1 = 0.1645351E+1f;
constexpr float E2 = -0.2236606E+0f;
constexpr float E3 = 0.3265851E-1f;
constexpr float E4 = -0.2790073E-2f;

__host__ __device__ constexpr float
cstg(int n)
{
    return n == 1 ? C1 : n == 2 ? C2 : n == 3 ? C3 : n == 4 ? C4 : 0.0f;
}
__host__ __device__ constexpr float
ecen(int n)
{
    return n == 0 ? E0 : n == 1 ? E1 : n == 2 ? E2 : n == 3 ? E3 : n == 4 ? E4 : 0.0f;
}

constexpr int R = 4; // stencil radius of order 8

struct ab2
{
    float a, b;
}; // sponge coefficient pair {A, B}, same layout as a float2

inline int
hip_status(hipError_t e)
{
    return e == hipSuccess ? TTI_OK : (TTI_EHIP_BASE - (int)e);
}

constexpr int CUS = 256; // compute units of one MI355X

// z planes per thread block of a z-marching kernel: nz planes of `tiles` x-y tiles cut into equal chunks. A block costs
// its planes plus `warm` (its prologue and the halo planes it recomputes, in planes), and the grid runs in rounds of
// `slots` resident blocks, so few deep blocks leave CUs idle (a 64^3 volume in chunks of 128 planes is 16 blocks, each
// marching 72 planes at 2 us) and a round that is barely begun costs a whole one; many shallow ones recompute halos.
// Returns the depth of the cheapest number of chunks, none deeper than `cap` (any value: the fused steps pass a caller's
// zblock, which may be the largest int for "no limit"); a shallower one has to gain 3% over the best so far, because
// deeper chunks also read less. Where several blocks fit a CU, a last round of at most one block per CU runs its planes
// faster and counts 0.85 of a round: only the elastic kernels have such rounds, and on the volumes where it changes the
// choice the mixed interpolations take 5.8 to 6.7 us with it and 6.9 to 7.5 without (40 to 180 points a side; chunks of 3
// and 4 planes instead of 2), the strains the same either way. The deepest chunk is taken at once where its blocks fill
// `full` of one round or more (see MIXED_CHUNK).
inline int
chunk_depth(int nz, long tiles, int slots, float warm, int cap, float full = 2.0f)
{
    cap = cap < 1 ? 1 : cap > nz ? nz : cap;
    int best = 0;
    float cost = 0.0f;
    for (int c = (nz + cap - 1) / cap;;) {
        const int bz = (nz + c - 1) / c;
        if (best && bz < 2)
            break;
        const long n = tiles * ((nz + bz - 1) / bz), r = n % slots;
        if (!best && n <= slots && (float)n >= full * (float)slots)
            return bz;
        const float rounds = (float)(n / slots) + (r == 0 ? 0.0f : r <= CUS && slots > CUS ? 0.85f : 1.0f);
        const float t = ((float)bz + warm) * rounds;
        if (!best || t < 0.97f * cost) {
            cost = t;
            best = bz;
        }
        if (bz < 2)
            break;
        c = (nz + bz - 2) / (bz - 1); // the next number of chunks that makes them shallower
    }
    return best;
}

// Status of the last launch on this thread.
inline int
launch_status()
{
    return hip_status(hipGetLastError());
}

} // namespace tti
