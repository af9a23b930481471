// Helpers shared by the 2.5-D stencil kernels (64-wide tiles staged in LDS, z-march with register queues).
#pragma once

#include <cstdint>
#include <initializer_list>
#include <type_traits>

#include "fd_tables.h"

namespace tti {

constexpr int BX = 64;

// x halo of a quad-staged tile of stencil radius RO: a whole number of quads, so the tile's rows start aligned
__host__ __device__ constexpr int
halo_x(int ro)
{
    return (ro + 3) / 4 * 4;
}

// Element offset of plane z, uniform over the wave and opaque to the optimiser: otherwise loop strength reduction turns
// base + z ldx ldy into one 64-bit per-lane pointer for every volume, two VGPRs each and a 64-bit vector add per plane.
__device__ __forceinline__ long
plane_off(int z, long sz)
{
    const long v = (long)z * sz;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (long)(((unsigned long)hi << 32) | lo);
}

// A lane offset, opaque in the block that uses it: instruction selection works block by block and folds a 32-bit offset
// into a load with a scalar base only where it sees the offset's extension to 64 bits, which is otherwise hoisted out
// of the loop (and every load then takes a 64-bit vector add).
__device__ __forceinline__ unsigned
here(unsigned off)
{
    asm volatile("" : "+v"(off));
    return off;
}

// Keeps v where it is computed: without it the compiler sinks a plane's sums to the end of the loop body, past the
// next plane's work, with every LDS word they need held in registers until then.
__device__ __forceinline__ void
hold(float& v)
{
    asm volatile("" : "+v"(v));
}

// a b + c as a three-address v_fma_f32. The compiler prefers v_fmac (result in c's register) and, where the result
// belongs elsewhere, a move: 18 of 236 VALU instructions a plane in the forward step.
__device__ __forceinline__ float
fma3(float a, float b, float c)
{
    float r;
    asm("v_fma_f32 %0, %1, %2, %3" : "=v"(r) : "s"(a), "v"(b), "v"(c));
    return r;
}

// Moves the queue of mixed partial sums one plane on and absorbs the differences d[1..RO] of that plane, in one FMA per
// slot: afterwards q[j] belongs to output plane p - RO + j (plane p at offset +n feeds output p - n, at -n output p + n
// with the sign flipped). Slots go upwards, so each is read by its left neighbour before it is written.
template <int RO>
__device__ __forceinline__ void
absorb(float (&q)[2 * RO + 1], const float (&d)[RO + 1])
{
#pragma unroll
    for (int j = 0; j < 2 * RO; ++j) {
        const int n = j < RO ? RO - j : j - RO;
        q[j] = n ? fma3(j < RO ? FD<RO>::e[n] : -FD<RO>::e[n], d[n], q[j + 1]) : q[j + 1];
        hold(q[j]);
    }
    q[2 * RO] = -FD<RO>::e[RO] * d[RO];
    hold(q[2 * RO]);
}

// Words of a plane: `plane` is a scalar (the volume plus a uniform plane or tile-origin offset), `off` a 32-bit byte
// offset of the lane, so a load needs one address register and no 64-bit vector arithmetic (64-bit offsets made the
// compiler keep one pointer per volume and lane: 222 VGPRs for the forward update where 18 volumes are touched).
__device__ __forceinline__ float
ldp(const float* __restrict__ plane, unsigned off)
{
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(plane) + off);
}
__device__ __forceinline__ float4
ldp4(const float* __restrict__ plane, unsigned off) // 16-byte aligned
{
    return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(plane) + off);
}
__device__ __forceinline__ void
stp(float* __restrict__ plane, unsigned off, float v)
{
    *reinterpret_cast<float*>(reinterpret_cast<char*>(plane) + off) = v;
}

// Cooperative load of one plane tile with halos into LDS. `origin` is the global index of tile element (0, 0), i.e.
// of the point (x0 - HX, y0 - HY, z). Elements whose tile column is >= xlim or row >= ylim are set to zero (they
// are outside the region any valid output reads).
template <int BY, int W, int H>
__device__ __forceinline__ void
load_tile(float (*t)[W], const float* __restrict__ src, long origin, long ldx, int xlim, int ylim)
{
    for (int k = threadIdx.y * BX + threadIdx.x; k < W * H; k += BX * BY) {
        const int ly = k / W;
        const int lx = k - ly * W;
        float v = 0.0f;
        if (lx < xlim && ly < ylim)
            v = src[origin + (long)ly * ldx + lx];
        t[ly][lx] = v;
    }
}

// The quads (4 consecutive x points) of a W x H plane tile that one thread of an NT-thread block moves: quad
// q = tid + k NT sits at tile row q / (W/4), column 4 (q mod W/4). Tile elements at columns >= xlim or rows >= ylim
// read as zero (no valid output reads them); quads wholly outside are not loaded, so no load leaves the rows of the
// allocation. The launchers check that ldx is a multiple of 4 and the volumes are 16-byte aligned, and every tile
// origin is a multiple of 4 columns, so each quad is one aligned float4 load and one aligned LDS store. fetch()
// issues the loads; commit() masks and stores them a plane later (a select right after a load would wait for it).
// LANE32: 32-bit byte offsets from a scalar plane pointer (planes of less than 4 GiB), which leave the type2 and type1
// kernels their registers; the elastic kernels have registers to spare and are faster with 64-bit element offsets (strains
// 1.81 -> 1.75 ms at 512^3, 34 -> 31 us at 150 x 203 x 117, velocity 42 -> 40 us there).
template <int W, int H, int NT, bool LANE32 = true>
struct TileQuads
{
    static constexpr int QPR = W / 4, NQ = QPR * H, QT = (NQ + NT - 1) / NT;
    std::conditional_t<LANE32, unsigned, long> off[QT]; // from the tile origin within a plane (64 bits: -1 not loaded)
    int lds[QT];      // first element of the quad in the W x H LDS tile, -1: no quad for this slot
    int keep[QT];     // elements of the quad inside xlim (0..4; 0: not loaded)

    __device__ TileQuads(int tid, long ldx, int xlim, int ylim)
    {
#pragma unroll
        for (int k = 0; k < QT; ++k) {
            const int q = tid + k * NT;
            const int row = q / QPR, lx = 4 * (q - row * QPR);
            const bool has = q < NQ;
            lds[k] = has ? row * W + lx : -1;
            keep[k] = has && row < ylim ? min(max(xlim - lx, 0), 4) : 0;
            if constexpr (LANE32)
                off[k] = ((unsigned)row * (unsigned)ldx + (unsigned)lx) * 4u;
            else
                off[k] = keep[k] > 0 ? (long)row * ldx + lx : -1;
        }
    }
    __device__ __forceinline__ void fetch(float4 (&r)[QT], const float* __restrict__ origin) const
    {
#pragma unroll
        for (int k = 0; k < QT; ++k)
            if constexpr (LANE32) {
                if (keep[k] > 0)
                    r[k] = ldp4(origin, here(off[k]));
            } else if (off[k] >= 0) {
                r[k] = *reinterpret_cast<const float4*>(origin + off[k]);
            }
    }
    __device__ __forceinline__ void commit(float* tile, const float4 (&r)[QT]) const
    {
#pragma unroll
        for (int k = 0; k < QT; ++k) {
            if (lds[k] < 0)
                continue;
            const int n = keep[k];
            const float4 v = make_float4(n > 0 ? r[k].x : 0.0f, n > 1 ? r[k].y : 0.0f, n > 2 ? r[k].z : 0.0f,
                                         n > 3 ? r[k].w : 0.0f);
            *reinterpret_cast<float4*>(tile + lds[k]) = v;
        }
    }
};

} // namespace tti

namespace tti {
constexpr int BYS = 8;  // rows per block of the reference-structure stencil kernels
constexpr int BYL = 16; // rows per block of the light ones (forward derivatives, adjoint update)

// Tile of a stencil block in a (gridDim.x, gridDim.y, gridDim.z) launch in XCD order. The dispatcher hands
// consecutive blocks (x fastest, then y, then z) to the 8 XCDs in turn; here each XCD instead takes a contiguous range
// of tiles in that order (any grid size: the first N mod 8 XCDs take one more), so blocks that run at the same time on
// one XCD are x and y neighbours and share their halo lines in its L2. (Measured at 512^3: derivatives 1.79 -> 1.38 ms
// with 16-row blocks and 256-plane chunks, adjoint derivatives 3.40 -> 3.09 ms, density gradient 3.54 -> 3.46 ms.)
__device__ __forceinline__ void
stencil_tile(int& bx, int& by, int& bz)
{
    const int gx = gridDim.x, gy = gridDim.y, n = gx * gy * gridDim.z;
    const int l = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const int q = n / 8, r = n % 8, k = l % 8;
    const int t = k * q + min(k, r) + l / 8;
    bx = t % gx;
    by = (t / gx) % gy;
    bz = t / (gx * gy);
}

// Validates the ghost requirement of the radius-ro stencils: the interior must sit at least ro points inside the
// allocated x and y extents (the z extent is the caller's contract, as in the reference launchers).
inline bool
ranges_ok(int ixbeg, int ixend, int iybeg, int iyend, int izbeg, int izend, int ldimx, int ldimy, int ro = R)
{
    return ixbeg >= ro && iybeg >= ro && izbeg >= ro && ixend >= ixbeg && iyend >= iybeg && izend >= izbeg &&
           ixend + ro < ldimx && iyend + ro < ldimy;
}

// Whether the quad-staged kernels apply: tile origins (ixbeg - 4 or - 8 + 64 k) and rows (ldimx) a multiple of 4 floats and
// every tile source 16-byte aligned, so each tile quad is one aligned float4 load, and planes of less than 4 GiB, which
// they address with 32-bit byte offsets. Otherwise the launchers use the
// element-wise kernels.
inline bool
quads_fit(int ixbeg, int ldimx, int ldimy, std::initializer_list<const float*> tiles)
{
    if (ixbeg % 4 || ldimx % 4 || (long)ldimx * ldimy >= (1L << 30))
        return false;
    for (const float* p : tiles)
        if (reinterpret_cast<uintptr_t>(p) % 16)
            return false;
    return true;
}

inline dim3
stencil_grid(int ixbeg, int ixend, int iybeg, int iyend, int izbeg, int izend, int bz, int by = BYS)
{
    const int nx = ixend - ixbeg + 1, ny = iyend - iybeg + 1, nz = izend - izbeg + 1;
    return dim3((nx + BX - 1) / BX, (ny + by - 1) / by, (nz + bz - 1) / bz);
}

// What chunk_depth needs of a z-marching kernel: the blocks per CU that make a round and the planes' worth of a chunk's
// prologue and recomputed halo, both from its sweep over chunk depths of 2 to 256 planes at 64^3 to 320 x 288 x 240. The
// element-wise kernels of the same operators take the constants of the tiled ones. The deepest chunk is 256 planes (4%
// more reads at 128; no faster at 512).
struct Chunk
{
    int per_cu;
    float warm;
    int cap = 256;
    float full = 2.0f; // share of one round that the deepest chunk's blocks have to fill to be taken (2: never)
};

inline int
stencil_bz(int ixbeg, int ixend, int iybeg, int iyend, int izbeg, int izend, Chunk k, int by = BYS)
{
    const dim3 g = stencil_grid(ixbeg, ixend, iybeg, iyend, izbeg, izend, 1, by);
    return chunk_depth((int)g.z, (long)g.x * g.y, k.per_cu * CUS, k.warm, k.cap, k.full);
}
} // namespace tti
