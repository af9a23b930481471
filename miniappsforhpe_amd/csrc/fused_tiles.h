#pragma once
// Fused single-pass TTI time steps for gfx950: one kernel per forward step and one per adjoint step.
//
// The reference runs a forward step as loop2 -> derivatives -> update (three passes, each a full HBM sweep,
// simulator2/simulator2SetUp.cu:530-599). Here one kernel reads sigma_{n+1} (2 fields), u_n (2), the 8 model words,
// and writes u_{n+1} and sigma_{n+2}: 16 words = 64 B per grid-point update. The time update of sigma is rotated
// into the same kernel (sigma_{n+2} = A sigma_{n+1} + B dt u_{n+1} is pointwise), so sigma ping-pongs between two
// buffers and u is updated in place.
//
// The adjoint step (simulator2/simulator2SetUp.cu:662-737: adjoint derivatives -> update -> loop2) is naturally a
// single pass: u' = u + dt L^T(sigma) (or the sponge form), sigma' = A sigma + B dt u'.  The zero-lag imaging
// condition g += u' * u_snap + w' * w_snap (kernels/kernel_type2_small.cu:42-59) is fused into it, accumulating in
// FP64, with the snapshot read in FP32, FP16 (per-64-point power-of-two scale) or BF16.
//
// Ghost semantics are those of the reference single-volume case: derivative fields are zero outside the interior
// (the reference writes them on the interior only and never fills their outer ghosts) and sigma ghosts hold what
// the caller stored there.
//
// A block marches over a chunk of z planes with one output column per pair of threads, one for each field (64 x 8 x 2
// threads). Per plane p it stages tiles with an 8-point halo in LDS, builds the staggered derivatives d = b D- sigma (of
// the adjoint's S) of plane p on the tile plus a 4-point rim, and absorbs plane p into register queues. Forward, output
// plane o = p - 4 is finalised with the z part coming from a per-thread column stream 7 planes ahead; the adjoint's S_z
// comes from the tile centres and its output plane is p - 7.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "stencil_common.h"
#include "tti_fused.h"

#include <initializer_list>
#include <type_traits>

namespace tti {

namespace fused {

constexpr int TW = BX + 16;               // width of a tile with halo 8
constexpr int BW = BX + 8;                // and with halo 4
constexpr int SNAP_SEG = 64;              // points per x-row segment of an FP16 snapshot (one scale each)

struct Snap
{
    int mode; // TTI_SNAP_NONE / FP32 / FP16 / BF16
    void* a;  // u
    void* b;  // w
    float* sa;
    float* sb;
    long ldx; // row length of the snapshot arrays (multiple of 64)
    long ldy;
    void* c;  // sigma_H of the step (density image), or null
    void* d;  // sigma_V
    float* sc;
    float* sd;
};

struct Box
{
    int ixbeg, ixend, iybeg, iyend, izbeg, izend;
    long ldx, ldy;
    int fs; // stress-free surface at plane izbeg (the z derivatives of planes <= izbeg mirrored, see mirror_dz)
};

// Free-surface mirror of the z-derivative queue (kernels/kernel_type2_small.cu:5-40): d_z is even about
// izbeg + 1/2, d_z(iz) = d_z(2 izbeg + 1 - iz) for every iz <= izbeg. When the queue window q[c .. c+7] holds
// d_z(izbeg - 3 .. izbeg + 4) (output plane o = izbeg), its first four slots take the last four in reverse; the
// outputs after it see the mirrored values as the window moves on.
template <int C, int N>
__device__ __forceinline__ void
mirror_dz(float (&q)[N])
{
#pragma unroll
    for (int k = 0; k < 4; ++k)
        q[C + k] = q[C + 7 - k];
}

// Block schedule within one z chunk: tile r -> (bxi, byi). strip <= 0 or >= ntx: x fastest over full rows; otherwise
// the chunk is cut into vertical strips of `strip` x tiles (the last one narrower), x fastest within a strip, then y,
// strip after strip. Narrow strips keep the blocks that run at the same time on one XCD closer together in x-y
// (their halos overlap in that XCD's L2); the autotuner picks the width.
__device__ __forceinline__ void
tile_xy(int r, int ntx, int nty, int strip, int& bxi, int& byi)
{
    if (strip <= 0 || strip >= ntx) {
        bxi = r % ntx;
        byi = r / ntx;
        return;
    }
    const int s = r / (strip * nty);
    const int w = min(strip, ntx - s * strip);
    const int q = r - s * strip * nty;
    byi = q / w;
    bxi = s * strip + q % w;
}

// XCD-aware tile decode: consecutive hardware blocks go round-robin over the 8 XCDs; each XCD gets a contiguous range
// of tiles (in the block schedule's order, then z chunk) so neighbouring tiles share halo lines in the same L2.
__device__ __forceinline__ bool
decode_tile(int ntx, int nty, int ntz, int strip, int& bxi, int& byi, int& bzi)
{
    const int nt = ntx * nty * ntz;
    const int bid = blockIdx.x;
    const int per = (nt + 7) / 8;
    const int t = (bid % 8) * per + bid / 8;
    if (t >= nt)
        return false;
    bzi = t / (ntx * nty);
    tile_xy(t - bzi * ntx * nty, ntx, nty, strip, bxi, byi);
    return true;
}

// v moved across lanes by the DPP control CTRL, into the rows selected by ROWS (lanes of other rows keep v)
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float
dpp(float v)
{
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false));
}

// Maximum over the 64 lanes of the wave, returned to every lane. DPP moves on the VALU (no LDS round trips): pairs
// and quads by quad_perm, 8 and 16 lanes by the half-row and row mirrors, then lane 15 of each row broadcast into
// rows 1 and 3 and lane 31 into rows 2 and 3, so lane 63 holds the maximum of all rows.
__device__ __forceinline__ float
wave_max(float v)
{
    v = fmaxf(v, dpp<0xb1>(v));       // quad_perm [1, 0, 3, 2]
    v = fmaxf(v, dpp<0x4e>(v));       // quad_perm [2, 3, 0, 1]
    v = fmaxf(v, dpp<0x141>(v));      // row_half_mirror
    v = fmaxf(v, dpp<0x140>(v));      // row_mirror
    v = fmaxf(v, dpp<0x142, 0xa>(v)); // row_bcast:15
    v = fmaxf(v, dpp<0x143, 0xc>(v)); // row_bcast:31
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Stores one 64-point row segment of a snapshot field (all 64 lanes of the wave call this). I = index type.
template <class I>
__device__ __forceinline__ void
snap_store(int mode, void* arr, float* scales, I idx, I sidx, bool act, float v)
{
    if (mode == TTI_SNAP_FP32) {
        if (act)
            reinterpret_cast<float*>(arr)[idx] = v;
    } else if (mode == TTI_SNAP_FP16) {
        const float m = wave_max(act ? fabsf(v) : 0.0f);
        int e = 0;
        frexpf(m, &e); // m < 2^e
        if (m == 0.0f)
            e = 0;
        if (act)
            reinterpret_cast<__half*>(arr)[idx] = __float2half(ldexpf(v, 14 - e));
        if (threadIdx.x == 0)
            scales[sidx] = ldexpf(1.0f, e - 14);
    } else if (mode == TTI_SNAP_BF16) {
        if (act)
            reinterpret_cast<__hip_bfloat16*>(arr)[idx] = __float2bfloat16(v);
    }
}

template <class I>
__device__ __forceinline__ float
snap_load(int mode, const void* arr, const float* scales, I idx, I sidx)
{
    if (mode == TTI_SNAP_FP32)
        return reinterpret_cast<const float*>(arr)[idx];
    if (mode == TTI_SNAP_FP16)
        return __half2float(reinterpret_cast<const __half*>(arr)[idx]) * scales[sidx];
    if (mode == TTI_SNAP_BF16)
        return __bfloat162float(reinterpret_cast<const __hip_bfloat16*>(arr)[idx]);
    return 0.0f;
}

// The stored words of one snapshot value, loaded one plane before they are used and decoded then by snap_decode
// (a decode right after the load would wait for that load, and for every memory operation issued before it)
struct SnapWord
{
    unsigned v; // FP32 bits, or the 16-bit FP16 / BF16 word
    float s;    // FP16: the segment's scale
};

template <class I>
__device__ __forceinline__ SnapWord
snap_fetch(int mode, const void* arr, const float* scales, I idx, I sidx)
{
    SnapWord r{ 0u, 1.0f };
    if (mode == TTI_SNAP_FP32) {
        r.v = reinterpret_cast<const unsigned*>(arr)[idx];
    } else if (mode == TTI_SNAP_FP16) {
        r.v = reinterpret_cast<const unsigned short*>(arr)[idx];
        r.s = scales[sidx];
    } else if (mode == TTI_SNAP_BF16) {
        r.v = reinterpret_cast<const unsigned short*>(arr)[idx];
    }
    return r;
}

// the value snap_load returns for the same words
__device__ __forceinline__ float
snap_decode(int mode, SnapWord r)
{
    if (mode == TTI_SNAP_FP32)
        return __uint_as_float(r.v);
    if (mode == TTI_SNAP_FP16)
        return __half2float(__ushort_as_half((unsigned short)r.v)) * r.s;
    if (mode == TTI_SNAP_BF16)
        return __uint_as_float(r.v << 16); // BF16 is the high half of the FP32 word
    return 0.0f;
}

constexpr int TQ_PER_ROW = TW / 4, BQ_PER_ROW = BW / 4; // quads per row of the two tile shapes

// ------------------------------------------------------------------------------------------------------------------
// Forward step: u += dt L(sigma) (+ source), sigma_out = A sigma + B dt u_new; optional snapshot of u_new.
// Same arithmetic as kernels/kernel_type2_fwd_drv.cu:148-362 + kernels/kernel_type2_fwd.cu:264-540 +
// kernels/kernel_base.cu:82-104, evaluated in one sweep.
//
// Pipeline per output plane o (tile plane p = o + 4): the tile of plane p is already in LDS buffer `par`;
//   A  load the column word of plane o + 8, store the prefetched tile of plane p + 1 into the other buffer, fetch the
//      tile of plane p + 2 (loads are issued before this plane's stores: one counter tracks both)
//   B  z-mixed partial sums, the x-y mixed term, and the staggered derivatives d_x, d_y of plane p -> LDS
//   C  d_z(o+4) from the column queue, V and H of plane o; H1 and V2 -> LDS for the other field's thread
//   -  the one barrier: every read of the tile comes before it, every read of d_x, d_y and H1, V2 after it, and those
//      alternate between two buffers as the tiles do
//   D  D+ of d_x, d_y; update and store plane o, load the pointwise words of plane o + 1
// Planes p outside the chunk feed only z stencils, so their bodies leave d_x, d_y and the x-y term out.
//
// What bounds it (512^3): VALU issue 66% and LDS 58% of the busy cycles in lock-step phases, and 11.1 GB moved, at 2.34 ms
// 4.7 TB/s, about what a copy reaches (with one volume in the place of seven models it runs 12% faster). One thread per
// column needed 253 VGPRs (8 waves a CU) where one per column and field takes 122 (16 waves); the tile of 8 rows instead of
// 4 reads 40% fewer halo quads and computes 2 instead of 3 d_y per column, the second barrier went, and the partial sums
// shift as they are summed. With the loads below, 2.78 -> 2.48 ms per step, 2.98 -> 2.74 ms with the FP16 snapshot (one
// box, in turn; other boxes take 2.3), and with the shortened rim planes 64^3 27 -> 17 us.
//
// Global addresses are 32-bit byte offsets from the (scalar) base pointers: the launcher checks that every volume is
// smaller than 4 GiB.
// ------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ float
ldf(const float* __restrict__ p, unsigned off)
{
    return *reinterpret_cast<const float*>(__builtin_assume_aligned(reinterpret_cast<const char*>(p) + off, 4));
}
__device__ __forceinline__ float4
ldf4(const float* __restrict__ p, unsigned off) // off = 0 mod 16
{
    return *reinterpret_cast<const float4*>(__builtin_assume_aligned(reinterpret_cast<const char*>(p) + off, 16));
}
__device__ __forceinline__ void
stf(float* __restrict__ p, unsigned off, float v)
{
    *reinterpret_cast<float*>(__builtin_assume_aligned(reinterpret_cast<char*>(p) + off, 4)) = v;
}

// Byte offset (within a plane) of the tile quad that starts at (gx, gy), clamped into the allocated rows
// [iybeg-4, iyend+4] and quad starts [ixbeg-4, ldx-4]. Clamped quads read real data of the volume that no output
// uses: values outside the allocated region only feed derivatives of non-interior points, which are zeroed.
__device__ __forceinline__ unsigned
quad_off(const Box& g, int gx, int gy)
{
    gx = min(max(gx, g.ixbeg - R), (int)g.ldx - 4);
    gy = min(max(gy, g.iybeg - R), g.iyend + R);
    return ((unsigned)gy * (unsigned)g.ldx + (unsigned)gx) * 4u;
}

// rho = 1/b by the hardware reciprocal (v_rcp_f32, 1 ulp) instead of an IEEE division sequence; zero where b is
// zero (outside the models' allocation)
__device__ __forceinline__ float
recip(float b)
{
    return b != 0.0f ? __builtin_amdgcn_rcpf(b) : 0.0f;
}

__device__ __forceinline__ bool
in_xy(const Box& g, int x, int y)
{
    return x >= g.ixbeg && x <= g.ixend && y >= g.iybeg && y <= g.iyend;
}

// staggered difference sum_n c_n (v[3+n] - v[4-n]) over 8 consecutive values v[0..7]
template <class F>
__device__ __forceinline__ float
stg8(F&& v)
{
    float a = 0.0f;
#pragma unroll
    for (int n = 1; n <= R; ++n)
        a += cstg(n) * (v(3 + n) - v(4 - n));
    return a;
}

constexpr int FWD_BY = 8; // rows per forward block (STEP_SLOTS, STEP_WARM and the launch bounds hold for these)
constexpr int FU = 2;     // forward planes per loop iteration

// One block's tile (bxi, byi, bzi) of a forward step; called by the single-volume kernel and the batched one. One thread
// per column and field (threadIdx.z: 0 sigma_H and u, 1 sigma_V and w).
template <int FBY, int SNAP, bool SPONGE, bool SIG = false>
__device__ __forceinline__ void
fwd_tile(const float* __restrict__ s1, const float* __restrict__ s2, float* __restrict__ s1o, float* __restrict__ s2o,
         float* __restrict__ u, float* __restrict__ w, const float* __restrict__ m1, const float* __restrict__ m2,
         const float* __restrict__ m3, const float* __restrict__ m4, const float* __restrict__ vrx,
         const float* __restrict__ vry, const float* __restrict__ vrz, const float* __restrict__ b,
         const ab2* __restrict__ abx, const ab2* __restrict__ aby, const ab2* __restrict__ abz, const Box& g, float dt,
         float invdx, float invdy, float invdz, float i4xy, float i4yz, float i4zx, unsigned src_off, float src_val,
         const Snap& snap, int bz, int bxi, int byi, int bzi)
{
    constexpr int NT = BX * FBY;                  // threads per field
    constexpr int FTH = FBY + 16, FBH = FBY + 8;  // tile heights (halo 8, halo 4)
    constexpr int FTQ = TQ_PER_ROW * FTH, FBQ = BQ_PER_ROW * FBH;
    constexpr int QT = (FTQ + NT - 1) / NT;                 // sigma quads per thread (of its field)
    constexpr int YI = FBH / FBY;                           // d_y items per thread
    static_assert(FBH % FBY == 0, "d_y rows split evenly over the thread rows");
    static_assert(FBQ <= 2 * NT, "one b quad per thread");
    __shared__ __align__(16) float T[2][2][FTH][TW]; // [parity][field] sigma, halo 8: (x0-8+lx, y0-8+ly)
    __shared__ __align__(16) float Bt[2][FBH][BW];   // b, halo 4: (x0-4+lx, y0-4+ly)
    __shared__ float X[2][2][FBY][BW];               // d_x at (x0-4+j, y0+r)
    __shared__ float Y[2][2][FBH][BX];               // d_y at (x0+c, y0-4+j)
    __shared__ float EX[2][2][FBY][BX];              // H1 and V2, which the other field's update needs

    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * BX + tx;
    const int F = __builtin_amdgcn_readfirstlane(threadIdx.z);
    const int x0 = g.ixbeg + bxi * BX, y0 = g.iybeg + byi * FBY, z0 = g.izbeg + bzi * bz;
    const int z1 = min(z0 + bz, g.izend + 1);
    const int ix = x0 + tx, iy = y0 + ty;
    const bool active = ix <= g.ixend && iy <= g.iyend;
    const unsigned PB = (unsigned)g.ldx * (unsigned)g.ldy * 4u; // bytes per plane
    const unsigned colb = active ? ((unsigned)iy * (unsigned)g.ldx + (unsigned)ix) * 4u : 0u;
    const float* const s = F ? s2 : s1;
    float *const so = F ? s2o : s1o, *const uw = F ? w : u;
    // u += dt (m1 H1 + m4 V1 + m2 V2), w += dt (m2 H1 + m3 V2 + m4 H2), summed in this order
    const float *const ma = F ? m2 : m1, *const mb = F ? m3 : m4, *const mc = F ? m4 : m2;
    // snapshot element offsets (32-bit: the launchers check that a snapshot field has < 2^32 elements): plane
    // stride and this thread's column within a plane; rows are whole 64-point segments, so an element's scale is its
    // offset / 64
    const unsigned s_plane = (unsigned)(snap.ldy * snap.ldx);
    const unsigned s_col = (unsigned)(iy - g.iybeg) * (unsigned)snap.ldx + (unsigned)(ix - g.ixbeg);
    float axy = 1.0f, bxy = 1.0f;
    if (SPONGE && active) {
        axy = fminf(abx[ix].a, aby[iy].a);
        bxy = fminf(abx[ix].b, aby[iy].b);
    }
    // tile quads (clamped into the allocation, see quad_off): sigma of this thread's field, b over all threads. Slots
    // past a tile's quad count load and store nothing, so whole waves skip them
    int tq_row[QT], tq_lx[QT];
    unsigned tqb[QT];
#pragma unroll
    for (int k = 0; k < QT; ++k) {
        const int q = min(tid + k * NT, FTQ - 1);
        tq_row[k] = q / TQ_PER_ROW;
        tq_lx[k] = 4 * (q - tq_row[k] * TQ_PER_ROW);
        tqb[k] = quad_off(g, x0 - 8 + tq_lx[k], y0 - 8 + tq_row[k]);
    }
    const int bq_id = tid + F * NT, bq_row = min(bq_id, FBQ - 1) / BQ_PER_ROW,
              bq_lx = 4 * (min(bq_id, FBQ - 1) - bq_row * BQ_PER_ROW);
    const unsigned bqb = quad_off(g, x0 - 4 + bq_lx, y0 - 4 + bq_row);
    auto tq_ok = [&](int k) { return k * NT + NT <= FTQ || tid + k * NT < FTQ; };
    float4 pt[QT], pb;
    auto fetch = [&](int pp) {
        const unsigned o = (unsigned)pp * PB;
#pragma unroll
        for (int k = 0; k < QT; ++k)
            if (tq_ok(k))
                pt[k] = ldf4(s, o + tqb[k]);
        if (bq_id < FBQ)
            pb = ldf4(b, o + bqb);
    };
    auto commit = [&](int buf) {
#pragma unroll
        for (int k = 0; k < QT; ++k)
            if (tq_ok(k))
                *reinterpret_cast<float4*>(&T[buf][F][tq_row[k]][tq_lx[k]]) = pt[k];
        if (bq_id < FBQ)
            *reinterpret_cast<float4*>(&Bt[buf][bq_row][bq_lx]) = pb;
    };
    // d_x items: the thread's own column, whose taps the z-x term needs as well, and the 4 rim columns on either side of
    // each row on the first threads; d_y items: rows ty + h * FBY of the halo-4 band, column tx (between them the taps
    // of the y-z term). The scale is 1/d for interior points and zero elsewhere (floats: no lane masks live across the
    // loop).
    constexpr int XE = 8 * FBY; // rim items
    static_assert(XE <= NT, "one rim item per thread");
    const int xe_r = min(tid, XE - 1) / 8, xe_k = min(tid, XE - 1) % 8, xe_j = xe_k < 4 ? xe_k : BX + xe_k;
    const float xs = in_xy(g, ix, iy) ? invdx : 0.0f;
    const float xes = in_xy(g, x0 - 4 + xe_j, y0 + xe_r) ? invdx : 0.0f;
    float ys[YI];
#pragma unroll
    for (int h = 0; h < YI; ++h)
        ys[h] = in_xy(g, x0 + tx, y0 - 4 + ty + h * FBY) ? invdy : 0.0f;

    // Register queues along z. The loop body is instantiated for FU consecutive planes; the body of plane o with
    // c = o - (z0 - 8) mod FU sees each delay queue through a window starting at slot c (FU - 1 spare slots per queue),
    // and after the FU-th plane the queues shift by FU. The partial sums shift as they are summed (absorb).
    float sq[8 + FU]; // sigma(o + k)   at [c + k], k = 0..7 (slot c + 8 receives sigma(o + 8))
    float dz[7 + FU]; // d_z(o - 3 + k) at [c + k], k = 0..7
    float xx[4 + FU]; // D+_x d_x (o + k), unscaled by rho, at [c + k], k = 0..4
    float yy[4 + FU]; // D+_y d_y
    float xy[4 + FU]; // X_xy sigma
    float bq[4 + FU]; // b(o + k), from the tile's centre: for d_z(o + 4) and the output plane
    float qx[9], qy[9]; // z-x and y-z mixed partial sums of output o + j
#pragma unroll
    for (int k = 0; k < 7 + FU; ++k)
        dz[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 4 + FU; ++k)
        xx[k] = yy[k] = xy[k] = bq[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 9; ++k)
        qx[k] = qy[k] = 0.0f;
    // column words: sigma at a plane clamped into the allocation (a clamped sigma only meets a zero b; b is zeroed
    // outside the interior planes where it is used)
    auto col = [&](int q) { return ldf(s, (unsigned)min(max(q, g.izbeg - R), g.izend + R) * PB + colb); };
#pragma unroll
    for (int k = 0; k < 8; ++k)
        sq[k] = col(z0 - 8 + k);
    // pointwise words of an output plane: rx ry rz are loaded again once their plane's V and H are formed, the model
    // words and u or w once its update is, so each has a whole plane to arrive
    // These loads are issued on every path (planes outside the block's read its nearest one), and so is the tile's fetch
    // in the block's own planes: past a load that may not have been issued, the wait for an earlier one (the tile, at the
    // next plane's stage A) drains everything in flight, down to the stores just made. 512^3 2.74 -> 2.47 ms per step.
    float pr[3], pm[4];
    auto fetch_r = [&](int o) {
        const unsigned io = (unsigned)min(max(o, z0), z1 - 1) * PB + colb;
        pr[0] = ldf(vrx, io);
        pr[1] = ldf(vry, io);
        pr[2] = ldf(vrz, io);
    };
    auto fetch_m = [&](int o) {
        const unsigned io = (unsigned)min(max(o, z0), z1 - 1) * PB + colb;
        pm[0] = ldf(ma, io);
        pm[1] = ldf(mb, io);
        pm[2] = ldf(mc, io);
        pm[3] = ldf(uw, io);
    };

    fetch(z0 - R);
    commit(0);
    fetch(z0 - R + 1);
    __syncthreads();

    auto body = [&](auto curc, auto ownc, int o) {
        constexpr int cur = decltype(curc)::value; // o - (z0 - 8) mod FU: queue window
        constexpr bool own = decltype(ownc)::value; // plane p = o + 4 is one of the block's output planes
        constexpr int par = cur & 1;               // parity of o: tile buffer of plane p (the other: p + 1)
        const int p = o + R;
        const bool pint = p >= g.izbeg && p <= g.izend;
        const float pin = pint ? 1.0f : 0.0f;
        // ---- A: this plane's loads first, so that waiting for them never waits for the stores below (one counter covers
        // loads and stores): the column word of plane o + 8; the tile of plane p + 1 goes to the other buffer (last read
        // before the previous plane's barrier) and the tile of plane p + 2 is fetched
        __builtin_amdgcn_s_setprio(3);
        sq[cur + 8] = col(o + 8);
        if (own || p + 1 <= z1 + R - 1)
            commit(par ^ 1);
        if (own || p + 2 <= z1 + R - 1)
            fetch(p + 2);
        __builtin_amdgcn_s_setprio(0);
        const float(*t)[TW] = T[par][F];
        // ---- B: the z-mixed partial sums; from the planes whose own outputs this block computes also the x-y mixed term,
        // d_x on rows of the tile (x' in [x0-4, x0+68)) and d_y on columns (y' in [y0-4, y0+BY+4)) (the scale is zero for
        // non-interior points: every tile value is finite)
        {
            float ddx[5], ddy[5];
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                ddx[n] = t[ty + 8][tx + 8 + n] - t[ty + 8][tx + 8 - n];
                ddy[n] = t[ty + 8 + n][tx + 8] - t[ty + 8 - n][tx + 8];
                hold(ddx[n]), hold(ddy[n]);
            }
            absorb<R>(qx, ddx);
            absorb<R>(qy, ddy);
        }
        if constexpr (own) {
            float fxy = 0;
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                fxy += ecen(n) * ((t[ty + 8 + n][tx + 8 + n] - t[ty + 8 - n][tx + 8 + n]) +
                                  (t[ty + 8 - n][tx + 8 - n] - t[ty + 8 + n][tx + 8 - n]));
                hold(fxy);
            }
            xy[cur + 4] = fxy * i4xy;
            hold(xy[cur + 4]);
            float xv = Bt[par][ty + 4][tx + 4] * (xs * pin) * stg8([&](int k) { return t[ty + 8][tx + 4 + k]; });
            hold(xv);
            X[par][F][ty][tx + 4] = xv;
            if (tid < XE) {
                xv = Bt[par][xe_r + 4][xe_j] * (xes * pin) * stg8([&](int k) { return t[xe_r + 8][xe_j + k]; });
                hold(xv);
                X[par][F][xe_r][xe_j] = xv;
            }
#pragma unroll
            for (int h = 0; h < YI; ++h) {
                const int j = ty + h * FBY;
                float yv = Bt[par][j][tx + 4] * (ys[h] * pin) * stg8([&](int k) { return t[j + k][tx + 8]; });
                hold(yv);
                Y[par][F][j][tx] = yv;
            }
        }
        // ---- C: d_z(o+4), then V and H of plane o
        bq[cur + 4] = Bt[par][ty + 4][tx + 4];
        dz[cur + 7] = (pint ? bq[cur + 4] : 0.0f) * invdz * stg8([&](int k) { return sq[cur + k]; });
        if (g.fs && o == g.izbeg)
            mirror_dz<cur>(dz);
        float V = 0.0f, Hf = 0.0f;
        if (o >= z0) {
            const float fz = stg8([&](int k) { return dz[cur + k]; });
            const float vx = pr[0], vy = pr[1], vz = pr[2];
            const float rho = recip(bq[cur]);
            const float fxx = xx[cur] * rho, fyy = yy[cur] * rho, fzz = fz * invdz * rho;
            const float fzx = qx[0] * i4zx, fyz = qy[0] * i4yz;
            const float rx2 = vx * vx, ry2 = vy * vy, rz2 = vz * vz;
            const float rxy = 2.0f * vx * vy, ryz = 2.0f * vy * vz, rzx = 2.0f * vz * vx;
            // sums of products are written as explicit fmaf chains (left to right): with contraction left to the
            // compiler, copies of this body (the loop's warm-up planes vs the rest) may fuse different products and
            // round differently, which would make a point's value depend on where its z chunk starts
            V = fmaf(ryz, fyz, fmaf(rzx, fzx, fmaf(rxy, xy[cur], fmaf(rz2, fzz, fmaf(ry2, fyy, rx2 * fxx)))));
            Hf = __fsub_rn(__fadd_rn(__fadd_rn(fxx, fyy), fzz), V); // plain adds: no product fused
            EX[par][F][ty][tx] = F ? V : Hf;
        }
        fetch_r(o + 1);
        // the one barrier of the plane: X, Y and EX of this plane are complete, and every read of tile buffer `par` and
        // of the previous plane's X, Y, EX buffers is done
        __syncthreads();
        // ---- D: D+ of d_x, d_y of plane p, and the update of plane o
        if constexpr (own) {
            float fx = 0, fy = 0;
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                const float c = cstg(n);
                fx += c * (X[par][F][ty][tx + 4 + n] - X[par][F][ty][tx + 5 - n]);
                fy += c * (Y[par][F][ty + 4 + n][tx] - Y[par][F][ty + 5 - n][tx]);
                hold(fx), hold(fy);
            }
            xx[cur + 4] = fx * invdx;
            yy[cur + 4] = fy * invdy;
            hold(xx[cur + 4]), hold(yy[cur + 4]);
        }
        const bool fin = o >= z0 && active;
        float unew = 0.0f, snew = 0.0f;
        const unsigned io = (unsigned)o * PB + colb;
        if (o >= z0) {
            const float e = EX[par][F ^ 1][ty][tx];
            const float r = F ? fmaf(pm[2], Hf, fmaf(pm[1], V, pm[0] * e)) : fmaf(pm[2], e, fmaf(pm[1], V, pm[0] * Hf));
            unew = pm[3] + r * dt;
            if (io == src_off)
                unew += src_val;
            float a = 1.0f, bb = 1.0f;
            if constexpr (SPONGE) {
                a = fminf(axy, abz[o].a);
                bb = fminf(bxy, abz[o].b);
            }
            snew = fmaf(bb * unew, dt, a * sq[cur]);
        }
        fetch_m(o + 1);
        // the stores of plane o
        if (fin) {
            stf(uw, io, unew);
            stf(so, io, snew);
        }
        if (SNAP != TTI_SNAP_NONE && o >= z0 && iy <= g.iyend) {
            const unsigned pz = (unsigned)(o - g.izbeg);
            const unsigned idx = pz * s_plane + s_col, sidx = idx / SNAP_SEG;
            snap_store(SNAP, F ? snap.b : snap.a, F ? snap.sb : snap.sa, idx, sidx, active, unew);
            if constexpr (SIG) // the sigma this step read (its u, w update used it)
                snap_store(SNAP, F ? snap.d : snap.c, F ? snap.sd : snap.sc, idx, sidx, active, sq[cur]);
        }
        if (cur == FU - 1) {
#pragma unroll
            for (int k = 0; k < 8; ++k)
                sq[k] = sq[k + FU];
#pragma unroll
            for (int k = 0; k < 7; ++k)
                dz[k] = dz[k + FU];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                xx[k] = xx[k + FU];
                yy[k] = yy[k + FU];
                xy[k] = xy[k + FU];
                bq[k] = bq[k + FU];
            }
        }
    };

    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    // planes that only feed the z stencils of the block's outputs: 4 before them and 4 after
    auto rim = [&](int o, int end) {
        for (; o < end; ++o)
            if (((o - z0) & 1) == 0)
                body(C0{}, std::false_type{}, o);
            else
                body(C1{}, std::false_type{}, o);
    };
    rim(z0 - 8, z0 - 4);
    for (int o = z0 - 4; o < z1 - 4; o += 2) {
        body(C0{}, std::true_type{}, o);
        if (o + 1 >= z1 - 4)
            break;
        body(C1{}, std::true_type{}, o + 1);
    }
    rim(z1 - 4, z1);
}

// ------------------------------------------------------------------------------------------------------------------
// Adjoint step (reference order, kernels/kernel_type2_grad_snap.cu:242-427 + kernels/kernel_type2_adj.cu:100-260 +
// kernels/kernel_base.cu:82-104):
//   r  = sum_a D+_a (b D-_a S_a) + sum_{a<b} X_ab M_ab,   S_a = rho (lap + r_a^2 hz), M_ab = 2 r_a r_b hz
//   u' = u + dt r            (sponge: u' = A u + B dt r)
//   sigma' = A sigma + B dt u'
//   grad += u' u_snap + w' w_snap   (FP64, when a snapshot is given)
// Same pipeline as the forward kernel; the tile stage holds the pointwise temporaries S_x, S_y, M_xy, M_zx, M_yz
// and b of plane p on a plus-shaped footprint, computed from the 10 prefetched input quads when they are stored.
// ------------------------------------------------------------------------------------------------------------------
struct Temps // lap2 = m4 f2 (see s2_of)
{
    float lap1, hz1, hz2;
};

__device__ __forceinline__ Temps
temps(float f1, float f2, float mm1, float mm2, float mm3, float mm4)
{
    Temps t;
    // explicit fmaf: one fixed rounding for every copy of the code (see the forward finalisation)
    t.lap1 = fmaf(mm2, f2, mm1 * f1);
    t.hz1 = fmaf(-mm2, f2, (-mm1 + mm4) * f1);
    t.hz2 = fmaf(-mm4 + mm3, f2, mm2 * f1);
    return t;
}

// S_a = rho (lap + r_a^2 hz) of either field, each with one fixed rounding (lap2 = m4 f2 is a product itself)
__device__ __forceinline__ float
s_of(float rho, float lap1, float r, float hz1)
{
    return rho * fmaf(r * r, hz1, lap1);
}
__device__ __forceinline__ float
s2_of(float rho, float m4, float f2, float r, float hz2)
{
    return rho * fmaf(m4, f2, __fmul_rn(r * r, hz2));
}

constexpr int ADJ_AX = BX, ADJ_AY = 8; // output columns per block, a pair of threads each

// Half-quads (2 consecutive x points) of the plus-shaped footprint of the adjoint tile, one per thread
template <int AY>
struct AdjShape
{
    static constexpr int NT = 2 * BX * AY;           // threads
    static constexpr int TH = AY + 16, BH = AY + 8;  // footprint with halo 8: (x0-8+lx, y0-8+ly); halo-4 region
    static constexpr int HR = TW / 2;                // half-quads per footprint row
    // rows [8, 8+AY) whole; rows [4, 8) and [8+AY, 12+AY) from x' = 4 (the halo-4 square); the 4 outermost rows on each
    // side from x' = 8 (the y halo of the block's own columns; these need S_y only)
    static constexpr int OUTER = 8 * (HR - 8), NH = OUTER + AY * HR + 8 * (HR - 4);
    static constexpr int YI = BH / AY; // d_y items per thread
    static_assert(NH <= NT && BH % AY == 0, "one footprint half-quad per thread");
};

// Footprint half-quad t (t < NH): its row and x' offset, bands of rows in order
template <int AY>
__device__ __forceinline__ void
adj_half(int t, int& row, int& lx)
{
    constexpr int HR = AdjShape<AY>::HR;
    // (first row, rows, half-quads per row, first one) of the five bands, the two outer ones first, so that the threads
    // of those bands fill whole waves
    constexpr int rs[5] = { 0, 12 + AY, 4, 8, 8 + AY }, br[5] = { 4, 4, 4, AY, 4 };
    constexpr int bq[5] = { HR - 8, HR - 8, HR - 4, HR, HR - 4 }, b0[5] = { 4, 4, 2, 0, 2 };
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const int n = br[k] * bq[k];
        if (t < n) {
            row = rs[k] + t / bq[k];
            lx = 2 * (b0[k] + t % bq[k]);
            return;
        }
        t -= n;
    }
    row = 0;
    lx = 0;
}

// One block's tile of an adjoint step; SNAP = snapshot mode of the imaging condition (TTI_SNAP_NONE: no imaging). One
// thread per column and field (threadIdx.z: 0 sigma_H and u, 1 sigma_V and w). At 512^3 it moves 96 B a point (12.9 GB of
// the 8.6 it needs: 10 words per footprint point), 3.8 TB/s or 0.8 of a copy's rate; VALU is busy 51% and LDS 43% of the
// cycles. With one volume in the place of seven models it takes 2.74 instead of 3.39 ms: a fifth of the time is the models'
// reads, the rest VALU, LDS and the latency between barriers, where what counts is waves to fill the gaps: one thread per
// column held both fields' queues in 256 registers, 8 waves per CU; this holds 16. Each temporary is formed
// once, by the thread that loaded its half-quad, for both fields. S_z comes with the tile, so no second stream of 6
// volumes runs 7 planes ahead, at the price of 3 more recomputed planes per chunk, which form S_z alone. One barrier per
// plane: X and Y are written before it and read after it, the tiles of the next plane go into the other buffer.
// 512^3 3.57 -> 3.37 ms, with FP16 imaging 4.08 -> 3.78 (64-column, 8-row blocks of either kind; 64^3 38 -> 30 us).
template <int SNAP, bool SPONGE>
__device__ __forceinline__ void
adj_tile(const float* __restrict__ a1, const float* __restrict__ a2, float* __restrict__ a1o, float* __restrict__ a2o,
         float* __restrict__ u, float* __restrict__ w, const float* __restrict__ m1, const float* __restrict__ m2,
         const float* __restrict__ m3, const float* __restrict__ m4, const float* __restrict__ vrx,
         const float* __restrict__ vry, const float* __restrict__ vrz, const float* __restrict__ b,
         const ab2* __restrict__ abx, const ab2* __restrict__ aby, const ab2* __restrict__ abz, const Box& g, float dt,
         float invdx, float invdy, float invdz, float i4xy, float i4yz, float i4zx, const Snap& snap,
         double* __restrict__ grad, int bz, int bxi, int byi, int bzi)
{
    constexpr int AY = ADJ_AY;
    using Sh = AdjShape<AY>;
    constexpr int NT = BX * AY, TH = Sh::TH, BH = Sh::BH; // NT: threads per field
    constexpr int DEP = 7;  // output plane o = p - DEP
    constexpr bool imaging = SNAP != TTI_SNAP_NONE;
    // The FP16 image (word and scale) with a sponge is the one form that does not fit 128 VGPRs: it spilled 7 and took 4.34
    // ms at 512^3, with the columns' x-y sponge values read back from LDS 3.78 ms. The other forms keep them in registers.
    constexpr bool tapers = SPONGE && SNAP == TTI_SNAP_FP16;
    // [parity][field] temporaries of plane p
    __shared__ __align__(16) float SX[2][2][AY][TW];  // S_x at (x0-8+lx, y0+r)
    __shared__ __align__(16) float SY[2][2][TH][BX];  // S_y at (x0+c, y0-8+ly)
    __shared__ __align__(16) float MXY[2][2][BH][BW]; // M_xy at (x0-4+lx, y0-4+ly)
    __shared__ __align__(16) float MZX[2][2][AY][BW]; // M_zx at (x0-4+lx, y0+r)
    __shared__ __align__(16) float MYZ[2][2][BH][BX]; // M_yz at (x0+c, y0-4+ly)
    __shared__ __align__(16) float SZ[2][2][AY][BX];  // S_z and sigma of the block's own columns
    __shared__ __align__(16) float SA[2][2][AY][BX];
    __shared__ __align__(16) float Bt[2][BH][BW];     // b at (x0-4+lx, y0-4+ly)
    __shared__ float X[2][2][AY][BW];                 // d_x, d_y
    __shared__ float Y[2][2][BH][BX];
    __shared__ double EX[imaging ? 2 : 1][imaging ? AY : 1][imaging ? BX : 1]; // w' w_snap
    __shared__ float2 AB[tapers ? AY : 1][tapers ? BX : 1];                    // x-y sponge values of the columns

    const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y), tid = ty * BX + tx;
    const int F = __builtin_amdgcn_readfirstlane(threadIdx.z);
    const int x0 = g.ixbeg + bxi * BX, y0 = g.iybeg + byi * AY, z0 = g.izbeg + bzi * bz;
    const int z1 = min(z0 + bz, g.izend + 1);
    const int ix = x0 + tx, iy = y0 + ty;
    const bool active = ix <= g.ixend && iy <= g.iyend;
    const unsigned PB = (unsigned)g.ldx * (unsigned)g.ldy * 4u;
    const unsigned colb = active ? ((unsigned)iy * (unsigned)g.ldx + (unsigned)ix) * 4u : 0u;
    float *const ao = F ? a2o : a1o, *const uw = F ? w : u;
    float axy = 1.0f, bxy = 1.0f;
    if (SPONGE && active) {
        axy = fminf(abx[ix].a, aby[iy].a);
        bxy = fminf(abx[ix].b, aby[iy].b);
    }
    if (tapers && !F)
        AB[ty][tx] = make_float2(axy, bxy); // read past the prologue's barrier
    // snapshot and image element offsets (32-bit: the launchers check both fit): plane strides and this thread's
    // column within a plane; snapshot rows are whole 64-point segments, so an element's scale is its offset / 64
    const unsigned s_plane = (unsigned)(snap.ldy * snap.ldx);
    const unsigned s_col = active ? (unsigned)(iy - g.iybeg) * (unsigned)snap.ldx + (unsigned)(ix - g.ixbeg) : 0u;
    const unsigned g_row = (unsigned)(g.ixend - g.ixbeg + 1);
    const unsigned g_plane = g_row * (unsigned)(g.iyend - g.iybeg + 1);
    const unsigned g_col = active && !F ? (unsigned)(iy - g.iybeg) * g_row + (unsigned)(ix - g.ixbeg) : 0u;

    // this thread's half-quad of the footprint: threads beyond the count load nothing
    const int ht = tid + F * NT;
    int hrow = 0, hlx = 0;
    const bool need = ht < Sh::NH;
    const bool sy_only = ht < Sh::OUTER;
    adj_half<AY>(need ? ht : 0, hrow, hlx);
    // What this thread's half-quad gives, as bits tested where they are used (kept as lane masks they filled the scalar
    // registers): 1 S_x and M_zx rows, 2 S_y and M_yz columns, 4 M_xy and b, 8 S_y alone, 16, 32, 64 a part in planes of
    // level 1, 2, 3
    int role = 0;
    if (need) {
        const bool r8 = hrow >= 8 && hrow < 8 + AY, c8 = hlx >= 8 && hlx < 8 + BX;
        const bool s4 = hlx >= 4 && hlx < 4 + BW && hrow >= 4 && hrow < 4 + BH;
        role = (r8 ? 1 : 0) | (c8 ? 2 : 0) | (s4 ? 4 : 0) | (sy_only ? 8 : 0) | (r8 && c8 ? 16 : 0) |
               (s4 && (r8 || c8) ? 32 : 0) | 64;
    }
    // byte offset within a plane, clamped into the allocation as quad_off does
    const unsigned hb = ((unsigned)min(max(y0 - 8 + hrow, g.iybeg - R), g.iyend + R) * (unsigned)g.ldx +
                         (unsigned)min(max(x0 - 8 + hlx, g.ixbeg - R), (int)g.ldx - 2)) *
                        4u;
    // What the planes outside [z0, z1) give: 2 M_zx, M_yz and S_z (p within 4 planes of the chunk), 1 S_z alone (the 3
    // planes after those); 3 everything; 4 past the last one, no thread's part
    auto level = [&](int p) { return p >= z1 + DEP ? 4 : p >= z1 + R ? 1 : p >= z0 && p < z1 ? 3 : 2; };
    float2 qa1, qa2, qm1, qm2, qm3, qm4, qrx, qry, qrz, qb;
    auto fetch = [&](int p) {
        const unsigned ro = here((unsigned)role);
        if (!(ro & (8u << level(p))))
            return;
        const unsigned i = (unsigned)min(p, g.izend + R) * PB + here(hb); // a clamped plane's S_z only meets a zero b
        auto ld = [&](const float* v) {
            return *reinterpret_cast<const float2*>(
                __builtin_assume_aligned(reinterpret_cast<const char*>(v) + i, 8));
        };
        qa1 = ld(a1);
        qa2 = ld(a2);
        qm1 = ld(m1);
        qm2 = ld(m2);
        qm3 = ld(m3);
        qm4 = ld(m4);
        qry = ld(vry);
        qb = ld(b);
        if (!(ro & 8u)) {
            qrx = ld(vrx);
            qrz = ld(vrz);
        }
    };
    auto commit = [&](int p, int buf) {
        const int lv = level(p);
        const unsigned ro = here((unsigned)role);
        if (!(ro & (8u << lv)))
            return;
        const bool row8 = ro & 1u, col8 = ro & 2u, sq4 = ro & 4u;
        const int hr = (int)here((unsigned)hrow), hl = (int)here((unsigned)hlx); // LDS places formed here, not kept
        const Temps t0 = temps(qa1.x, qa2.x, qm1.x, qm2.x, qm3.x, qm4.x);
        const Temps t1 = temps(qa1.y, qa2.y, qm1.y, qm2.y, qm3.y, qm4.y);
        const float r0 = recip(qb.x), r1 = recip(qb.y);
        auto st = [](float* dst, float e0, float e1) { *reinterpret_cast<float2*>(dst) = make_float2(e0, e1); };
        // S of both fields for the direction cosines v, M for the pairs va, vb
        auto S = [&](float* d1, float* d2, float2 v) {
            st(d1, s_of(r0, t0.lap1, v.x, t0.hz1), s_of(r1, t1.lap1, v.y, t1.hz1));
            st(d2, s2_of(r0, qm4.x, qa2.x, v.x, t0.hz2), s2_of(r1, qm4.y, qa2.y, v.y, t1.hz2));
        };
        auto M = [&](float* d1, float* d2, float2 va, float2 vb) {
            st(d1, 2.0f * va.x * vb.x * t0.hz1, 2.0f * va.y * vb.y * t1.hz1);
            st(d2, 2.0f * va.x * vb.x * t0.hz2, 2.0f * va.y * vb.y * t1.hz2);
        };
        if (lv == 3 && col8)
            S(&SY[buf][0][hr][hl - 8], &SY[buf][1][hr][hl - 8], qry);
        if (ro & 8u)
            return;
        if (lv == 3 && row8)
            S(&SX[buf][0][hr - 8][hl], &SX[buf][1][hr - 8][hl], qrx);
        if (sq4) {
            if (lv == 3)
                M(&MXY[buf][0][hr - 4][hl - 4], &MXY[buf][1][hr - 4][hl - 4], qrx, qry);
            if (lv >= 2) {
                st(&Bt[buf][hr - 4][hl - 4], qb.x, qb.y);
                if (row8)
                    M(&MZX[buf][0][hr - 8][hl - 4], &MZX[buf][1][hr - 8][hl - 4], qrz, qrx);
                if (col8)
                    M(&MYZ[buf][0][hr - 4][hl - 8], &MYZ[buf][1][hr - 4][hl - 8], qry, qrz);
            }
            if (row8 && col8) {
                S(&SZ[buf][0][hr - 8][hl - 8], &SZ[buf][1][hr - 8][hl - 8], qrz);
                if (lv == 3) {
                    st(&SA[buf][0][hr - 8][hl - 8], qa1.x, qa1.y);
                    st(&SA[buf][1][hr - 8][hl - 8], qa2.x, qa2.y);
                }
            }
        }
    };
    // d_x items: the thread's own column and the 4 rim columns on either side of each row on the first threads; d_y items:
    // rows ty + h AY of the BH band, column tx. The scale is 1/d for interior points and zero elsewhere (floats: no lane
    // masks live across the loop).
    constexpr int XE = 8 * AY;
    static_assert(XE <= NT, "one rim item per thread");
    const int xe_r = min(tid, XE - 1) / 8, xe_k = min(tid, XE - 1) % 8, xe_j = xe_k < 4 ? xe_k : BX + xe_k;
    const float xs = in_xy(g, ix, iy) ? invdx : 0.0f;
    const float xes = in_xy(g, x0 - 4 + xe_j, y0 + xe_r) ? invdx : 0.0f;
    float ys[Sh::YI];
#pragma unroll
    for (int h = 0; h < Sh::YI; ++h)
        ys[h] = in_xy(g, x0 + tx, y0 - 4 + ty + h * AY) ? invdy : 0.0f;

    // z queues; the delay queues are seen through a window at slot c = p - (z0 - 4) mod 2 and shift by 2 every second plane,
    // the right-hand side sums shift as they are summed
    float sz[9], sa[9]; // S_z and sigma of plane p - 7 + k  at [c + k], k = 0..7
    float dz[9];        // d_z(p - 10 + k) = d_z(o - 3 + k)  at [c + k], k = 0..7
    float sb[5];        // b(p - 3 + k)                      at [c + k], k = 0..3
    // right-hand side sums of output p - 7 + j, j = 0..11: the X_zx + X_yz terms of the planes around it and, when plane
    // p is the output itself, its in-plane terms D+_x d_x + D+_y d_y + X_xy M_xy
    float q[12];
#pragma unroll
    for (int k = 0; k < 9; ++k)
        sz[k] = sa[k] = dz[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 5; ++k)
        sb[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < 12; ++k)
        q[k] = 0.0f;
    // S_z of the 3 planes before the first tile plane, clamped into the allocation (a clamped value only meets a zero b)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const unsigned i = (unsigned)max(z0 - 7 + k, g.izbeg - R) * PB + colb;
        const float c2 = ldf(a2, i), c4 = ldf(m4, i);
        const Temps t = temps(ldf(a1, i), c2, ldf(m1, i), ldf(m2, i), ldf(m3, i), c4);
        const float rho = recip(ldf(b, i)), vz = ldf(vrz, i);
        sz[4 + k] = F ? s2_of(rho, c4, c2, vz, t.hz2) : s_of(rho, t.lap1, vz, t.hz1);
    }
    // pointwise words of an output plane: u or w (+ the snapshot word and, in the first field's thread, the image value)
    float pu = 0.0f;
    SnapWord sw{ 0u, 1.0f };
    double g0 = 0.0;
    // An imaging step issues these loads on every path (planes outside the block's read its nearest one): past loads that
    // may not have been issued, the wait for a tile quad drains everything in flight, and with the extra words in registers
    // too the loop spilled (512^3 FP16 4.17 -> 3.78 ms). Without imaging it is the branch that is faster (3.47 -> 3.37 ms).
    auto own_plane = [&](int o) { return min(max(o, z0), z1 - 1); };
    auto fetch_point = [&](int o) {
        if (!imaging && (o < z0 || o >= z1))
            return;
        o = own_plane(o);
        pu = ldf(uw, (unsigned)o * PB + here(colb));
        if (imaging) {
            const unsigned idx = (unsigned)(o - g.izbeg) * s_plane + here(s_col);
            sw = snap_fetch(SNAP, F ? snap.b : snap.a, F ? snap.sb : snap.sa, idx, idx / SNAP_SEG);
        }
    };
    auto fetch_image = [&](int o) {
        if (imaging)
            g0 = grad[(unsigned)(own_plane(o) - g.izbeg) * g_plane + here(g_col)];
    };

    fetch_point(z0);
    fetch_image(z0);
    fetch(z0 - R);
    commit(z0 - R, 0);
    fetch(z0 - R + 1);
    __syncthreads();

    auto body = [&](auto curc, auto ownc, int p) {
        constexpr int cur = decltype(curc)::value;   // queue window, tile buffer
        constexpr bool own = decltype(ownc)::value;  // plane p is one of the block's output planes
        const int o = p - DEP, c = p - 3;
        const float pin = (p >= g.izbeg && p <= g.izend) ? 1.0f : 0.0f;
        // ---- A: this plane's loads before its stores (one counter tracks both): the temporaries of plane p + 1 into the
        // other buffer (last read before the previous plane's barrier), tile of plane p + 2
        if (p + 1 < z1 + DEP)
            commit(p + 1, cur ^ 1);
        fetch(p + 2);
        // ---- B: X_yz + X_zx of plane p into the sums; from the block's output planes also X_xy, d_x and d_y
        sz[cur + 7] = SZ[cur][F][ty][tx];
        sb[cur + 3] = Bt[cur][ty + 4][tx + 4];
        {
            float d[R + 1];
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                d[n] = fmaf(i4yz, MYZ[cur][F][ty + 4 + n][tx] - MYZ[cur][F][ty + 4 - n][tx],
                            i4zx * (MZX[cur][F][ty][tx + 4 + n] - MZX[cur][F][ty][tx + 4 - n]));
                hold(d[n]);
            }
            // plane p at offset +n feeds output p - n (slot 7 - n), at -n output p + n (slot 7 + n), sign flipped
#pragma unroll
            for (int j = 0; j < 11; ++j) {
                const int n = j < 7 ? 7 - j : j - 7;
                q[j] = n >= 1 && n <= R ? fma3(j < 7 ? ecen(n) : -ecen(n), d[n], q[j + 1]) : q[j + 1];
                hold(q[j]);
            }
            q[11] = -ecen(R) * d[R];
            hold(q[11]);
        }
        float hxy = 0.0f;
        if constexpr (own) {
            sa[cur + 7] = SA[cur][F][ty][tx];
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                hxy += ecen(n) * (MXY[cur][F][ty + 4 + n][tx + 4 + n] - MXY[cur][F][ty + 4 + n][tx + 4 - n] +
                                  MXY[cur][F][ty + 4 - n][tx + 4 - n] - MXY[cur][F][ty + 4 - n][tx + 4 + n]);
                hold(hxy);
            }
            // (the scale is zero for non-interior points: every tile value is finite)
            float v = Bt[cur][ty + 4][tx + 4] * (xs * pin) * stg8([&](int k) { return SX[cur][F][ty][tx + 4 + k]; });
            hold(v);
            X[cur][F][ty][tx + 4] = v;
            if (tid < XE) {
                v = Bt[cur][xe_r + 4][xe_j] * (xes * pin) * stg8([&](int k) { return SX[cur][F][xe_r][xe_j + k]; });
                hold(v);
                X[cur][F][xe_r][xe_j] = v;
            }
#pragma unroll
            for (int h = 0; h < Sh::YI; ++h) {
                const int j = ty + h * AY;
                v = Bt[cur][j][tx + 4] * (ys[h] * pin) * stg8([&](int k) { return SY[cur][F][j + k][tx]; });
                hold(v);
                Y[cur][F][j][tx] = v;
            }
        }
        // ---- C: d_z(p - 3), then plane o = p - 7
        dz[cur + 7] = ((c >= g.izbeg && c <= g.izend) ? sb[cur] : 0.0f) * invdz * stg8([&](int k) { return sz[cur + k]; });
        if (g.fs && o == g.izbeg)
            mirror_dz<cur>(dz);
        const bool fin = o >= z0 && active;
        const float gz = stg8([&](int k) { return dz[cur + k]; });
        // fixed rounding whichever products the compiler can see (see the forward finalisation)
        const float r = fmaf(gz, invdz, q[0]);
        float a = 1.0f, bb = 1.0f;
        if constexpr (SPONGE) {
            const ab2 z = abz[own_plane(o)];
            const float2 xy = tapers ? AB[ty][tx] : make_float2(axy, bxy);
            a = fminf(xy.x, z.a);
            bb = fminf(xy.y, z.b);
        }
        const float un = SPONGE ? fmaf(bb * dt, r, a * pu) : fmaf(r, dt, pu);
        const float an = fmaf(bb * un, dt, a * sa[cur]);
        double prod = 0.0;
        if (imaging) {
            prod = (double)un * (double)snap_decode(SNAP, sw); // exact
            if (F)
                EX[cur][ty][tx] = prod;
        }
        // the pointwise words of plane o + 1 (their registers are free now), then the stores of plane o
        fetch_point(o + 1);
        if (fin) {
            const unsigned io = (unsigned)o * PB + here(colb);
            stf(uw, io, un);
            stf(ao, io, an);
        }
        // the one barrier of the plane: d_x, d_y (and w' w_snap) are complete, every read of tile buffer `cur` is done
        __syncthreads();
        // ---- D: in-plane terms of output p; the image of plane o
        if constexpr (own) {
            float gx = 0, gy = 0;
#pragma unroll
            for (int n = 1; n <= R; ++n) {
                const float cc = cstg(n);
                gx += cc * (X[cur][F][ty][tx + 4 + n] - X[cur][F][ty][tx + 5 - n]);
                gy += cc * (Y[cur][F][ty + 4 + n][tx] - Y[cur][F][ty + 5 - n][tx]);
                hold(gx), hold(gy);
            }
            // explicit roundings: no product is fused into these sums
            q[7] = __fadd_rn(q[7], __fadd_rn(__fadd_rn(__fmul_rn(gx, invdx), __fmul_rn(gy, invdy)), __fmul_rn(hxy, i4xy)));
            hold(q[7]);
        }
        if (imaging) {
            const double gn = g0 + (prod + EX[cur][ty][tx]);
            fetch_image(o + 1);
            if (fin && !F)
                grad[(unsigned)(o - g.izbeg) * g_plane + here(g_col)] = gn;
        }
        if (cur == 1) {
#pragma unroll
            for (int k = 0; k < 7; ++k) {
                sz[k] = sz[k + 2];
                sa[k] = sa[k + 2];
                dz[k] = dz[k + 2];
            }
#pragma unroll
            for (int k = 0; k < 3; ++k)
                sb[k] = sb[k + 2];
        }
    };

    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    // planes that only feed the z stencils of the block's outputs: 4 before them and 7 after
    auto rim = [&](int p, int end) {
        for (; p < end; ++p)
            if (((p - z0) & 1) == 0)
                body(C0{}, std::false_type{}, p);
            else
                body(C1{}, std::false_type{}, p);
    };
    rim(z0 - R, z0);
    for (int p = z0; p < z1; p += 2) {
        body(C0{}, std::true_type{}, p);
        if (p + 1 >= z1)
            break;
        body(C1{}, std::true_type{}, p + 1);
    }
    rim(z1, z1 + DEP);
}


// ------------------------------------------------------------------------------------------------------------------
// Receivers
// ------------------------------------------------------------------------------------------------------------------

// pressure -(2 s1 + s2)/3 at linear index i (simulator2/simulator2SetUp.cu:31-42)
__device__ __forceinline__ float
pressure_at(const float* __restrict__ s1, const float* __restrict__ s2, long i)
{
    return -(2.0f * s1[i] + s2[i]) / 3.0f;
}

// Transpose of the pressure recording at receiver k, applied after an adjoint step: u += -2/3 r, w += -1/3 r and the
// already-updated sigma_out gets B dt times the same increment (the adjoint step's sigma' = A sigma + B dt u').
// Optionally adds the increment's share of the imaging condition.
__device__ __forceinline__ void
inject_point(float* __restrict__ u, float* __restrict__ w, float* __restrict__ a1o, float* __restrict__ a2o,
             const long* __restrict__ idx, const int* __restrict__ ijk, int k, const float* __restrict__ res, float dt,
             const ab2* __restrict__ abx, const ab2* __restrict__ aby, const ab2* __restrict__ abz, const Box& g,
             const Snap& snap, double* __restrict__ grad)
{
    const long i = idx[k];
    const int x = ijk[3 * k], y = ijk[3 * k + 1], z = ijk[3 * k + 2];
    const float du = -2.0f / 3.0f * res[k], dw = -1.0f / 3.0f * res[k];
    float bb = 1.0f;
    if (abx != nullptr)
        bb = fminf(fminf(abx[x].b, aby[y].b), abz[z].b);
    u[i] += du;
    w[i] += dw;
    a1o[i] += bb * du * dt;
    a2o[i] += bb * dw * dt;
    if (snap.mode != TTI_SNAP_NONE && grad != nullptr) {
        const long row = (long)(z - g.izbeg) * snap.ldy + (y - g.iybeg);
        const long sidx = row * (snap.ldx / SNAP_SEG) + (x - g.ixbeg) / SNAP_SEG;
        const long si = row * snap.ldx + (x - g.ixbeg);
        const float su = snap_load(snap.mode, snap.a, snap.sa, si, sidx);
        const float sw = snap_load(snap.mode, snap.b, snap.sb, si, sidx);
        const long gstride_y = (long)(g.ixend - g.ixbeg + 1), gstride_z = gstride_y * (g.iyend - g.iybeg + 1);
        const long gi = (long)(z - g.izbeg) * gstride_z + (long)(y - g.iybeg) * gstride_y + (x - g.ixbeg);
        grad[gi] += fma((double)dw, (double)sw, (double)du * (double)su);
    }
}


// ------------------------------------------------------------------------------------------------------------------
// Host-side argument checks shared by the launchers
// ------------------------------------------------------------------------------------------------------------------

// Resident blocks on the whole GPU (one 1024-thread block per CU, by their registers) and
// the cost, in planes, of a chunk's recomputed rim planes (8 and 11) and prologue, for chunk_depth; [0] forward, [1]
// adjoint. Fitted over z depths of 1 to 256 planes on volumes of 40^3 to 400^3: a plane takes 1.82 and 2.06 us where few
// blocks run (64^3: 17.0 us forward at 2 planes, 129.7 at 64; 29.5 and 157.5 adjoint) and 2.3 and 3.1 us on a full GPU,
// and no fixed depth of the sweep beats the chosen one by more than 2% from 96 points a side up. 128-plane chunks
// throughout: 64^3 130 and 158 us against 17 and 30, 128^3 253 and 304 against 46 and 63.
constexpr int STEP_SLOTS[2] = { CUS, CUS };
constexpr float STEP_WARM[2] = { 7.5f, 12.5f };

// The fused kernels stage tiles with 16-byte loads: the interior must start on a 4-float boundary, rows must be a
// multiple of 4 floats and every volume 16-byte aligned.
inline bool
box_ok(int ixbeg, int ixend, int iybeg, int iyend, int izbeg, int izend, int ldimx, int ldimy)
{
    return ixbeg >= R && iybeg >= R && izbeg >= R && ixend >= ixbeg && iyend >= iybeg && izend >= izbeg &&
           ixend + R < ldimx && iyend + R < ldimy && ixbeg % 4 == 0 && ldimx % 4 == 0;
}

// Every volume (allocated planes up to izend + 4) must be smaller than 4 GiB: the kernels address it with 32-bit
// byte offsets.
inline bool
small_volume(int ldimx, int ldimy, int izend)
{
    return (long)ldimx * ldimy * (izend + R + 1) * (long)sizeof(float) < (1L << 32);
}

inline bool
aligned16(std::initializer_list<const void*> ps)
{
    for (const void* p : ps)
        if (reinterpret_cast<uintptr_t>(p) % 16 != 0)
            return false;
    return true;
}

inline bool
snap_ok(const tti_snapshot* s, int nx, int ny, int nz)
{
    if (s == nullptr || s->mode == TTI_SNAP_NONE)
        return true;
    if (s->mode < TTI_SNAP_FP32 || s->mode > TTI_SNAP_BF16 || !s->field3 || !s->field4)
        return false;
    if (s->ldimx % 64 != 0 || s->ldimx < nx || s->ldimy < ny)
        return false;
    if (s->mode == TTI_SNAP_FP16 && (!s->scale3 || !s->scale4))
        return false;
    if ((s->field1 == nullptr) != (s->field2 == nullptr))
        return false;
    if (s->field1 && s->mode == TTI_SNAP_FP16 && (!s->scale1 || !s->scale2))
        return false;
    // the kernels address a snapshot field with 32-bit element offsets
    return (long)nz * s->ldimy * s->ldimx < (1L << 32);
}

inline Snap
to_snap(const tti_snapshot* s)
{
    Snap r{ TTI_SNAP_NONE, nullptr, nullptr, nullptr, nullptr, 64, 1, nullptr, nullptr, nullptr, nullptr };
    if (s && s->mode != TTI_SNAP_NONE) {
        r.mode = s->mode;
        r.a = s->field3;
        r.b = s->field4;
        r.sa = s->scale3;
        r.sb = s->scale4;
        r.ldx = s->ldimx;
        r.ldy = s->ldimy;
        r.c = s->field1;
        r.d = s->field2;
        r.sc = s->scale1;
        r.sd = s->scale2;
    }
    return r;
}


} // namespace fused
} // namespace tti
