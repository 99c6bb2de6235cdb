// Red-black half-sweeps, several per launch, for one simulation (gfx950):
// the reference's in-place SOR on face velocities (smokeSimulation.cu:356-394).
// Included by step_kernels.hip.
//
// One half-sweep per launch costs a launch and a trip of the fields to memory
// for a few operations per cell.  Here a workgroup takes a part of the grid
// grown by H cells and runs up to H half-sweeps on it; each makes one more
// layer of the grown part stale.  The faces it owns are written to a second
// set of fields, so that neighbouring workgroups, which read the same faces,
// are not disturbed, and the launches of a solve alternate between the two
// sets.  Every cell that counts sees exactly the operands the one-half-sweep
// kernel gives it: the bits are the same.
//
// Grids of at most one box per CU (k_ref_faces_box): the launch is a chain of
// latencies, and a box in LDS with all CUs busy is the shortest one.  80^3:
// 13.3 us per launch of 4 half-sweeps (2.3 the launch itself, 5 the loads and
// stores, 1.4 each half-sweep), 4 x 4.5 us one by one, 19.3 us marched.
// Larger grids (k_ref_faces_march): a column marched up z re-reads far less
// halo.  Empty 256x240x248, 5 half-sweeps per launch: 127 us against 5 x 80 us;
// boxes 306 us per 4.  150x96x121, 4 per launch: 21.5 us against 4 x 10.5 us (boxes
// 42 per 4): there FP64 conversions and VALU issue bind, memory at 256.  Cells next
// to a solid take longer (256^3, 5 a launch: 138 us empty, 141 with 5 % solid boxes).
// Grids thin in x or y keep one half-sweep per launch (reference_in_place).
#pragma once

#include "step_device.h"

namespace smk {
namespace {

// The diagonal of a cell by its flags: RN(1 / fluid neighbours) in FP64, one
// entry per combination of the six neighbour bits.
struct FaceDiagonal {
    double inv[64];
    __device__ __forceinline__ double of(uint32_t c) const { return inv[(c & F_NBRS) >> 1]; }
    __device__ __forceinline__ void fill(int tid)
    {
        if (tid < 64) inv[tid] = tid ? 1.0 / (double)__popc((unsigned)tid) : 0.0;
    }
};

// Relaxes an active cell with flags c on its six faces f (u low, u high, v low,
// ...), as k_project_ref_half does; other cells keep theirs.
//
// -dv / n is RN(double(-dv) * RN(1/n)): the FP64 product is within 2^-52 of the
// quotient, and no quotient by n = 1..6 comes that near a rounding boundary of
// FP32 without lying on it exactly (all 2^32 floats compared on the CPU for 3,
// 5 and 6; 1, 2 and 4 are exact).  Cells with six fluid neighbours (nearly
// all) move every face, in straight-line code for every lane: others subtract
// +0 and add -0, which leave any face as it was.  Next to a solid a face moves
// by p * 0, a zero of p's sign or NaN, as the reference's product does.
__device__ __forceinline__ void relax_faces(uint32_t c, double inv, double omega, float (&f)[6])
{
    const float dv = -f[0] + f[1] + -f[2] + f[3] + -f[4] + f[5];
    const float q = (float)((double)(-dv) * inv);
    const float p = (float)((double)q * omega);
    constexpr uint32_t kFull = F_ACTIVE | F_SELF | F_NBRS;
    const bool full = c == kFull;
    const float sub = full ? p : 0.0f, add = full ? p : -0.0f;
#pragma unroll
    for (int k = 0; k < 6; k += 2) {
        f[k] = f[k] - sub;
        f[k + 1] = f[k + 1] + add;
    }
    if (c >= F_ACTIVE && !full) {
        const uint32_t on = __float_as_uint(p), off = __float_as_uint(p * 0.0f);
        auto step = [&](int bit) {
            const uint32_t m = (uint32_t)((int32_t)(c << (31 - bit)) >> 31);
            return __uint_as_float((on & m) | (off & ~m));
        };
#pragma unroll
        for (int k = 0; k < 6; k += 2) {
            f[k] = f[k] - step(k + 1);
            f[k + 1] = f[k + 1] + step(k + 2);
        }
    }
}

// A box of faces grown by H on every side, in LDS: x pairs split into even and
// odd x (a colour's cells of a row are one of the two), so the lanes of a wave
// read consecutive words.
template <int IX, int IY, int IZ, int H>
struct FaceBox {
    static_assert(IX % 4 == 0 && H % 4 == 0, "whole quads of x");
    static constexpr int SX = IX + 2 * H, SY = IY + 2 * H, SZ = IZ + 2 * H;
    static constexpr int TP = SX / 2;      // x pairs per row
    static constexpr int ROWS = SY * SZ;   // rows (y, z)
    static constexpr int N = ROWS * TP;    // pairs
    static constexpr int ZS = SY * TP;     // stride of z
};
constexpr int kBoxThreads = 1024;

template <int IX, int IY, int IZ, int H>
__global__ __launch_bounds__(kBoxThreads) void k_ref_faces_box(
    Grid g, const float* __restrict__ ui, const float* __restrict__ vi,
    const float* __restrict__ wi, float* __restrict__ uo, float* __restrict__ vo,
    float* __restrict__ wo, const uint8_t* __restrict__ flags, int colour, int sweeps, double omega)
{
    using S = FaceBox<IX, IY, IZ, H>;
    __shared__ __align__(16) float f[3][2][S::N];
    __shared__ __align__(16) uint16_t fl[S::N];  // the pair's two flags bytes
    __shared__ FaceDiagonal diag;
    const int tid = (int)threadIdx.x;
    diag.fill(tid);
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int b = dev::xcd_tile_order();
    const int xa = IX * (b % nbx) - H, ya = IY * ((b / nbx) % nby) - H, za = IZ * (b / (nbx * nby)) - H;
    {
        // Quads of four x (16 bytes of a field); every load of the thread is
        // issued before the first LDS store.
        constexpr int Q = S::SX / 4, QN = Q * S::ROWS, QT = (QN + kBoxThreads - 1) / kBoxThreads;
        float4 a[QT][3];
        uint32_t c[QT];
#pragma unroll
        for (int j = 0; j < QT; ++j) {
            const int k = tid + j * kBoxThreads;
            const int row = k / Q;
            const int x = xa + 4 * (k % Q), y = ya + row % S::SY, z = za + row / S::SY;
            c[j] = 0;
            a[j][0] = a[j][1] = a[j][2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            // Rows hold a multiple of 32 elements, at least nx + 1: the quad of
            // an x < nx lies inside its row (flags past nx are 0).
            if (k < QN && x >= 0 && x < g.nx && y >= 0 && y < g.ny && z >= 0 && z < g.nz) {
                const int i = g.idx(x, y, z);
                __builtin_memcpy(&c[j], flags + i, 4);
                a[j][0] = *reinterpret_cast<const float4*>(ui + i);
                a[j][1] = *reinterpret_cast<const float4*>(vi + i);
                a[j][2] = *reinterpret_cast<const float4*>(wi + i);
            }
        }
#pragma unroll
        for (int j = 0; j < QT; ++j) {
            const int k = tid + j * kBoxThreads;
            if (k >= QN) continue;
            *reinterpret_cast<uint32_t*>(&fl[2 * k]) = c[j];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                *reinterpret_cast<float2*>(&f[m][0][2 * k]) = make_float2(a[j][m].x, a[j][m].z);
                *reinterpret_cast<float2*>(&f[m][1][2 * k]) = make_float2(a[j][m].y, a[j][m].w);
            }
        }
    }
    __syncthreads();
    // Pair k = tid + j * kBoxThreads of the grown box, the same for every
    // half-sweep, so that its LDS indices are constants apart.
    constexpr int PT = (S::N + kBoxThreads - 1) / kBoxThreads;
    uint32_t cell[PT];  // flags byte of this half-sweep's colour, the other's << 8, (1 + last) << 16
    int own[PT];        // index in f[m] of this half-sweep's cell
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const int k = tid + j * kBoxThreads;
        const int t = k % S::TP, row = k / S::TP, ly = row % S::SY, lz = row / S::SY;
        // Half-sweep s of the launch updates the cells of the layers
        // lo .. S-2-lo of each axis, lo = H - sweeps + s: those that still
        // have all their operands (the last layer lacks its high faces).
        const int last = min(min(ly, lz), min(S::SY - 2 - ly, S::SZ - 2 - lz));
        uint32_t c = k < S::N && last >= 0 ? fl[k] : 0u;
        if (t == S::TP - 1) c &= 0xffu;  // the odd cell of a row's last pair lacks its high x face
        const bool odd = (ya + ly + za + lz + colour) & 1;
        if (odd) c = c >> 8 | (c & 0xffu) << 8;
        cell[j] = c | (uint32_t)(last + 1) << 16;
        own[j] = odd ? k + S::N : k;
    }
    float* const F = &f[0][0][0];
    for (int s = 0; s < sweeps; ++s) {
        const uint32_t lo = (uint32_t)(H - sweeps + s + 1) << 16;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const uint32_t c = cell[j];
            const int k = tid + j * kBoxThreads;
            const int other = 2 * k + S::N - own[j];  // the other cell of the pair
            if ((c & F_ACTIVE) && c >= lo) {
                // The high x face: in the same pair (even x) or the next.
                float* const u0 = F + own[j];
                float* const u1 = F + other + (other == k ? 1 : 0);
                float* const v0 = u0 + 2 * S::N;
                float* const w0 = u0 + 4 * S::N;
                float face[6] = {u0[0], u1[0], v0[0], v0[S::TP], w0[0], w0[S::ZS]};
                relax_faces(c & 0xffu, diag.of(c), omega, face);
                u0[0] = face[0];
                u1[0] = face[1];
                v0[0] = face[2];
                v0[S::TP] = face[3];
                w0[0] = face[4];
                w0[S::ZS] = face[5];
            }
            own[j] = other;
            cell[j] = (c & 0xffff0000u) | ((c >> 8) & 0xffu) | ((c & 0xffu) << 8);
        }
        __syncthreads();
    }
    // The owned box, in quads.
    constexpr int OQ = IX / 4, ON = OQ * IY * IZ;
    for (int k = tid; k < ON; k += kBoxThreads) {
        const int r = k / OQ, lx = H + 4 * (k % OQ), ly = H + r % IY, lz = H + r / IY;
        const int x = xa + lx, y = ya + ly, z = za + lz;
        if (x >= g.nx || y >= g.ny || z >= g.nz) continue;
        const int i = g.idx(x, y, z), l = (ly + lz * S::SY) * S::TP + lx / 2;
        float* const out[3] = {uo, vo, wo};
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const float2 e = *reinterpret_cast<const float2*>(&f[m][0][l]);
            const float2 o = *reinterpret_cast<const float2*>(&f[m][1][l]);
            *reinterpret_cast<float4*>(out[m] + i) = make_float4(e.x, o.x, e.y, o.y);
        }
    }
}

// A column of faces marched up z: half-sweep h trails half-sweep h-1 by two
// planes, so that the half-sweeps of one step touch no common face and one
// barrier per plane separates the steps.
//
// The grown column: TP x pairs by TY rows.  Pair t of row y holds the cells
// x0 = xa + 2t + (y & 1) and x0 + 1: with the rows skewed so, the colour of a
// half-sweep is the same cell of every pair of a plane.  The first cell of an
// even row and the last of an odd row have no y neighbours in the column, so
// there one pair more than H cells goes stale.
template <int TP, int TY, int H>
struct FaceColumn {
    static_assert(64 % TP == 0, "whole rows per wave");
    static constexpr int IX = 2 * TP - 2 * H - 2, IY = TY - 2 * H;  // owned faces
    // First owned pair of a row (whole pairs: with an even H the odd rows'
    // owned pairs start and end one earlier).
    static __device__ __forceinline__ int first(int skew) { return (H + 2) / 2 - (H % 2 == 0 ? skew : 0); }
    // Planes in flight: k+1 (entering) down to k-2H+1 (leaving), and one more
    // for an even count, so that a slot's colour does not change.
    static constexpr int W = 2 * H + 2;
    static constexpr int ROW = 2 * (TP + 1);      // LDS words of a row: even x, odd x
    static constexpr int SLOT = (TY + 1) * ROW;   // of a plane
};

// The y faces of the planes in flight live in LDS, where the cells on both
// sides of a face update it in turn; x faces (shared by adjacent lanes, DPP)
// and z faces (this thread's own) in registers.
template <int TP, int TY, int H>
__global__ __launch_bounds__(TP * TY) void k_ref_faces_march(
    Grid g, const float* __restrict__ ui, const float* __restrict__ vi,
    const float* __restrict__ wi, float* __restrict__ uo, float* __restrict__ vo,
    float* __restrict__ wo, const uint8_t* __restrict__ flags, int zc, int colour, int sweeps,
    double omega)
{
    using S = FaceColumn<TP, TY, H>;
    constexpr int W = S::W, D = 2;  // D planes of prefetch (W % D == 0)
    __shared__ float lv[W * S::SLOT];
    __shared__ FaceDiagonal diag;
    const int t = (int)threadIdx.x, r = (int)threadIdx.y;
    diag.fill(t + TP * r);
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int b = dev::xcd_tile_order();
    const int xa = S::IX * (b % nbx) - (H + 2) / 2 * 2, ya = S::IY * ((b / nbx) % nby) - H;
    const int z0 = zc * (b / (nbx * nby)), z1 = min(z0 + zc, g.nz);
    const int y = ya + r, skew = y & 1, x0 = xa + 2 * t + skew;
    const bool inside = x0 >= 0 && x0 < g.nx && y >= 0 && y < g.ny;
    // Lanes outside the grid read its first cells and have no flags.
    const uint32_t lane = inside ? (uint32_t)g.idx(x0, y, 0) : 0u;
    const uint32_t fmask = inside ? 0xffffu : 0u;
    const bool owner = inside && t >= S::first(skew) && t < S::first(skew) + S::IX / 2 && r >= H && r < TY - H;
    // LDS index of the y face of the pair's first and second cell in slot 0.
    const int l0 = r * S::ROW + t + (skew ? TP + 1 : 0);
    const int l1 = r * S::ROW + t + (skew ? 1 : TP + 1);

    float u0[W], u1[W], w0[W], w1[W];
    uint32_t fl[W];
    float2 pu[D], pv[D], pw[D];
    uint16_t pf[D];
    auto load = [&](int z, int s) {
        const size_t at = (size_t)min(max(z, 0), g.nz - 1) * (size_t)g.plane;
        __builtin_memcpy(&pu[s], ui + at + lane, 8);
        __builtin_memcpy(&pv[s], vi + at + lane, 8);
        __builtin_memcpy(&pw[s], wi + at + lane, 8);
        __builtin_memcpy(&pf[s], flags + at + lane, 2);
    };
    auto enter = [&](int z, int slot) {  // plane z, prefetched in slot % D
        const int s = slot % D;
        u0[slot] = pu[s].x;
        u1[slot] = pu[s].y;
        w0[slot] = pw[s].x;
        w1[slot] = pw[s].y;
        lv[slot * S::SLOT + l0] = pv[s].x;
        lv[slot * S::SLOT + l1] = pv[s].y;
        fl[slot] = pf[s] & (z >= 0 && z < g.nz ? fmask : 0u);
    };
#pragma unroll
    for (int s = 0; s < W; ++s) {
        u0[s] = u1[s] = w0[s] = w1[s] = 0.0f;
        fl[s] = 0;
    }
    // Step k relaxes plane k - 2(h-1) for half-sweep h = 1..sweeps; the first
    // step's plane is z0 - sweeps, or one before for a fixed colour of step 0.
    // (With fewer half-sweeps than H the trailing ones do nothing.)
    int k0 = z0 - sweeps;
    k0 -= (xa + k0 + colour) & 1;
    const int kend = z1 + 2 * H - 1;  // one past the step that writes plane z1 - 1
#pragma unroll
    for (int s = 0; s < D; ++s) load(k0 + s, s);
    enter(k0, 0);
    load(k0 + D, 0);
    __syncthreads();
    for (int kb = k0; kb < kend; kb += W) {
#pragma unroll
        for (int u = 0; u < W; ++u) {
            const int k = kb + u;  // in slot u
            if (k >= kend) break;
            enter(k + 1, (u + 1) % W);
            load(k + 1 + D, (u + 1) % W % D);
#pragma unroll
            for (int h = 1; h <= H; ++h) {
                const int z = k - 2 * (h - 1);
                // Planes whose cells half-sweep h must relax.
                if (h > sweeps || z < z0 - 1 - (sweeps - h) || z > z1 - 1 + (sweeps - h)) continue;
                const int s = (u - 2 * (h - 1) + 2 * W) % W, s1 = (s + 1) % W;
                const bool second = (u + h - 1) & 1;  // constant once unrolled
                const uint32_t c = second ? fl[s] >> 8 : fl[s] & 0xffu;
                float* const v = lv + s * S::SLOT + (second ? l1 : l0);
                float* const w = second ? w1 : w0;
                float f[6] = {second ? u1[s] : u0[s], second ? dev::lane_next(u0[s]) : u1[s],
                              v[0], v[S::ROW], w[s], w[s1]};
                relax_faces(c, diag.of(c), omega, f);
                v[0] = f[2];
                v[S::ROW] = f[3];
                w[s] = f[4];
                w[s1] = f[5];
                if (second) {
                    u1[s] = f[0];
                    u0[s] = dev::lane_prev(f[1]);
                } else {
                    u0[s] = f[0];
                    u1[s] = f[1];
                }
            }
            const int zo = k - 2 * H + 1;
            if (zo >= z0 && owner) {
                const int s = (u - 2 * H + 1 + 2 * W) % W;
                const size_t at = (size_t)zo * (size_t)g.plane;
                const float2 ou = make_float2(u0[s], u1[s]), ow = make_float2(w0[s], w1[s]);
                const float2 ov = make_float2(lv[s * S::SLOT + l0], lv[s * S::SLOT + l1]);
                __builtin_memcpy(uo + at + lane, &ou, 8);
                __builtin_memcpy(vo + at + lane, &ov, 8);
                __builtin_memcpy(wo + at + lane, &ow, 8);
            }
            __syncthreads();
        }
    }
}

// The pressure form's half-sweeps on a column marched up z: half-sweep h trails
// half-sweep h-1 by one plane, its cells' z neighbours in this thread's
// registers, x neighbours in adjacent lanes (DPP), y neighbours in LDS, and
// one barrier per plane.  The pairs are skewed as above; a cell needs only its
// neighbours' pressures, so exactly H cells go stale on every side.
//
// us per half-sweep, one per launch -> here: 113x90x101 6.1 -> 3.2, 80^3 4.1 ->
// 2.5, 256x240x248 51 -> 11.6.  Small grids are a chain of LDS latencies and
// barriers (16-pair columns of half the threads then beat 32-pair ones: 48x40x57
// 1.9 against 2.5), large ones 3.5 TB/s of loads and stores over VALU issue.
template <int TP, int TY, int H>
struct PressureColumn {
    static_assert(H % 2 == 0 && 64 % TP == 0, "whole pairs, whole rows per wave");
    static constexpr int IX = 2 * TP - 2 * H, IY = TY - 2 * H;  // owned cells
    // Planes in flight: k+1 (entering) down to k-H (below the last relaxed).
    static constexpr int W = H + 2;
    static constexpr int ROW = 2 * (TP + 1);     // LDS words of a row: even x, odd x
    static constexpr int SLOT = (TY + 2) * ROW;  // of a plane, a row more on each side
};

// `cold`: the pressure starts at zero and is not read.  Cells that are not
// active are taken, and written, as zero.
template <int TP, int TY, int H>
__global__ __launch_bounds__(TP * TY) void k_ref_pressure_march(
    Grid g, const float* __restrict__ pi, float* __restrict__ po, const float* __restrict__ d,
    const uint8_t* __restrict__ flags, int zc, int colour, int sweeps, float omega, int cold)
{
    using S = PressureColumn<TP, TY, H>;
    constexpr int W = S::W, D = 2;  // D planes of prefetch
    __shared__ float lp[W * S::SLOT];
    __shared__ float inv[256];
    const int t = (int)threadIdx.x, r = (int)threadIdx.y;
    for (int f = t + TP * r; f < 256; f += TP * TY) inv[f] = dev::cell_inv((uint8_t)f);
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int b = dev::xcd_tile_order();
    const int xa = S::IX * (b % nbx) - H, ya = 1 + S::IY * ((b / nbx) % nby) - H;
    const int z0 = 1 + zc * (b / (nbx * nby)), z1 = min(z0 + zc, g.nz - 1);
    const int y = ya + r, skew = y & 1, x0 = xa + 2 * t + skew;
    const bool inside = x0 >= 0 && x0 < g.nx && y >= 0 && y < g.ny;
    // Lanes outside the grid read its first cells and have no flags.
    const uint32_t lane = inside ? (uint32_t)g.idx(x0, y, 0) : 0u;
    const uint32_t fmask = inside ? 0xffffu : 0u;
    const bool owner = inside && y <= g.ny - 2 && t >= H / 2 && t < TP - H / 2 && r >= H && r < TY - H;
    // LDS index of the pair's first and second cell in slot 0 (rows from 1).
    const int l0 = (r + 1) * S::ROW + t + (skew ? TP + 1 : 0);
    const int l1 = (r + 1) * S::ROW + t + (skew ? 1 : TP + 1);

    float2 p[W], q[W], iv[W];  // pressure, 0 - d * inv, inv (0: not active)
    float2 np[D], nd[D];
    uint16_t nf[D];
    auto load = [&](int z, int s) {
        const size_t at = (size_t)min(max(z, 0), g.nz - 1) * (size_t)g.plane;
        if (!cold) __builtin_memcpy(&np[s], pi + at + lane, 8);
        __builtin_memcpy(&nd[s], d + at + lane, 8);
        __builtin_memcpy(&nf[s], flags + at + lane, 2);
    };
    auto enter = [&](int z, int slot) {  // plane z, prefetched in slot % D
        const int s = slot % D;
        const uint32_t c = nf[s] & (z >= 0 && z < g.nz ? fmask : 0u);
        iv[slot] = make_float2(inv[c & 0xffu], inv[c >> 8]);
        q[slot] = make_float2(dev::neg_scaled_rhs(nd[s].x, iv[slot].x),
                              dev::neg_scaled_rhs(nd[s].y, iv[slot].y));
        p[slot] = make_float2(iv[slot].x > 0.0f ? np[s].x : 0.0f, iv[slot].y > 0.0f ? np[s].y : 0.0f);
        lp[slot * S::SLOT + l0] = p[slot].x;
        lp[slot * S::SLOT + l1] = p[slot].y;
    };
#pragma unroll
    for (int s = 0; s < W; ++s) p[s] = q[s] = iv[s] = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int s = 0; s < D; ++s) np[s] = make_float2(0.0f, 0.0f);
    // Step k relaxes plane k - (h-1) for half-sweep h = 1..sweeps.  The first
    // step's plane is z0 - sweeps (whose plane below is never needed), or one
    // before for a fixed colour of step 0.
    int k0 = z0 - sweeps;
    k0 -= (xa + k0 + colour) & 1;
    const int kend = z1 + H - 1;  // one past the step that writes plane z1 - 1
#pragma unroll
    for (int s = 0; s < D; ++s) load(k0 + s, s);
    __syncthreads();  // inv
    enter(k0, 0);
    load(k0 + D, 0);
    __syncthreads();
    for (int kb = k0; kb < kend; kb += W) {
#pragma unroll
        for (int u = 0; u < W; ++u) {
            const int k = kb + u;  // in slot u
            if (k >= kend) break;
            enter(k + 1, (u + 1) % W);
            load(k + 1 + D, (u + 1) % W % D);
            const bool second = u & 1;  // the pair's cell of this step's colour
            // The y neighbours of every half-sweep's cell, none of which this
            // step changes, in one go.
            float yn[H][2];
#pragma unroll
            for (int h = 1; h <= H; ++h) {
                const float* const at = lp + (u - (h - 1) + W) % W * S::SLOT + (second ? l1 : l0);
                yn[h - 1][0] = at[-S::ROW];
                yn[h - 1][1] = at[S::ROW];
            }
#pragma unroll
            for (int h = 1; h <= H; ++h) {
                const int z = k - (h - 1);
                // Planes whose cells half-sweep h must relax.
                if (h > sweeps || z < z0 - (sweeps - h) || z > z1 - 1 + (sweeps - h)) continue;
                const int s = (u - (h - 1) + W) % W, lo = (s + W - 1) % W, hi = (s + 1) % W;
                const float left = second ? p[s].x : dev::lane_prev(p[s].y);
                const float right = second ? dev::lane_next(p[s].x) : p[s].y;
                const float pc = second ? p[s].y : p[s].x;
                const float w = second ? iv[s].y : iv[s].x;
                const float sum = dev::sum6(left, right, yn[h - 1][0], yn[h - 1][1],
                                            second ? p[lo].y : p[lo].x, second ? p[hi].y : p[hi].x);
                const float G = __builtin_fmaf(sum, w, second ? q[s].y : q[s].x);
                const float v = pc + omega * (G - pc);
                const float out = w > 0.0f ? v : pc;
                if (second) p[s].y = out;
                else p[s].x = out;
                lp[s * S::SLOT + (second ? l1 : l0)] = out;
            }
            const int zo = k - (H - 1);
            if (zo >= z0 && owner)
                __builtin_memcpy(po + (size_t)zo * (size_t)g.plane + lane, &p[(u - (H - 1) + W) % W], 8);
            __syncthreads();
        }
    }
}

// Launch of a marched form: columns in x and y, chunks of zc planes in z.
struct MarchPlan {
    dim3 grid;
    int zc;
    long long steps;
};
inline MarchPlan march_plan(int nx, int ny, int planes, int fill)
{
    const MarchChunk c = fit_march((long long)nx * ny, planes, fill);
    return {dim3((unsigned)nx, (unsigned)ny, (unsigned)((planes + c.zc - 1) / c.zc)), c.zc, c.steps};
}

constexpr int kMarchTP = 32, kMarchTY = 32;

template <int H>
MarchPlan faces_plan(const Grid& g)
{
    using S = FaceColumn<kMarchTP, kMarchTY, H>;
    // Odd rows may own one x less on the right: columns for nx + 1.
    return march_plan((g.nx + S::IX) / S::IX, (g.ny + S::IY - 1) / S::IY, g.nz, 3 * H);
}

struct FaceSets {
    const float *ui, *vi, *wi;
    float *uo, *vo, *wo;
};

template <int H>
hipError_t launch_faces_march(const Grid& g, const MarchPlan& p, const FaceSets& f, const uint8_t* flags,
                              int colour, int sweeps, double omega, hipStream_t st)
{
    hipLaunchKernelGGL((k_ref_faces_march<kMarchTP, kMarchTY, H>), p.grid, dim3(kMarchTP, kMarchTY), 0,
                       st, g, f.ui, f.vi, f.wi, f.uo, f.vo, f.wo, flags, p.zc, colour, sweeps, omega);
    return hipGetLastError();
}

template <int TP, int H>
MarchPlan pressure_plan(const Grid& g)
{
    using S = PressureColumn<TP, kMarchTY, H>;
    return march_plan((g.nx - 1 + S::IX - 1) / S::IX, (g.ny - 2 + S::IY - 1) / S::IY, g.nz - 2, 2 * H);
}

template <int TP, int H>
hipError_t launch_pressure_march(const Grid& g, const MarchPlan& p, const float* pi, float* po,
                                 const float* d, const uint8_t* flags, int colour, int sweeps,
                                 float omega, int cold, hipStream_t st)
{
    hipLaunchKernelGGL((k_ref_pressure_march<TP, kMarchTY, H>), p.grid, dim3(TP, kMarchTY), 0, st, g, pi,
                       po, d, flags, p.zc, colour, sweeps, omega, cold);
    return hipGetLastError();
}

}  // namespace
}  // namespace smk
