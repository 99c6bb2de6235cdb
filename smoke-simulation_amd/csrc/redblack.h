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
// stores, 1.4 each half-sweep), 4 x 4.6 us one by one, 16.4 us marched.
// Larger grids (k_ref_faces_march): a column marched up z re-reads far less
// halo.  256x240x248, 6 half-sweeps per launch: 134 us against 6 x 85 us; 4
// per launch: 119 us (memory-bound, 4.8 TB/s); boxes: 306 us per 4.
// 150x96x121, 4 per launch: 22.5 us against 4 x 11.2 us (6 per launch 35.5,
// boxes 42 per 4): there FP64 conversions and VALU issue bind.
#pragma once

#include "step_device.h"

namespace smk {
namespace {

// Relaxes a cell on its six faces f (u low, u high, v low, ...), as
// k_project_ref_half does, in two parts.
//
// Cells with six fluid neighbours (nearly all): the divisor is 6 and every face
// moves.  -dv / 6 is RN(double(-dv) * RN(1/6)): the FP64 product is within
// 2^-52 of the quotient, and no quotient by 6 comes that near a rounding
// boundary of FP32 without lying on it exactly (all 2^32 floats compared on
// the CPU).  Straight-line code for every lane: others subtract +0 and add
// -0, which leave every face as it was.
__device__ __forceinline__ void relax_full(bool full, double omega, float (&f)[6])
{
    const float dv = -f[0] + f[1] + -f[2] + f[3] + -f[4] + f[5];
    const float q = (float)((double)(-dv) * (1.0 / 6.0));
    const float p = (float)((double)q * omega);
    const float sub = full ? p : 0.0f, add = full ? p : -0.0f;
#pragma unroll
    for (int k = 0; k < 6; k += 2) {
        f[k] = f[k] - sub;
        f[k + 1] = f[k + 1] + add;
    }
}
// Cells next to a solid.
__device__ __forceinline__ void relax_partial(uint32_t c, double omega, float (&f)[6])
{
    const float dv = -f[0] + f[1] + -f[2] + f[3] + -f[4] + f[5];
    const float p = (float)((double)(-dv / (float)__popc(c & F_NBRS)) * omega);
#pragma unroll
    for (int k = 0; k < 6; k += 2) {
        f[k] = f[k] - p * (float)((c >> (k + 1)) & 1);
        f[k + 1] = f[k + 1] + p * (float)((c >> (k + 2)) & 1);
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
    const int tid = (int)threadIdx.x;
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
                if ((c & F_NBRS) == F_NBRS) relax_full(true, omega, face);
                else relax_partial(c & 0xffu, omega, face);
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
    static_assert(H % 2 == 0 && 64 % TP == 0, "whole pairs, whole rows per wave");
    static constexpr int IX = 2 * TP - 2 * H - 2, IY = TY - 2 * H;  // owned faces
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
    const int t = (int)threadIdx.x, r = (int)threadIdx.y;
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int b = dev::xcd_tile_order();
    const int xa = S::IX * (b % nbx) - H - 2, ya = S::IY * ((b / nbx) % nby) - H;
    const int z0 = zc * (b / (nbx * nby)), z1 = min(z0 + zc, g.nz);
    const int y = ya + r, skew = y & 1, x0 = xa + 2 * t + skew;
    const bool inside = x0 >= 0 && x0 < g.nx && y >= 0 && y < g.ny;
    // Lanes outside the grid read its first cells and have no flags.
    const uint32_t lane = inside ? (uint32_t)g.idx(x0, y, 0) : 0u;
    const uint32_t fmask = inside ? 0xffffu : 0u;
    const bool owner = inside && t >= H / 2 + 1 - skew && t < TP - H / 2 - skew && r >= H && r < TY - H;
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
                constexpr uint32_t kFull = F_ACTIVE | F_SELF | F_NBRS;
                relax_full(c == kFull, omega, f);
                if (c >= F_ACTIVE && c != kFull) relax_partial(c, omega, f);
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

// Half-sweeps per launch and z planes per workgroup of the marched form:
// one workgroup per CU (1024 threads), whose steps are its planes and the
// 3H of the pipeline's fill.
inline int march_planes(const Grid& g, int columns, int h)
{
    int best = g.nz;
    long long best_cost = -1;
    for (int chunks = 1; chunks <= (g.nz + 1) / 2; ++chunks) {
        const int zc = (g.nz + chunks - 1) / chunks;
        const long long rounds = ((long long)columns * ((g.nz + zc - 1) / zc) + kCUs - 1) / kCUs;
        const long long cost = rounds * (zc + 3 * h);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = zc;
        }
    }
    return best;
}

struct FaceSets {
    const float *ui, *vi, *wi;
    float *uo, *vo, *wo;
};

template <int H>
hipError_t launch_faces_march(const Grid& g, const FaceSets& f, const uint8_t* flags, int colour,
                              int sweeps, double omega, hipStream_t st)
{
    constexpr int TP = 32, TY = 32;
    using S = FaceColumn<TP, TY, H>;
    // Odd rows own one x less on the right: columns for nx + 1.
    const int nx = (g.nx + S::IX) / S::IX, ny = (g.ny + S::IY - 1) / S::IY;
    const int zc = march_planes(g, nx * ny, H);
    const dim3 grid((unsigned)nx, (unsigned)ny, (unsigned)((g.nz + zc - 1) / zc));
    hipLaunchKernelGGL((k_ref_faces_march<TP, TY, H>), grid, dim3(TP, TY), 0, st, g, f.ui, f.vi,
                       f.wi, f.uo, f.vo, f.wo, flags, zc, colour, sweeps, omega);
    return hipGetLastError();
}

}  // namespace
}  // namespace smk
