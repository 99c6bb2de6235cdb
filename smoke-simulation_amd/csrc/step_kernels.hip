// HIP kernels of one smoke time step for one simulation, for gfx950: FP32
// fields, or BF16 fields with FP32 arithmetic (the mixed-precision form; the
// per-field kernels are templates over the storage element).
//
// The arithmetic lives in step_device.h (shared with the batched kernels);
// the kernels here map threads to cells.  Thread blocks are 64 x 4 x 1: one
// wave64 covers 64 consecutive x of one row starting at a multiple of 64 (a
// stage that starts at x = 1 idles lane 0 of a row's first wave), so a
// wave's own-cell accesses are one contiguous 256-byte run (FP32) on two
// 128-byte lines of a 128-byte-aligned row, shared with no other wave;
// blockIdx.z walks z planes (kZ planes per thread in the streaming stages).
// Compiled with -ffp-contract=off: results are bit-identical to the oracle's
// FP32 mode.
#include <algorithm>

#include "redblack.h"
#include "step_device.h"

namespace smk {

namespace {

using dev::BX;
using dev::BY;

inline dim3 grid_for(int wx, int wy, int wz)
{
    return dim3((unsigned)((wx + BX - 1) / BX), (unsigned)((wy + BY - 1) / BY), (unsigned)wz);
}

// Cells per thread of the streaming stages (force, divergence, gradient,
// density advection): kZ consecutive planes of one column, so each thread
// has kZ cells' loads in flight (the *_col bodies of step_device.h).
constexpr int kZ = kColZ;
inline dim3 grid_col(int wx, int wy, int wz)
{
    return dim3((unsigned)((wx + BX - 1) / BX), (unsigned)((wy + BY - 1) / BY),
                (unsigned)((wz + kZ - 1) / kZ));
}

// ------------------------------------------------------------ utilities

__global__ void k_fill_f32(float* __restrict__ p, long long n, float value)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = value;
}

__global__ void k_fill_u8(uint8_t* __restrict__ p, long long n, uint8_t value)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = value;
}

// Contiguous index of the reference layout with row length rx and rows ry.
__device__ __forceinline__ long long cidx(int x, int y, int z, int rx, int ry)
{
    return x + (long long)rx * (y + (long long)ry * z);
}

// FP32 values of the reference layout <-> a padded field stored as T.
template <bool TO_PADDED, typename T>
__global__ void k_convert(Grid g, const void* __restrict__ src_, void* __restrict__ dst_, int wx,
                          int wy, int wz)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= wx || y >= wy || z >= wz) return;
    int i = g.idx(x, y, z);
    long long c = cidx(x, y, z, wx, wy);
    if (TO_PADDED)
        dev::stf(static_cast<T*>(dst_), i, static_cast<const float*>(src_)[c]);
    else
        static_cast<float*>(dst_)[c] = dev::ldf(static_cast<const T*>(src_), i);
}

template <bool TO_PADDED, typename T>
__global__ void k_repack(Grid g, const T* __restrict__ src, T* __restrict__ dst, int wx, int wy,
                         int wz)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= wx || y >= wy || z >= wz) return;
    int i = g.idx(x, y, z);
    long long c = cidx(x, y, z, wx, wy);
    if (TO_PADDED) dst[i] = src[c];
    else dst[c] = src[i];
}

// Padded FP32 cells -> contiguous 16-bit values: format 1 FP16 (hardware
// conversion, round to nearest even), format 2 BF16 (round to nearest even on
// the FP32 bits; NaN stays a quiet NaN).
template <typename T>
__global__ void k_pack_half(Grid g, const T* __restrict__ src, uint16_t* __restrict__ dst, int format)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    const float f = dev::ldf(src, g.idx(x, y, z));
    uint16_t h;
    if (format == 1) {
        h = __builtin_bit_cast(uint16_t, dev::to_f16(f));
    } else {
        h = dev::bf16_rne(f);
    }
    dst[cidx(x, y, z, g.nx, g.ny)] = h;
}

__global__ void k_unpack_solid(Grid g, const uint8_t* __restrict__ solid, uint8_t* __restrict__ base)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    base[g.idx(x, y, z)] = solid[cidx(x, y, z, g.nx, g.ny)] ? 0 : 1;
}

// Initial mask: fluid everywhere, solid floor y = 0 (smokeSimulation.cu:200-207).
__global__ void k_floor_mask(Grid g, uint8_t* __restrict__ base)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    base[g.idx(x, y, z)] = (y == 0) ? 0 : 1;
}

// --------------------------------------------------------------- scene

// fillObstacle (smokeSimulation.cu:289-313) over a base mask: interior cells
// only; LAST_WINS keeps the reference's overwrite-per-obstacle result.
__global__ void k_mask(Grid g, const uint8_t* __restrict__ base, uint8_t* __restrict__ s,
                       SphereList obst, int mode)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    int i = g.idx(x, y, z);
    uint8_t v = base[i];
    if (obst.count > 0 && dev::is_interior(g, x, y, z)) {
        bool solid;
        if (mode == SMOKE_OBSTACLES_LAST_WINS) {
            solid = dev::inside(obst.s[obst.count - 1], x, y, z);
        } else {
            solid = false;
            for (int k = 0; k < obst.count; ++k) solid = solid || dev::inside(obst.s[k], x, y, z);
        }
        if (solid) v = 0;
    }
    s[i] = v;
}

__global__ void k_flags(Grid g, const uint8_t* __restrict__ s, uint8_t* __restrict__ flags)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    int i = g.idx(x, y, z);
    uint8_t fl = s[i] ? F_SELF : 0;
    if (x > 0 && s[i - 1]) fl |= F_XM;
    if (x < g.nx - 1 && s[i + 1]) fl |= F_XP;
    if (y > 0 && s[i - g.px]) fl |= F_YM;
    if (y < g.ny - 1 && s[i + g.px]) fl |= F_YP;
    if (z > 0 && s[i - g.plane]) fl |= F_ZM;
    if (z < g.nz - 1 && s[i + g.plane]) fl |= F_ZP;
    if (dev::is_interior(g, x, y, z) && (fl & F_SELF) && (fl & F_NBRS)) fl |= F_ACTIVE;
    flags[i] = fl;
}

// Owner of each cell for the moving-obstacle boundary condition: the index
// of the obstacle whose sphere makes it solid under k_mask's rule (LAST_WINS:
// the last obstacle; UNION: the last one containing the cell), or kNoOwner.
__global__ void k_owner(Grid g, uint8_t* __restrict__ owner, SphereList obst, int mode)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    uint8_t who = kNoOwner;
    if (obst.count > 0 && dev::is_interior(g, x, y, z)) {
        if (mode == SMOKE_OBSTACLES_LAST_WINS) {
            if (dev::inside(obst.s[obst.count - 1], x, y, z)) who = (uint8_t)(obst.count - 1);
        } else {
            for (int k = 0; k < obst.count; ++k)
                if (dev::inside(obst.s[k], x, y, z)) who = (uint8_t)k;
        }
    }
    owner[g.idx(x, y, z)] = who;
}

// The low faces of cell (x,y,z) next to an owned cell take the owner's
// velocity component (this cell's owner first, else the low neighbour's).
template <typename T>
__global__ void k_obstacle_bc(Grid g, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                              const uint8_t* __restrict__ owner, SphereList vel)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    const int i = g.idx(x, y, z);
    const uint8_t self = owner[i];
    if (x >= 1) {
        const uint8_t o = self != kNoOwner ? self : owner[i - 1];
        if (o != kNoOwner) dev::stf(u, i, vel.s[o].x);
    }
    if (y >= 1) {
        const uint8_t o = self != kNoOwner ? self : owner[i - g.px];
        if (o != kNoOwner) dev::stf(v, i, vel.s[o].y);
    }
    if (z >= 1) {
        const uint8_t o = self != kNoOwner ? self : owner[i - g.plane];
        if (o != kNoOwner) dev::stf(w, i, vel.s[o].z);
    }
}

// fillSmoke (smokeSimulation.cu:251-273) for every source in one launch,
// restricted to the sources' bounding boxes (clipped to the interior by the
// launcher): blockIdx.z counts their planes, source after source.
struct SourceBoxes {
    int count;
    int first[SMOKE_MAX_OBJECTS + 1];  // planes of the sources before
    int lo[SMOKE_MAX_OBJECTS][3], ext[SMOKE_MAX_OBJECTS][2];
    float4 s[SMOKE_MAX_OBJECTS];
};
template <typename T>
__global__ void k_source(Grid g, T* __restrict__ r0, T* __restrict__ r1, SourceBoxes b)
{
    int k = 0;
    while (b.first[k + 1] <= (int)blockIdx.z) ++k;
    const int lx = blockIdx.x * BX + threadIdx.x, ly = blockIdx.y * BY + threadIdx.y;
    if (lx >= b.ext[k][0] || ly >= b.ext[k][1]) return;
    dev::source_at(g, r0, r1, b.s[k], b.lo[k][0] + lx, b.lo[k][1] + ly,
                   b.lo[k][2] + (int)blockIdx.z - b.first[k]);
}

// ---------------------------------------------------------- step stages

template <typename T, typename TR>
__global__ void k_force(Grid g, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                        const TR* __restrict__ rho, const uint8_t* __restrict__ flags, ForceArgs a)
{
    dev::force_col<kZ>(g, u, v, w, rho, flags, a, blockIdx.x * BX + threadIdx.x,
                       blockIdx.y * BY + threadIdx.y + 1, blockIdx.z * kZ);
}

// Vorticity confinement (an extension with no reference code; the bodies in
// step_device.h define it): curl, force and face passes over one simulation.
template <typename T>
__global__ void k_vort_curl(Grid g, const T* __restrict__ u, const T* __restrict__ v,
                            const T* __restrict__ w, const uint8_t* __restrict__ flags,
                            VortBufs b)
{
    dev::vort_curl_at(g, u, v, w, flags, b.mag, b.f[0], b.f[1], b.f[2],
                      blockIdx.x * BX + threadIdx.x, blockIdx.y * BY + threadIdx.y, blockIdx.z);
}

__global__ void k_vort_force(Grid g, const uint8_t* __restrict__ flags, VortBufs b, float eps)
{
    dev::vort_force_at(g, flags, b.mag, b.f[0], b.f[1], b.f[2], eps,
                       blockIdx.x * BX + threadIdx.x + 1, blockIdx.y * BY + threadIdx.y + 1,
                       blockIdx.z + 1);
}

template <typename T>
__global__ void k_vort_apply(Grid g, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                             const uint8_t* __restrict__ flags, VortBufs b, float dt)
{
    dev::vort_apply_at(g, u, v, w, flags, b.f[0], b.f[1], b.f[2], dt,
                       blockIdx.x * BX + threadIdx.x, blockIdx.y * BY + threadIdx.y, blockIdx.z);
}

// divergence (smokeSimulation.cu:356-394): one red-black SOR half-sweep in
// place on the face velocities.  Same-colour cells share no face, so the
// in-place update is race-free, and any assignment of the colour's cells to
// threads gives the same bits.  The (column pair, row) index is flat over the
// block's lanes (no idle lanes when a row holds fewer pairs than a wave), and
// each thread takes kRefZ consecutive planes, loading every cell's six faces
// and flags before it updates any (one wait for memory; every interior cell's
// faces lie inside the arrays).
constexpr int kRefZ = 2;

__global__ __launch_bounds__(BX * BY) void k_project_ref_half(
    Grid g, float* __restrict__ u, float* __restrict__ v, float* __restrict__ w,
    const uint8_t* __restrict__ flags, int colour, double omega, int pairs)
{
    const int f = (int)blockIdx.x * (BX * BY) + (int)threadIdx.y * BX + (int)threadIdx.x;
    if (f >= pairs * (g.ny - 2)) return;
    const int t = f % pairs, y = f / pairs + 1;
    const int z0 = (int)blockIdx.y * kRefZ + 1;
    float u0[kRefZ], u1[kRefZ], v0[kRefZ], v1[kRefZ], w0[kRefZ], w1[kRefZ];
    uint8_t fl[kRefZ];
    int ic[kRefZ];
#pragma unroll
    for (int j = 0; j < kRefZ; ++j) {
        const int z = z0 + j, x = dev::colour_x(t, y, z, colour);
        fl[j] = 0;
        ic[j] = 0;
        u0[j] = u1[j] = v0[j] = v1[j] = w0[j] = w1[j] = 0.0f;
        if (z > g.nz - 2 || x > g.nx - 2) continue;
        const int i = g.idx(x, y, z);
        ic[j] = i;
        u0[j] = u[i];
        u1[j] = u[i + 1];
        v0[j] = v[i];
        v1[j] = v[i + g.px];
        w0[j] = w[i];
        w1[j] = w[i + g.plane];
        fl[j] = flags[i];
    }
#pragma unroll
    for (int j = 0; j < kRefZ; ++j) {
        const uint8_t c = fl[j];
        if (!(c & F_ACTIVE)) continue;  // solid (:365), no fluid neighbour (:377), or no cell
        const int i = ic[j];
        int sx0 = (c >> 1) & 1, sx1 = (c >> 2) & 1;
        int sy0 = (c >> 3) & 1, sy1 = (c >> 4) & 1;
        int sz0 = (c >> 5) & 1, sz1 = (c >> 6) & 1;
        int acc = sx0 + sx1 + sy0 + sy1 + sz0 + sz1;
        float dv = -u0[j] + u1[j] + -v0[j] + v1[j] + -w0[j] + w1[j];
        float p = (float)((double)(-dv / (float)acc) * omega);
        u[i] = u0[j] - p * (float)sx0;
        u[i + 1] = u1[j] + p * (float)sx1;
        v[i] = v0[j] - p * (float)sy0;
        v[i + g.px] = v1[j] + p * (float)sy1;
        w[i] = w0[j] - p * (float)sz0;
        w[i + g.plane] = w1[j] + p * (float)sz1;
    }
}

template <typename T>
__global__ void k_divergence(Grid g, const T* __restrict__ u, const T* __restrict__ v,
                             const T* __restrict__ w, const uint8_t* __restrict__ flags,
                             float* __restrict__ d)
{
    dev::divergence_col<kZ>(g, u, v, w, flags, d, blockIdx.x * BX + threadIdx.x,
                            blockIdx.y * BY + threadIdx.y + 1, blockIdx.z * kZ + 1);
}

__global__ void k_jacobi(Grid g, const float* __restrict__ pin, float* __restrict__ pout,
                         const float* __restrict__ d, const uint8_t* __restrict__ flags,
                         float omega, int plain, int zero_in)
{
    dev::jacobi_at(g, pin, pout, d, flags, omega, plain, zero_in, blockIdx.x * BX + threadIdx.x,
                   blockIdx.y * BY + threadIdx.y + 1, blockIdx.z + 1);
}

// T fused Jacobi sweeps, one TX x TY tile per block of TX x (TY / R) threads
// (dev::jacobi_fused_tile).  One row per thread: at most 64 VGPRs, two
// 1024-thread blocks per CU; two rows per thread: at most 128 VGPRs.
template <int TX, int TY, int T, bool DAMPED, int R>
__global__ __launch_bounds__(TX * TY / R, 8 / R) void k_jacobi_fused(
    Grid g, const float* __restrict__ pin, float* __restrict__ pout, const float* __restrict__ d,
    const uint8_t* __restrict__ flags, int zc, int zero_in, float omega)
{
    __shared__ dev::FusedLds<TX, TY, T> sh;
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int L = dev::xcd_tile_order();
    dev::jacobi_fused_tile<TX, TY, T, DAMPED, R>(g, pin, pout, d, flags, zc, zero_in, omega,
                                                 L % nbx, (L / nbx) % nby, L / (nbx * nby), sh);
}

// One red-black SOR half-sweep of the pressure form, in place (on grids thin in
// x or y, rbsor_in_place).
__global__ __launch_bounds__(BX * BY) void k_rbsor_half(Grid g, float* __restrict__ p,
                                                    const float* __restrict__ d,
                                                    const uint8_t* __restrict__ flags, int colour,
                                                    float omega, int pairs)
{
    // The same thread layout as k_project_ref_half: a flat (column pair, row)
    // index and kRefZ consecutive planes per thread, every load issued before
    // any update.  The neighbours are of the other colour, which this launch
    // leaves alone, and every interior cell's neighbours lie inside the array.
    const int f = (int)blockIdx.x * (BX * BY) + (int)threadIdx.y * BX + (int)threadIdx.x;
    if (f >= pairs * (g.ny - 2)) return;
    const int t = f % pairs, y = f / pairs + 1;
    const int z0 = (int)blockIdx.y * kRefZ + 1;
    float nb[kRefZ][6], pc[kRefZ], di[kRefZ];
    uint8_t fl[kRefZ];
    int ic[kRefZ];
#pragma unroll
    for (int j = 0; j < kRefZ; ++j) {
        const int z = z0 + j, x = dev::colour_x(t, y, z, colour);
        fl[j] = 0;
        ic[j] = 0;
        pc[j] = di[j] = 0.0f;
#pragma unroll
        for (int k = 0; k < 6; ++k) nb[j][k] = 0.0f;
        if (z > g.nz - 2 || x > g.nx - 2) continue;
        const int i = g.idx(x, y, z);
        ic[j] = i;
        nb[j][0] = p[i - 1];
        nb[j][1] = p[i + 1];
        nb[j][2] = p[i - g.px];
        nb[j][3] = p[i + g.px];
        nb[j][4] = p[i - g.plane];
        nb[j][5] = p[i + g.plane];
        pc[j] = p[i];
        di[j] = d[i];
        fl[j] = flags[i];
    }
#pragma unroll
    for (int j = 0; j < kRefZ; ++j) {
        if (!(fl[j] & F_ACTIVE)) continue;
        const float G = dev::pressure_update(
            dev::sum6(nb[j][0], nb[j][1], nb[j][2], nb[j][3], nb[j][4], nb[j][5]),
            dev::inv_acc(__popc(fl[j] & F_NBRS)), di[j]);
        p[ic[j]] = pc[j] + omega * (G - pc[j]);
    }
}

// Warm start: zero the pressure of cells that are not active.
__global__ void k_mask_pressure(Grid g, float* __restrict__ p, const uint8_t* __restrict__ flags)
{
    int x = blockIdx.x * BX + threadIdx.x;
    int y = blockIdx.y * BY + threadIdx.y;
    int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny || z >= g.nz) return;
    int i = g.idx(x, y, z);
    if (!(flags[i] & F_ACTIVE)) p[i] = 0.0f;
}

template <typename T>
__global__ void k_gradient(Grid g, T* __restrict__ u, T* __restrict__ v, T* __restrict__ w,
                           const float* __restrict__ p, const uint8_t* __restrict__ flags)
{
    dev::gradient_col<kZ>(g, u, v, w, p, flags, blockIdx.x * BX + threadIdx.x,
                          blockIdx.y * BY + threadIdx.y + 1, blockIdx.z * kZ + 1);
}

// Velocity advection: a block of BX x BY threads marches a column of BX x BY
// cells through zc planes (dev::advect_velocity_march), in XCD tile order.
template <typename T>
__global__ __launch_bounds__(BX * BY, 8) void k_advect_velocity(
    Grid g, const T* __restrict__ u0, const T* __restrict__ v0, const T* __restrict__ w0,
    T* __restrict__ u1, T* __restrict__ v1, T* __restrict__ w1, const uint8_t* __restrict__ flags,
    float dt, int zc)
{
    __shared__ dev::AdvRing<BX, BY, 4, 3> ring;
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int L = dev::xcd_tile_order();
    dev::advect_velocity_march<BY>(g, u0, v0, w0, u1, v1, w1, flags, dt, 1 + BX * (L % nbx),
                                   1 + BY * ((L / nbx) % nby), 1 + zc * (L / (nbx * nby)), zc, ring);
}

// Density advection: a block of BX x BY threads marches a column of BX x BY
// cells through zc planes (dev::advect_density_march), in XCD tile order.
template <typename T, typename TV>
__global__ __launch_bounds__(BX * BY, sizeof(T) == 2 ? 8 : 1) void k_advect_density(
    Grid g, const T* __restrict__ r0, T* __restrict__ r1, const TV* __restrict__ u,
    const TV* __restrict__ v, const TV* __restrict__ w, const uint8_t* __restrict__ flags, float dt,
    int zc)
{
    __shared__ dev::AdvRing<BX, BY, 4, 1, 2> ring;
    const int nbx = (int)gridDim.x, nby = (int)gridDim.y;
    const int L = dev::xcd_tile_order();
    dev::advect_density_march<BY>(g, r0, r1, u, v, w, flags, dt, BX * (L % nbx),
                                  1 + BY * ((L / nbx) % nby), 1 + zc * (L / (nbx * nby)), zc, ring);
}

// Planes per block of the marched advection: kAdvChunkZ, fewer (down to 2)
// while the blocks would not give every CU four.  A block's planes are a serial
// chain of about 1.4 us each, so a grid that does not fill the GPU takes less
// time in shorter chunks although their window planes are loaded more often.
// Velocity / density, chunks of 16 -> this rule, us: 48x40x57 23.0 -> 6.0 / 15.7
// -> 4.1, 80^3 26.1 -> 11.0 / 16.9 -> 7.2, 113x90x101 28.8 -> 15.3 / 18.5 -> 9.1,
// 150x96x121 33.1 -> 25.1 / 20.4 -> 14.7 (two per CU: 13.8 / 7.6 at 80^3).
inline int advect_chunk(const dim3& columns, int planes)
{
    int zc = kAdvChunkZ;
    while (zc > 2 && (long long)columns.x * columns.y * ((planes + zc - 1) / zc) < 4 * kCUs) zc /= 2;
    return zc;
}

}  // namespace

// ------------------------------------------------------------- launchers

hipError_t fill_f32(float* p, long long n, float value, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    long long blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)blocks), dim3(256), 0, st, p, n, value);
    return hipGetLastError();
}

hipError_t fill_u8(uint8_t* p, long long n, uint8_t value, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    long long blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_fill_u8, dim3((unsigned)blocks), dim3(256), 0, st, p, n, value);
    return hipGetLastError();
}

hipError_t unpack_cells_f32(const Grid& g, const float* src, float* dst, hipStream_t st)
{
    hipLaunchKernelGGL((k_repack<true, float>), grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st,
                       g, src, dst, g.nx, g.ny, g.nz);
    return hipGetLastError();
}

hipError_t pack_cells_f32(const Grid& g, const float* src, float* dst, hipStream_t st)
{
    hipLaunchKernelGGL((k_repack<false, float>), grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st,
                       g, src, dst, g.nx, g.ny, g.nz);
    return hipGetLastError();
}

hipError_t unpack_faces_f32(const Grid& g, const float* src, float* dst, hipStream_t st)
{
    hipLaunchKernelGGL((k_repack<true, float>), grid_for(g.nx + 1, g.ny + 1, g.nz + 1),
                       dim3(BX, BY), 0, st, g, src, dst, g.nx + 1, g.ny + 1, g.nz + 1);
    return hipGetLastError();
}

hipError_t pack_faces_f32(const Grid& g, const float* src, float* dst, hipStream_t st)
{
    hipLaunchKernelGGL((k_repack<false, float>), grid_for(g.nx + 1, g.ny + 1, g.nz + 1),
                       dim3(BX, BY), 0, st, g, src, dst, g.nx + 1, g.ny + 1, g.nz + 1);
    return hipGetLastError();
}

hipError_t unpack_cells_solid(const Grid& g, const uint8_t* solid, uint8_t* base, hipStream_t st)
{
    hipLaunchKernelGGL(k_unpack_solid, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, solid,
                       base);
    return hipGetLastError();
}

hipError_t pack_cells_u8(const Grid& g, const uint8_t* src, uint8_t* dst, hipStream_t st)
{
    hipLaunchKernelGGL((k_repack<false, uint8_t>), grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st,
                       g, src, dst, g.nx, g.ny, g.nz);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_pack_half(const Grid& g, const T* src, uint16_t* dst, int format,
                                   hipStream_t st)
{
    hipLaunchKernelGGL(k_pack_half<T>, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, src, dst,
                       format);
    return hipGetLastError();
}
hipError_t pack_cells_half(const Grid& g, const float* src, uint16_t* dst, int format,
                           hipStream_t st)
{
    return launch_pack_half(g, src, dst, format, st);
}


hipError_t floor_mask(const Grid& g, uint8_t* base, hipStream_t st)
{
    hipLaunchKernelGGL(k_floor_mask, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, base);
    return hipGetLastError();
}

hipError_t build_mask(const Grid& g, const uint8_t* base, uint8_t* s, const SphereList& obst,
                      int mode, hipStream_t st)
{
    hipLaunchKernelGGL(k_mask, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, base, s, obst,
                       mode);
    return hipGetLastError();
}

hipError_t build_owner(const Grid& g, uint8_t* owner, const SphereList& obst, int mode,
                       hipStream_t st)
{
    hipLaunchKernelGGL(k_owner, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, owner, obst,
                       mode);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_obstacle_bc(const Grid& g, T* u, T* v, T* w, const uint8_t* owner,
                                     const SphereList& vel, hipStream_t st)
{
    hipLaunchKernelGGL(k_obstacle_bc<T>, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, u, v,
                       w, owner, vel);
    return hipGetLastError();
}
hipError_t obstacle_velocity_bc(const Grid& g, float* u, float* v, float* w, const uint8_t* owner,
                                const SphereList& vel, hipStream_t st)
{
    return launch_obstacle_bc(g, u, v, w, owner, vel, st);
}

hipError_t build_flags(const Grid& g, const uint8_t* s, uint8_t* flags, hipStream_t st)
{
    hipLaunchKernelGGL(k_flags, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, s, flags);
    return hipGetLastError();
}

bool source_box(const Grid& g, float4 sph, int lo[3], int ext[3])
{
    // Any cell with d^2 < r^2 lies within ceil(|r|) + 1 of the centre on each
    // axis; clipped to the interior [1, n-2].
    double r = fabs((double)sph.w);
    double c[3] = {(double)sph.x, (double)sph.y, (double)sph.z};
    int n[3] = {g.nx, g.ny, g.nz};
    for (int k = 0; k < 3; ++k) {
        if (!(c[k] == c[k]) || !(r == r)) return false;  // NaN: nothing inside
        double l = std::floor(c[k] - r) - 1.0, h = std::ceil(c[k] + r) + 1.0;
        int lk = l < 1.0 ? 1 : (l > n[k] - 2 ? n[k] - 1 : (int)l);
        int hk = h > n[k] - 2 ? n[k] - 2 : (h < 1.0 ? 0 : (int)h);
        if (lk > hk) return false;
        lo[k] = lk;
        ext[k] = hk - lk + 1;
    }
    return true;
}

template <typename T>
static hipError_t launch_sources(const Grid& g, T* rho0, T* rho1, const SphereList& src,
                                 hipStream_t st, int* launched)
{
    *launched = 0;
    SourceBoxes b;
    b.count = 0;
    b.first[0] = 0;
    int wx = 0, wy = 0;
    auto launch = [&]() {
        if (b.count == 0) return hipSuccess;
        hipLaunchKernelGGL(k_source<T>, grid_for(wx, wy, b.first[b.count]), dim3(BX, BY), 0, st, g, rho0,
                           rho1, b);
        *launched += 1;
        b.count = wx = wy = 0;
        return hipGetLastError();
    };
    for (int k = 0; k < src.count; ++k) {
        int lo[3], ext[3];
        if (!source_box(g, src.s[k], lo, ext)) continue;
        if (b.first[b.count] + (long long)ext[2] > 65535) {  // a grid's z extent
            const hipError_t e = launch();
            if (e != hipSuccess) return e;
        }
        const int n = b.count++;
        for (int a = 0; a < 3; ++a) b.lo[n][a] = lo[a];
        b.ext[n][0] = ext[0];
        b.ext[n][1] = ext[1];
        b.s[n] = src.s[k];
        b.first[n + 1] = b.first[n] + ext[2];
        wx = std::max(wx, ext[0]);
        wy = std::max(wy, ext[1]);
    }
    return launch();
}

hipError_t fill_sources(const Grid& g, float* rho0, float* rho1, const SphereList& src, hipStream_t st,
                        int* launched)
{
    return launch_sources(g, rho0, rho1, src, st, launched);
}

template <typename T, typename TR>
static hipError_t launch_force(const Grid& g, T* u, T* v, T* w, const TR* rho, const uint8_t* flags,
                               const ForceArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL((k_force<T, TR>), grid_col(g.nx, g.ny - 1, g.nz), dim3(BX, BY), 0, st, g, u,
                       v, w, rho, flags, a);
    return hipGetLastError();
}
hipError_t force(const Grid& g, float* u, float* v, float* w, const float* rho,
                 const uint8_t* flags, const ForceArgs& a, hipStream_t st)
{
    return launch_force(g, u, v, w, rho, flags, a, st);
}

template <typename T>
static hipError_t launch_vorticity(const Grid& g, T* u, T* v, T* w, const uint8_t* flags,
                                   const VortBufs& b, float eps, float dt, hipStream_t st)
{
    hipLaunchKernelGGL(k_vort_curl<T>, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, u, v, w,
                       flags, b);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_vort_force, grid_for(g.nx - 2, g.ny - 2, g.nz - 2), dim3(BX, BY), 0, st, g,
                       flags, b, eps);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_vort_apply<T>, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, u, v, w,
                       flags, b, dt);
    return hipGetLastError();
}
hipError_t vorticity(const Grid& g, float* u, float* v, float* w, const uint8_t* flags,
                     const VortBufs& b, float eps, float dt, hipStream_t st)
{
    return launch_vorticity(g, u, v, w, flags, b, eps, dt, st);
}

void forget_last_error() { (void)hipGetLastError(); }

hipError_t project_reference_half(const Grid& g, float* u, float* v, float* w,
                                  const uint8_t* flags, int colour, double omega, hipStream_t st)
{
    const int pairs = (g.nx - 2 + 1) / 2;  // cells of one colour per row, at most
    const long long items = (long long)pairs * (g.ny - 2);
    const dim3 grid((unsigned)((items + BX * BY - 1) / (BX * BY)),
                    (unsigned)((g.nz - 2 + kRefZ - 1) / kRefZ));
    hipLaunchKernelGGL(k_project_ref_half, grid, dim3(BX, BY), 0, st, g, u, v, w, flags, colour,
                       omega, pairs);
    return hipGetLastError();
}

// How the reference form's half-sweeps run.  At most one box per CU: boxes
// (redblack.h has both sides).  Else columns, 4 half-sweeps per launch, or where
// the two sets of faces and the flags approach the 256 MB memory-side cache (a
// launch is then bound by memory and fewer passes pay for the larger halo) the
// better fitting of 5 and 6.  us per half-sweep of empty grids with 4 / 5 / 6:
// 160^3 (125 MB) 7.8 / 9.0 / 8.7, 192x180x188 (191 MB) 10.7 / 11.0 / 10.6,
// 224x200x210 (271 MB) 19.5 / 15.7 / 14.4, 256x240x248 29.0 / 25.5 / 26.7 (one
// column more for 6).
constexpr int kBoxX = 24, kBoxY = 10, kBoxZ = 10;
struct FacesRoute {
    bool boxed;
    dim3 boxes;
    int H;
    MarchPlan plan;  // of the columns
};
static FacesRoute faces_route(const Grid& g)
{
    FacesRoute r{};
    r.boxes = dim3((unsigned)((g.nx + kBoxX - 1) / kBoxX), (unsigned)((g.ny + kBoxY - 1) / kBoxY),
                   (unsigned)((g.nz + kBoxZ - 1) / kBoxZ));
    r.boxed = (long long)r.boxes.x * r.boxes.y * r.boxes.z <= kCUs;
    r.H = 4;
    if (r.boxed) return r;
    if ((long long)g.elems * 25 > (180LL << 20)) {
        const MarchPlan five = faces_plan<5>(g), six = faces_plan<6>(g);
        r.H = five.steps * 6 < six.steps * 5 ? 5 : 6;
        r.plan = r.H == 5 ? five : six;
    } else {
        r.plan = faces_plan<4>(g);
    }
    return r;
}
// An even number of launches, so that the last one writes the first set again.
static int faces_launches(const FacesRoute& r, int sweeps) { return 2 * ((sweeps + 2 * r.H - 1) / (2 * r.H)); }

// The 128-byte lines of a field that a half-sweep visits.
static double half_sweep_lines(const Grid& g) { return (double)(g.ny - 2) * (g.nz - 2) * ((g.nx + 31) / 32); }
static double interior_cells(const Grid& g) { return (double)(g.nx - 2) * (g.ny - 2) * (g.nz - 2); }

// A column of the marched launches costs the same however few of its cells the
// grid has, and a grid thin in x or y fills little of it: one half-sweep per
// launch in place is then faster.  Both by their measured times (400 random
// grids, extents 3..20000, within 5 % for most): a marched launch 2.5 us, and 0.6
// and 0.125 for each half-sweep a step; a half-sweep 2.8 us, 6.9 per 10^5
// 128-byte lines and 3.4 per 10^6 cells.  The march has to gain 15 % by these.
// us for 40 half-sweeps, in place /
// marched: 18072x3x56 290 / 1290, 59x4x19372 569 / 1864, 10x4x3220 146 / 299,
// 129x9x882 249 / 282, 130x3308x6 388 / 412; 28x120x289 326 / 226, 150x96x121
// 431 / 226 (4 of them 43 / 34).  Of the boxes' two launches, 4 half-sweeps in
// place are faster or as fast: 16x16x40 12 / 15, 80^3 21 / 21.
bool reference_in_place(const Grid& g, int sweeps)
{
    if (sweeps < 4) return true;
    if ((g.nz - 2 + kRefZ - 1) / kRefZ > 65535) return false;  // a grid's y extent
    const FacesRoute r = faces_route(g);
    if (r.boxed) return sweeps < 6;
    const double in_place = sweeps * (2.8 + 6.9e-5 * half_sweep_lines(g) + 3.4e-6 * interior_cells(g));
    const int n = faces_launches(r, sweeps);
    return in_place < 1.15 * n * (2.5 + (0.6 + 0.125 * sweeps / n) * (double)r.plan.steps);
}

hipError_t project_reference_sweeps(const Grid& g, float* const (&a)[3], float* const (&b)[3],
                                    const uint8_t* flags, int sweeps, double omega, hipStream_t st,
                                    int* launches)
{
    const FacesRoute r = faces_route(g);
    const int n = faces_launches(r, sweeps);
    *launches = 0;
    for (int l = 0, done = 0; l < n; ++l) {
        const int m = sweeps / n + (l < sweeps % n ? 1 : 0), colour = done & 1;
        float* const* in = l & 1 ? b : a;
        float* const* out = l & 1 ? a : b;
        const FaceSets f = {in[0], in[1], in[2], out[0], out[1], out[2]};
        hipError_t e;
        if (r.boxed) {
            hipLaunchKernelGGL((k_ref_faces_box<kBoxX, kBoxY, kBoxZ, 4>), r.boxes, dim3(kBoxThreads), 0,
                               st, g, f.ui, f.vi, f.wi, f.uo, f.vo, f.wo, flags, colour, m, omega);
            e = hipGetLastError();
        } else {
            e = r.H == 6   ? launch_faces_march<6>(g, r.plan, f, flags, colour, m, omega, st)
                : r.H == 5 ? launch_faces_march<5>(g, r.plan, f, flags, colour, m, omega, st)
                           : launch_faces_march<4>(g, r.plan, f, flags, colour, m, omega, st);
        }
        if (e != hipSuccess) return e;
        done += m;
        ++*launches;
    }
    return hipSuccess;
}

template <typename T>
static hipError_t launch_divergence(const Grid& g, const T* u, const T* v, const T* w,
                                    const uint8_t* flags, float* d, hipStream_t st)
{
    hipLaunchKernelGGL(k_divergence<T>, grid_col(g.nx - 1, g.ny - 2, g.nz - 2), dim3(BX, BY), 0, st,
                       g, u, v, w, flags, d);
    return hipGetLastError();
}
hipError_t divergence(const Grid& g, const float* u, const float* v, const float* w,
                      const uint8_t* flags, float* d, hipStream_t st)
{
    return launch_divergence(g, u, v, w, flags, d, st);
}

hipError_t jacobi_sweep(const Grid& g, const float* pin, float* pout, const float* d,
                        const uint8_t* flags, float omega, int plain, int zero_in, hipStream_t st)
{
    hipLaunchKernelGGL(k_jacobi, grid_for(g.nx - 1, g.ny - 2, g.nz - 2), dim3(BX, BY), 0, st, g,
                       pin, pout, d, flags, omega, plain, zero_in);
    return hipGetLastError();
}

template <int TX, int TY, int R, int T>
static hipError_t launch_fused(const Grid& g, const float* pin, float* pout, const float* d,
                               const uint8_t* flags, int zc, int zero_in, float omega, bool damped,
                               hipStream_t st)
{
    constexpr int OX = TX - 2 * T, OY = TY - 2 * T;
    const int m[3] = {g.nx - 2, g.ny - 2, g.nz - 2};
    dim3 grid((unsigned)((m[0] + OX - 1) / OX), (unsigned)((m[1] + OY - 1) / OY),
              (unsigned)((m[2] + zc - 1) / zc));
    const dim3 block(TX, TY / R);
    if (damped)
        hipLaunchKernelGGL((k_jacobi_fused<TX, TY, T, true, R>), grid, block, 0, st, g, pin, pout,
                           d, flags, zc, zero_in, omega);
    else
        hipLaunchKernelGGL((k_jacobi_fused<TX, TY, T, false, R>), grid, block, 0, st, g, pin,
                           pout, d, flags, zc, zero_in, omega);
    return hipGetLastError();
}

template <int TX, int TY, int R>
static hipError_t launch_fused_t(const Grid& g, const float* pin, float* pout, const float* d,
                                 const uint8_t* flags, int t, int zc, int zero_in, float omega,
                                 bool damped, hipStream_t st)
{
    switch (t) {
    case 2: return launch_fused<TX, TY, R, 2>(g, pin, pout, d, flags, zc, zero_in, omega, damped, st);
    case 3: return launch_fused<TX, TY, R, 3>(g, pin, pout, d, flags, zc, zero_in, omega, damped, st);
    case 4: return launch_fused<TX, TY, R, 4>(g, pin, pout, d, flags, zc, zero_in, omega, damped, st);
    case 5: return launch_fused<TX, TY, R, 5>(g, pin, pout, d, flags, zc, zero_in, omega, damped, st);
    case 6: return launch_fused<TX, TY, R, 6>(g, pin, pout, d, flags, zc, zero_in, omega, damped, st);
    default: return hipErrorInvalidValue;
    }
}

// A plan that was never set follows the grid: with the plan's own 64 planes per
// workgroup a small grid occupies a handful of CUs (48x40x57: 4 workgroups,
// 30.6 us per 4 sweeps; fitted 8.2 us per 5) and a middling one fills the last
// round of CUs badly (197x131x243: 36.5 us per 4, fitted 30.1 per 5).  Five
// sweeps per launch, whose loop is unrolled by 6 planes only, were the fastest
// per sweep at every size measured (48x40x57 to 512^3), in 32x32 tiles (two
// workgroups per CU) on small grids and 64x32 tiles on large ones.  The step
// times are measured on full-size tiles of those grids; where the fields
// outgrow the 256 MB memory-side cache, a launch takes at least the tiles'
// re-read bytes at 4.9 TB/s.
JacobiPlan fitted_plan(const Grid& g, bool refined)
{
    JacobiPlan plan;
    const int m[3] = {g.nx - 2, g.ny - 2, g.nz - 2};
    const int most = std::max(1, fused_max_zc(g.plane));
    auto columns = [&](int w, int h, int ox, int oy) { return (w + ox - 1) / ox * ((h + oy - 1) / oy); };
    double us = 0.0;
    if (refined) {
        // FP16 pairs: 64x32-cell tiles (two per CU) of 4 sweeps, as unset plans had.
        constexpr int T = 4;
        const ChunkModel half{2 * T, 6, 2, 0.45, 0.70};
        plan.zc = fit_chunk(half, columns(g.nx, m[1], 64 - 2 * T, 32 - 2 * T), m[2], std::min(64, most), &us);
        return plan;
    }
    constexpr int T = 5;
    plan.sweeps_per_launch = T;
    const double cells = (double)m[0] * m[1] * m[2];
    const double memory = cells * 13.0 > 256e6 ? cells * 13.0 / 4.9e6 : 0.0;  // us, halo apart
    const ChunkModel one_row{2 * T, 6, 2, 0.42, 0.66}, two_rows{2 * T, 6, 1, 0.72, 0.73};
    plan.zc = fit_chunk(one_row, columns(m[0], m[1], 32 - 2 * T, 32 - 2 * T), m[2], most, &us);
    const double one_us = std::max(us, 1.6 * memory);
    const int zc = fit_chunk(two_rows, columns(m[0], m[1], 64 - 2 * T, 32 - 2 * T), m[2], most, &us);
    if (std::max(us, 1.27 * memory) < one_us) {
        plan.tile = JacobiPlan::TILE_64x32;
        plan.zc = zc;
    }
    return plan;
}

hipError_t jacobi_fused(const Grid& g, const float* pin, float* pout, const float* d,
                        const uint8_t* flags, const JacobiPlan& plan, int sweeps, float omega,
                        int plain, int zero_in, hipStream_t st)
{
    if (sweeps == 1)
        return jacobi_sweep(g, pin, pout, d, flags, omega, plain, zero_in, st);
    if (plan.zc < 1) return hipErrorInvalidValue;
    // The z-chunk is a speed parameter (every chunk gives the same bits): cap
    // it so a block's span of planes fits the 32-bit buffer offsets.
    const int zc = std::min(plan.zc, fused_max_zc(g.plane));
    if (zc < 1) return hipErrorInvalidValue;  // enqueue_jacobi runs single sweeps then
    const bool damped = !plain;
    switch (plan.tile) {
    case JacobiPlan::TILE_32x32:
        return launch_fused_t<32, 32, 1>(g, pin, pout, d, flags, sweeps, zc, zero_in, omega, damped, st);
    case JacobiPlan::TILE_64x16:
        return launch_fused_t<64, 16, 1>(g, pin, pout, d, flags, sweeps, zc, zero_in, omega, damped, st);
    case JacobiPlan::TILE_64x32:
        return launch_fused_t<64, 32, 2>(g, pin, pout, d, flags, sweeps, zc, zero_in, omega, damped, st);
    case JacobiPlan::TILE_32x64:
        return launch_fused_t<32, 64, 2>(g, pin, pout, d, flags, sweeps, zc, zero_in, omega, damped, st);
    default: return hipErrorInvalidValue;
    }
}

// 4 or 6 half-sweeps per launch, whichever takes fewer steps per half-sweep;
// narrow columns where the grid is too small to fill the CUs with wide ones.
// us per half-sweep, narrow 4 / 4 / 6: 48x40x57 1.9 / 2.5 / 2.5, 80^3 2.5 / 2.8
// / 2.7, 113x90x101 3.2 / 3.2 / 3.3, 150^3 6.0 / 4.8 / 4.5, 256x240x248 19.2 /
// 11.8 / 11.6.
struct PressureRoute {
    bool narrow;
    int H;
    MarchPlan plan;
};
static PressureRoute pressure_route(const Grid& g)
{
    PressureRoute r{(long long)g.nx * g.ny * g.nz <= 1500000, 4, MarchPlan{}};
    if (r.narrow) {
        r.plan = pressure_plan<16, 4>(g);
        return r;
    }
    const MarchPlan four = pressure_plan<32, 4>(g), six = pressure_plan<32, 6>(g);
    r.H = four.steps * 6 <= six.steps * 4 ? 4 : 6;
    r.plan = r.H == 4 ? four : six;
    return r;
}

// As reference_in_place, by the pressure form's times (1200 random grids): a
// marched launch 2.5 us and 0.86 a step of wide columns, 0.535 of narrow ones
// (0.39 where two of those share a CU); a half-sweep 2.35 us, 4.2 per 10^5
// 128-byte lines and 2.3 per 10^6 cells, and one pass to mask or clear the
// pressure.  The march has to gain 10 %.  us for 40 half-sweeps with divergence
// and gradient, in place / marched: 18072x3x56 249 / 728, 51x4x6934 221 / 522,
// 3944x209x3 207 / 270, 256x6x235 139 / 143; 24^3 122 / 93, 113x90x101 265 / 147.
bool rbsor_in_place(const Grid& g, int sweeps)
{
    if (sweeps == 0) return true;
    if ((g.nz - 2 + kRefZ - 1) / kRefZ > 65535) return false;  // a grid's y extent
    const PressureRoute r = pressure_route(g);
    const double in_place = sweeps * (2.35 + 4.2e-5 * half_sweep_lines(g) + 2.3e-6 * interior_cells(g)) +
                            2.3 + 1e-6 * g.elems;
    const bool shared = (long long)r.plan.grid.x * r.plan.grid.y * r.plan.grid.z > kCUs;
    const double step = r.narrow ? (shared ? 0.39 : 0.535) : 0.86;
    return in_place < 1.1 * sweeps / r.H * (2.5 + step * (double)r.plan.steps);
}

hipError_t rbsor_half(const Grid& g, float* p, const float* d, const uint8_t* flags, int colour,
                      float omega, hipStream_t st)
{
    const int pairs = (g.nx - 2 + 1) / 2;
    const long long items = (long long)pairs * (g.ny - 2);
    const dim3 grid((unsigned)((items + BX * BY - 1) / (BX * BY)),
                    (unsigned)((g.nz - 2 + kRefZ - 1) / kRefZ));
    hipLaunchKernelGGL(k_rbsor_half, grid, dim3(BX, BY), 0, st, g, p, d, flags, colour, omega,
                       pairs);
    return hipGetLastError();
}

hipError_t rbsor_sweeps(const Grid& g, float* const (&p)[2], int* cur, const float* d,
                        const uint8_t* flags, int sweeps, float omega, int cold, hipStream_t st,
                        int* launches)
{
    const PressureRoute r = pressure_route(g);
    const int n = (sweeps + r.H - 1) / r.H;
    *launches = 0;
    for (int l = 0, done = 0; l < n; ++l) {
        const int m = sweeps / n + (l < sweeps % n ? 1 : 0), colour = done & 1;
        const float* pi = p[*cur];
        float* po = p[*cur ^ 1];
        const int zero_in = cold && l == 0;
        const hipError_t e =
            r.narrow ? launch_pressure_march<16, 4>(g, r.plan, pi, po, d, flags, colour, m, omega, zero_in, st)
            : r.H == 4
                ? launch_pressure_march<32, 4>(g, r.plan, pi, po, d, flags, colour, m, omega, zero_in, st)
                : launch_pressure_march<32, 6>(g, r.plan, pi, po, d, flags, colour, m, omega, zero_in, st);
        if (e != hipSuccess) return e;
        *cur ^= 1;
        done += m;
        ++*launches;
    }
    return hipSuccess;
}

hipError_t mask_pressure(const Grid& g, float* p, const uint8_t* flags, hipStream_t st)
{
    hipLaunchKernelGGL(k_mask_pressure, grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, g, p,
                       flags);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_gradient(const Grid& g, T* u, T* v, T* w, const float* p,
                                  const uint8_t* flags, hipStream_t st)
{
    hipLaunchKernelGGL(k_gradient<T>, grid_col(g.nx, g.ny - 1, g.nz - 1), dim3(BX, BY), 0, st,
                       g, u, v, w, p, flags);
    return hipGetLastError();
}
hipError_t gradient(const Grid& g, float* u, float* v, float* w, const float* p,
                    const uint8_t* flags, hipStream_t st)
{
    return launch_gradient(g, u, v, w, p, flags, st);
}

template <typename T>
static hipError_t launch_advect_velocity(const Grid& g, const T* u0, const T* v0, const T* w0,
                                         T* u1, T* v1, T* w1, const uint8_t* flags, float dt,
                                         hipStream_t st)
{
    dim3 grid((unsigned)((g.nx - 1 + BX - 1) / BX), (unsigned)((g.ny - 1 + BY - 1) / BY));
    const int zc = advect_chunk(grid, g.nz - 1);
    grid.z = (unsigned)((g.nz - 1 + zc - 1) / zc);
    hipLaunchKernelGGL(k_advect_velocity<T>, grid, dim3(BX, BY), 0, st, g, u0, v0, w0, u1, v1, w1,
                       flags, dt, zc);
    return hipGetLastError();
}
hipError_t advect_velocity(const Grid& g, const float* u0, const float* v0, const float* w0,
                           float* u1, float* v1, float* w1, const uint8_t* flags, float dt,
                           hipStream_t st)
{
    return launch_advect_velocity(g, u0, v0, w0, u1, v1, w1, flags, dt, st);
}

template <typename T, typename TV>
static hipError_t launch_advect_density(const Grid& g, const T* r0, T* r1, const TV* u, const TV* v,
                                        const TV* w, const uint8_t* flags, float dt, hipStream_t st)
{
    dim3 grid((unsigned)((g.nx - 1 + BX - 1) / BX), (unsigned)((g.ny - 2 + BY - 1) / BY));
    const int zc = advect_chunk(grid, g.nz - 2);
    grid.z = (unsigned)((g.nz - 2 + zc - 1) / zc);
    hipLaunchKernelGGL((k_advect_density<T, TV>), grid, dim3(BX, BY), 0, st, g, r0, r1, u, v, w,
                       flags, dt, zc);
    return hipGetLastError();
}
hipError_t advect_density(const Grid& g, const float* r0, float* r1, const float* u,
                          const float* v, const float* w, const uint8_t* flags, float dt,
                          hipStream_t st)
{
    return launch_advect_density(g, r0, r1, u, v, w, flags, dt, st);
}

// The stages and conversions for 16-bit stored fields H (declared in
// smoke_internal.h), density stored as H or as FP32.
#define SMK_HALF_STORAGE_DEFS(H)                                                                   \
    hipError_t pack_cells_half(const Grid& g, const H* src, uint16_t* dst, int format,             \
                               hipStream_t st)                                                     \
    {                                                                                              \
        return launch_pack_half(g, src, dst, format, st);                                          \
    }                                                                                              \
    hipError_t unpack_cells_f32(const Grid& g, const float* src, H* dst, hipStream_t st)           \
    {                                                                                              \
        hipLaunchKernelGGL((k_convert<true, H>), grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st,  \
                           g, (const void*)src, (void*)dst, g.nx, g.ny, g.nz);                     \
        return hipGetLastError();                                                                  \
    }                                                                                              \
    hipError_t pack_cells_f32(const Grid& g, const H* src, float* dst, hipStream_t st)             \
    {                                                                                              \
        hipLaunchKernelGGL((k_convert<false, H>), grid_for(g.nx, g.ny, g.nz), dim3(BX, BY), 0, st, \
                           g, (const void*)src, (void*)dst, g.nx, g.ny, g.nz);                     \
        return hipGetLastError();                                                                  \
    }                                                                                              \
    hipError_t unpack_faces_f32(const Grid& g, const float* src, H* dst, hipStream_t st)           \
    {                                                                                              \
        hipLaunchKernelGGL((k_convert<true, H>), grid_for(g.nx + 1, g.ny + 1, g.nz + 1),           \
                           dim3(BX, BY), 0, st, g, (const void*)src, (void*)dst, g.nx + 1,         \
                           g.ny + 1, g.nz + 1);                                                    \
        return hipGetLastError();                                                                  \
    }                                                                                              \
    hipError_t pack_faces_f32(const Grid& g, const H* src, float* dst, hipStream_t st)             \
    {                                                                                              \
        hipLaunchKernelGGL((k_convert<false, H>), grid_for(g.nx + 1, g.ny + 1, g.nz + 1),          \
                           dim3(BX, BY), 0, st, g, (const void*)src, (void*)dst, g.nx + 1,         \
                           g.ny + 1, g.nz + 1);                                                    \
        return hipGetLastError();                                                                  \
    }                                                                                              \
    hipError_t fill_sources(const Grid& g, H* rho0, H* rho1, const SphereList& src,                \
                            hipStream_t st, int* launched)                                         \
    {                                                                                              \
        return launch_sources(g, rho0, rho1, src, st, launched);                                   \
    }                                                                                              \
    hipError_t force(const Grid& g, H* u, H* v, H* w, const H* rho, const uint8_t* flags,          \
                     const ForceArgs& a, hipStream_t st)                                           \
    {                                                                                              \
        return launch_force(g, u, v, w, rho, flags, a, st);                                        \
    }                                                                                              \
    hipError_t force(const Grid& g, H* u, H* v, H* w, const float* rho, const uint8_t* flags,      \
                     const ForceArgs& a, hipStream_t st)                                           \
    {                                                                                              \
        return launch_force(g, u, v, w, rho, flags, a, st);                                        \
    }                                                                                              \
    hipError_t obstacle_velocity_bc(const Grid& g, H* u, H* v, H* w, const uint8_t* owner,         \
                                    const SphereList& vel, hipStream_t st)                         \
    {                                                                                              \
        return launch_obstacle_bc(g, u, v, w, owner, vel, st);                                     \
    }                                                                                              \
    hipError_t vorticity(const Grid& g, H* u, H* v, H* w, const uint8_t* flags,                    \
                         const VortBufs& b, float eps, float dt, hipStream_t st)                   \
    {                                                                                              \
        return launch_vorticity(g, u, v, w, flags, b, eps, dt, st);                                \
    }                                                                                              \
    hipError_t divergence(const Grid& g, const H* u, const H* v, const H* w,                       \
                          const uint8_t* flags, float* d, hipStream_t st)                          \
    {                                                                                              \
        return launch_divergence(g, u, v, w, flags, d, st);                                        \
    }                                                                                              \
    hipError_t gradient(const Grid& g, H* u, H* v, H* w, const float* p, const uint8_t* flags,     \
                        hipStream_t st)                                                            \
    {                                                                                              \
        return launch_gradient(g, u, v, w, p, flags, st);                                          \
    }                                                                                              \
    hipError_t advect_velocity(const Grid& g, const H* u0, const H* v0, const H* w0, H* u1,        \
                               H* v1, H* w1, const uint8_t* flags, float dt, hipStream_t st)       \
    {                                                                                              \
        return launch_advect_velocity(g, u0, v0, w0, u1, v1, w1, flags, dt, st);                   \
    }                                                                                              \
    hipError_t advect_density(const Grid& g, const H* r0, H* r1, const H* u, const H* v,           \
                              const H* w, const uint8_t* flags, float dt, hipStream_t st)          \
    {                                                                                              \
        return launch_advect_density(g, r0, r1, u, v, w, flags, dt, st);                           \
    }                                                                                              \
    hipError_t advect_density(const Grid& g, const float* r0, float* r1, const H* u, const H* v,   \
                              const H* w, const uint8_t* flags, float dt, hipStream_t st)          \
    {                                                                                              \
        return launch_advect_density(g, r0, r1, u, v, w, flags, dt, st);                           \
    }
SMK_HALF_STORAGE_DEFS(bf16s)
SMK_HALF_STORAGE_DEFS(f16s)
#undef SMK_HALF_STORAGE_DEFS

}  // namespace smk
