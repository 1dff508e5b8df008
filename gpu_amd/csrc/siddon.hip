// siddon.hip - ray-driven Siddon projector for gfx950.
//
// One ray per lane.  A 256-thread workgroup owns a 16x16 tile of detector
// pixels and each wave64 an 8x8 sub-tile, so the 64 rays of a wave stay
// within a few voxels of each other along the whole traversal and their
// gathers share cache lines.
//
// The traversal restates forward_ray_driven_3d_kernel_correction
// (V63/kernel_IterativeRecon_universal.cu:14-551; multi-source variant
// TB/voxel/kernel_IterativeRecon_TBCT_voxel.cu:1-545) with the same FP
// operation order, so with contraction off the FP32 path reproduces the
// reference arithmetic.  The reference's seven tie branches (:307-549) are
// one branch-free step here: every axis whose next crossing equals the
// minimum steps, which is the same set of cases without wave divergence.
#include "ct_internal.hpp"
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <mutex>
#include <string>

namespace ct {

template <typename T> __device__ __forceinline__ T dfloor(T x);
template <> __device__ __forceinline__ float dfloor<float>(float x) { return floorf(x); }
template <> __device__ __forceinline__ double dfloor<double>(double x) { return floor(x); }
template <typename T> __device__ __forceinline__ T dmin(T a, T b);
template <> __device__ __forceinline__ float dmin<float>(float a, float b) { return fminf(a, b); }
template <> __device__ __forceinline__ double dmin<double>(double a, double b) { return fmin(a, b); }
template <typename T> __device__ __forceinline__ T dmax(T a, T b);
template <> __device__ __forceinline__ float dmax<float>(float a, float b) { return fmaxf(a, b); }
template <> __device__ __forceinline__ double dmax<double>(double a, double b) { return fmax(a, b); }
template <typename T> __device__ __forceinline__ T dabs(T a);
template <> __device__ __forceinline__ float dabs<float>(float a) { return fabsf(a); }
template <> __device__ __forceinline__ double dabs<double>(double a) { return fabs(a); }
template <typename T> __device__ __forceinline__ T dsqrt(T a);
template <> __device__ __forceinline__ float dsqrt<float>(float a) { return sqrtf(a); }
template <> __device__ __forceinline__ double dsqrt<double>(double a) { return sqrt(a); }
template <typename T> __device__ __forceinline__ T dinf();
template <> __device__ __forceinline__ float dinf<float>() { return __builtin_inff(); }
template <> __device__ __forceinline__ double dinf<double>() { return __builtin_inf(); }
template <typename T> __device__ __forceinline__ T loop_eps();
template <> __device__ __forceinline__ float loop_eps<float>() { return 1e-16f; }
template <> __device__ __forceinline__ double loop_eps<double>() { return 1e-16; }

// Traverses the ray detector pixel (col,row) -> source `src`; visit(index, len)
// per segment.  Returns the summed length.
template <typename T, typename F>
__device__ __forceinline__ T siddon_traverse(const DGeo<T> &d, T s, T c, int col, int row, int src, F &&visit) {
    const int M = d.M, N = d.N, Z = d.Z;
    const T u = d.ymin + (T)col * d.du;
    const T x1x = d.dod * c - u * s;
    const T x1y = d.dod * s + u * c;
    const T x1z = d.zmin + (T)row * d.dv;
    T x2x, x2y, x2z;
    ray_source(d, s, c, u, x1z, src, x2x, x2y, x2z);
    const T ixd = (T)1 / (x2x - x1x);
    const T iyd = (T)1 / (x2y - x1y);
    const T izd = (T)1 / (x2z - x1z);

    T a0, a1;
    a0 = (d.bx - x1x) * ixd;
    a1 = (d.bx + d.vx * (T)M - x1x) * ixd;
    const T axmin = dmin(a0, a1), axmax = dmax(a0, a1);
    a0 = (d.by - x1y) * iyd;
    a1 = (d.by + d.vy * (T)N - x1y) * iyd;
    const T aymin = dmin(a0, a1), aymax = dmax(a0, a1);
    a0 = (d.bz - x1z) * izd;
    a1 = (d.bz + d.vz * (T)Z - x1z) * izd;
    const T azmin = dmin(a0, a1), azmax = dmax(a0, a1);
    const T amin = dmax(dmax(axmin, aymin), dmax(aymin, azmin));
    const T amax = dmin(dmin(axmax, aymax), dmin(aymax, azmax));

    T len = 0;
    if (amax <= amin) return len;

    int imin, imax, jmin, jmax, kmin, kmax;
    const T ex = x2x - x1x, ey = x2y - x1y, ez = x2z - x1z;
    if (x1x < x2x) {
        imin = (amin == axmin) ? 1 : (int)dfloor((amin * ex + x1x - d.bx) * d.ivx) + 1;
        imax = (amax == axmax) ? M : (int)dfloor((amax * ex + x1x - d.bx) * d.ivx);
    } else {
        imax = (amin == axmin) ? M - 1 : (int)dfloor((amin * ex + x1x - d.bx) * d.ivx);
        imin = (amax == axmax) ? 0 : (int)dfloor((amax * ex + x1x - d.bx) * d.ivx) + 1;
    }
    if (x1y < x2y) {
        jmin = (amin == aymin) ? 1 : (int)dfloor((amin * ey + x1y - d.by) * d.ivy) + 1;
        jmax = (amax == aymax) ? N : (int)dfloor((amax * ey + x1y - d.by) * d.ivy);
    } else {
        jmax = (amin == aymin) ? N - 1 : (int)dfloor((amin * ey + x1y - d.by) * d.ivy);
        jmin = (amax == aymax) ? 0 : (int)dfloor((amax * ey + x1y - d.by) * d.ivy) + 1;
    }
    const bool zpar = dabs(x1z - x2z) < d.vz * (T)1e-6;
    if (zpar) {
        kmin = (int)dfloor((x1z - d.bz) * d.ivz) + 1;
        kmax = (int)dfloor((x1z - d.bz) * d.ivz);
    } else if (x1z < x2z) {
        kmin = (amin == azmin) ? 1 : (int)dfloor((amin * ez + x1z - d.bz) * d.ivz) + 1;
        kmax = (amax == azmax) ? Z : (int)dfloor((amax * ez + x1z - d.bz) * d.ivz);
    } else {
        kmax = (amin == azmin) ? Z - 1 : (int)dfloor((amin * ez + x1z - d.bz) * d.ivz);
        kmin = (amax == azmax) ? 0 : (int)dfloor((amax * ez + x1z - d.bz) * d.ivz) + 1;
    }

    // next-plane index n* and the crossing a* of that plane (:218-266)
    const int sgx = (x1x < x2x) ? 1 : ((x1x > x2x) ? -1 : 0);
    const int sgy = (x1y < x2y) ? 1 : ((x1y > x2y) ? -1 : 0);
    const int sgz = (x1z < x2z) ? 1 : ((x1z > x2z) ? -1 : 0);
    int nx, ny, nz;
    T ax, ay, az;
    if (dabs(x1x - x2x) < d.vx * (T)1e-6) { ax = dinf<T>(); nx = imin; }
    else { nx = (sgx > 0) ? imin : imax; ax = (d.vx * (T)nx + d.bx - x1x) * ixd; }
    if (dabs(x1y - x2y) < d.vy * (T)1e-6) { ay = dinf<T>(); ny = jmin; }
    else { ny = (sgy > 0) ? jmin : jmax; ay = (d.vy * (T)ny + d.by - x1y) * iyd; }
    if (zpar) { az = dinf<T>(); nz = kmin; }
    else { nz = (sgz > 0) ? kmin : kmax; az = (d.vz * (T)nz + d.bz - x1z) * izd; }
    int vi = (x1x < x2x) ? imin - 1 : imax;   // (:271-284)
    int vj = (x1y < x2y) ? jmin - 1 : jmax;
    int vk = (x1z < x2z) ? kmin - 1 : kmax;

    const T dist = dsqrt(ex * ex + ey * ey + ez * ez);
    T ac = amin;
    // the traversal visits at most M+N+Z+1 voxels; the cap only guarantees
    // termination for non-finite inputs
    int guard = M + N + Z + 4;
    while (amax - ac > loop_eps<T>() && guard-- > 0) {
        if ((unsigned)vi >= (unsigned)M || (unsigned)vj >= (unsigned)N || (unsigned)vk >= (unsigned)Z) break;
        const T m = dmin(dmin(ax, ay), az);
        const T seg = dist * (m - ac);
        len += seg;
        visit(vk * (M * N) + vj * M + vi, seg);
        ac = m;
        if (ax == m) { vi += sgx; nx += sgx; ax = (d.vx * (T)nx + d.bx - x1x) * ixd; }
        if (ay == m) { vj += sgy; ny += sgy; ay = (d.vy * (T)ny + d.by - x1y) * iyd; }
        if (az == m) { vk += sgz; nz += sgz; az = (d.vz * (T)nz + d.bz - x1z) * izd; }
    }
    return len;
}

// Ray setup shared by the batched forward sum: the reference's entry point,
// plane indices and first crossings (:20-292), kept operation for operation.
template <typename T> struct RayState {
    T amax, ac, ax, ay, az, dist, x1x, x1y, x1z, x2x, x2y, x2z, ixd, iyd, izd;
    int nx, ny, nz, vi, vj, vk, sgx, sgy, sgz;
    bool hit;
};

template <typename T>
__device__ __forceinline__ RayState<T> ray_setup(const DGeo<T> &d, T s, T c, int col, int row, int src) {
    RayState<T> r;
    const int M = d.M, N = d.N, Z = d.Z;
    const T u = d.ymin + (T)col * d.du;
    const T x1x = d.dod * c - u * s;
    const T x1y = d.dod * s + u * c;
    const T x1z = d.zmin + (T)row * d.dv;
    T x2x, x2y, x2z;
    ray_source(d, s, c, u, x1z, src, x2x, x2y, x2z);
    r.x2x = x2x; r.x2y = x2y; r.x2z = x2z;
    const T ixd = (T)1 / (x2x - x1x);
    const T iyd = (T)1 / (x2y - x1y);
    const T izd = (T)1 / (x2z - x1z);
    r.x1x = x1x; r.x1y = x1y; r.x1z = x1z; r.ixd = ixd; r.iyd = iyd; r.izd = izd;
    T a0, a1;
    a0 = (d.bx - x1x) * ixd;
    a1 = (d.bx + d.vx * (T)M - x1x) * ixd;
    const T axmin = dmin(a0, a1), axmax = dmax(a0, a1);
    a0 = (d.by - x1y) * iyd;
    a1 = (d.by + d.vy * (T)N - x1y) * iyd;
    const T aymin = dmin(a0, a1), aymax = dmax(a0, a1);
    a0 = (d.bz - x1z) * izd;
    a1 = (d.bz + d.vz * (T)Z - x1z) * izd;
    const T azmin = dmin(a0, a1), azmax = dmax(a0, a1);
    const T amin = dmax(dmax(axmin, aymin), dmax(aymin, azmin));
    const T amax = dmin(dmin(axmax, aymax), dmin(aymax, azmax));
    r.amax = amax; r.ac = amin;
    r.hit = !(amax <= amin);
    if (!r.hit) return r;
    int imin, imax, jmin, jmax, kmin, kmax;
    const T ex = x2x - x1x, ey = x2y - x1y, ez = x2z - x1z;
    if (x1x < x2x) {
        imin = (amin == axmin) ? 1 : (int)dfloor((amin * ex + x1x - d.bx) * d.ivx) + 1;
        imax = (amax == axmax) ? M : (int)dfloor((amax * ex + x1x - d.bx) * d.ivx);
    } else {
        imax = (amin == axmin) ? M - 1 : (int)dfloor((amin * ex + x1x - d.bx) * d.ivx);
        imin = (amax == axmax) ? 0 : (int)dfloor((amax * ex + x1x - d.bx) * d.ivx) + 1;
    }
    if (x1y < x2y) {
        jmin = (amin == aymin) ? 1 : (int)dfloor((amin * ey + x1y - d.by) * d.ivy) + 1;
        jmax = (amax == aymax) ? N : (int)dfloor((amax * ey + x1y - d.by) * d.ivy);
    } else {
        jmax = (amin == aymin) ? N - 1 : (int)dfloor((amin * ey + x1y - d.by) * d.ivy);
        jmin = (amax == aymax) ? 0 : (int)dfloor((amax * ey + x1y - d.by) * d.ivy) + 1;
    }
    const bool zpar = dabs(x1z - x2z) < d.vz * (T)1e-6;
    if (zpar) {
        kmin = (int)dfloor((x1z - d.bz) * d.ivz) + 1;
        kmax = (int)dfloor((x1z - d.bz) * d.ivz);
    } else if (x1z < x2z) {
        kmin = (amin == azmin) ? 1 : (int)dfloor((amin * ez + x1z - d.bz) * d.ivz) + 1;
        kmax = (amax == azmax) ? Z : (int)dfloor((amax * ez + x1z - d.bz) * d.ivz);
    } else {
        kmax = (amin == azmin) ? Z - 1 : (int)dfloor((amin * ez + x1z - d.bz) * d.ivz);
        kmin = (amax == azmax) ? 0 : (int)dfloor((amax * ez + x1z - d.bz) * d.ivz) + 1;
    }
    r.sgx = (x1x < x2x) ? 1 : ((x1x > x2x) ? -1 : 0);
    r.sgy = (x1y < x2y) ? 1 : ((x1y > x2y) ? -1 : 0);
    r.sgz = (x1z < x2z) ? 1 : ((x1z > x2z) ? -1 : 0);
    if (dabs(x1x - x2x) < d.vx * (T)1e-6) { r.ax = dinf<T>(); r.nx = imin; }
    else { r.nx = (r.sgx > 0) ? imin : imax; r.ax = (d.vx * (T)r.nx + d.bx - x1x) * ixd; }
    if (dabs(x1y - x2y) < d.vy * (T)1e-6) { r.ay = dinf<T>(); r.ny = jmin; }
    else { r.ny = (r.sgy > 0) ? jmin : jmax; r.ay = (d.vy * (T)r.ny + d.by - x1y) * iyd; }
    if (zpar) { r.az = dinf<T>(); r.nz = kmin; }
    else { r.nz = (r.sgz > 0) ? kmin : kmax; r.az = (d.vz * (T)r.nz + d.bz - x1z) * izd; }
    r.vi = (x1x < x2x) ? imin - 1 : imax;
    r.vj = (x1y < x2y) ? jmin - 1 : jmax;
    r.vk = (x1z < x2z) ? kmin - 1 : kmax;
    r.dist = dsqrt(ex * ex + ey * ey + ez * ez);
    return r;
}

// Ray sum with B steps generated per batch and their B gathers issued
// together: the steps, segment lengths and the order of the two sums are
// those of siddon_traverse, so with COMP = false the result is identical; only
// the loads are in flight together instead of one at a time.  COMP = true
// (fast mode) adds Kahan compensation to the ray sum and length, which keeps
// long FP32 rays at FP64-like accuracy.
template <typename T, typename SV, int B, bool COMP>
__device__ __forceinline__ T siddon_sum(const DGeo<T> &d, T s, T c, int col, int row, int src,
                                        const SV *__restrict__ f, T &len_out) {
    RayState<T> r = ray_setup(d, s, c, col, row, src);
    T sum = 0, len = 0, csum = 0, clen = 0;
    if (r.hit) {
        const unsigned M = d.M, N = d.N, Z = d.Z, MN = M * N;
        int guard = d.M + d.N + d.Z + 4;
        bool alive = true;
        while (alive) {
            unsigned idx[B];
            T seg[B];
            bool act[B];
            // step generation, branch-free: every state update is a select
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const bool ok = alive && (r.amax - r.ac > loop_eps<T>()) && (guard > 0) &&
                                (unsigned)r.vi < M && (unsigned)r.vj < N && (unsigned)r.vk < Z;
                const T m = dmin(dmin(r.ax, r.ay), r.az);
                act[u] = ok;
                seg[u] = r.dist * (m - r.ac);
                idx[u] = ok ? (unsigned)r.vk * MN + (unsigned)r.vj * M + (unsigned)r.vi : 0u;
                const bool sx = ok && (r.ax == m), sy = ok && (r.ay == m), sz = ok && (r.az == m);
                const int nx1 = r.nx + r.sgx, ny1 = r.ny + r.sgy, nz1 = r.nz + r.sgz;
                const T ax1 = (d.vx * (T)nx1 + d.bx - r.x1x) * r.ixd;
                const T ay1 = (d.vy * (T)ny1 + d.by - r.x1y) * r.iyd;
                const T az1 = (d.vz * (T)nz1 + d.bz - r.x1z) * r.izd;
                r.vi = sx ? r.vi + r.sgx : r.vi;
                r.nx = sx ? nx1 : r.nx;
                r.ax = sx ? ax1 : r.ax;
                r.vj = sy ? r.vj + r.sgy : r.vj;
                r.ny = sy ? ny1 : r.ny;
                r.ay = sy ? ay1 : r.ay;
                r.vk = sz ? r.vk + r.sgz : r.vk;
                r.nz = sz ? nz1 : r.nz;
                r.az = sz ? az1 : r.az;
                r.ac = ok ? m : r.ac;
                guard -= ok ? 1 : 0;
                alive = ok;
            }
            T fv[B];
#pragma unroll
            for (int u = 0; u < B; ++u) fv[u] = (T)ldf(f, idx[u]);
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if constexpr (COMP) {
                    const T yl = seg[u] - clen;
                    const T tl = len + yl;
                    const T cl = (tl - len) - yl;
                    const T ys = seg[u] * fv[u] - csum;
                    const T ts = sum + ys;
                    const T cs = (ts - sum) - ys;
                    len = act[u] ? tl : len;
                    clen = act[u] ? cl : clen;
                    sum = act[u] ? ts : sum;
                    csum = act[u] ? cs : csum;
                } else {
                    len = act[u] ? len + seg[u] : len;
                    sum = act[u] ? sum + seg[u] * fv[u] : sum;
                }
            }
        }
    }
    len_out = len;
    return sum;
}

// Fast-mode FP32 traversal (CT_MATH_FAST).  Same walk as siddon_traverse
// with the instruction count of one step cut from ~59 to ~30 VALU:
//  * the crossing of plane n is fma(n, vx*ixd, (bx - x1x)*ixd) (one rounding
//    per term instead of four), with n kept as a float counter;
//  * one linear voxel offset (in units of ES bytes) with per-axis strides
//    replaces the three voxel coordinates; the first voxel is bounds-checked
//    once (a ray entering outside the grid is empty, as in the reference),
//    and the walk ends at alpha_max, clipped to the grid's exit planes as the
//    walk itself computes them, instead of bounds-checking every step (steps
//    past the end have length 0; the forward still reads them in bounds or
//    gets 0 from the range-checked load, the adjoint skips them);
//  * min/min3 are issued directly (no per-use NaN canonicalisation);
//  * steps carry alpha lengths; the forward multiplies its sum by dist once;
//  * the ray length is the closed form dist*(alpha_max - alpha_min), the
//    telescoped sum of the segments without their rounding.
// The forward (siddon_walk_fast) and the matched adjoint (k_adjoint) both
// step through this walker, so their segments are the same numbers.
//
// ZQ: the volume is in the z-quad layout of the SART sweep,
// [z/4][y][x][z%4] (four z-neighbours share 16 bytes, so the 64 rays of a
// wave - a few voxels apart in the lateral and z directions - hit a few cache
// lines per gather instead of one each).  An x or y step moves the offset by
// a constant; a z step moves it by +-1 inside a quad and by +-(4MN - 3)
// across a quad boundary, i.e. when the plane crossed has an index that is a
// multiple of 4.
// One axis of the fast walk's plane model: plane n is crossed at
// alpha = fma(n, k, b0) with k = v/(x2 - x1) and b0 = (b - x1)/(x2 - x1).  An
// axis whose ray component is below 1e-6 of a voxel (the reference's parallel
// test) never steps; the ray then stays in slab i0 = floor((x1 - b)/v).
// The matched gather adjoint evaluates the same planes per detector column
// and row, so every segment is the same number in both.
struct PlaneAxis {
    float k, b0;
    int sg, i0;
    bool par;
    // clip [lo, hi] to the grid's planes 0 and n
    __device__ __forceinline__ void clip(float &lo, float &hi, int n) const {
        if (par) return;
        const float g0 = b0, gn = fmaf((float)n, k, b0);
        lo = hmax(lo, hmin(g0, gn));
        hi = hmin(hi, hmax(g0, gn));
    }
    // the slab holding alpha lo, starting from the reference setup's index
    __device__ __forceinline__ bool start(int v0, float lo, int n, int &v) const {
        if (par) { v = i0; return (unsigned)v < (unsigned)n; }
        v = v0;
        if (fmaf((float)(v + (sg < 0)), k, b0) > lo) v -= sg;        // lo lies before the entry plane
        else if (fmaf((float)(v + (sg > 0)), k, b0) < lo) v += sg;   // lo lies past the exit plane
        return (unsigned)v < (unsigned)n;
    }
};
__device__ __forceinline__ PlaneAxis plane_axis(float v, float iv, float b, float x1, float id, int sg, bool par) {
    PlaneAxis a;
    a.k = v * id; a.b0 = (b - x1) * id; a.sg = sg; a.par = par;
    a.i0 = (int)floorf((x1 - b) * iv);
    return a;
}

template <int ES, bool ZQ = false> struct FastWalk {
    float kx, ky, kz, bx0, by0, bz0, sgxf, sgyf, sgzf, nfx, nfy, nfz, ax, ay, az, ac, amax, dist, len;
    int dix, diy, diz, dizb;
    unsigned idx;
    // returns false for an empty ray (the forward yields 0 for it)
    __device__ __forceinline__ bool init(const DGeo<float> &d, float s, float c, int col, int row, int src) {
        RayState<float> r = ray_setup(d, s, c, col, row, src);
        if (!r.hit) return false;
        const unsigned M = d.M, N = d.N, Z = d.Z, MN = M * N;
        // The reference's walk begins in the voxel its FP32 setup names and
        // stops before the first segment when that voxel lies outside the
        // grid, so the ray comes out as 0 (V63/kernel_IterativeRecon_universal.cu
        // :271-284, :297-303, :554-563).  This happens at exact ties, where
        // the entry point rounds onto the outer side of an edge plane; such
        // rays are empty here too, in the forward and the matched adjoint.
        if ((unsigned)r.vi >= M || (unsigned)r.vj >= N || (unsigned)r.vk >= Z) return false;
        const PlaneAxis X = plane_axis(d.vx, d.ivx, d.bx, r.x1x, r.ixd, r.sgx, d.vx * 1e-6f > fabsf(r.x1x - r.x2x));
        const PlaneAxis Y = plane_axis(d.vy, d.ivy, d.by, r.x1y, r.iyd, r.sgy, d.vy * 1e-6f > fabsf(r.x1y - r.x2y));
        const PlaneAxis Zx = plane_axis(d.vz, d.ivz, d.bz, r.x1z, r.izd, r.sgz, d.vz * 1e-6f > fabsf(r.x1z - r.x2z));
        // the walk runs over [alpha_min, alpha_max] of the reference setup,
        // clipped to the grid's entry and exit planes as this walk computes
        // them (so no step past the grid carries a nonzero length)
        float lo = r.ac, hi = r.amax;
        X.clip(lo, hi, (int)M); Y.clip(lo, hi, (int)N); Zx.clip(lo, hi, (int)Z);
        if (!(hi > lo)) return false;
        // start voxel: the slab that holds alpha_min under these planes
        int vi, vj, vk;
        if (!X.start(r.vi, lo, (int)M, vi) || !Y.start(r.vj, lo, (int)N, vj) || !Zx.start(r.vk, lo, (int)Z, vk))
            return false;
        // a parallel axis gets k = 0, b0 = +inf: its pending crossing is +inf
        kx = X.par ? 0.0f : X.k; bx0 = X.par ? __builtin_inff() : X.b0;
        ky = Y.par ? 0.0f : Y.k; by0 = Y.par ? __builtin_inff() : Y.b0;
        kz = Zx.par ? 0.0f : Zx.k; bz0 = Zx.par ? __builtin_inff() : Zx.b0;
        sgxf = (float)r.sgx; sgyf = (float)r.sgy; sgzf = (float)r.sgz;
        nfx = (float)(vi + (r.sgx > 0)); nfy = (float)(vj + (r.sgy > 0)); nfz = (float)(vk + (r.sgz > 0));
        ax = fmaf(nfx, kx, bx0); ay = fmaf(nfy, ky, by0); az = fmaf(nfz, kz, bz0);
        if constexpr (ZQ) {
            dix = r.sgx * 4 * ES; diy = r.sgy * (int)M * 4 * ES;
            diz = r.sgz * ES; dizb = r.sgz * (4 * (int)MN - 3) * ES;
            idx = (((unsigned)(vk >> 2) * MN + (unsigned)vj * M + (unsigned)vi) * 4u + ((unsigned)vk & 3u)) * (unsigned)ES;
        } else {
            dix = r.sgx * ES; diy = r.sgy * (int)M * ES; diz = r.sgz * (int)MN * ES; dizb = diz;
            idx = ((unsigned)vk * MN + (unsigned)vj * M + (unsigned)vi) * (unsigned)ES;
        }
        ac = lo; amax = hi; dist = r.dist;
        len = dist * (hi - lo);
        return true;
    }
    // one step: the segment's alpha length (times dist = its length in mm)
    // and the offset of the voxel it lies in.  alpha_min <= every pending
    // crossing, so once ac reaches alpha_max every later step has length 0;
    // the caller tests for the end of the ray once per batch (ended()).
    __device__ __forceinline__ float step(unsigned &id) {
        // the crossings are fma results (canonical), so the compiler's
        // minimum is the bare v_min3/v_min pair with no hazard padding
        const float m = __builtin_fminf(__builtin_fminf(__builtin_fminf(ax, ay), az), amax);
        const float dl = m - ac;
        id = idx;
        const bool sx = ax == m, sy = ay == m, sz = az == m;
        // ZQ: the z plane about to be crossed bounds a quad
        const bool qb = ZQ && __builtin_amdgcn_fractf(nfz * 0.25f) == 0.0f;
        // the stepped axes move to their next plane; every pending crossing
        // is re-evaluated from its plane index (the same value when unmoved)
        nfx += sx ? sgxf : 0.0f; nfy += sy ? sgyf : 0.0f; nfz += sz ? sgzf : 0.0f;
        ax = fmaf(nfx, kx, bx0); ay = fmaf(nfy, ky, by0); az = fmaf(nfz, kz, bz0);
        idx += (unsigned)((sx ? dix : 0) + (sy ? diy : 0) + (sz ? (qb ? dizb : diz) : 0));
        ac = m;
        return dl;
    }
    // z planes counted from the multiple of four next to the first crossing,
    // whose alpha has no cancellation left: on nearly level rays, where a plane
    // spans much alpha, the rounding of plane 0's would move every crossing.
    // Returns that plane (restart takes it).
    __device__ __forceinline__ int rebase_z(const DGeo<float> &d, int row) {
        if (kz == 0.0f) return 0;
        const float n0 = 4.0f * floorf(nfz * 0.25f);
        bz0 = (fmaf(n0, d.vz, d.bz) - (d.zmin + (float)row * d.dv)) * d.ivz * kz;
        nfz -= n0;
        az = fmaf(nfz, kz, bz0);
        return (int)n0;
    }
    __device__ __forceinline__ bool ended() const { return !(amax - ac > loop_eps<float>()); }
    // continue the walk from alpha a in [ac, amax]: the slab of each
    // stepping axis that holds a (as start() finds it), its pending crossing
    // and the voxel offset
    // (zq: the plane index that nfz and bz0 count from, see rebase_z)
    __device__ __forceinline__ void restart(const DGeo<float> &d, float a, int zq = 0) {
        const int vi = restart_axis(kx, bx0, sgxf, nfx, a, d.M);
        const int vj = restart_axis(ky, by0, sgyf, nfy, a, d.N);
        const int vk = restart_axis(kz, bz0, sgzf, nfz, a, d.Z - zq, -zq) + zq;
        ax = fmaf(nfx, kx, bx0); ay = fmaf(nfy, ky, by0); az = fmaf(nfz, kz, bz0);
        const unsigned M = d.M, MN = (unsigned)d.M * (unsigned)d.N;
        if constexpr (ZQ)
            idx = (((unsigned)(vk >> 2) * MN + (unsigned)vj * M + (unsigned)vi) * 4u + ((unsigned)vk & 3u)) * (unsigned)ES;
        else
            idx = ((unsigned)vk * MN + (unsigned)vj * M + (unsigned)vi) * (unsigned)ES;
        ac = a;
    }
    __device__ __forceinline__ static int restart_axis(float k, float b0, float sg, float &nf, float a, int n, int first = 0) {
        const int up = sg > 0.0f;
        if (k == 0.0f) return (int)nf - up;   // parallel axis: its slab never changes
        const int sgi = up ? 1 : -1;
        int v = min(max((int)floorf((a - b0) / k), first), n - 1);
        if (fmaf((float)(v + 1 - up), k, b0) > a) v -= sgi;     // a lies before the entry plane
        else if (fmaf((float)(v + up), k, b0) < a) v += sgi;    // a lies past the exit plane
        v = min(max(v, first), n - 1);
        nf = (float)(v + up);
        return v;
    }
};

constexpr int FAST_B = 16;  // steps per batch: their gathers are in flight together

// Fast-mode ray sum: batches of FAST_B steps whose loads are issued together;
// each batch is summed in FP32 and the batch sums accumulate in FP32 with
// Kahan compensation.
// Volumes under 4 GiB are read with range-checked buffer loads on 32-bit
// byte offsets; larger ones use 64-bit addresses with an explicit range test.
// The batch loop of the fast ray sum over an initialised walker: batches of
// FAST_B steps whose loads are issued together, each batch summed in FP32 and
// the batch sums accumulated Kahan-compensated in FP32.  Returns the sum of
// alpha-length x value
// (times dist = the ray sum).  Volumes under 4 GiB are read with
// range-checked buffer loads on 32-bit byte offsets; larger ones use 64-bit
// addresses with an explicit range test.
template <typename SV, bool BUF, bool ZQ>
__device__ __forceinline__ float walk_sum(FastWalk<BUF ? (int)sizeof(SV) : 1, ZQ> &w, const DGeo<float> &d,
                                          const SV *__restrict__ f) {
    // elements of the array (the z-quad layout pads z to a multiple of 4)
    const unsigned nvox = (unsigned)d.M * (unsigned)d.N * (ZQ ? (unsigned)((d.Z + 3) & ~3) : (unsigned)d.Z);
    // (for the 64-bit path the resource is built but never used)
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(f, BUF ? nvox * (unsigned)sizeof(SV) : 0u);
    float sum = 0.0f, comp = 0.0f;   // Kahan-compensated total of the batch sums
    int guard = d.M + d.N + d.Z + 4;
    do {
        unsigned ids[FAST_B];
        float dl[FAST_B];
#pragma unroll
        for (int u = 0; u < FAST_B; ++u) dl[u] = w.step(ids[u]);
        guard -= FAST_B;
        float fv[FAST_B];
#pragma unroll
        for (int u = 0; u < FAST_B; ++u) {
            if constexpr (BUF) fv[u] = bload<SV>(rs, ids[u]);
            else fv[u] = ids[u] < nvox ? (float)ldf(f, (int64_t)ids[u]) : 0.0f;
        }
        float ps = dl[0] * fv[0];
#pragma unroll
        for (int u = 1; u < FAST_B; ++u) ps = fmaf(dl[u], fv[u], ps);
        const float y = ps - comp, t = sum + y;
        comp = (t - sum) - y;
        sum = t;
    } while (!w.ended() && guard > 0);
    return sum - comp;
}

template <typename SV, bool BUF, bool ZQ = false>
__device__ __forceinline__ float siddon_walk_fast(const DGeo<float> &d, float s, float c, int col, int row, int src,
                                                  const SV *__restrict__ f, float &len_out) {
    FastWalk<BUF ? (int)sizeof(SV) : 1, ZQ> w;
    len_out = 0.0f;
    if (!w.init(d, s, c, col, row, src)) return 0.0f;
    len_out = w.len;
    return walk_sum<SV, BUF, ZQ>(w, d, f) * w.dist;
}

template <typename SV>
__device__ __forceinline__ float siddon_sum_fast(const DGeo<float> &d, float s, float c, int col, int row, int src,
                                                 const SV *__restrict__ f, float &len_out) {
    if ((uint64_t)d.M * d.N * d.Z * sizeof(SV) < (1ull << 32))
        return siddon_walk_fast<SV, true>(d, s, c, col, row, src, f, len_out);
    return siddon_walk_fast<SV, false>(d, s, c, col, row, src, f, len_out);
}

// 16x16-pixel tile per workgroup (XCD-aware tile order), 8x8 per wave;
// returns the tile's image slot
__device__ __forceinline__ int tile_coords(int &col, int &row) {
    const int tid = threadIdx.x;
    const int w = tid >> 6, l = tid & 63;
    const int3 t = xcd_tile();
    col = t.x * 16 + (w & 1) * 8 + (l & 7);
    row = t.y * 16 + (w >> 1) * 8 + (l >> 3);
    return t.z;
}

// CMD 0: ray sum; CMD 1: SART correction (b - sum)/len
// (V63/kernel_IterativeRecon_universal.cu:554-563).  image slot = q*NS + src
// for batch slot q; view = first + q*stride; meas is indexed by view - mv0.
template <typename T, typename SV, typename SO, typename SM, int CMD, bool COMP>
__global__ __launch_bounds__(256) void k_forward(DGeo<T> d, const T *__restrict__ ang,
                                                 const SV *__restrict__ f, SO *__restrict__ out,
                                                 const SM *__restrict__ meas, int first, int stride,
                                                 int mv0, int z0) {
    int col, row;
    const int slot = tile_coords(col, row);
    if (col >= d.R || row >= d.ZP) return;
    const int img = slot + z0;
    const int q = img / d.NS, src = img - q * d.NS;
    const int v = first + q * stride;
    const T s = ang[2 * v], c = ang[2 * v + 1];
    T len;
    T sum;
    if constexpr (COMP && std::is_same<T, float>::value) sum = siddon_sum_fast<SV>(d, s, c, col, row, src, f, len);
    else sum = siddon_sum<T, SV, 4, false>(d, s, c, col, row, src, f, len);
    const int64_t P = (int64_t)d.R * d.ZP;
    const int64_t pix = (int64_t)row * d.R + col;
    T r;
    if (len < d.vz * (T)1e-6) r = 0;
    else if (CMD == 0) r = sum;
    else {
        const T b = (T)ldf(meas, ((int64_t)(v - mv0) * d.NS + src) * P + pix);
        r = (b - sum) / len;
    }
    St<SO>::st(out, (int64_t)img * P + pix, r);
}

// SART correction (CMD 1) of the sweep on a z-quad-layout volume (fast
// mode, FP32 arithmetic, volume under 4 GiB): the same rays, segments and
// output as k_forward<float, SV, float, SM, 1, true>.
// Projection on a z-quad-layout volume (fast mode, FP32 arithmetic, volume
// under 4 GiB): CMD 0 ray sums, CMD 1 SART corrections (b - sum)/len, the same
// rays and segments as k_forward.  S parts per ray: a workgroup holds 256 / S
// rays (16x16 pixels for S = 1, 16x8 for 2, 8x8 for 4); part p walks alpha in
// [lo + (hi - lo) p / S, lo + (hi - lo) (p + 1) / S] and the partial sums meet
// in LDS, added in part order.  Splitting gives more waves per view and parts
// of equal length, so more gathers are in flight; it also splits the segment
// that holds each cut point, so the SART correction uses it (S = 2) and the ray
// sums of the autograd pair do not (their segments stay those of the matched
// adjoint).
constexpr int CORR_SPLIT = 2;

template <typename SV, typename SO, typename SM, int CMD, int S>
__global__ __launch_bounds__(256) void k_project_zq(DGeo<float> d, const float *__restrict__ ang,
                                                    const SV *__restrict__ fq, SO *__restrict__ out,
                                                    const SM *__restrict__ meas, int first, int stride, int mv0,
                                                    int z0) {
    constexpr int NR = 256 / S, WPP = 4 / S;   // rays and waves per part
    constexpr int TW = WPP >= 2 ? 16 : 8, TH = WPP == 4 ? 16 : 8;
    __shared__ float part[S > 1 ? 256 : 1];
    const int tid = threadIdx.x, p = tid / NR, rr = tid % NR;
    const int w = rr >> 6, l = rr & 63;
    const int3 t = xcd_tile();
    const int col = t.x * TW + (w & 1) * 8 + (l & 7), row = t.y * TH + (w >> 1) * 8 + (l >> 3);
    const int img = t.z + z0;
    const bool inb = col < d.R && row < d.ZP;
    const int q = img / d.NS, src = img - q * d.NS;
    const int v = first + q * stride;
    float sum = 0.0f;
    float len = 0.0f, dist = 0.0f;
    if (inb) {
        const float s = ang[2 * v], c = ang[2 * v + 1];
        FastWalk<(int)sizeof(SV), true> fw;
        if (fw.init(d, s, c, col, row, src)) {
            len = fw.len;
            dist = fw.dist;
            if constexpr (S > 1) {
                // (16-bit volumes, whose storage rounding hides it and whose
                // stored updates are dithered from the sums' low bits, do without)
                int zq = 0;
                if constexpr (std::is_same<SV, float>::value) zq = fw.rebase_z(d, row);
                const float lo = fw.ac, span = fw.amax - fw.ac;
                if (p + 1 < S) fw.amax = fmaf(span, (float)(p + 1) / (float)S, lo);
                if (p > 0) fw.restart(d, fmaf(span, (float)p / (float)S, lo), zq);
            }
            sum = walk_sum<SV, true, true>(fw, d, fq);
        }
    }
    if constexpr (S > 1) {
        part[tid] = sum;
        __syncthreads();
        if (p != 0) return;
#pragma unroll
        for (int k = 1; k < S; ++k) sum += part[k * NR + rr];
    }
    if (!inb) return;
    const int64_t P = (int64_t)d.R * d.ZP;
    const int64_t pix = (int64_t)row * d.R + col;
    float r = 0.0f;
    if (!(len < d.vz * 1e-6f)) {
        const float ax = sum * dist;
        if constexpr (CMD == 0) r = ax;
        else r = ((float)ldf(meas, ((int64_t)(v - mv0) * d.NS + src) * P + pix) - ax) / len;
    }
    St<SO>::st(out, (int64_t)img * P + pix, r);
}

// Column walk (fast mode, z-quad volume).  Every ray of one detector column
// runs from a point of the column to the column's source point, and for all
// three beam styles those points share their x and y: the rays of a column
// lie in one vertical plane and cross the x and y planes at the same alpha
// (fma(n, k, b0) over the same k and b0, so the same FP32 numbers).  A
// workgroup takes 256 rows (or 128) of one column and merges the column's x and y
// crossings once into an LDS list; each list segment is one x/y voxel, and at
// a segment all 256 rays read that voxel column of z, within a window the
// list also records (the extreme rows at the segment's ends, one voxel of
// margin).  The workgroup stages those windows into LDS with coalesced
// 16-byte quad loads, double-buffered over batches of segments, and every
// lane walks the list in step with the others, clipped to its own
// [alpha_min, alpha_max], tracking only its own z slab and reading its voxels
// from the staged window.  A segment holds at most one z crossing when
// |dz|/vz < max(|dx|/vx, |dy|/vy) along every ray (the host checks a bound);
// the part after the crossing reads the next z voxel.  The segments are those
// of the per-ray walk (same alphas, same voxels; a tie there is one step, here
// a zero-length segment), and the sums keep its FP32 batches with a
// Kahan-compensated FP32 total.  Per segment ~14 VALU (staging included), one
// LDS pair read and no per-lane gather, against ~25 VALU and one scattered
// gather per step of the per-ray walk.  Views whose rays run along y walk a
// transposed copy of the volume (see col_walk_view).
// Whether the rays of a view at angle cosine c run along x rather than y (to
// within ~41 degrees of it).
__host__ __device__ __forceinline__ bool col_along_x(float c) { return fabsf(c) >= 0.75f; }

// RW, the rays per workgroup (rows of one column): 256, or 128 where that
// leaves fewer lanes without a row, or where 256 rows span too tall a window
// (col_plan).
constexpr int COL_B = 16;       // list padding: a multiple of every staged batch (col_batch)
template <int RW> constexpr int col_nq() { return RW == 256 ? 48 : 32; }   // largest staged window, in z-quads
// LDS elements per staged window: col_nq quads and one quad of padding, so
// that the windows of a batch's segments start on different banks (the
// staging writes of eight segments' same quad are then conflict-free)
template <int RW> constexpr int col_w() { return 4 * col_nq<RW>() + 4; }
// List segments per staged batch: 16 (one barrier per 16 segments, and a
// staging load's eight-lane groups cover 16 segments), or 8 for BF16
// volumes, whose FP32 windows at 16 would leave four workgroups per CU
// instead of six (correction per view at 512^3 / 1024^2: FP32 0.382 -> 0.342
// ms and FP16 0.286 -> 0.261 ms from 8 to 16; BF16 0.263 ms at either).
template <typename SV> constexpr int col_batch() { return std::is_same<SV, __hip_bfloat16>::value ? 8 : 16; }
// staged quads per thread and batch
template <typename SV, int RW> constexpr int col_sp() { return (col_batch<SV>() * col_nq<RW>() + RW - 1) / RW; }

// LDS: two staging buffers of col_batch windows in a static array (fixed
// address and stride, so every staged read has a constant offset; FP32
// elements, or the volume's own halves for FP16); the list in dynamic LDS as
// three arrays of at most M + N - 1 entries padded to a multiple of COL_B:
// alpha, the window's first quad times the staged bytes per quad (its byte
// offset in a staged row), and the x/y byte offset for the staging loads.
// (The entry count is a multiple of 4, so the alpha and window arrays stay
// 16-byte aligned for their vector reads; col_lds_bytes bounds the largest
// workgroup.)
static inline size_t col_list_entries(int M, int N) { return (size_t)((M + N + COL_B + 3) & ~3); }
static inline size_t col_dyn_bytes(int M, int N) { return 12 * col_list_entries(M, N); }
static inline size_t col_lds_bytes(int M, int N) {
    return sizeof(float) * 2 * COL_B * col_w<256>() + col_dyn_bytes(M, N);
}

// Element type of the staged windows: FP16 volumes stage their halves as
// loaded (the walk's FMAs take FP16 operands directly), the others FP32.
template <typename SV> struct StageOf { using type = float; };
template <> struct StageOf<__half> { using type = _Float16; };

// fq is the volume in the z-quad layout and ft in its lateral transpose
// [z/4][x][y][z%4], either of them null; a view reads the one along whose fast
// axis its rays run (col_walk_view: the staged quads of consecutive segments
// then share cache lines) if both are there, so one launch takes views of both
// directions.
template <typename SV, typename SO, typename SM, int CMD, int RW>
__global__ __launch_bounds__(RW) void k_project_col(DGeo<float> d, const float *__restrict__ ang,
                                                          const SV *__restrict__ fq, const SV *__restrict__ ft,
                                                          SO *__restrict__ out, const SM *__restrict__ meas, int first,
                                                          int stride, int mv0, int z0, int NQ) {
    using SE = typename StageOf<SV>::type;
    constexpr int SB = (int)sizeof(SE);                // staged bytes per voxel
    constexpr int QSH = SB == 4 ? 4 : 3;               // log2 of the staged bytes per quad
    constexpr int CB = col_batch<SV>(), SP = col_sp<SV, RW>(), CW = col_w<RW>();
    __shared__ __align__(16) SE stg[2 * CB * CW];
    extern __shared__ __align__(16) unsigned char col_smem[];
    const int LE = (d.M + d.N + COL_B + 3) & ~3;   // col_list_entries
    float *const la = reinterpret_cast<float *>(col_smem);             // alpha
    int *const lw = reinterpret_cast<int *>(col_smem + 4 * LE);          // first quad x 4 SB
    unsigned *const ls = reinterpret_cast<unsigned *>(col_smem + 8 * LE); // x/y byte offset
    constexpr int ES = (int)sizeof(SV);
    const int tid = (int)threadIdx.x;
    const int3 t = xcd_tile<true>();
    const int col = t.x, row0 = t.y * RW, row = row0 + tid;
    const int rowL = min(row0 + RW, d.ZP) - 1;
    const int img = t.z + z0;
    const int q = img / d.NS, src = img - q * d.NS;
    const int v = first + q * stride;
    const float s = ang[2 * v], c = ang[2 * v + 1];
    const bool tr = !fq || (ft && !col_along_x(c));
    const unsigned M = d.M, MN = (unsigned)d.M * (unsigned)d.N;
    const int ZQ4 = (d.Z + 3) >> 2;                        // quads per (x, y)
    const unsigned QS = MN * 4u * (unsigned)ES;            // bytes between z-quad planes

    // the column's x/y walk (the x and y terms of ray_setup and FastWalk::init)
    const float u = d.ymin + (float)col * d.du;
    const float x1x = d.dod * c - u * s, x1y = d.dod * s + u * c;
    float x2x, x2y, x2z0, x2zL;
    const float z1a = d.zmin + (float)row0 * d.dv, z1b = d.zmin + (float)rowL * d.dv;
    ray_source(d, s, c, u, z1a, src, x2x, x2y, x2z0);
    ray_source(d, s, c, u, z1b, src, x2x, x2y, x2zL);
    const float ixd = 1.0f / (x2x - x1x), iyd = 1.0f / (x2y - x1y);
    float a0 = (d.bx - x1x) * ixd, a1 = (d.bx + d.vx * (float)d.M - x1x) * ixd;
    const float axmin = fminf(a0, a1), axmax = fmaxf(a0, a1);
    a0 = (d.by - x1y) * iyd; a1 = (d.by + d.vy * (float)d.N - x1y) * iyd;
    const float aymin = fminf(a0, a1), aymax = fmaxf(a0, a1);
    const int sgx = (x1x < x2x) ? 1 : ((x1x > x2x) ? -1 : 0);
    const int sgy = (x1y < x2y) ? 1 : ((x1y > x2y) ? -1 : 0);
    const PlaneAxis X = plane_axis(d.vx, d.ivx, d.bx, x1x, ixd, sgx, d.vx * 1e-6f > fabsf(x1x - x2x));
    const PlaneAxis Y = plane_axis(d.vy, d.ivy, d.by, x1y, iyd, sgy, d.vy * 1e-6f > fabsf(x1y - x2y));
    float lxy = fmaxf(axmin, aymin), hxy = fminf(axmax, aymax);
    X.clip(lxy, hxy, d.M); Y.clip(lxy, hxy, d.N);
    int vi0 = X.i0, vj0 = Y.i0, NX = 0, NY = 0;
    bool cmiss = !(hxy > lxy);
    if (!cmiss) {
        float nf;
        if (!X.par) {
            vi0 = FastWalk<ES, true>::restart_axis(X.k, X.b0, (float)sgx, nf, lxy, d.M);
            NX = max((FastWalk<ES, true>::restart_axis(X.k, X.b0, (float)sgx, nf, hxy, d.M) - vi0) * sgx, 0);
        }
        if (!Y.par) {
            vj0 = FastWalk<ES, true>::restart_axis(Y.k, Y.b0, (float)sgy, nf, lxy, d.N);
            NY = max((FastWalk<ES, true>::restart_axis(Y.k, Y.b0, (float)sgy, nf, hxy, d.N) - vj0) * sgy, 0);
        }
        cmiss = (unsigned)vi0 >= M || (unsigned)vj0 >= (unsigned)d.N;
    }
    const int K = cmiss ? 0 : NX + NY;                       // crossings; entry K ends at hxy
    const int KP = cmiss ? 0 : (K + COL_B) / COL_B * COL_B;  // entries incl. padding
    if (!cmiss) {
        const float px0 = (float)(vi0 + (sgx > 0)), py0 = (float)(vj0 + (sgy > 0));
        const float fsx = (float)sgx, fsy = (float)sgy;
        auto XA = [&](int i) { return fmaf(fmaf((float)i, fsx, px0), X.k, X.b0); };
        auto YA = [&](int j) { return fmaf(fmaf((float)j, fsy, py0), Y.k, Y.b0); };
        const int ox = (tr ? d.N : 1) * 4 * ES, oy = (tr ? 1 : (int)M) * 4 * ES;
        const int ox1 = sgx * ox, oy1 = sgy * oy, o0 = vi0 * ox + vj0 * oy;
        auto OFF = [&](int i, int j) { return (unsigned)(o0 + i * ox1 + j * oy1); };
        // first staged quad of a segment [ap, a]: the z voxel range of the
        // workgroup's first and last rows at both ends, one voxel of margin
        auto QLO = [&](float ap, float a) {
            const float za = fminf(fmaf(ap, x2z0 - z1a, z1a), fmaf(a, x2z0 - z1a, z1a));
            const float zb = fminf(fmaf(ap, x2zL - z1b, z1b), fmaf(a, x2zL - z1b, z1b));
            const int vlo = (int)floorf((fminf(za, zb) - d.bz) * d.ivz) - 1;
            return vlo >> 2;   // floor division by 4 (arithmetic shift)
        };
        // merge path: thread t writes entries [t C, t C + C); ties take x first
        const int C = (KP + RW - 1) / RW;
        const int e0 = tid * C;
        if (e0 < KP) {
            const int ee = min(e0, K);
            int ilo = max(0, ee - NY), ihi = min(ee, NX);
            while (ilo < ihi) {
                const int mid = (ilo + ihi) >> 1;
                if (XA(mid) <= YA(ee - mid - 1)) ilo = mid + 1;
                else ihi = mid;
            }
            int i = ilo, j = ee - ilo;
            // alpha at which this thread's first segment starts
            float ap = lxy;
            if (ee > 0) ap = fmaxf(i > 0 ? XA(i - 1) : -__builtin_inff(), j > 0 ? YA(j - 1) : -__builtin_inff());
            if (e0 > K) ap = hxy;
            for (int e = e0; e < min(e0 + C, KP); ++e) {
                float a;
                const unsigned off = OFF(i, j);
                if (e >= K) a = hxy;
                else if (i < NX && (j >= NY || XA(i) <= YA(j))) { a = XA(i); ++i; }
                else { a = YA(j); ++j; }
                const int ql = QLO(ap, a);
                la[e] = a;
                lw[e] = ql * (1 << QSH);
                ls[e] = off;
                ap = a;
            }
        }
    }

    // this ray: its length as the per-ray walk forms it (0 for the rays the
    // reference leaves empty), and its height in voxel units along the
    // column's alpha, zeta(alpha) = (z1 + alpha (z2 - z1) - bz)/vz, as one FMA
    // zeta is kept relative to the slab kb the ray enters in, so that it
    // stays small and its rounding does not move the crossings of nearly
    // level rays; kbb = SB kb (bytes) re-bases the window offsets.
    FastWalk<ES, true> fw;
    float len = 0.0f, dist = 0.0f;
    float cz = 0.0f, z0c = 0.0f, icz = 0.0f;
    int kbb = 0;
    {
        const float z1 = d.zmin + (float)row * d.dv;
        float sx, sy, z2;
        ray_source(d, s, c, u, z1, src, sx, sy, z2);
        cz = (z2 - z1) * d.ivz;
        const float kb = floorf(fmaf(lxy, cz, (z1 - d.bz) * d.ivz));
        kbb = SB * (int)kb;
        z0c = fmaf(z1 - d.bz, d.ivz, -kb);
        // alpha per unit of zeta (0 for a level ray, which never changes slab)
        icz = fabsf(cz) > 1e-30f ? 1.0f / fabsf(cz) : 0.0f;
    }
    // CMD 0 and 2 (ray sums of the autograd pair, and the objective's residual
    // of the same sums): the per-ray walk's own segments, so that the matched adjoint stays its exact transpose.  The lane clips
    // the list to its [alpha_min, alpha_max] and tracks its next z-plane
    // crossing fma(nfz, kz, bz0); zrb is its slab relative to kb, times SB.
    float lo = 0.0f, hi = 0.0f, az = __builtin_inff(), nfz = 0.0f, kz = 0.0f, bz0 = __builtin_inff(), sgzf = 0.0f;
    int zrb = 0, dzb = 0;
    if (!cmiss && row < d.ZP && fw.init(d, s, c, col, row, src)) {
        len = fw.len; dist = fw.dist;
        if constexpr (CMD == 1) {
            // a level ray (kz = 0) keeps the slab the walk puts it in, which
            // the rounding of zeta would decide where it lies in a slice plane
            if (fw.kz == 0.0f) {
                cz = 0.0f; icz = 0.0f;
                z0c = fw.nfz - (fw.sgzf > 0.0f ? 1.0f : 0.0f) - (float)(kbb / SB) + 0.5f;
            }
        } else {
            lo = fw.ac; hi = fw.amax;
            az = fw.az; nfz = fw.nfz; kz = fw.kz; bz0 = fw.bz0; sgzf = fw.sgzf;
            zrb = ((int)nfz - (sgzf > 0.0f ? 1 : 0)) * SB - kbb;
            dzb = (int)sgzf * SB;
        }
    }
    const bool up = cz >= 0.0f;
    const unsigned nbytes = MN * (unsigned)ZQ4 * 4u * (unsigned)ES;
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(tr ? ft : fq, nbytes);
    // this thread's staged quads (the same in every batch): segment k of the
    // batch and quad qi of its window (sk = -1: none), and where they go
    const int nst = CB * NQ;   // quads staged per batch (at most SP * RW)
    // Segment-fastest: lanes 8q .. 8q + 7 load quad q of the batch's eight
    // segments.  Consecutive segments are mostly neighbours along the
    // layout's fast axis, whose quads share a 128-byte line, so a wave's load
    // touches ~8-16 lines instead of one per lane (the quads of one segment
    // lie a z-quad plane, M N quads, apart).
    int sk[SP], sq[SP], so[SP];
#pragma unroll
    for (int p = 0; p < SP; ++p) {
        const int sidx = tid + p * RW;
        sk[p] = sidx < nst ? sidx % CB : -1;
        sq[p] = sidx / CB;
        so[p] = (sidx % CB) * CW + 4 * sq[p];
    }
    // a quad outside the volume reads as zeros: its index is clamped to -1 or
    // ZQ4, whose offsets lie past the buffer's end (the volume is under 2 GiB)
    // Staged quads stay in registers as loaded (FP32 quads, or the 16-bit
    // volume's raw halves; BF16 is widened only at the LDS write), so no
    // instruction waits for them before the commit.
    using SR = typename std::conditional<ES == 2, uint2, float4>::type;
    SR sreg[SP];
    auto issue = [&](int b) {
#pragma unroll
        for (int p = 0; p < SP; ++p) {
            if (sk[p] >= 0) {
                const int e = b * CB + sk[p];
                const int qz = min(max((lw[e] >> QSH) + sq[p], -1), ZQ4);
                const uint32_t off = ls[e] + (unsigned)qz * QS;
                if constexpr (ES == 2) {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
                    sreg[p] = make_uint2(v[0], v[1]);
                } else {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
                    sreg[p] = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                                          __uint_as_float(v[3]));
                }
            }
        }
    };
    auto commit = [&](auto bufc) {
        constexpr int buf = decltype(bufc)::value;
#pragma unroll
        for (int p = 0; p < SP; ++p) {
            if (sk[p] < 0) continue;
            SE *const dst = stg + (buf * CB * CW + so[p]);
            if constexpr (std::is_same<SV, __hip_bfloat16>::value) {
                const uint2 r = sreg[p];
                *reinterpret_cast<float4 *>(dst) = make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u),
                                                               __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
            } else {
                *reinterpret_cast<SR *>(dst) = sreg[p];
            }
        }
    };
    __syncthreads();   // the list is complete
    const int nb = KP / CB;
    if (nb > 0) { issue(0); commit(std::integral_constant<int, 0>()); }
    // the lower element of a segment's slab pair lies at most 4 NQ - 2 into
    // its window (one voxel of margin each way by construction; clamped)
    const unsigned wmax2 = (unsigned)((4 * NQ - 2) * SB);
    // Kahan-compensated FP32 total of the batches' FP32 sums
    float sum = 0.0f, comp = 0.0f;
    float as = lxy, zs = fmaf(lxy, cz, z0c);
    // CMD 1 (SART corrections): a segment [as, ae] of the column's list lies
    // in one x/y voxel; this ray
    // enters it in slab k = floor(zeta(as)) and, as |dzeta| < 1 per segment
    // (col_plan), crosses at most one z plane in it.  The crossing part,
    // in zeta units clamp(zeta(ae) - (k + 1), 0, 1) for a rising ray or
    // clamp(k - zeta(ae), 0, 1) for a falling one, times alpha per unit of
    // zeta, belongs to the next slab and the rest of the segment to slab k;
    // both slabs are one LDS pair read.  Parts below or above the volume read
    // the window's zeros, so no per-ray clipping is needed: the sum is the
    // per-ray walk's to rounding.
    auto segs = [&](auto upc, const char *sb, const float *ea, const int *ew) {
        constexpr bool UP = decltype(upc)::value;
        float ps = 0.0f;
#pragma unroll
        for (int k = 0; k < CB; ++k) {
            const float ae = ea[k];
            const float ze = fmaf(ae, cz, z0c);
            const float kf = floorf(zs);
            const float wx = (UP ? __builtin_amdgcn_fmed3f(ze - kf - 1.0f, 0.0f, 1.0f)
                                 : __builtin_amdgcn_fmed3f(kf - ze, 0.0f, 1.0f)) * icz;
            const float wy = (ae - as) - wx;
            const int klo = (int)kf - (UP ? 0 : 1);
            const unsigned a = min((unsigned)(klo * SB + ew[k]), wmax2);
            const SE *pr = reinterpret_cast<const SE *>(sb + k * CW * SB + a);
            const float f0 = (float)pr[0], f1 = (float)pr[1];
            ps = fmaf(UP ? wy : wx, f0, ps);
            ps = fmaf(UP ? wx : wy, f1, ps);
            as = ae;
            zs = ze;
        }
        return ps;
    };
    const unsigned wmax = (unsigned)((4 * NQ - 1) * SB);
    float asx = lo;
    auto segs_exact = [&](const char *sb, const float *ea, const int *ew) {
        float ps = 0.0f;
#pragma unroll
        for (int k = 0; k < CB; ++k) {
            const float ae = __builtin_amdgcn_fmed3f(ea[k], lo, hi);
            const float m = fminf(az, ae);
            const float d0 = m - asx, d1 = ae - m;
            const bool cr = az < ae;
            // the slab before and after the crossing, as byte offsets in the
            // window (an idle lane's slab may lie outside it: clamped, and its
            // segment lengths are 0)
            const unsigned r0 = min((unsigned)(zrb + ew[k]), wmax);
            zrb += cr ? dzb : 0;
            nfz += cr ? sgzf : 0.0f;
            az = fmaf(nfz, kz, bz0);
            const unsigned r1 = min((unsigned)(zrb + ew[k]), wmax);
            ps = fmaf(d0, (float)*reinterpret_cast<const SE *>(sb + k * CW * SB + r0), ps);
            ps = fmaf(d1, (float)*reinterpret_cast<const SE *>(sb + k * CW * SB + r1), ps);
            asx = ae;
        }
        return ps;
    };
    // one batch from staging buffer BUF; the next batch's quads are loaded
    // meanwhile and go to the other buffer
    auto batch = [&](auto bufc, int b) {
        constexpr int BUF = decltype(bufc)::value;
        __syncthreads();   // batch b staged; batch b - 1's readers are done with the other buffer
        if (b + 1 < nb) issue(b + 1);
        const char *sb = reinterpret_cast<const char *>(stg + BUF * CB * CW);
        float ea[CB];
        int ew[CB];
#pragma unroll
        for (int k = 0; k < CB; k += 4) {
            const float4 a4 = *reinterpret_cast<const float4 *>(la + b * CB + k);
            const int4 w4 = *reinterpret_cast<const int4 *>(lw + b * CB + k);
            ea[k] = a4.x; ea[k + 1] = a4.y; ea[k + 2] = a4.z; ea[k + 3] = a4.w;
            // this ray's slab kb at the window's byte 0
            ew[k] = kbb - w4.x; ew[k + 1] = kbb - w4.y; ew[k + 2] = kbb - w4.z; ew[k + 3] = kbb - w4.w;
        }
        // rising and falling rays (all but one wave per column are uniform)
        float ps;
        if constexpr (CMD != 1) ps = segs_exact(sb, ea, ew);
        else ps = up ? segs(std::true_type(), sb, ea, ew) : segs(std::false_type(), sb, ea, ew);
        const float yk = ps - comp;
        const float tk = sum + yk;
        comp = (tk - sum) - yk;
        sum = tk;
        if (b + 1 < nb) commit(std::integral_constant<int, 1 - BUF>());
    };
    for (int b = 0; b < nb; b += 2) {
        batch(std::integral_constant<int, 0>(), b);
        if (b + 1 < nb) batch(std::integral_constant<int, 1>(), b + 1);
    }
    const int64_t P = (int64_t)d.R * d.ZP;
    const int64_t pix = (int64_t)row * d.R + col;
    const float ax = len < d.vz * 1e-6f ? 0.0f : (sum - comp) * dist;
    if constexpr (CMD == 2) {
        // FP64 sum of the workgroup's squared residuals, one slot per workgroup
        __shared__ double wsum[RW / 64];
        double e2 = 0.0;
        if (row < d.ZP) {
            const double e = (double)ax - (double)ldf(meas, ((int64_t)(v - mv0) * d.NS + src) * P + pix);
            e2 = e * e;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) e2 += __shfl_down(e2, o, 64);
        if ((tid & 63) == 0) wsum[tid >> 6] = e2;
        __syncthreads();
        if (tid == 0)
            out[((int64_t)img * gridDim.y + t.y) * gridDim.x + t.x] =
                RW == 256 ? (wsum[0] + wsum[1]) + (wsum[RW / 64 - 2] + wsum[RW / 64 - 1]) : wsum[0] + wsum[1];
        return;
    }
    if (row >= d.ZP) return;
    float r = ax;
    if constexpr (CMD == 1)
        r = len < d.vz * 1e-6f ? 0.0f : ((float)ldf(meas, ((int64_t)(v - mv0) * d.NS + src) * P + pix) - ax) / len;
    if constexpr (CMD != 2) St<SO>::st(out, (int64_t)img * P + pix, r);
}

// SART correction of fan- and parallel-beam views whose detector rows lie at
// the slice centres (planar_sweep_fits): a ray then stays in its row's slice,
// and all rows of a detector column cross the same x/y cells over the same
// alphas.  The volume is in the z-fastest layout [y][x][z], so a cell's slices
// are contiguous: zw lanes (a power of two from 64 to 256) take one column's
// slices, the column's cells and alpha lengths are listed once in LDS (the
// merge of k_project_col, clipped to the ray's [alpha_min, alpha_max]), and a
// segment costs every lane one coalesced load and one FMA, whatever the ray's
// direction.  Batches of 16 segments are summed in FP32 and the batch sums
// Kahan-compensated, as in the other walks.  The corrections are stored
// [image][column][row], as k_planar_update reads them.
//
// Bound by memory, the volume read once: 512 x 512 x 256 / 1024 x 256 0.055 ms
// and 272 MB of HBM per view (5.0 TB/s; VALU issue 27%), against 0.28 ms for one
// per-ray walk per lane.
template <typename SV, typename SM>
__global__ __launch_bounds__(256) void k_planar_corr(DGeo<float> d, const float *__restrict__ ang,
                                                     const SV *__restrict__ fz, float *__restrict__ corr,
                                                     const SM *__restrict__ meas, int first, int stride, int zsh) {
    extern __shared__ __align__(16) unsigned char pl_smem[];
    constexpr int B = 16, ES = (int)sizeof(SV);
    const int zw = 1 << zsh, cpw = 256 >> zsh;
    const int LE = (d.M + d.N + B) & ~(B - 1);           // list entries of a column, padded (at most M + N - 1 used)
    const int tid = threadIdx.x, c = tid >> zsh, zt = tid & (zw - 1);
    const int3 t = xcd_tile();
    const int col = t.x * cpw + c, z = t.y * zw + zt, img = t.z;
    const int v = first + img * stride;
    const float s = ang[2 * v], cs = ang[2 * v + 1];
    uint2 *const list = reinterpret_cast<uint2 *>(pl_smem) + (size_t)c * LE;   // (alpha length, byte offset of the cell)
    FastWalk<1> fw;
    // (the column's rays differ in the slice alone)
    const bool hit = col < d.R && fw.init(d, s, cs, col, t.y * zw, 0);
    int KP = 0;
    if (hit) {
        const float u = d.ymin + (float)col * d.du;
        const float x1x = d.dod * cs - u * s, x1y = d.dod * s + u * cs;
        float x2x, x2y, x2z;
        ray_source(d, s, cs, u, 0.0f, 0, x2x, x2y, x2z);
        const int sgx = (x1x < x2x) ? 1 : ((x1x > x2x) ? -1 : 0), sgy = (x1y < x2y) ? 1 : ((x1y > x2y) ? -1 : 0);
        const PlaneAxis X = plane_axis(d.vx, d.ivx, d.bx, x1x, 1.0f / (x2x - x1x), sgx, d.vx * 1e-6f > fabsf(x1x - x2x));
        const PlaneAxis Y = plane_axis(d.vy, d.ivy, d.by, x1y, 1.0f / (x2y - x1y), sgy, d.vy * 1e-6f > fabsf(x1y - x2y));
        const float lo = fw.ac, hi = fw.amax;
        float nf;
        int vi0 = X.i0, vj0 = Y.i0, NX = 0, NY = 0;
        if (!X.par) {
            vi0 = FastWalk<1>::restart_axis(X.k, X.b0, (float)sgx, nf, lo, d.M);
            NX = max((FastWalk<1>::restart_axis(X.k, X.b0, (float)sgx, nf, hi, d.M) - vi0) * sgx, 0);
        }
        if (!Y.par) {
            vj0 = FastWalk<1>::restart_axis(Y.k, Y.b0, (float)sgy, nf, lo, d.N);
            NY = max((FastWalk<1>::restart_axis(Y.k, Y.b0, (float)sgy, nf, hi, d.N) - vj0) * sgy, 0);
        }
        const int K = NX + NY;                  // crossings; entry K ends at hi
        KP = (K + B) / B * B;
        const float px0 = (float)(vi0 + (sgx > 0)), py0 = (float)(vj0 + (sgy > 0));
        const float fsx = (float)sgx, fsy = (float)sgy;
        auto XA = [&](int i) { return fmaf(fmaf((float)i, fsx, px0), X.k, X.b0); };
        auto YA = [&](int j) { return fmaf(fmaf((float)j, fsy, py0), Y.k, Y.b0); };
        const int C = (KP + zw - 1) >> zsh, e0 = zt * C;
        if (e0 < KP) {
            const int ee = min(e0, K);
            int ilo = max(0, ee - NY), ihi = min(ee, NX);
            while (ilo < ihi) {
                const int mid = (ilo + ihi) >> 1;
                if (XA(mid) <= YA(ee - mid - 1)) ilo = mid + 1;
                else ihi = mid;
            }
            int i = ilo, j = ee - ilo;
            float ap = lo;
            if (e0 > K) ap = hi;
            else if (ee > 0)
                ap = __builtin_amdgcn_fmed3f(fmaxf(i > 0 ? XA(i - 1) : -__builtin_inff(), j > 0 ? YA(j - 1) : -__builtin_inff()), lo, hi);
            for (int e = e0; e < min(e0 + C, KP); ++e) {
                const unsigned off = ((unsigned)(vj0 + j * sgy) * (unsigned)d.M + (unsigned)(vi0 + i * sgx)) * (unsigned)d.Z * (unsigned)ES;
                float a = hi;
                if (e < K) {
                    if (i < NX && (j >= NY || XA(i) <= YA(j))) { a = XA(i); ++i; }
                    else { a = YA(j); ++j; }
                    a = __builtin_amdgcn_fmed3f(a, lo, hi);
                }
                list[e] = make_uint2(__float_as_uint(a - ap), off);
                ap = a;
            }
        }
    }
    __syncthreads();
    if (col >= d.R) return;
    float sum = 0.0f, comp = 0.0f;
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(fz, (uint32_t)d.M * (uint32_t)d.N * (uint32_t)d.Z * (uint32_t)ES);
    const uint32_t zo = (uint32_t)z * (uint32_t)ES;
    for (int e = 0; e < KP; e += B) {
        float dl[B], fv[B];
#pragma unroll
        for (int k = 0; k < B; k += 2) {
            const uint4 w = *reinterpret_cast<const uint4 *>(list + e + k);
            dl[k] = __uint_as_float(w.x); dl[k + 1] = __uint_as_float(w.z);
            fv[k] = bload<SV>(rs, w.y + zo);
            fv[k + 1] = bload<SV>(rs, w.w + zo);
        }
        float ps = dl[0] * fv[0];
#pragma unroll
        for (int k = 1; k < B; ++k) ps = fmaf(dl[k], fv[k], ps);
        const float y = ps - comp, tt = sum + y;
        comp = (tt - sum) - y;
        sum = tt;
    }
    if (z >= d.Z) return;
    float r = 0.0f;
    if (hit && !(fw.len < d.vz * 1e-6f))
        r = ((float)ldf(meas, ((int64_t)v * d.ZP + z) * d.R + col) - (sum - comp) * fw.dist) / fw.len;
    corr[((int64_t)img * d.R + col) * d.Z + z] = r;
}

// Data fidelity sum (Ax - b)^2 fused into the ray traversal: Ax never goes to
// memory.  Geometries that admit the column walk take it (CMD 2 of
// k_project_col); this per-ray form serves the others, exact mode and FP64.
// Each 256-ray block writes one FP64 partial (wave64 shuffles, then
// LDS across the 4 waves); the partials are folded in fixed order afterwards.
// (L2_norm_gpu + the objective's Forward_3D_ray_driven_siddon,
// V63/host_tool_functions.cu:28-58 and V63/main_recon.cu:401-407.)
template <typename T, typename SV, typename SM, bool COMP>
__global__ __launch_bounds__(256) void k_residual(DGeo<T> d, const T *__restrict__ ang, const SV *__restrict__ f,
                                                  const SM *__restrict__ meas, int view0, int z0,
                                                  double *__restrict__ part) {
    int col, row;
    const int slot = tile_coords(col, row);
    const int img = slot + z0;
    double e2 = 0.0;
    if (col < d.R && row < d.ZP) {
        const int q = img / d.NS, src = img - q * d.NS;
        const int v = view0 + q;
        const T s = ang[2 * v], c = ang[2 * v + 1];
        T len;
        T sum;
        if constexpr (COMP && std::is_same<T, float>::value) sum = siddon_sum_fast<SV>(d, s, c, col, row, src, f, len);
        else sum = siddon_sum<T, SV, 4, false>(d, s, c, col, row, src, f, len);
        const T ax = (len < d.vz * (T)1e-6) ? (T)0 : sum;
        const int64_t P = (int64_t)d.R * d.ZP;
        const double e = (double)ax - (double)ldf(meas, (int64_t)img * P + (int64_t)row * d.R + col);
        e2 = e * e;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e2 += __shfl_down(e2, o, 64);
    __shared__ double wsum[4];
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = e2;
    __syncthreads();
    // one slot per workgroup: launches cover images [z0, z0 + gridDim.z)
    if (threadIdx.x == 0)
        part[((int64_t)z0 * gridDim.y + blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] =
            (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

template <typename A> __device__ __forceinline__ void atomic_add(A *p, A v);
template <> __device__ __forceinline__ void atomic_add<float>(float *p, float v) { unsafeAtomicAdd(p, v); }
template <> __device__ __forceinline__ void atomic_add<double>(double *p, double v) { unsafeAtomicAdd(p, v); }

// Matched adjoint: scatter the forward's segments (scatter form of
// V63/pixel_driven_backprj/kernel_IterativeRecon_CBCT.cu:563-1116).  Rays the
// forward zeroes (len < 1e-6*vz) scatter nothing, so the pair is an exact
// transpose.  FAST pairs with the fast forward: the same FastWalk steps, its
// closed-form length, and no scatter for an offset past the grid (the
// forward reads 0 there).  Otherwise a first pass measures the ray length
// of the reference traversal.
template <typename T, typename SP, typename A, bool FAST, bool ZQ = false>
__global__ __launch_bounds__(256) void k_adjoint(DGeo<T> d, const T *__restrict__ ang,
                                                 const SP *__restrict__ proj, A *__restrict__ acc,
                                                 int view0, int z0) {
    int col, row;
    const int slot = tile_coords(col, row);
    if (col >= d.R || row >= d.ZP) return;
    const int img = slot + z0;
    const int q = img / d.NS, src = img - q * d.NS;
    const int v = view0 + q;
    const int64_t P = (int64_t)d.R * d.ZP;
    const T y = (T)ldf(proj, (int64_t)img * P + (int64_t)row * d.R + col);
    if (y == (T)0) return;
    const T s = ang[2 * v], c = ang[2 * v + 1];
    if constexpr (FAST) {
        FastWalk<1, ZQ> w;
        if (!w.init(d, s, c, col, row, src)) return;
        if (w.len < d.vz * 1e-6f) return;
        const unsigned nvox = (unsigned)d.M * (unsigned)d.N * (ZQ ? (unsigned)((d.Z + 3) & ~3) : (unsigned)d.Z);
        int guard = d.M + d.N + d.Z + 4;
        do {
#pragma unroll
            for (int u = 0; u < FAST_B; ++u) {
                unsigned id;
                const float dl = w.step(id);
                if (dl != 0.0f && id < nvox) atomic_add<A>(acc + id, (A)(w.dist * dl) * (A)y);
            }
            guard -= FAST_B;
        } while (!w.ended() && guard > 0);
    } else {
        const T len = siddon_traverse(d, s, c, col, row, src, [](int, T) {});
        if (len < d.vz * (T)1e-6) return;
        siddon_traverse(d, s, c, col, row, src, [&](int idx, T seg) { atomic_add<A>(acc + idx, (A)seg * (A)y); });
    }
}

// ------------------------------------------------- gather form of the adjoint
// Aᵀy without atomics, for the fast walk.  The walk's segment in voxel
// (i, j, k) is max(0, min(exit planes, alpha_hi) - max(entry planes,
// alpha_lo)) - it is in that voxel exactly while it is inside all three
// slabs - and every term is separable: the x/y plane models and the x/y parts
// of [alpha_lo, alpha_hi] depend on the detector column, the z ones on the
// row.  So each voxel gathers over the pixels of its detector footprint
// exactly the numbers the walk scatters, in any order and without atomics.
//
// Per-view tables: column  (kx, bx0, ky, by0) (lo_xy, hi_xy)
//                  row     (kz, bz0) (lo_z, hi_z)
//                  pixel   w = dist*y (0 for a ray the forward zeroes)
// A parallel axis (the ray stays in slab i0) gets planes at alpha
// (n - i0 - 1/2) ADJ_FAR: voxel i0 holds every alpha and any other none.
struct AdjCol { float4 a; float2 b; };
constexpr float ADJ_FAR = 1e25f;   // times 2^31 voxels still finite

__device__ __forceinline__ void axis_bounds(float v, float b, int n, float x1, float x2, float &k, float &b0, float &lo,
                                            float &hi, float iv) {
    const float id = 1.0f / (x2 - x1);
    const bool par = v * 1e-6f > fabsf(x1 - x2);
    const PlaneAxis P = plane_axis(v, iv, b, x1, id, 0, par);
    if (par) {
        // a ray outside the grid's slabs has pixel weight 0
        k = ADJ_FAR;
        b0 = -((float)P.i0 + 0.5f) * ADJ_FAR;
        lo = -__builtin_inff(); hi = __builtin_inff();
        return;
    }
    // the reference setup's slab interval along this axis
    // (V63/kernel_IterativeRecon_universal.cu:77-104)
    const float a0 = (b - x1) * id, a1 = (b + v * (float)n - x1) * id;
    k = P.k; b0 = P.b0;
    const float g0 = b0, gn = fmaf((float)n, k, b0);
    lo = hmax(fminf(a0, a1), hmin(g0, gn));
    hi = hmin(fmaxf(a0, a1), hmax(g0, gn));
}

// tables for images [0, nimg) of views view0 + q (q = img / NS)
template <typename SP>
__global__ __launch_bounds__(256) void k_adj_prep(DGeo<float> d, const float *__restrict__ ang, int view0,
                                                  const SP *__restrict__ proj, int nimg, float *__restrict__ pixw,
                                                  AdjCol *__restrict__ colT, float4 *__restrict__ rowT) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, img = blockIdx.z;
    if (i >= d.R) return;
    const int q = img / d.NS, src = img - q * d.NS;
    const int v = view0 + q;
    const float s = ang[2 * v], c = ang[2 * v + 1];
    const int64_t P = (int64_t)d.R * d.ZP;
    const float y = (float)ldf(proj, (int64_t)img * P + (int64_t)j * d.R + i);
    float w = 0.0f;
    if (y != 0.0f) {
        FastWalk<1> fw;
        if (fw.init(d, s, c, i, j, src) && !(fw.len < d.vz * 1e-6f)) w = fw.dist * y;
    }
    pixw[(int64_t)img * P + (int64_t)j * d.R + i] = w;
    // the detector pixel and source, as ray_setup forms them
    const float x2x = d.sx * c - d.sy * s, x2y = d.sx * s + d.sy * c;
    if (j == 0 && src == 0) {
        const float u = d.ymin + (float)i * d.du;
        const float x1x = d.dod * c - u * s, x1y = d.dod * s + u * c;
        float kx, bx0, lx, hx, ky, by0, ly, hy;
        axis_bounds(d.vx, d.bx, d.M, x1x, x2x, kx, bx0, lx, hx, d.ivx);
        axis_bounds(d.vy, d.by, d.N, x1y, x2y, ky, by0, ly, hy, d.ivy);
        AdjCol e;
        e.a = make_float4(kx, bx0, ky, by0);
        e.b = make_float2(hmax(lx, ly), hmin(hx, hy));
        colT[(int64_t)q * d.R + i] = e;
    }
    if (i == 0) {
        const float x1z = d.zmin + (float)j * d.dv;
        const float x2z = d.tb ? (float)(d.sz0 + (float)src * d.sdz) : d.sz0;
        float kz, bz0, lz, hz;
        axis_bounds(d.vz, d.bz, d.Z, x1z, x2z, kz, bz0, lz, hz, d.ivz);
        rowT[(int64_t)img * d.ZP + j] = make_float4(kz, bz0, lz, hz);
    }
}

constexpr int AZR = 8;          // z-run per lane
constexpr int ALW = 80;         // staged footprint columns
constexpr int ALP = ALW + 8;    // row pitch (zero columns for the NC overrun)
constexpr int ALH = 48;         // staged footprint rows (48 sources 3 mm apart need 36)
constexpr int ANC = 8;          // bounding-box columns per voxel

// One voxel's sum over the rows [z0, z1] of its footprint: per row the slab
// interval of voxel n along z (planes n and n + 1), per pixel the overlap with
// the column's x/y interval.  The grid clip of the reference's setup moves a
// plane only at the grid's own faces (by rounding), so EDGE, the runs that
// hold a first or last slice, alone applies it.
template <int NC, bool EDGE>
__device__ __forceinline__ float adj_rows(const float *__restrict__ sw, const float2 *__restrict__ srk,
                                          const float2 *__restrict__ srl, int z0, int z1, int cbase, float n, float n1,
                                          const float *xin, const float *xout) {
    float acc = 0.0f;
    if (z1 < z0) return acc;   // (a slice past the volume or the staged rows: no pointer to form)
    const float *prow = sw + (__umul24((uint32_t)z0, ALP) + cbase);
    const float2 *lp = srl + z0;
    for (const float2 *rp = srk + z0, *const re = srk + z1; rp <= re; ++rp, prow += ALP) {
        const float2 rk = *rp;
        float pw[NC];
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) pw[cc] = prow[cc];
        const float a0 = fmaf(n, rk.x, rk.y), a1 = fmaf(n1, rk.x, rk.y);
        float zi = fminf(a0, a1), zo = fmaxf(a0, a1);
        if constexpr (EDGE) {
            const float2 l = *lp++;
            zi = hmax(zi, l.x);
            zo = hmin(zo, l.y);
        }
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) {
            // alpha lengths are below 1
            acc = fmaf(hspan(xout[cc], zo, xin[cc], zi), pw[cc], acc);
        }
    }
    return acc;
}

// The gather's tiles: two rows of tiles to each XCD in turn.  Whole eighths of
// the volume (xcd_tile) leave the XCDs of the end slices idle where the detector
// does not reach them, single tiles share no lines of the tables (gradient of many
// sources in BF16 4.43 ms by eighths, 2.60 by tile, 2.53, 2.49 and
// 2.53 by one, two and four rows; 512^3 / 1024^2, 24 views 12.3, 12.6, 12.3,
// 12.0, 12.0).  The rest past a multiple of eight such chunks keeps its order.
__device__ __forceinline__ int3 xcd_rows() {
    const unsigned gx = gridDim.x, gy = gridDim.y, T = gx * gy * gridDim.z, C = gx * 2;
    const unsigned L = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned i = L >> 3, q = i / C;
    const unsigned t = (q + 1) * 8 * C <= T ? (q * 8 + (L & 7u)) * C + (i - q * C) : L;
    const unsigned z = t / (gx * gy), r = t - z * (gx * gy);
    const unsigned y = r / gx;
    return make_int3((int)(r - y * gx), (int)y, (int)z);
}

// one lane per (x, y) and its AZR z-voxels; a 16x16 (x, y) tile per
// workgroup; per image the tile's detector footprint of weights is staged in
// LDS.  Each image's per-voxel sum (FP32, ~10 terms) is added into an FP32
// total with Kahan compensation; the volume is written once.
//
// Bound by VALU issue: 4 per (voxel, footprint pixel), 9 per row and ~20 per
// voxel.  The columns' x/y intervals are formed once per view and lane, for
// as many columns as the wave needs, and shared by the run of 8 slices and by
// the view's sources; each z face's shadow is evaluated once for the two
// voxels it bounds.  0.32 ms per view at 512^3 / 1024^2 in batches of 16
// (0.63 ms when every voxel formed all eight columns' and both faces' terms
// itself), 48 sources x 2 views of 1024 x 128 on 256^3 2.6 ms (5.8).  Four
// waves per SIMD: five spill (0.41 ms), and a run of 16 slices is no faster
// (0.33 ms) and needs a third more staged rows.
//
// PART: the grid's z axis also splits the views into parts of vpp, for
// volumes whose tiles leave the chip idle; part p's sums and their
// compensations go to part[p V + voxel] and k_adj_fold adds them in FP64.
// 64^3 from 90 views of 96^2: 730 us on its 128 tiles, 80 us in 1024 parts.
template <typename SO, bool PART>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_adjoint_gather(DGeo<float> d, const float *__restrict__ ang, int view0,
                                                        int nv, int vpp, const float *__restrict__ pixw,
                                                        const AdjCol *__restrict__ colT,
                                                        const float4 *__restrict__ rowT, SO *__restrict__ vol,
                                                        float2 *__restrict__ part) {
    __shared__ float sw[ALH * ALP];
    __shared__ float4 sca[ALP];
    __shared__ float2 scb[ALP];
    __shared__ float2 srk[ALH], srl[ALH];
    const int tid = threadIdx.y * 16 + threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int3 tile = xcd_rows();
    const int tz = PART ? (d.Z + AZR - 1) / AZR : 1;
    const int pt = PART ? tile.z / tz : 0;
    const int ix = tile.x * 16 + threadIdx.x, iy = tile.y * 16 + threadIdx.y, iz0 = (tile.z - pt * tz) * AZR;
    const int nz = min(AZR, d.Z - iz0);
    const bool active = ix < d.M && iy < d.N;
    float cx = 0, cy = 0;
    if (!d.tb) {
        cx = d.bx + d.vx * 0.5f + (float)ix * d.vx;
        cy = d.by + d.vy * 0.5f + (float)iy * d.vy;
    } else {
        cx = d.bx + d.vx * (0.5f + (float)ix);
        cy = d.by + d.vy * (0.5f + (float)iy);
    }
    const float hvx = 0.5f * d.vx, hvy = 0.5f * d.vy;
    const float xl = cx - hvx, xh = cx + hvx, yl = cy - hvy, yh = cy + hvy;
    const float nx = (float)ix, ny = (float)iy;
    const int tx0 = tile.x * 16, ty0 = tile.y * 16;
    const float TX0 = d.bx + (float)tx0 * d.vx, TX1 = d.bx + (float)min(tx0 + 16, d.M) * d.vx;
    const float TY0 = d.by + (float)ty0 * d.vy, TY1 = d.by + (float)min(ty0 + 16, d.N) * d.vy;
    const float TZ0 = d.bz + (float)iz0 * d.vz, TZ1 = d.bz + (float)(iz0 + nz) * d.vz;
    const bool edge = iz0 == 0 || iz0 + AZR >= d.Z;
    // per-voxel sums over the images, Kahan-compensated FP32
    float W[AZR], Wc[AZR];
#pragma unroll
    for (int k = 0; k < AZR; ++k) { W[k] = 0.0f; Wc[k] = 0.0f; }
    const int64_t P = (int64_t)d.R * d.ZP;
    const int q1 = PART ? min(nv, (pt + 1) * vpp) : nv;
    for (int q = PART ? pt * vpp : 0; q < q1; ++q) {
        const int v = view0 + q;
        const float s = ang[2 * v], c = ang[2 * v + 1];
        // the tile's footprint
        float Tumin = __builtin_inff(), Tumax = -__builtin_inff(), Trmin = __builtin_inff(), Trmax = -__builtin_inff();
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
                const float px = ii ? TX1 : TX0, py = jj ? TY1 : TY0;
                const float t = px * c + py * s;
                const float sv = -px * s + py * c;
                const float ratio = (t - d.dod) * frcp(d.dso - t);
                const float u = fmaf(ratio, sv - d.sy, sv);
                Tumin = fminf(Tumin, u); Tumax = fmaxf(Tumax, u);
                Trmin = fminf(Trmin, ratio); Trmax = fmaxf(Trmax, ratio);
            }
        const int C0 = max((int)floorf(fmaf(Tumin - d.ymin, d.idu, 0.5f)) - 1, 0);
        const int C1 = min(min((int)floorf(fmaf(Tumax - d.ymin, d.idu, 0.5f)) + 1, d.R - 1), C0 + ALW - 1);
        const int ncw = C1 - C0 + 1;
        if (ncw <= 0) continue;   // uniform
        // this lane's voxel column: corner ratios and detector-column box
        float rmin = __builtin_inff(), rmax = -__builtin_inff(), minY = __builtin_inff(), maxY = -__builtin_inff();
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
                const float px = ii ? xh : xl, py = jj ? yh : yl;
                const float t = px * c + py * s;
                const float sv = -px * s + py * c;
                const float ratio = (t - d.dod) * frcp(d.dso - t);
                const float u = fmaf(ratio, sv - d.sy, sv);
                minY = fminf(minY, u); maxY = fmaxf(maxY, u);
                rmin = fminf(rmin, ratio); rmax = fmaxf(rmax, ratio);
            }
        const int y0r = shadow_lo((minY - d.ymin) * d.idu);
        const int y1r = shadow_hi((maxY - d.ymin) * d.idu);
        const int y0 = max(y0r, C0), y1 = min(min(y1r, C1), y0 + ANC - 1);
        // (a lane off the volume or the detector has no columns; it still reads
        // its wave's NC, and takes them from ncw on: of the staged rows only the
        // footprint and the eight zero columns after it are written, and a
        // pixel that is not finite must not reach it, not even times 0)
        const int ncol = active ? max(y1 - y0 + 1, 0) : 0;
        const int cbase = ncol > 0 ? y0 - C0 : ncw;
        int NC = 0;   // uniform over the wave
        bool fresh = true;
        float xin[ANC], xout[ANC];
        for (int src = 0; src < d.NS; ++src) {
            const int img = q * d.NS + src;
            const float szs = d.tb ? (float)(d.sz0 + (float)src * d.sdz) : d.sz0;
            const float e0 = TZ0 - szs, e1 = TZ1 - szs;
            const float Tw0 = fminf(fmaf(Trmin, e0, TZ0), fmaf(Trmax, e0, TZ0));
            const float Tw1 = fmaxf(fmaf(Trmin, e1, TZ1), fmaf(Trmax, e1, TZ1));
            const int R0 = max((int)floorf(fmaf(Tw0 - d.zmin, d.idv, 0.5f)) - 1, 0);
            const int R1 = min(min((int)floorf(fmaf(Tw1 - d.zmin, d.idv, 0.5f)) + 1, d.ZP - 1), R0 + ALH - 1);
            const int nrow = R1 - R0 + 1;
            if (nrow <= 0) continue;   // uniform
            __syncthreads();   // the previous image's readers are done
            {
                // a wave per row, a lane per column; the columns past the
                // footprint that a voxel's NC columns can reach are zero
                const float *g = pixw + (int64_t)img * P + (int64_t)R0 * d.R + C0;
                const bool wide = ncw + 8 > 64;   // uniform
                for (int r = wave; r < nrow; r += 4) {
                    sw[r * ALP + lane] = lane < ncw ? g[(int64_t)r * d.R + lane] : 0.0f;
                    if (wide && lane < ALP - 64)
                        sw[r * ALP + 64 + lane] = lane + 64 < ncw ? g[(int64_t)r * d.R + 64 + lane] : 0.0f;
                }
                if (fresh && tid < ncw) {
                    const AdjCol e = colT[(int64_t)q * d.R + C0 + tid];
                    sca[tid] = e.a;
                    scb[tid] = e.b;
                }
                if (tid < nrow) {
                    const float4 e = rowT[(int64_t)img * d.ZP + R0 + tid];
                    srk[tid] = make_float2(e.x, e.y);
                    srl[tid] = make_float2(e.z, e.w);
                }
            }
            __syncthreads();
            if (fresh) {
                fresh = false;
                if (__builtin_amdgcn_ballot_w64(ncol > 6)) NC = 8;
                else if (__builtin_amdgcn_ballot_w64(ncol > 5)) NC = 6;
                else if (__builtin_amdgcn_ballot_w64(ncol > 4)) NC = 5;
                else if (__builtin_amdgcn_ballot_w64(ncol > 3)) NC = 4;
                else if (__builtin_amdgcn_ballot_w64(ncol > 0)) NC = 3;
                // x/y slab interval of this voxel column for each footprint
                // column
#pragma unroll
                for (int cc = 0; cc < ANC; ++cc) {
                    xin[cc] = __builtin_inff();
                    xout[cc] = -__builtin_inff();
                    if (cc >= NC) continue;
                    const int ci = min(cbase + cc, ncw - 1);
                    const float4 a = sca[ci];
                    const float2 b = scb[ci];
                    const float ax0 = fmaf(nx, a.x, a.y), ax1 = fmaf(nx + 1.0f, a.x, a.y);
                    const float ay0 = fmaf(ny, a.z, a.w), ay1 = fmaf(ny + 1.0f, a.z, a.w);
                    if (cc < ncol) {
                        xin[cc] = hmax(hmax(hmin(ax0, ax1), hmin(ay0, ay1)), b.x);
                        xout[cc] = hmin(hmin(hmax(ax0, ax1), hmax(ay0, ay1)), b.y);
                    }
                }
            }
            if (NC == 0) continue;   // uniform over the wave
            // The faces' shadow rows, counted from the staged window's first
            // row, with shadow_lo / shadow_hi's margins folded into the
            // offset: w = z + r (z - z_source) is monotone in the corner
            // ratio r, so the extreme ratios give its extremes.
            const float zrow = -d.zmin * d.idv - (float)R0;
            const float zrow_lo = zrow - 0.01f, zrow_hi = zrow + 0.01f;
            auto voxels = [&](auto ncc, auto edgec) {
                constexpr int N = decltype(ncc)::value;
                constexpr bool E = decltype(edgec)::value;
                float zk = (float)iz0;
                asm volatile("" : "+v"(zk));   // the faces are formed here, not kept over the images
                float zf = fmaf(zk, d.vz, d.bz);
                float wl = fminf(fmaf(rmin, zf - szs, zf), fmaf(rmax, zf - szs, zf));
#pragma unroll
                for (int k = 0; k < AZR; ++k) {
                    const float n = zk;
                    zk += 1.0f;
                    zf = fmaf(zk, d.vz, d.bz);
                    const float e = zf - szs;
                    const float wa = fmaf(rmin, e, zf), wb = fmaf(rmax, e, zf);
                    const int z0 = max((int)ceilf(fmaf(wl, d.idv, zrow_lo)), 0);
                    // (slices past the volume have no rows)
                    const int z1 = min((int)floorf(fmaf(fmaxf(wa, wb), d.idv, zrow_hi)), k < nz ? nrow - 1 : -1);
                    wl = fminf(wa, wb);
                    const float a = adj_rows<N, E>(sw, srk, srl, z0, z1, cbase, n, zk, xin, xout);
                    const float y = a - Wc[k], t = W[k] + y;
                    Wc[k] = (t - W[k]) - y;
                    W[k] = t;
                }
            };
            auto by_edge = [&](auto ncc) {
                if (edge) voxels(ncc, std::true_type());
                else voxels(ncc, std::false_type());
            };
            if (NC == 3) by_edge(std::integral_constant<int, 3>());
            else if (NC == 4) by_edge(std::integral_constant<int, 4>());
            else if (NC == 5) by_edge(std::integral_constant<int, 5>());
            else if (NC == 6) by_edge(std::integral_constant<int, 6>());
            else by_edge(std::integral_constant<int, 8>());
        }
    }
    if (!active) return;
#pragma unroll
    for (int k = 0; k < AZR; ++k) {
        if (k >= nz) break;
        const int64_t idx = ((int64_t)(iz0 + k) * d.N + iy) * d.M + ix;
        if constexpr (PART) part[(int64_t)pt * ((int64_t)d.M * d.N * d.Z) + idx] = make_float2(W[k], Wc[k]);
        else St<SO>::st(vol, idx, W[k] - Wc[k]);
    }
}

// the parts' sums, in part order, in FP64
template <typename SO>
__global__ __launch_bounds__(256) void k_adj_fold(const float2 *__restrict__ part, int parts, int64_t V,
                                                  SO *__restrict__ vol) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= V) return;
    double a = 0.0;
    for (int p = 0; p < parts; ++p) {
        const float2 w = part[(int64_t)p * V + i];
        a += (double)w.x - (double)w.y;
    }
    St<SO>::st(vol, i, (float)a);
}

// Host bound for k_adjoint_gather: every tile footprint fits ALW x ALH and
// every voxel box ANC columns (the bound of bp_lds_fits without the
// reconstruction cylinder: the adjoint covers every voxel).
static bool adj_gather_fits(const DGeo<float> &d) {
    if (d.style != CT_CONE) return false; // the column/row tables assume one source per view
    const double vx = d.vx, vy = d.vy, vz = d.vz, dso = d.dso, dod = d.dod;
    const double xs[2] = {(double)d.bx, (double)d.bx + d.M * vx}, ys[2] = {(double)d.by, (double)d.by + d.N * vy};
    double rho = 0;
    for (double x : xs)
        for (double y : ys) rho = std::max(rho, std::sqrt(x * x + y * y));
    if (!(dso - rho > 0)) return false;
    const double r_lo = (-rho - dod) / (dso + rho), r_hi = (rho - dod) / (dso - rho);
    const double rmax = std::max(std::fabs(r_lo), std::fabs(r_hi));
    const double dr = (dso - dod) / ((dso - rho) * (dso - rho));
    double zs_lo = d.sz0, zs_hi = d.sz0 + (double)(d.NS - 1) * d.sdz;
    if (zs_lo > zs_hi) std::swap(zs_lo, zs_hi);
    const double z_lo = d.bz, z_hi = (double)d.bz + d.Z * vz;
    const double zrel = std::max({std::fabs(z_lo - zs_lo), std::fabs(z_lo - zs_hi), std::fabs(z_hi - zs_lo),
                                  std::fabs(z_hi - zs_hi)});
    const double lat = rho + std::fabs((double)d.sy);
    auto cols = [&](double D) { return ((1.0 + rmax) * D + dr * D * lat) / (double)d.du; };
    auto rows = [&](double D, double H) { return ((1.0 + rmax) * H + dr * D * zrel) / (double)d.dv; };
    const double DT = std::hypot(16 * vx, 16 * vy), DV = std::hypot(vx, vy);
    return cols(DT) + 4.0 <= ALW && rows(DT, AZR * vz) + 4.0 <= ALH && cols(DV) + 2.0 <= ANC;
}

// Host conditions of k_project_col; gives the rows per workgroup and the
// staged window NQ (quads per segment).  The list and two staging buffers fit the workgroup's LDS,
// the z-quad volume is under 2 GiB, and no list segment holds two z
// crossings: along every ray |dz|/vz < max(|dx|/vx, |dy|/vy), checked with
// |dz| at its largest (rows against the farthest source height) and the
// in-plane length at its smallest (|dso - dod|), with margin.  The window
// covers the z range of a workgroup's rows at any alpha inside the volume:
// for cone beam the rows fan out from the source, so their spread at a point
// is (1 - alpha) times the spread on the detector, and 1 - alpha (the
// point's share of the source-to-pixel distance) is at most
// (r_xy + |S|) / |dso - dod| with r_xy the volume's largest in-plane radius;
// fan and parallel rays keep their row height.  One voxel of the segment's
// own z travel, one of rounding margin on each side and the quad alignment
// are added.
// Of the two workgroup sizes 256, unless 128 leaves enough fewer lanes past
// the last row to pay for its second list: any on 16-bit volumes, a quarter on
// FP32 ones, whose staging weighs more (corrections of 24 views, FP32: 840
// rows on 420^3, 7/8 of the lanes, 11.2 -> 11.7 ms with 128; 560 on 280^3, 5/6,
// 4.1 -> 4.0; FP16: 640 on 320^3, 5/6, 4.7 -> 4.4; gradient of 90 views of 96
// rows on 64^3 217 -> 163 us).  Where 256 rows overrun the window, 128 serve;
// not for corrections with more than an eighth of the lanes past the last row, of
// FP32 volumes beyond the 32 MB of the XCDs' L2, or of fewer than four images on
// 16-bit ones: the per-ray walk is then the faster one (dv/vz = 1, FP32, four
// views at a time: 200^3 0.82 -> 0.78 ms by column, 512^3 10.4 -> 11.3; ten at a
// time with 152 rows on 128^3 0.316 -> 0.329; FP16: 512^3 10.2 -> 9.7, one at a
// time 4.4 -> 5.4; 420^3 with 504 rows 5.5 -> 5.0, six at a time with 525 rows
// 8.5 -> 9.2).
struct ColPlan { int rows, nq; };   // nq 0: the walk is not admitted
static int col_quads(const DGeo<float> &d, int rw, int max_nq) {
    if ((d.ZP + rw - 1) / rw > 65535) return 0;
    const double inplane = std::fabs((double)d.dso - (double)d.dod);
    const int rows = std::min(rw, d.ZP) - 1;
    double span;
    if (d.style == CT_CONE) {
        const double X0 = d.bx, X1 = d.bx + (double)d.M * d.vx, Y0 = d.by, Y1 = d.by + (double)d.N * d.vy;
        const double rxy = std::sqrt(std::max(X0 * X0, X1 * X1) + std::max(Y0 * Y0, Y1 * Y1));
        const double rho = (rxy + std::hypot((double)d.dso, (double)d.sy)) / inplane;
        span = rho * rows * (double)d.dv / (double)d.vz + 1.0;
    } else {
        span = rows * (double)d.dv / (double)d.vz;
    }
    const double nq = std::ceil((span + 8.0) / 4.0);
    return nq >= 1.0 && nq <= max_nq ? (int)nq : 0;
}
// The windows of 256 and 128 rows a launch would stage; 0 where they are not
// admitted.
struct ColQuads { int n256, n128; };
static ColQuads col_fits(const DGeo<float> &d) {
    const ColQuads none = {0, 0};
    if ((uint64_t)d.M * d.N * (uint64_t)((d.Z + 3) & ~3) * 4 >= (1ull << 31)) return none;
    double dzmax = 0.0;
    const double inplane = std::fabs((double)d.dso - (double)d.dod);
    if (d.style == CT_CONE) {
        const double s0 = d.sz0, s1 = d.tb ? d.sz0 + (double)(d.NS - 1) * d.sdz : d.sz0;
        dzmax = std::max(std::max(std::fabs(d.zmin - s0), std::fabs(d.zmax - s0)),
                         std::max(std::fabs(d.zmin - s1), std::fabs(d.zmax - s1)));
    }
    const double vxy = std::max((double)d.vx, (double)d.vy);
    if (!(dzmax / (double)d.vz < 0.9 * inplane / (std::sqrt(2.0) * vxy))) return none;
    // (the padding of col_dyn_lds keeps a workgroup under 33 KiB)
    if (col_lds_bytes(d.M, d.N) > 65536) return none;
    return {col_quads(d, 256, col_nq<256>()), col_quads(d, 128, col_nq<128>())};
}
static ColPlan col_plan(const DGeo<float> &d, size_t es, int nimg, bool corrections) {
    const ColPlan none = {0, 0};
    const ColQuads q = col_fits(d);
    const int n256 = q.n256, n128 = q.n128;
    const int pad256 = (d.ZP + 255) / 256 * 256, pad128 = (d.ZP + 127) / 128 * 128;
    if (n256 == 0) {
        const bool ray = corrections && (8 * pad128 > 9 * d.ZP
                                         || (es == 4 ? (uint64_t)d.M * d.N * d.Z * es > (32u << 20) : nimg < 4));
        return n128 > 0 && !ray ? ColPlan{128, n128} : none;
    }
    if (n128 > 0 && (es == 2 ? pad128 < pad256 : 4 * pad256 >= 5 * pad128)) return {128, n128};
    return {256, n256};
}

// Dynamic LDS of a launch: the list, padded so that a workgroup of 256 holds
// at least col_lds_floor bytes in all, which caps the workgroups per CU.
// Measured per view at 512^3 / 1024^2 (a one-view launch is 4096
// workgroups): FP32 volumes 0.457 ms at four per CU against 0.464 at five and
// 0.485 at six; FP16 0.331 ms at four against 0.376 at seven; BF16 (windows
// staged as FP32) 0.378 ms at six against 0.436 at four.
template <typename SV, int RW> constexpr size_t col_lds_floor() {
    return std::is_same<SV, __hip_bfloat16>::value || RW != 256 ? 0 : 32 * 1024 + 512;   // > 160 KiB / 5
}
template <typename SV, int RW> static size_t col_dyn_lds(int M, int N) {
    const size_t stat = sizeof(typename StageOf<SV>::type) * 2 * col_batch<SV>() * col_w<RW>() + 16;
    const size_t want = col_lds_floor<SV, RW>();
    const size_t list = col_dyn_bytes(M, N);
    return stat + list >= want ? list : want - stat;
}
template <typename SV, typename SO, typename SM, int CMD, int RW>
static void launch_col_rw(ct_context *ctx, const DGeo<float> &d, int nq, const float *ang, const void *const vols[2],
                          void *out, const void *meas, int first, int stride, int mv0, int nimg) {
    for (int z0 = 0; z0 < nimg; z0 += 65535) {
        const int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
        dim3 grid(d.R, (d.ZP + RW - 1) / RW, nz);
        hipLaunchKernelGGL((k_project_col<SV, SO, SM, CMD, RW>), grid, dim3(RW), (col_dyn_lds<SV, RW>(d.M, d.N)),
                           ctx->stream, d, ang, (const SV *)vols[0], (const SV *)vols[1], (SO *)out, (const SM *)meas,
                           first, stride, mv0, z0, nq);
    }
}

// (ray, x/y plane) pairs of a launch.  The column walk's lists, barriers and
// volume copies pay from 3 * 2^24 on, twice that for the objective, whose
// alternative reads the linear volume.  Corrections of 24 views, FP32, one at a
// time: 200^3 / 400^2 (2^25.9) 1.91 ms by column, 1.87 by ray, 240^3 / 480^2
// (2^26.7) 2.48 and 2.92; four at a time: 96^3 / 192^2 (2^24.8) 0.73 and 0.71,
// 160^3 / 256 x 192 (2^25.9) 0.45 and 0.51; eight single views of 128^3 / 204 x
// 152 0.35 and 0.25.  Ray sums of 24 views on 96^3 with the adjoint 0.136 and
// 0.157 ms.  Objective: 119 x 133 x 119, 6 views of 237 x 196 in FP16 (2^26.1)
// 115 us by column, 108 by ray; 120 x 127 x 79, 20 views of 200 x 123 in FP32
// (2^26.9) 128 and 146.
static double col_pairs(const DGeo<float> &d, int nimg) { return (double)d.R * d.ZP * nimg * (d.M + d.N); }
constexpr double COL_MIN = (double)(3 << 24);

// The plan of corrections.  A BF16 sweep's updates are stored with a
// dither from the low bits of their sums, so that another order of summing a ray
// changes the volume by up to 2% of its norm in 60 views (FP16 0.3%): BF16 keeps
// one walk at all sizes, by column wherever 256 rows fit.
static ColPlan sweep_plan(const DGeo<float> &d, ct_dtype vdt, int nimg) {
    if (vdt == CT_BF16) {
        const int n = col_fits(d).n256;
        return {n > 0 ? 256 : 0, n};
    }
    return col_pairs(d, nimg) >= COL_MIN ? col_plan(d, dtype_size(vdt), nimg, true) : ColPlan{0, 0};
}

// The column walk stages, per segment, one z-quad of each (x, y) on the
// column's path; a 128-byte line holds eight neighbours along the layout's
// fast axis, so paths that run along it use whole lines and paths across it
// one quad per line.  Measured at 512^3 / 1024^2 per view: 0.39 ms along the
// fast axis, even near 40 degrees, 0.67 ms across it.  Views whose central
// ray is within ~41 degrees of the x axis (|cos| >= 0.75) walk the z-quad
// copy, the others its lateral transpose.
static bool col_walk_view(const ct_geometry &g, int v) { return col_along_x(view_cos(g, v)); }

// Per-ray walk on the z-quad layout (k_project_zq): one walk per ray for ray
// sums, each ray split in two for corrections.
template <typename SV, typename SO, typename SM, int CMD>
static void launch_zq(ct_context *ctx, const DGeo<float> &d, const float *ang, const void *volq, SO *out,
                      const void *meas, int first, int stride, int nimg, int mv0) {
    constexpr int S = CMD == 1 ? CORR_SPLIT : 1;
    constexpr int tw = S <= 2 ? 16 : 8, th = S == 1 ? 16 : 8;
    for (int z0 = 0; z0 < nimg; z0 += 65535) {
        const int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
        dim3 grid((d.R + tw - 1) / tw, (d.ZP + th - 1) / th, nz);
        hipLaunchKernelGGL((k_project_zq<SV, SO, SM, CMD, S>), grid, dim3(256), 0, ctx->stream, d, ang,
                           (const SV *)volq, out, (const SM *)meas, first, stride, mv0, z0);
    }
}

// Walks the views first, first + stride, ... of a z-quad volume by column.
// volq is in the plain layout or, with `tr`, the transposed one (each in its
// own slot of the context); views that run the other way take the other copy.
template <typename SV, typename SO, typename SM, int CMD>
static ct_status launch_col(ct_context *ctx, const ct_geometry &g, const DGeo<float> &d, ColPlan cp, const float *ang,
                            const void *volq, bool tr, void *out, const void *meas, int first, int stride, int nv,
                            int mv0) {
    const void *vols[2] = {tr ? nullptr : volq, tr ? volq : nullptr};
    auto walk = [&](int q0, int n, void *o) {
        if (cp.rows == 256) launch_col_rw<SV, SO, SM, CMD, 256>(ctx, d, cp.nq, ang, vols, o, meas, first + q0 * stride, stride, mv0, n * d.NS);
        else launch_col_rw<SV, SO, SM, CMD, 128>(ctx, d, cp.nq, ang, vols, o, meas, first + q0 * stride, stride, mv0, n * d.NS);
    };
    int others = 0;
    for (int q = 0; q < nv; ++q) others += col_walk_view(g, first + q * stride) == tr;
    // Fewer than four images of the other direction do without the copy: in the
    // transposed layout (which the sweep takes by the middle view) and for the
    // objective they walk the layout that is there, in the plain one by ray
    // (FP32, 263 x 261 x 251 / 549 x 459, three views and two: 0.19 ms, 0.23 on
    // the layout that is there; 512^3 / 1024^2 in subsets of four 22.4 ms, 23.0
    // with the copy).  So do all of a BF16 sweep's, at all sizes (sweep_plan).
    // And so does any launch for which there is no memory for the other copy.
    const bool few = others * d.NS < 4 || (CMD == 1 && std::is_same<SV, __hip_bfloat16>::value);
    const uint64_t bytes = (uint64_t)d.M * d.N * (uint64_t)((d.Z + 3) & ~3) * sizeof(SV);
    void *t = few ? nullptr : slot_or_null(ctx, tr ? SLOT_ZQVOL : SLOT_ZQVOL_T, bytes);
    if constexpr (CMD != 2) {
        if (others > 0 && !t && !tr) {
            const int64_t P = (int64_t)d.R * d.ZP * d.NS;
            for (int q0 = 0, q1; q0 < nv; q0 = q1) {
                const bool w = col_walk_view(g, first + q0 * stride);
                for (q1 = q0 + 1; q1 < nv && col_walk_view(g, first + q1 * stride) == w; ++q1) {}
                SO *o = (SO *)out + q0 * P;
                if (w) walk(q0, q1 - q0, o);
                else launch_zq<SV, SO, SM, CMD>(ctx, d, ang, volq, o, meas, first + q0 * stride, stride, (q1 - q0) * d.NS, mv0);
            }
            return CT_OK;
        }
    }
    if (t) {
        const ct_status st = launch_zq_transpose(ctx, volq, dtype_of<SV>(), t, d.M, d.N, d.Z, !tr);
        if (st != CT_OK) return st;
        vols[!tr] = t;
    }
    walk(0, nv, out);
    return CT_OK;
}

// ---------------------------------------------------------------- launchers
template <typename T, typename SV, typename SM>
static ct_status run_residual(ct_context *ctx, const ct_geometry &g, const void *vol, const void *meas, double *out) {
    ct_status st;
    const T *ang = (const T *)angle_table(ctx, g, sizeof(T) == 8, false, &st);
    if (!ang) return st;
    DGeo<T> d = derive<T>(g);
    const int nimg = g.nviews * d.NS;
    const bool comp = std::is_same<T, float>::value && ctx->math == CT_MATH_FAST;
    if constexpr (std::is_same<T, float>::value) {
        // the batched ray sums' column walk where it outweighs the copies of
        // the volume, and there is memory for one
        const uint64_t qbytes = (uint64_t)d.M * d.N * (uint64_t)((d.Z + 3) & ~3) * sizeof(SV);
        const bool large = col_pairs(d, nimg) >= 2 * COL_MIN;
        const ColPlan cp = comp && large && nimg >= 4 && qbytes < (1ull << 32) ? col_plan(d, sizeof(SV), nimg, false) : ColPlan{0, 0};
        void *volq = cp.nq > 0 ? slot_or_null(ctx, SLOT_ZQVOL, qbytes) : nullptr;
        if (volq) {
            const int64_t per = (int64_t)d.R * ((d.ZP + cp.rows - 1) / cp.rows);   // workgroups per image
            double *part = (double *)slot(ctx, SLOT_TMP_PROJ2, sizeof(double) * per * nimg, &st);
            if (!part) return st;
            {
                ProfScope ps(ctx, CT_K_FORWARD);
                st = launch_zq_pack(ctx, vol, dtype_of<SV>(), volq, d.M, d.N, d.Z);
                if (st != CT_OK) return st;
                st = launch_col<SV, double, SM, 2>(ctx, g, d, cp, ang, volq, false, part, meas, 0, 1, g.nviews, 0);
                if (st != CT_OK) return st;
            }
            st = launch_check(ctx, "residual");
            if (st != CT_OK) return st;
            return reduce_dot(ctx, part, nullptr, per * nimg, CT_F64, 2, out);
        }
    }
    const int gx = (d.R + 15) / 16, gy = (d.ZP + 15) / 16;
    const int64_t nblk = (int64_t)gx * gy * nimg;
    double *part = (double *)slot(ctx, SLOT_TMP_PROJ2, sizeof(double) * nblk, &st);
    if (!part) return st;
    {
        ProfScope ps(ctx, CT_K_FORWARD);
        for (int z0 = 0; z0 < nimg; z0 += 65535) {
            const int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
            dim3 grid(gx, gy, nz);
            if (comp)
                hipLaunchKernelGGL((k_residual<T, SV, SM, true>), grid, dim3(256), 0, ctx->stream, d, ang,
                                   (const SV *)vol, (const SM *)meas, 0, z0, part);
            else
                hipLaunchKernelGGL((k_residual<T, SV, SM, false>), grid, dim3(256), 0, ctx->stream, d, ang,
                                   (const SV *)vol, (const SM *)meas, 0, z0, part);
        }
    }
    st = launch_check(ctx, "residual");
    if (st != CT_OK) return st;
    return reduce_dot(ctx, part, nullptr, nblk, CT_F64, 2, out);
}

template <typename T, typename SV>
static ct_status residual_meas(ct_context *ctx, const ct_geometry &g, const void *vol, const void *meas, ct_dtype mdt,
                               double *out) {
    switch (mdt) {
    case CT_F32: return run_residual<T, SV, float>(ctx, g, vol, meas, out);
    case CT_F16: return run_residual<T, SV, __half>(ctx, g, vol, meas, out);
    case CT_BF16: return run_residual<T, SV, __hip_bfloat16>(ctx, g, vol, meas, out);
    case CT_F64: return run_residual<T, SV, double>(ctx, g, vol, meas, out);
    }
    return fail(ctx, CT_ERR_DTYPE, "residual: bad measurement dtype");
}

ct_status launch_residual(ct_context *ctx, const ct_geometry &g, const void *vol, ct_dtype vdt, const void *meas,
                          ct_dtype mdt, double *out) {
    switch (vdt) {
    case CT_F32: return residual_meas<float, float>(ctx, g, vol, meas, mdt, out);
    case CT_F16: return residual_meas<float, __half>(ctx, g, vol, meas, mdt, out);
    case CT_BF16: return residual_meas<float, __hip_bfloat16>(ctx, g, vol, meas, mdt, out);
    case CT_F64: return residual_meas<double, double>(ctx, g, vol, meas, mdt, out);
    }
    return fail(ctx, CT_ERR_DTYPE, "residual: bad volume dtype");
}

template <typename T, typename SV, typename SO, typename SM, int CMD>
static ct_status run_forward(ct_context *ctx, const ct_geometry &g, const void *vol, void *out, const void *meas,
                             int first, int stride, int nv, int mv0) {
    ct_status st;
    const T *ang = (const T *)angle_table(ctx, g, sizeof(T) == 8, false, &st);
    if (!ang) return st;
    DGeo<T> d = derive<T>(g);
    const int nimg = nv * d.NS;
    dim3 block(256);
    // compensated FP32 ray sums in fast mode; the exact mode keeps the
    // reference's plain accumulation
    const bool comp = std::is_same<T, float>::value && ctx->math == CT_MATH_FAST;
    if constexpr (std::is_same<T, float>::value) {
        // four or more images: copy the volume once into the z-quad layout
        // and walk by detector column (k_project_col) where the geometry
        // admits it; otherwise one walk per ray for ray sums and each ray
        // split in two for corrections
        const uint64_t qbytes = (uint64_t)d.M * d.N * (uint64_t)((d.Z + 3) & ~3) * sizeof(SV);
        if (comp && nimg >= 4 && qbytes < (1ull << 32) && (CMD == 1 || col_pairs(d, nimg) >= COL_MIN)) {
            void *volq = slot(ctx, SLOT_ZQVOL, qbytes, &st);
            if (!volq) return st;
            ProfScope ps(ctx, CT_K_FORWARD);   // the copy is part of the call's cost
            st = launch_zq_pack(ctx, vol, dtype_of<SV>(), volq, d.M, d.N, d.Z);
            if (st != CT_OK) return st;
            const ColPlan cp = CMD == 1 ? sweep_plan(d, dtype_of<SV>(), nimg) : col_plan(d, sizeof(SV), nimg, false);
            if (cp.nq > 0) {
                st = launch_col<SV, SO, SM, CMD>(ctx, g, d, cp, ang, volq, false, out, meas, first, stride, nv, mv0);
                if (st != CT_OK) return st;
            } else {
                launch_zq<SV, SO, SM, CMD>(ctx, d, ang, volq, (SO *)out, meas, first, stride, nimg, mv0);
            }
            return launch_check(ctx, "forward");
        }
    }
    ProfScope ps(ctx, CT_K_FORWARD);
    for (int z0 = 0; z0 < nimg; z0 += 65535) {
        int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
        dim3 grid((d.R + 15) / 16, (d.ZP + 15) / 16, nz);
        if (comp)
            hipLaunchKernelGGL((k_forward<T, SV, SO, SM, CMD, true>), grid, block, 0, ctx->stream, d, ang,
                               (const SV *)vol, (SO *)out, (const SM *)meas, first, stride, mv0, z0);
        else
            hipLaunchKernelGGL((k_forward<T, SV, SO, SM, CMD, false>), grid, block, 0, ctx->stream, d, ang,
                               (const SV *)vol, (SO *)out, (const SM *)meas, first, stride, mv0, z0);
    }
    return launch_check(ctx, "forward");
}

template <typename T, typename SV, typename SO, int CMD>
static ct_status fwd_meas(ct_context *ctx, const ct_geometry &g, const void *vol, void *out, const void *meas,
                          ct_dtype mdt, int first, int stride, int nv, int mv0) {
    if constexpr (CMD == 0) return run_forward<T, SV, SO, SO, CMD>(ctx, g, vol, out, meas, first, stride, nv, mv0);
    switch (mdt) {
    case CT_F32: return run_forward<T, SV, SO, float, CMD>(ctx, g, vol, out, meas, first, stride, nv, mv0);
    case CT_F16: return run_forward<T, SV, SO, __half, CMD>(ctx, g, vol, out, meas, first, stride, nv, mv0);
    case CT_BF16: return run_forward<T, SV, SO, __hip_bfloat16, CMD>(ctx, g, vol, out, meas, first, stride, nv, mv0);
    case CT_F64: return run_forward<T, SV, SO, double, CMD>(ctx, g, vol, out, meas, first, stride, nv, mv0);
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported measurement dtype");
}

template <typename T, typename SV, int CMD>
static ct_status fwd_out(ct_context *ctx, const ct_geometry &g, const void *vol, void *out, ct_dtype odt,
                         const void *meas, ct_dtype mdt, int first, int stride, int nv, int mv0) {
    if constexpr (CMD == 1) {   // corrections are in the arithmetic type
        if (odt != dtype_of<T>()) return fail(ctx, CT_ERR_DTYPE, "unsupported output dtype");
        return fwd_meas<T, SV, T, CMD>(ctx, g, vol, out, meas, mdt, first, stride, nv, mv0);
    } else switch (odt) {
    case CT_F32: return fwd_meas<T, SV, float, CMD>(ctx, g, vol, out, meas, mdt, first, stride, nv, mv0);
    case CT_F16: return fwd_meas<T, SV, __half, CMD>(ctx, g, vol, out, meas, mdt, first, stride, nv, mv0);
    case CT_BF16: return fwd_meas<T, SV, __hip_bfloat16, CMD>(ctx, g, vol, out, meas, mdt, first, stride, nv, mv0);
    case CT_F64: return fwd_meas<T, SV, double, CMD>(ctx, g, vol, out, meas, mdt, first, stride, nv, mv0);
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported output dtype");
}

// first/stride select the batch's views; for CMD 1 meas is indexed by view - mv0
// (the sweep passes the whole stack with mv0 = 0).
ct_status launch_forward_mv(ct_context *ctx, const ct_geometry &g, const void *vol, ct_dtype vdt, void *out,
                            ct_dtype odt, const void *meas, ct_dtype mdt, int32_t first, int32_t stride,
                            int32_t nv, int cmd, int32_t mv0) {
    if (nv <= 0) return CT_OK;
    if (vdt == CT_F64) {
        if (cmd == 0) return fwd_out<double, double, 0>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0);
        return fwd_out<double, double, 1>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0);
    }
    switch (vdt) {
    case CT_F32:
        return cmd == 0 ? fwd_out<float, float, 0>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0)
                        : fwd_out<float, float, 1>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0);
    case CT_F16:
        return cmd == 0 ? fwd_out<float, __half, 0>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0)
                        : fwd_out<float, __half, 1>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0);
    case CT_BF16:
        return cmd == 0 ? fwd_out<float, __hip_bfloat16, 0>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0)
                        : fwd_out<float, __hip_bfloat16, 1>(ctx, g, vol, out, odt, meas, mdt, first, stride, nv, mv0);
    default: break;
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported volume dtype");
}

// ---------------------------------------------------------------------------
// Allocation-free forward projection (ct_forward_noalloc).  Its only scratch
// is the per-view (sin, cos) table the kernels read, which ct_forward keeps
// in a context buffer allocated on first use.  Here the table lives in the
// file-scope array `scratch` (256 KiB: up to 16384 views, in FP64 or FP32),
// one copy per GPU, held until the process ends.  Its device address
// is looked up once per device at context creation (noalloc_init) and only
// that address is passed to kernels and copies.  Calls that overlap on one
// GPU (two streams or two contexts) race on the table; a call first waits for
// its own stream, so back-to-back calls on one stream are ordered.
constexpr int NOALLOC_MAX_VIEWS = 16384;
static __device__ __align__(256) double scratch[2 * NOALLOC_MAX_VIEWS];

static std::mutex g_noalloc_mtx;
static void *g_noalloc_ptr[64] = {};

ct_status noalloc_init(ct_context *ctx) {
    if (ctx->device < 0 || ctx->device >= 64) return fail(ctx, CT_ERR_DEVICE, "device index beyond 63");
    ctx->noalloc_host.assign(sizeof(scratch), 0);   // the host side of the table, allocated here once
    std::lock_guard<std::mutex> l(g_noalloc_mtx);
    if (g_noalloc_ptr[ctx->device]) return CT_OK;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        hipGetLastError();
        return fail(ctx, CT_ERR_DEVICE, std::string("scratch symbol lookup failed: ") + hipGetErrorString(e));
    }
    g_noalloc_ptr[ctx->device] = p;
    return CT_OK;
}

// The per-ray forward walk of run_forward (no z-quad copy) on a caller-given
// angle table.
template <typename T, typename SV, typename SO>
static ct_status run_forward_table(ct_context *ctx, const ct_geometry &g, const T *ang, const void *vol, void *out,
                                   int first, int nv) {
    DGeo<T> d = derive<T>(g);
    const int nimg = nv * d.NS;
    const bool comp = std::is_same<T, float>::value && ctx->math == CT_MATH_FAST;
    for (int z0 = 0; z0 < nimg; z0 += 65535) {
        const int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
        dim3 grid((d.R + 15) / 16, (d.ZP + 15) / 16, nz);
        if (comp)
            hipLaunchKernelGGL((k_forward<T, SV, SO, float, 0, true>), grid, dim3(256), 0, ctx->stream, d, ang,
                               (const SV *)vol, (SO *)out, (const float *)nullptr, first, 1, first, z0);
        else
            hipLaunchKernelGGL((k_forward<T, SV, SO, float, 0, false>), grid, dim3(256), 0, ctx->stream, d, ang,
                               (const SV *)vol, (SO *)out, (const float *)nullptr, first, 1, first, z0);
    }
    return launch_check(ctx, "forward (allocation-free)");
}

template <typename T, typename SV>
static ct_status noalloc_out(ct_context *ctx, const ct_geometry &g, const T *ang, const void *vol, void *out,
                             ct_dtype odt, int first, int nv) {
    switch (odt) {
    case CT_F32: return run_forward_table<T, SV, float>(ctx, g, ang, vol, out, first, nv);
    case CT_F16: return run_forward_table<T, SV, __half>(ctx, g, ang, vol, out, first, nv);
    case CT_BF16: return run_forward_table<T, SV, __hip_bfloat16>(ctx, g, ang, vol, out, first, nv);
    case CT_F64: return run_forward_table<T, SV, double>(ctx, g, ang, vol, out, first, nv);
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported output dtype");
}

ct_status launch_forward_noalloc(ct_context *ctx, const ct_geometry &g, const void *vol, ct_dtype vdt, void *out,
                                 ct_dtype odt, int32_t view0, int32_t nv) {
    if (g.nviews > NOALLOC_MAX_VIEWS)
        return fail(ctx, CT_ERR_INVALID_ARG, "allocation-free forward: nviews " + std::to_string(g.nviews) +
                                                 " exceeds its limit of " + std::to_string(NOALLOC_MAX_VIEWS));
    if (nv <= 0) return CT_OK;
    void *tab = nullptr;
    {
        std::lock_guard<std::mutex> l(g_noalloc_mtx);
        if (ctx->device >= 0 && ctx->device < 64) tab = g_noalloc_ptr[ctx->device];
    }
    if (!tab) return fail(ctx, CT_ERR_DEVICE, "allocation-free forward: scratch not set up on this device");
    // the previous call on this stream may still read the table
    ct_status st = hip_check(ctx, hipStreamSynchronize(ctx->stream), "stream synchronize");
    if (st != CT_OK) return st;
    const bool dbl = vdt == CT_F64;
    const size_t bytes = (size_t)g.nviews * 2 * (dbl ? 8 : 4);
    // sized for NOALLOC_MAX_VIEWS at context creation (noalloc_init)
    if (ctx->noalloc_host.size() < bytes) return fail(ctx, CT_ERR_INVALID_ARG, "allocation-free forward: host table");
    fill_angle_table(g, dbl, false, ctx->noalloc_host.data());
    st = hip_check(ctx, hipMemcpyAsync(tab, ctx->noalloc_host.data(), bytes, hipMemcpyHostToDevice, ctx->stream),
                   "angle table upload");
    if (st != CT_OK) return st;
    switch (vdt) {
    case CT_F32: return noalloc_out<float, float>(ctx, g, (const float *)tab, vol, out, odt, view0, nv);
    case CT_F16: return noalloc_out<float, __half>(ctx, g, (const float *)tab, vol, out, odt, view0, nv);
    case CT_BF16: return noalloc_out<float, __hip_bfloat16>(ctx, g, (const float *)tab, vol, out, odt, view0, nv);
    case CT_F64: return noalloc_out<double, double>(ctx, g, (const double *)tab, vol, out, odt, view0, nv);
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported volume dtype");
}

template <typename SV, typename SM>
static ct_status run_correction_zq(ct_context *ctx, const ct_geometry &g, const void *volq, float *corr,
                                   const void *meas, int first, int stride, int nv, bool tr) {
    ct_status st;
    const float *ang = (const float *)angle_table(ctx, g, false, false, &st);
    if (!ang) return st;
    DGeo<float> d = derive<float>(g);
    ProfScope ps(ctx, CT_K_FORWARD);
    const ColPlan cp = sweep_plan(d, dtype_of<SV>(), nv * d.NS);
    if (cp.nq > 0) {
        // (a subset's views may run both ways; the update that follows works
        // on volq, so the other copy serves this correction alone)
        st = launch_col<SV, float, SM, 1>(ctx, g, d, cp, ang, volq, tr, corr, meas, first, stride, nv, 0);
        return st != CT_OK ? st : launch_check(ctx, "correction");
    }
    // (only with the column walk does the sweep use the transposed layout)
    if (tr) return fail(ctx, CT_ERR_INVALID_ARG, "transposed correction without the column walk");
    launch_zq<SV, float, SM, 1>(ctx, d, ang, volq, corr, meas, first, stride, nv * d.NS, 0);
    return launch_check(ctx, "correction");
}

template <typename SV>
static ct_status corr_zq_meas(ct_context *ctx, const ct_geometry &g, const void *volq, float *corr, const void *meas,
                              ct_dtype mdt, int first, int stride, int nv, bool tr) {
    switch (mdt) {
    case CT_F32: return run_correction_zq<SV, float>(ctx, g, volq, corr, meas, first, stride, nv, tr);
    case CT_F16: return run_correction_zq<SV, __half>(ctx, g, volq, corr, meas, first, stride, nv, tr);
    case CT_BF16: return run_correction_zq<SV, __hip_bfloat16>(ctx, g, volq, corr, meas, first, stride, nv, tr);
    case CT_F64: return run_correction_zq<SV, double>(ctx, g, volq, corr, meas, first, stride, nv, tr);
    }
    return fail(ctx, CT_ERR_DTYPE, "unsupported measurement dtype");
}

// The sweep's SART correction on a z-quad-layout volume (views first,
// first + stride, ...; the measurement stack is indexed by view).
ct_status launch_correction_zq(ct_context *ctx, const ct_geometry &g, const void *volq, ct_dtype vdt, float *corr,
                               const void *meas, ct_dtype mdt, int32_t first, int32_t stride, int32_t nv, bool tr) {
    if (nv <= 0) return CT_OK;
    switch (vdt) {
    case CT_F32: return corr_zq_meas<float>(ctx, g, volq, corr, meas, mdt, first, stride, nv, tr);
    case CT_F16: return corr_zq_meas<__half>(ctx, g, volq, corr, meas, mdt, first, stride, nv, tr);
    case CT_BF16: return corr_zq_meas<__hip_bfloat16>(ctx, g, volq, corr, meas, mdt, first, stride, nv, tr);
    default: break;
    }
    return fail(ctx, CT_ERR_DTYPE, "z-quad correction: unsupported volume dtype");
}

template <typename SV>
static ct_status planar_corr_meas(ct_context *ctx, const DGeo<float> &d, const float *ang, const void *volz, float *corr,
                                  const void *meas, ct_dtype mdt, int first, int stride, int nv) {
    const int zsh = planar_zshift(d.Z);
    const int cpw = 256 >> zsh, LE = (d.M + d.N + 16) & ~15;
    dim3 grid((d.R + cpw - 1) / cpw, (d.Z + (1 << zsh) - 1) >> zsh, nv);
    const size_t lds = sizeof(uint2) * (size_t)LE * cpw;
    auto go = [&](auto m) {
        using SM = decltype(m);
        hipLaunchKernelGGL((k_planar_corr<SV, SM>), grid, dim3(256), lds, ctx->stream, d, ang, (const SV *)volz, corr,
                           (const SM *)meas, first, stride, zsh);
    };
    switch (mdt) {
    case CT_F32: go(float()); break;
    case CT_F16: go(__half()); break;
    case CT_BF16: go(__hip_bfloat16()); break;
    case CT_F64: go(double()); break;
    }
    return launch_check(ctx, "planar correction");
}

ct_status launch_planar_corr(ct_context *ctx, const ct_geometry &g, const void *volz, ct_dtype vdt, float *corr,
                             const void *meas, ct_dtype mdt, int32_t first, int32_t stride, int32_t nv) {
    if (nv <= 0) return CT_OK;
    ct_status st;
    const float *ang = (const float *)angle_table(ctx, g, false, false, &st);
    if (!ang) return st;
    const DGeo<float> d = derive<float>(g);
    ProfScope ps(ctx, CT_K_FORWARD);
    switch (vdt) {
    case CT_F32: return planar_corr_meas<float>(ctx, d, ang, volz, corr, meas, mdt, first, stride, nv);
    case CT_F16: return planar_corr_meas<__half>(ctx, d, ang, volz, corr, meas, mdt, first, stride, nv);
    default: break;
    }
    return fail(ctx, CT_ERR_DTYPE, "planar correction: unsupported volume dtype");
}

// The sweep walks views whose rays run along y on the transposed z-quad
// layout, so that every view takes the column walk with line-sharing staging.
bool sweep_view_transposed(const ct_geometry &g, ct_dtype vdt, int v, int nv) {
    const DGeo<float> d = derive<float>(g);
    return !col_walk_view(g, v) && sweep_plan(d, vdt, nv * d.NS).nq > 0;
}

ct_status launch_forward(ct_context *ctx, const ct_geometry &g, const void *vol, ct_dtype vdt, void *out,
                         ct_dtype odt, const void *meas, ct_dtype mdt, int32_t first, int32_t stride,
                         int32_t nv, int cmd) {
    return launch_forward_mv(ctx, g, vol, vdt, out, odt, meas, mdt, first, stride, nv, cmd, first);
}

template <typename T, typename SP, typename A>
static ct_status run_adjoint(ct_context *ctx, const ct_geometry &g, const void *proj, A *acc, int view0, int nv) {
    ct_status st;
    const T *ang = (const T *)angle_table(ctx, g, sizeof(T) == 8, false, &st);
    if (!ang) return st;
    DGeo<T> d = derive<T>(g);
    const int nimg = nv * d.NS;
    dim3 block(256);
    ProfScope ps(ctx, CT_K_ADJOINT);
    for (int z0 = 0; z0 < nimg; z0 += 65535) {
        int nz = nimg - z0 < 65535 ? nimg - z0 : 65535;
        dim3 grid((d.R + 15) / 16, (d.ZP + 15) / 16, nz);
        // the fast forward's walk in fast mode, so the pair stays matched; the
        // accumulator is then in the z-quad layout (neighbouring rays' atomics
        // share cache lines)
        if (std::is_same<T, float>::value && ctx->math == CT_MATH_FAST)
            hipLaunchKernelGGL((k_adjoint<T, SP, A, std::is_same<T, float>::value, true>), grid, block, 0,
                               ctx->stream, d, ang, (const SP *)proj, acc, view0, z0);
        else
            hipLaunchKernelGGL((k_adjoint<T, SP, A, false>), grid, block, 0, ctx->stream, d, ang, (const SP *)proj,
                               acc, view0, z0);
    }
    return launch_check(ctx, "adjoint");
}

// Parts the gather's views are split into: enough workgroups for four per CU
// (what the kernel's registers admit) where the tiles alone give fewer.  Under
// eight images a workgroup is done with them sooner than another launch starts.
static int adj_parts(const DGeo<float> &d, int nv) {
    const int64_t tiles = (int64_t)((d.M + 15) / 16) * ((d.N + 15) / 16) * ((d.Z + AZR - 1) / AZR);
    if (tiles >= 512 || nv < 2 || nv * d.NS < 8) return 1;
    const int64_t want = std::min<int64_t>((1024 + tiles - 1) / tiles, nv);
    const int64_t vpp = (nv + want - 1) / want;
    return (int)((nv + vpp - 1) / vpp);
}

template <typename SO>
static void launch_gather(ct_context *ctx, const DGeo<float> &d, const float *ang, int view0, int nv, int parts,
                          const float *pixw, const AdjCol *colT, const float4 *rowT, void *vol, float2 *part) {
    dim3 grid((d.M + 15) / 16, (d.N + 15) / 16, (d.Z + AZR - 1) / AZR * parts);
    if (parts == 1) {
        hipLaunchKernelGGL((k_adjoint_gather<SO, false>), grid, dim3(16, 16, 1), 0, ctx->stream, d, ang, view0, nv, nv,
                           pixw, colT, rowT, (SO *)vol, part);
        return;
    }
    hipLaunchKernelGGL((k_adjoint_gather<SO, true>), grid, dim3(16, 16, 1), 0, ctx->stream, d, ang, view0, nv,
                       (nv + parts - 1) / parts, pixw, colT, rowT, (SO *)vol, part);
    const int64_t V = (int64_t)d.M * d.N * d.Z;
    hipLaunchKernelGGL((k_adj_fold<SO>), dim3((unsigned)((V + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const float2 *)part, parts, V, (SO *)vol);
}

static ct_status run_adjoint_gather(ct_context *ctx, const ct_geometry &g, const DGeo<float> &d, const void *proj,
                                    ct_dtype pdt, void *vol, ct_dtype vdt, int view0, int nv) {
    ct_status st;
    const float *ang = (const float *)angle_table(ctx, g, false, false, &st);
    if (!ang) return st;
    const int nimg = nv * d.NS;
    const size_t P = (size_t)d.R * d.ZP;
    int parts = adj_parts(d, nv);
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t pw_b = up(sizeof(float) * P * nimg), col_b = up(sizeof(AdjCol) * (size_t)d.R * nv);
    const size_t row_b = up(sizeof(float4) * (size_t)d.ZP * nimg);
    const size_t part_b = parts > 1 ? sizeof(float2) * (size_t)d.M * d.N * d.Z * parts : 0;
    char *tab = parts > 1 ? (char *)slot_or_null(ctx, SLOT_TMP_VOL, pw_b + col_b + row_b + part_b) : nullptr;
    if (!tab) {   // in one part if it has to be
        parts = 1;
        tab = (char *)slot(ctx, SLOT_TMP_VOL, pw_b + col_b + row_b, &st);
        if (!tab) return st;
    }
    float *pixw = (float *)tab;
    AdjCol *colT = (AdjCol *)(tab + pw_b);
    float4 *rowT = (float4 *)(tab + pw_b + col_b);
    float2 *part = (float2 *)(tab + pw_b + col_b + row_b);
    ProfScope ps(ctx, CT_K_ADJOINT);
    dim3 pg((d.R + 255) / 256, d.ZP, nimg);
    switch (pdt) {
    case CT_F32: hipLaunchKernelGGL((k_adj_prep<float>), pg, dim3(256), 0, ctx->stream, d, ang, view0, (const float *)proj, nimg, pixw, colT, rowT); break;
    case CT_F16: hipLaunchKernelGGL((k_adj_prep<__half>), pg, dim3(256), 0, ctx->stream, d, ang, view0, (const __half *)proj, nimg, pixw, colT, rowT); break;
    case CT_BF16: hipLaunchKernelGGL((k_adj_prep<__hip_bfloat16>), pg, dim3(256), 0, ctx->stream, d, ang, view0, (const __hip_bfloat16 *)proj, nimg, pixw, colT, rowT); break;
    default: return fail(ctx, CT_ERR_DTYPE, "unsupported projection dtype");
    }
    switch (vdt) {
    case CT_F32: launch_gather<float>(ctx, d, ang, view0, nv, parts, pixw, colT, rowT, vol, part); break;
    case CT_F16: launch_gather<__half>(ctx, d, ang, view0, nv, parts, pixw, colT, rowT, vol, part); break;
    case CT_BF16: launch_gather<__hip_bfloat16>(ctx, d, ang, view0, nv, parts, pixw, colT, rowT, vol, part); break;
    default: return fail(ctx, CT_ERR_DTYPE, "unsupported volume dtype");
    }
    return launch_check(ctx, "adjoint");
}

ct_status launch_adjoint(ct_context *ctx, const ct_geometry &g, const void *proj, ct_dtype pdt, void *vol,
                         ct_dtype vdt, int32_t view0, int32_t nv) {
    const int64_t V = (int64_t)g.nx * g.ny * g.nz;
    if (vdt == CT_F64) {
        if (pdt != CT_F64) return fail(ctx, CT_ERR_DTYPE, "F64 volume needs F64 projections");
        ct_status st = launch_fill(ctx, vol, CT_F64, V, 0.0);
        if (st != CT_OK) return st;
        return run_adjoint<double, double, double>(ctx, g, proj, (double *)vol, view0, nv);
    }
    if (pdt == CT_F64) return fail(ctx, CT_ERR_DTYPE, "F64 projections need an F64 volume");
    // FP32 segments scattered into an FP64 accumulator (f64 atomics): the
    // ~10^2 contributions per voxel are summed without FP32 rounding, then
    // rounded once to the output type.  Fast mode accumulates in the z-quad
    // layout and unpacks while converting.
    const bool zq = ctx->math == CT_MATH_FAST;
    if (zq) {
        // gather form: the walk's segments summed per voxel, no atomics
        const DGeo<float> d = derive<float>(g);
        const int nimg = nv * d.NS;
        if (nimg <= 65535 && adj_gather_fits(d)) return run_adjoint_gather(ctx, g, d, proj, pdt, vol, vdt, view0, nv);
    }
    const int64_t Va = zq ? (int64_t)g.nx * g.ny * ((g.nz + 3) & ~3) : V;
    ct_status st;
    double *acc = (double *)slot(ctx, SLOT_TMP_VOL, sizeof(double) * Va, &st);
    if (!acc) return st;
    st = launch_fill(ctx, acc, CT_F64, Va, 0.0);
    if (st != CT_OK) return st;
    switch (pdt) {
    case CT_F32: st = run_adjoint<float, float, double>(ctx, g, proj, acc, view0, nv); break;
    case CT_F16: st = run_adjoint<float, __half, double>(ctx, g, proj, acc, view0, nv); break;
    case CT_BF16: st = run_adjoint<float, __hip_bfloat16, double>(ctx, g, proj, acc, view0, nv); break;
    default: return fail(ctx, CT_ERR_DTYPE, "unsupported projection dtype");
    }
    if (st != CT_OK) return st;
    if (zq) return launch_zq_unpack_f64(ctx, acc, vol, vdt, g.nx, g.ny, g.nz);
    return launch_convert(ctx, acc, CT_F64, vol, vdt, V);
}

} // namespace ct
