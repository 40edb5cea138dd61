// Device helpers shared by the kernel files: obstacle staging in LDS,
// oriented-box frame changes and per-link constants.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rvs_geometry.hpp"
#include "rvs_internal.hpp"

namespace rvs {

// LDS image of an obstacle set:
//   xf   [M][12]  centre, rotation rows (oriented boxes only; 16-byte aligned)
//   box  [M]      AABB, or [-h, h] in the box frame for oriented boxes
//   tol  [M]      min_dist_tol
//   gnd  [M]      ground flag
template <typename T>
struct Staged {
    const float* xf;
    Box<T>* box;
    T* tol;
    uint8_t* gnd;
    bool obb;
};

template <typename T>
__host__ __device__ inline size_t staged_bytes(const EnvDev& env) {
    const size_t M = (size_t)env.num_obj;
    return M * ((env.use_obb ? 12 * sizeof(float) : 0) + sizeof(Box<T>) + sizeof(T) + 1);
}

// Copy the obstacle set into LDS (whole workgroup participates).  OBB is a
// compile-time choice so that the axis-aligned kernels keep a constant layout;
// it must equal env.use_obb.
template <typename T, bool OBB>
__device__ inline Staged<T> stage_env(const EnvDev& env, unsigned char* smem) {
    const int M = env.num_obj;
    constexpr bool obb = OBB;
    float* xf = reinterpret_cast<float*>(smem);
    Staged<T> s;
    s.xf = xf;
    s.box = reinterpret_cast<Box<T>*>(smem + (obb ? (size_t)M * 12 * sizeof(float) : 0));
    s.tol = reinterpret_cast<T*>(s.box + M);
    s.gnd = reinterpret_cast<uint8_t*>(s.tol + M);
    s.obb = obb;
    for (int j = threadIdx.x; j < M; j += blockDim.x) {
        Box<T> b;
        if (obb) {
            const float* o = env.obb + 15 * j;
#pragma unroll
            for (int k = 0; k < 12; ++k) xf[12 * j + k] = o[k];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b.lo[k] = -(T)o[12 + k];
                b.hi[k] = (T)o[12 + k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b.lo[k] = (T)env.aabb[6 * j + k];
                b.hi[k] = (T)env.aabb[6 * j + 3 + k];
            }
        }
        s.box[j] = b;
        s.tol[j] = (T)env.tol[j];
        s.gnd[j] = env.flags[j] & kObjGround;
    }
    __syncthreads();
    return s;
}

// World point -> box frame: local_k = R[0][k] (x - c_x) + R[1][k] (y - c_y)
// + R[2][k] (z - c_z), summed left to right (x = centre, rotation rows).
template <typename T>
__device__ __attribute__((always_inline)) inline Vec3<T> to_box(const float* x, const Vec3<T>& P) {
    const T vx = P.x - (T)x[0], vy = P.y - (T)x[1], vz = P.z - (T)x[2];
    return Vec3<T>{(T)x[3] * vx + (T)x[6] * vy + (T)x[9] * vz, (T)x[4] * vx + (T)x[7] * vy + (T)x[10] * vz,
                   (T)x[5] * vx + (T)x[8] * vy + (T)x[11] * vz};
}

// Box frame -> world: c_i + (R[i][0] l_0 + R[i][1] l_1 + R[i][2] l_2).
template <typename T>
__device__ __attribute__((always_inline)) inline Vec3<T> from_box(const float* x, const Vec3<T>& l) {
    return Vec3<T>{(T)x[0] + ((T)x[3] * l.x + (T)x[4] * l.y + (T)x[5] * l.z),
                   (T)x[1] + ((T)x[6] * l.x + (T)x[7] * l.y + (T)x[8] * l.z),
                   (T)x[2] + ((T)x[9] * l.x + (T)x[10] * l.y + (T)x[11] * l.z)};
}

// Broad phase.  The distance the case tree returns for a (capsule, box) pair
// is at least the raw segment-box distance minus r, except for its snaps to
// 0 / -r, which need a raw distance below EQUALITY_THRESHOLD (or contact).
// The gap between the segment's bounding box [slo, shi] and a box containing
// the obstacle (cb = lo[3], hi[3]) is a lower bound of the raw distance, so a
// pair whose gap exceeds max(running link minimum + r, EQUALITY_THRESHOLD)
// plus a margin that covers float rounding can neither lower the link's
// minimum nor end the loop: skipping it leaves every result unchanged.
// Compares squared values (no square root); a NaN end point never culls.
constexpr float kCullMargin = 1e-5f;

// Orders the LDS accesses of a wave's lanes (LDS that one wave alone uses).
__device__ __attribute__((always_inline)) inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Squared gap between the segment's bounding box and the box cb (0 on an
// axis where they overlap or a coordinate is NaN).
template <typename T>
__device__ __attribute__((always_inline)) inline T gap_squared(const float* __restrict__ cb, const Vec3<T>& slo,
                                                               const Vec3<T>& shi) {
    T g2 = T(0);
    {
        T g = (T)cb[0] - shi.x;
        const T g1 = slo.x - (T)cb[3];
        g = g1 > g ? g1 : g;
        g2 = g > T(0) ? g * g : T(0);
    }
    {
        T g = (T)cb[1] - shi.y;
        const T g1 = slo.y - (T)cb[4];
        g = g1 > g ? g1 : g;
        g2 = g > T(0) ? g2 + g * g : g2;
    }
    {
        T g = (T)cb[2] - shi.z;
        const T g1 = slo.z - (T)cb[5];
        g = g1 > g ? g1 : g;
        g2 = g > T(0) ? g2 + g * g : g2;
    }
    return g2;
}

template <typename T>
__device__ __attribute__((always_inline)) inline bool cull_pair(const float* __restrict__ cb, const Vec3<T>& slo,
                                                                 const Vec3<T>& shi, T bound) {
    return gap_squared(cb, slo, shi) > bound * bound;
}

template <typename T>
__device__ __attribute__((always_inline)) inline T cull_bound(T prof, T r, T eq) {
    const T a = prof + r;
    return (a > eq ? a : eq) + (T)kCullMargin;
}

template <typename T>
__device__ __attribute__((always_inline)) inline void seg_bounds(const Vec3<T>& A, const Vec3<T>& B, Vec3<T>& lo,
                                                                 Vec3<T>& hi) {
    lo = Vec3<T>{A.x < B.x ? A.x : B.x, A.y < B.y ? A.y : B.y, A.z < B.z ? A.z : B.z};
    hi = Vec3<T>{A.x < B.x ? B.x : A.x, A.y < B.y ? B.y : A.y, A.z < B.z ? B.z : A.z};
}

// The planes of one nearest-point set ([M][L][6], RealVectorSpace.cpp:402-446)
// in LDS, links i0 .. i1 - 1 as [i1 - i0][M]: O and the unit normal of each
// (obstacle, link) pair, worked out by the threads of the workgroup (all of
// them call; the caller synchronizes before the planes are read and before
// they are staged again).  A pair the reference skips (|O| = maxd) gets a NaN
// normal: its term is NaN and never enters a minimum.  With max_vel [M] the
// planes first move towards the robot for delta_t.
struct alignas(16) Plane {
    Vec3<float> O;
    float nx, ny, nz;
    float pad[2];
};
static_assert(sizeof(Plane) == 32, "two 16-byte LDS reads per plane");

__device__ inline void stage_planes(Plane* planes, const float* __restrict__ set, int M, int L, int i0, int i1,
                                    float maxd, const float* __restrict__ max_vel, float delta_t) {
    for (int k = threadIdx.x; k < (i1 - i0) * M; k += blockDim.x) {
        const int i = i0 + k / M, j = k % M;
        const float* e = set + ((int64_t)j * L + i) * 6;
        Vec3<float> R{e[0], e[1], e[2]}, O{e[3], e[4], e[5]};
        const bool skip = vnorm(O) == maxd;
        if (max_vel) plane_move(R, O, max_vel[j], delta_t);
        const Vec3<float> nv = plane_normal(R, O);
        planes[k] = Plane{O, skip ? NAN : nv.x, skip ? NAN : nv.y, skip ? NAN : nv.z, {0.0f, 0.0f}};
    }
}

// Smallest term of one link (P0, P1) over its row of M staged planes, from
// infinity: its sign alone says whether any term was negative, and
// MAX_DISTANCE, the start of the reference's minimum, enters afterwards.
__device__ __attribute__((always_inline)) inline float planes_min(const Plane* row, int M, const Vec3<float>& P0,
                                                                  const Vec3<float>& P1, float r) {
    float low = INFINITY;
#pragma unroll 2
    for (int j = 0; j < M; ++j) {
        const Plane pl = row[j];
        low = smin(low, plane_value(P0, P1, pl.O, Vec3<float>{pl.nx, pl.ny, pl.nz}, r));
    }
    return low;
}

// Entry k of the refinement's work: configuration c and the first link to
// recompute, k0 (entry k itself and k0 = 0 for a direct call, idx null; k0
// = 0 too without a profile, which holds the values of the links before it).
__device__ __attribute__((always_inline)) inline void flag_decode(const int32_t* idx, int64_t k, const QueryParams& qp,
                                                                  const DistOut& out, int64_t& c, int& k0) {
    if (!idx) {
        c = k;
        k0 = 0;
        return;
    }
    const int64_t e = (int64_t)idx[k];
    if (qp.flag_link) {
        c = e & (((int64_t)1 << kFlagLinkShift) - 1);
        k0 = out.profile ? (int)(e >> kFlagLinkShift) : 0;
    } else {
        c = e;
        k0 = 0;
    }
}

// Bound of a self pair's computed distance by the bounding boxes of its
// segments.  distanceLineSegToLineSeg (CollisionAndDistance.cpp:217-320)
// returns 0 (below the equality threshold eq), max_distance (degenerate
// input), or the float norm of p1 - p0 for points that are end points or
// a + o (b - a) with o in [0, 1], each within 5 eps C of its segment
// (eps = 2^-24, C the largest coordinate magnitude), so the returned distance
// is at least (D - 21 eps C)(1 - 2 eps) with D the distance of the two
// segments' bounding boxes.  A D, computed in float, above
// R = max(lo + r_a + r_b, eq) by 4e-6 (C + R) (about 67 eps (C + R), which also
// covers the rounding of D and of the radii's subtraction) therefore leaves
// it at lo + r_a + r_b or more, provided max_distance is at least that bound.
// apart_bound2 is the square of that bound (infinite when max_distance is
// smaller, NaN when cmax is: nothing is ruled out then); a pair whose
// boxes_gap2 exceeds it has a capsule distance of at least lo.
__device__ __attribute__((always_inline)) inline float apart_bound2(float rsum, float lo, float cmax,
                                                                    const Params<float>& p) {
    const float R = fmaxf(lo + rsum, p.eq);
    const float thr = R + 4e-6f * (cmax + R);
    return thr <= p.maxd ? thr * thr : (thr == thr ? INFINITY : NAN);
}
struct SegBox {
    float lx, ly, lz, hx, hy, hz;
    __device__ SegBox(const Vec3<float>& A, const Vec3<float>& B)
        : lx(fminf(A.x, B.x)), ly(fminf(A.y, B.y)), lz(fminf(A.z, B.z)),
          hx(fmaxf(A.x, B.x)), hy(fmaxf(A.y, B.y)), hz(fmaxf(A.z, B.z)) {}
};
__device__ __attribute__((always_inline)) inline float boxes_gap2(const SegBox& a, const SegBox& c) {
    const float gx = fmaxf(fmaxf(c.lx - a.hx, a.lx - c.hx), 0.0f);
    const float gy = fmaxf(fmaxf(c.ly - a.hy, a.ly - c.hy), 0.0f);
    const float gz = fmaxf(fmaxf(c.lz - a.hz, a.lz - c.hz), 0.0f);
    return __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
}

template <typename T> __device__ inline T rnew_of(const RobotDev& rb, int i);
template <> __device__ inline float rnew_of<float>(const RobotDev& rb, int i) { return rb.rnew32[i]; }
template <> __device__ inline double rnew_of<double>(const RobotDev& rb, int i) { return rb.rnew64[i]; }

}  // namespace rvs
