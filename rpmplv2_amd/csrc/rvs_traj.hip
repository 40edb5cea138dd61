// Trajectory safety kernel (gfx950): AbstractTrajectory::isSafe
// (src/planners/trajectory/AbstractTrajectory.cpp:212-256) for a batch of
// candidate trajectories that leave one current state, one wave per
// trajectory.
//
// Along the trajectory points the lane keeps a reference state q_temp with a
// distance profile (first the current state's, from computeDistance).  A
// point is accepted while, for every skeleton point j, the distance it can
// cover from q_temp (enclosing radii R.col(j) . |q - q_temp|) plus the
// distance the obstacles can cover since q_temp's profile was taken
// (max_obs_vel * elapsed time) stays below the link's clearance.  Otherwise
// the point becomes the new q_temp and gets a fresh profile from the
// moving-plane underestimation (planes through the current state's nearest
// points, moved towards the robot for the elapsed time at each obstacle's
// maximal speed); a non-positive result makes the trajectory unsafe.
// Optionally every point is also tested for self-collision (capsule pairs).
//
// No FMA contraction anywhere in this translation unit, headers included:
// the float arithmetic must keep the reference's rounding.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "rvs_fk.hpp"
#include "rvs_geometry.hpp"
#include "rvs_internal.hpp"
#include "rvs_radii.hpp"
#include "rvs_stage.hpp"

namespace rvs {

namespace {

// LDS of one workgroup (one wave, one trajectory): the reference state (D),
// its profile (L = D), its skeleton 3 (D+1) and its radii D (D+1), in floats;
// then a skeleton slice per lane for the self-collision test, 64 x 3 (D+1)
// floats, whose place the walk takes over: segment poses, skeleton recipe,
// every lane's joint distances to the reference state (D x 64 floats) and the
// points' times.
constexpr int kTrajTimes = 1024;   // points with a time in the table
__host__ __device__ inline size_t traj_walk_off(int D) {
    return ((size_t)(2 * D + 3 * (D + 1) + D * (D + 1)) * sizeof(float) + 15) & ~size_t(15);
}
__host__ __device__ inline size_t traj_walk_bytes(const RobotDev& rb, int times) {
    return (size_t)96 * rb.num_segments + sizeof(PointDev) * (rb.num_links + 1) + (size_t)256 * rb.num_dofs +
           4 * (size_t)times;
}

// One wave per trajectory.  The bubble test of a point only reads the
// reference state, so the wave tests 64 points at once and re-anchors at
// the first point that fails; the lanes share the new reference state's work:
// segment poses and frame rows (skeleton_row), a row of radii each, and the
// moving-plane underestimation, a (link, obstacle) pair each.  The outcome is
// the reference's sequential walk: a point is tested against the reference
// state the walk would hold there, a minimum of floats is exact in any order,
// and any term that is not positive ends the walk as unsafe whichever comes
// first (a negative one returns early, a zero leaves a distance of 0).
// Self-collision of any point makes the trajectory unsafe, as the walk would
// stop there or earlier; pairs whose bounding boxes are farther apart than
// their radii (apart_bound2) skip the segment-segment test.
// Bound by latency (a chain of short steps per re-anchoring).  8,192 xArm6
// trajectories of 60 points, 16 boxes: 0.35 ms (1.04 ms with the reference
// state's kinematics and radii in lane 0).
__global__ __launch_bounds__(64) void k_traj_safe(RobotDev rb, QueryParams qp, TrajArgs a, int64_t T) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int D = rb.num_dofs, L = rb.num_links;
    const int t = threadIdx.x;
    const int64_t c = blockIdx.x;
    if (c >= T) return;   // uniform across the workgroup
    const int M = a.num_obj, K = a.num_points;
    float* qa = reinterpret_cast<float*>(smem);          // [D]
    float* pr = qa + D;                                   // [L]
    float* ska = pr + L;                                  // [3 (D+1)]
    float* Rm = ska + 3 * (D + 1);                        // [D][D+1]
    unsigned char* const area = smem + traj_walk_off(D);
    float* skl = reinterpret_cast<float*>(area);          // [3 (D+1)][64]
    double* segs = reinterpret_cast<double*>(area);       // [S][12], the walk's part of the area
    PointDev* pts = reinterpret_cast<PointDev*>(segs + 12 * rb.num_segments);   // [L + 1]
    float* dq = reinterpret_cast<float*>(pts + L + 1);    // [D][64]
    float* times = dq + 64 * D;                           // [K], K <= kTrajTimes
    const bool table = K <= kTrajTimes;
    const Params<float> p{qp.eq, qp.maxd};
    const float* points = a.points + c * (int64_t)K * D;
    auto PA = [&](int k) { return Vec3<float>{ska[3 * k], ska[3 * k + 1], ska[3 * k + 2]}; };
    auto PL = [&](int k) { return Vec3<float>{skl[(3 * k) * 64 + t], skl[(3 * k + 1) * 64 + t], skl[(3 * k + 2) * 64 + t]}; };
    float max_obs_vel = 0.0f;   // AbstractTrajectory.cpp:44-49
    for (int o = t; o < M; o += 64)
        if (a.max_vel[o] > max_obs_vel) max_obs_vel = a.max_vel[o];
    for (int o = 32; o > 0; o >>= 1) max_obs_vel = max_std(max_obs_vel, __shfl_xor(max_obs_vel, o, 64));

    bool unsafe = false;
    // robot->checkSelfCollision(q_final) at every point: capsule pairs
    if (a.self_collision && rb.num_pairs > 0) {
        bool hit = false;
        for (int i = t; i < K; i += 64) {
            float cmax = 0.0f, csum = 0.0f;
            FKStream fk;
            fk_init(fk);
            for (int k = 0; k <= D; ++k) {
                const Vec3<float> v = skel_point<float>(fk, rb, points + (int64_t)i * D, k);
                skl[(3 * k) * 64 + t] = v.x;
                skl[(3 * k + 1) * 64 + t] = v.y;
                skl[(3 * k + 2) * 64 + t] = v.z;
                cmax = fmaxf(cmax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fabsf(v.z)));
                csum = csum + ((v.x + v.y) + v.z);
            }
            if (!(csum == csum)) cmax = NAN;
            for (int m = 0; m < rb.num_pairs; ++m) {
                const int u = rb.pairs[2 * m], w = rb.pairs[2 * m + 1];
                const Vec3<float> A = PL(u), B = PL(u + 1), C = PL(w), E = PL(w + 1);
                const float ru = rb.radius[u], rw = rb.radius[w];
                if (boxes_gap2(SegBox(A, B), SegBox(C, E)) > apart_bound2(ru + rw, 0.0f, cmax, p)) continue;
                if (seg_seg<float, false>(A, B, C, E, p, nullptr) - ru - rw < 0.0f) hit = true;
            }
        }
        unsafe = __any(hit);
    }
    __syncthreads();   // the skeleton slices are free
    for (int k = t; k <= L; k += 64) pts[k] = rb.pts[k];
    for (int k = t; k < D; k += 64) qa[k] = a.q_current[k];
    for (int k = t; k < L; k += 64) pr[k] = a.profile_current[k];
    if (table) {
        float ti = a.t_iter;
        for (int k = 0; k < K; ++k) {
            if ((k & 63) == t) times[k] = ti;
            ti += a.time_step;
        }
    }
    __syncthreads();
    // skeleton of the reference state
    auto anchor = [&]() {
        for (int m = t; m < rb.num_segments; m += 64) seg_pose_store(segs + 12 * m, rb.seg[m], qa);
        wave_sync();
        skeleton_row(segs, pts, L, t < 3 ? t : 0, ska, t < 3);
        wave_sync();
    };
    if (!unsafe) anchor();
    float t_init = 0.0f;
    int s = 0;
    float ts = a.t_iter;   // time at point s
    while (!unsafe) {
        // radii of the reference state, a row a lane (D <= 64 rows)
        if (t < D) {
            float acc = 0.0f;
            Rm[t * (D + 1)] = 0.0f;
            for (int j = 1; j <= D; ++j) {
                float v;
                if (t < j && radii_distance(rb, PA, t, j, PA(j), v)) acc = max_std(acc, v + rb.rad_enc[j - 1]);
                Rm[t * (D + 1) + j] = acc;
            }
        }
        wave_sync();
        int f = K;
        float tf = 0.0f;   // time at point f
        float tb = ts;     // time at the chunk's first point
        for (int b = s; b < K; b += 64) {
            const int i = b + t;
            bool fail = false;
            // time at point i: t_iter + time_step added i times, in order;
            // without the table the additions go on from the chunk before
            // (from t_iter each time a trajectory of 10,000 points took 20 ms
            // instead of 0.8)
            float ti = tb;
            if (table) {
                if (i < K) ti = times[i];
            } else {
                for (int k = 0; k < t; ++k) ti += a.time_step;
                tb = __shfl(ti, 63) + a.time_step;
            }
            if (i < K) {
                const float* qf = points + (int64_t)i * D;
                const float rho_obs = max_obs_vel * (ti - t_init);
                for (int k = 0; k < D; ++k) dq[k * 64 + t] = fabsf(qf[k] - qa[k]);
                for (int j = 0; j < D && !fail; ++j) {
                    const float rho_robot =
                        eigen_dyn_sum([&](int k) { return Rm[k * (D + 1) + j + 1] * dq[k * 64 + t]; }, D);
                    if (rho_robot + rho_obs >= pr[j]) fail = true;
                }
            }
            const uint64_t m = __ballot(fail);
            if (m) {
                const int lane = __ffsll((unsigned long long)m) - 1;
                f = b + lane;
                tf = __shfl(ti, lane);
                break;
            }
        }
        if (f >= K) break;   // every remaining point inside the bubble
        // possible collision at point f: it becomes the reference state
        wave_sync();
        for (int k = t; k < D; k += 64) qa[k] = points[(int64_t)f * D + k];
        for (int l = t; l < L; l += 64) pr[l] = qp.maxd;
        wave_sync();
        anchor();
        bool bad = qp.maxd <= 0.0f;   // some term, or the distance without any, is not positive
        for (int k = t; k < L * M; k += 64) {
            const int o = k / L, l = k - o * L;
            const float* e = a.nearest_current + (int64_t)k * 6;
            const Vec3<float> O{e[3], e[4], e[5]};
            if (vnorm(O) == qp.maxd) continue;
            const Vec3<float> R{e[0], e[1], e[2]};
            const float tm = plane_term_moving(PA(l), PA(l + 1), R, O, rb.radius[l], a.max_vel[o], tf);
            if (tm <= 0.0f) bad = true;
            else if (tm < qp.maxd) atomicMin(reinterpret_cast<uint32_t*>(pr) + l, __float_as_uint(tm));   // positive floats order as their bits
        }
        if (__any(bad)) unsafe = true;
        t_init = tf;
        s = f + 1;
        ts = tf + a.time_step;
        wave_sync();
    }
    if (t == 0) a.safe[c] = unsafe ? 0 : 1;
}

}  // namespace

size_t traj_lds_bytes(const RobotDev& rb) {
    const size_t slices = (size_t)64 * 3 * (rb.num_dofs + 1) * sizeof(float);
    return traj_walk_off(rb.num_dofs) + std::max(slices, traj_walk_bytes(rb, 0));
}

hipError_t launch_traj_safe(const RobotDev& rb, const QueryParams& qp, const TrajArgs& a, int64_t T, hipStream_t st) {
    if (T <= 0) return hipSuccess;
    const size_t sm = std::max(traj_lds_bytes(rb), traj_walk_off(rb.num_dofs) +
                                                       traj_walk_bytes(rb, a.num_points <= kTrajTimes ? a.num_points : 0));
    hipLaunchKernelGGL(k_traj_safe, dim3((unsigned)T), dim3(64), sm, st, rb, qp, a, T);
    return hipGetLastError();
}

}  // namespace rvs
