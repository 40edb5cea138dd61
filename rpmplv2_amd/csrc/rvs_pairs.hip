// Reference-arithmetic distances by pairs (gfx950): k_distance_pairs, the
// low-latency form of computeDistance (RealVectorSpace.cpp:318-392) for small
// batches and for the configurations that the FP32 bulk pass flags.
//
// No FMA contraction anywhere in this translation unit, headers included:
// the float kernels must keep the reference's rounding.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "rvs_fk.hpp"
#include "rvs_geometry.hpp"
#include "rvs_internal.hpp"
#include "rvs_stage.hpp"

namespace rvs {

namespace {

// A configuration's row of LDS: the segments' rotations and origins, the
// nearest pair (squared gap, obstacle) and the first hit (obstacle, value) of
// every link, the skeleton, the links' smallest positive values, broad-phase
// bounds and the first link with a hit, and every pair's squared gap.
struct PairRow {
    double* seg;                    // [S][12] rotation (row major), origin
    unsigned long long* near_key;   // [L] squared gap bits << 32 | obstacle
    unsigned long long* hit_key;    // [L] obstacle << 32 | value bits; ~0 none
    float* skel;                    // [L + 1][3]
    uint32_t* low;                  // [L] bits of the smallest positive value
    float* bound2;                  // [L] square of the broad-phase bound
    int* first_link;
    float* gap2;                    // [L][M]
    __device__ PairRow(unsigned char* p, int S, int L) {
        seg = reinterpret_cast<double*>(p);
        near_key = reinterpret_cast<unsigned long long*>(seg + 12 * S);
        hit_key = near_key + L;
        skel = reinterpret_cast<float*>(hit_key + L);
        low = reinterpret_cast<uint32_t*>(skel + 3 * (L + 1));
        bound2 = reinterpret_cast<float*>(low + L);
        first_link = reinterpret_cast<int*>(bound2 + L);
        gap2 = reinterpret_cast<float*>(first_link + 1);
    }
};
// Rows are an odd number of 16-byte pieces apart, so that the groups of a
// wave, which read the same place of their rows together, hit different banks.
inline size_t pair_row_bytes(int S, int L, int M) {
    const size_t b = 96 * (size_t)S + 16 * (size_t)L + 12 * (size_t)(L + 1) + 8 * (size_t)L + 4 + 4 * (size_t)L * M;
    return ((b + 15) / 16 | 1) * 16;
}
// The wave's queue of pairs to evaluate: group << 16 | link << 10 | obstacle.
// Room for a nearest pair of each link (64) of each group (4) and one more
// step of the scan.
constexpr int kPairQueue = 320;

// The workgroup's LDS after the staged obstacles: the skeleton recipe, the
// radii, the queue, the rows.
struct PairLds {
    size_t pts, rad, queue, rows, row, total;
};
inline PairLds pair_lds(const RobotDev& rb, const EnvDev& env, bool want_np, int groups) {
    auto up = [](size_t b) { return (b + 15) & ~size_t(15); };
    PairLds l;
    l.pts = up(staged_bytes<float>(env));
    l.rad = l.pts + (size_t)(rb.num_links + 1) * sizeof(PointDev);
    l.queue = up(l.rad + 4 * (size_t)rb.num_links);
    l.rows = l.queue + (want_np ? 0 : 4 * kPairQueue);
    l.row = pair_row_bytes(rb.num_segments, rb.num_links, want_np ? 0 : env.num_obj);
    l.total = l.rows + groups * l.row;
    return l;
}

// G lanes per configuration (16 or 64), 64 / G configurations per wave; a
// workgroup is one wave.
//   1. Lane m of the group works out segment m's rotation (and m + G's, ...),
//      the same double operations as the serial stream, so the same bits.
//   2. The frames' product is a chain over the segments, but row by row: lane
//      r of the group carries row r of the frame and coordinate r of its
//      origin, 21 operations a segment instead of 133.
//   3. Without nearest points, the pair of each link with the smallest gap
//      between the segment's bounding box and the obstacle's cull box is
//      evaluated first; its value bounds the link's minimum.
//   4. The pairs that the broad phase does not rule out with that bound
//      (cull_pair's rule; a link with a hit takes the bound of a minimum of
//      0, which never skips a pair whose distance can be <= 0), of the links up
//      to the first with a hit so far, are queued, all of the wave's
//      configurations together, and evaluated one a lane.
//   5. The values meet in the rows by atomics: the smallest positive value of
//      each link, and the smallest obstacle index with a value <= 0.
// That gives what the reference's loop gives: its running minimum starts at
// MAX_DISTANCE, so a NaN distance never enters it, and it stops at the first
// pair in obstacle order whose minimum is <= 0, which is then the link's
// value; a minimum of floats is exact in any order, and a skipped pair can
// neither lower it nor end the loop.  With nearest points every pair is
// evaluated and its points stored (NaN for all when any pair hits).
//
// Bound by the latency of a wave's chain of steps (a batch of 16 fills 4 of
// the 1,024 SIMDs) and by the divergence of the case tree: a wave pays for
// every case that any of its lanes meets, so the fewer, fuller evaluation
// steps the better.  xArm6 and 17 boxes, a call: 1 configuration 24 us, 4,096
// 44 us, 16,384 60 us (one wave per configuration with every pair evaluated:
// 30, 60 and 121 us; the serial kinematics alone took 13,000 of a wave's 39,000
// cycles, now 6,000), one state with its nearest points 75 us from copied host
// arrays (90 us with a link at a time) and 30 us in place.  The times of both
// widths stand at launch_distance_pairs.
template <bool OBB, bool WANT_NP, int G>
__global__ __launch_bounds__(64) void k_distance_pairs(RobotDev rb, EnvDev env, QueryParams qp,
                                                       const float* __restrict__ q, DistOut out,
                                                       const int32_t* __restrict__ idx,
                                                       const uint32_t* __restrict__ count, int64_t n_direct,
                                                       uint32_t* count_out, PairLds lds) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kGroups = 64 / G;   // configurations of a wave
    const int64_t total = idx ? (int64_t)*count : n_direct;
    if (count_out && blockIdx.x == 0 && threadIdx.x == 0) *count_out = (uint32_t)total;
    if ((int64_t)blockIdx.x * kGroups >= total) return;   // uniform over the workgroup
    const int M = env.num_obj, L = rb.num_links, D = rb.num_dofs, S = rb.num_segments;
    const int lane = threadIdx.x;
    PointDev* const pts = reinterpret_cast<PointDev*>(smem + lds.pts);
    float* const rad = reinterpret_cast<float*>(smem + lds.rad);
    uint32_t* const queue = reinterpret_cast<uint32_t*>(smem + lds.queue);
    for (int k = lane; k <= L; k += 64) pts[k] = rb.pts[k];
    for (int k = lane; k < L; k += 64) rad[k] = rb.radius[k];
    const Staged<float> s = stage_env<float, OBB>(env, smem);   // ends with a barrier
    const int t = lane & (G - 1);
    const int grp = lane / G;
    const PairRow row(smem + lds.rows + grp * lds.row, S, L);
    const Params<float> p{qp.eq, qp.maxd};
    const uint64_t below = (1ull << lane) - 1;
    const int di = M > 0 ? G / M : 0, dj = M > 0 ? G % M : 0;   // one step of a lane's walk over the pairs

    for (int64_t kb = (int64_t)blockIdx.x * kGroups; kb < total; kb += (int64_t)gridDim.x * kGroups) {
        // a group past the end rides along on the last configuration
        const bool live = kb + grp < total;
        int64_t c = 0;
        int k0 = 0;   // the first link to compute
        flag_decode(idx, live ? kb + grp : total - 1, qp, out, c, k0);
        const float* qc = q + c * D;
        for (int m = t; m < S; m += G) seg_pose_store(row.seg + 12 * m, rb.seg[m], qc);
        for (int i = t; i < L; i += G) {
            row.near_key[i] = ~0ull;
            row.hit_key[i] = ~0ull;
            row.low[i] = __float_as_uint(INFINITY);
        }
        if (t == 0) *row.first_link = L;
        wave_sync();
        skeleton_row(row.seg, pts, L, t < 3 ? t : 0, row.skel, t < 3);   // lanes 3 and up follow row 0
        wave_sync();
        // the loop's view of pair (i, j) of a row: min(MAX_DISTANCE, filtered
        // distance), MAX_DISTANCE for a NaN; and its place in the row
        auto evaluate = [&](const PairRow& w, int i, int j, NP<float>& np) {
            const Vec3<float> A{w.skel[3 * i], w.skel[3 * i + 1], w.skel[3 * i + 2]};
            const Vec3<float> B{w.skel[3 * i + 3], w.skel[3 * i + 4], w.skel[3 * i + 5]};
            float dt;
            if (s.gnd[j] && i < rb.ground_included) {
                dt = p.maxd;
                if (WANT_NP) {
                    np.r = Vec3<float>{0.0f, 0.0f, 0.0f};
                    np.o = Vec3<float>{0.0f, 0.0f, -p.maxd};
                    np.valid = true;
                }
            } else if (OBB) {
                const float* x = s.xf + 12 * j;
                dt = capsule_box<float, WANT_NP>(to_box(x, A), to_box(x, B), rad[i], s.box[j], p, &np, nullptr);
                if (WANT_NP && np.valid) {
                    np.r = from_box(x, np.r);
                    np.o = from_box(x, np.o);
                }
            } else {
                dt = capsule_box<float, WANT_NP>(A, B, rad[i], s.box[j], p, &np, nullptr);
            }
            if (dt > s.tol[j]) dt = p.maxd;
            const float v = smin(p.maxd, dt);
            if (v <= 0) {
                atomicMin(w.hit_key + i, ((unsigned long long)(uint32_t)j << 32) | __float_as_uint(v));
                atomicMin(w.first_link, i);
            } else {
                atomicMin(w.low + i, __float_as_uint(v));   // positive floats order as their bits
            }
        };
        // this lane's walk over the pairs (i, j), links from k0 on, G at a time
        int i = M > 0 ? k0 + t / M : L, j = M > 0 ? t % M : 0;
        const int i0 = i, j0 = j;
        auto advance = [&]() {
            i += di;
            j += dj;
            if (j >= M) {
                j -= M;
                ++i;
            }
        };
        if (WANT_NP) {
            for (; i < L; advance()) {
                NP<float> np;
                evaluate(row, i, j, np);
                if (live) {
                    float* e = out.nearest + ((c * M + j) * L + i) * 6;
                    if (np.valid) {
                        e[0] = np.r.x; e[1] = np.r.y; e[2] = np.r.z;
                        e[3] = np.o.x; e[4] = np.o.y; e[5] = np.o.z;
                    } else {
                        for (int k = 0; k < 6; ++k) e[k] = NAN;
                    }
                }
            }
            wave_sync();
        } else {
            // 3. gaps, and each link's nearest obstacle
            for (; i < L; advance()) {
                float g2 = INFINITY;   // a ground box that the link skips
                if (!(s.gnd[j] && i < rb.ground_included)) {
                    const float* P = row.skel + 3 * i;
                    Vec3<float> slo, shi;
                    seg_bounds(Vec3<float>{P[0], P[1], P[2]}, Vec3<float>{P[3], P[4], P[5]}, slo, shi);
                    g2 = gap_squared(OBB ? env.cull + 6 * j : s.box[j].lo, slo, shi);
                    atomicMin(row.near_key + i, ((unsigned long long)__float_as_uint(g2) << 32) | (uint32_t)j);
                }
                row.gap2[i * M + j] = g2;
            }
            i = i0;
            j = j0;
            wave_sync();
            // the queue holds those pairs first, then the pairs that their
            // values leave; one copy of the case tree serves both
            int last = L;   // the links up to the first with a hit
#pragma clang loop unroll(disable)
            for (bool first = true;; first = false) {
                int qn = 0;
                if (first) {
                    for (int m = k0 + t; __any(m < L); m += G) {
                        const unsigned long long key = m < L ? row.near_key[m] : ~0ull;
                        const uint64_t take = __ballot(key != ~0ull);
                        if (key != ~0ull)
                            queue[__popcll(take & below) + qn] = (uint32_t)(grp << 16 | m << 10) | (uint32_t)key;
                        qn += __popcll(take);
                    }
                } else {
                    while (qn <= kPairQueue - 64 && __any(i <= last)) {
                        bool tk = i <= last;
                        if (tk) tk = (uint32_t)row.near_key[i] != (uint32_t)j && !(row.gap2[i * M + j] > row.bound2[i]);
                        const uint64_t take = __ballot(tk);
                        if (tk) queue[__popcll(take & below) + qn] = (uint32_t)(grp << 16 | i << 10 | j);
                        qn += __popcll(take);
                        advance();
                    }
                }
                wave_sync();
                for (int k = lane; k < qn; k += 64) {
                    const uint32_t e = queue[k];
                    NP<float> np;
                    evaluate(PairRow(smem + lds.rows + (e >> 16) * lds.row, S, L), (e >> 10) & 63, e & 1023, np);
                }
                wave_sync();
                last = min(L - 1, *row.first_link);
                if (first) {
                    for (int m = k0 + t; m < L; m += G) {
                        const float prof =
                            row.hit_key[m] != ~0ull ? 0.0f : smin(p.maxd, __uint_as_float(row.low[m]));
                        const float b = cull_bound(prof, rad[m], p.eq);
                        // (a MAX_DISTANCE of 0 or less makes every pair a hit)
                        row.bound2[m] = p.maxd > 0 ? b * b : INFINITY;
                    }
                    wave_sync();
                } else if (!__any(i <= last)) {
                    break;
                }
            }
        }
        const int first_hit = *row.first_link;
        float d = p.maxd;
        for (int m = t; m < L; m += G) {
            float prof;
            if (m < k0) prof = out.profile[c * L + m];   // the bulk pass's value, no hit
            else if (m == first_hit) prof = __uint_as_float((uint32_t)row.hit_key[m]);
            else prof = m < first_hit ? smin(p.maxd, __uint_as_float(row.low[m])) : 0.0f;
            if (live && m >= k0 && out.profile) out.profile[c * L + m] = prof;
            if (m < first_hit) d = smin(d, prof);
        }
        for (int o = G / 2; o > 0; o >>= 1) d = smin(d, __shfl_xor(d, o, G));
        if (live && t == 0) {
            if (out.d) out.d[c] = first_hit < L ? 0.0f : d;
            if (out.verdict) out.verdict[c] = first_hit < L ? 0 : 1;
        }
        if (WANT_NP && first_hit < L && live) {
            // the points this wave stored for the pairs must land before the
            // NaN fill of the same addresses by other lanes
            __builtin_amdgcn_s_waitcnt(0);
            float* e = out.nearest + c * (int64_t)M * L * 6;
            for (int k = t; k < M * L * 6; k += G) e[k] = NAN;
        }
        wave_sync();   // the row is written again by the next round
    }
}

constexpr int kPairsMax = 1024;   // links x obstacles of a configuration's row

template <bool OBB, bool WANT_NP, int G>
hipError_t launch_shape(const RobotDev& rb, const EnvDev& env, const QueryParams& qp, const float* q,
                        const DistOut& out, const int32_t* idx, const uint32_t* count, int64_t n, int64_t max_waves,
                        uint32_t* count_out, hipStream_t st) {
    constexpr int groups = 64 / G;
    const PairLds lds = pair_lds(rb, env, WANT_NP, groups);
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min((n + groups - 1) / groups, max_waves));
    hipLaunchKernelGGL((k_distance_pairs<OBB, WANT_NP, G>), dim3(grid), dim3(64), lds.total, st, rb, env, qp, q, out,
                       idx, count, idx ? (int64_t)0 : n, count_out, lds);
    return hipGetLastError();
}

}  // namespace

bool pairs_fit(const RobotDev& rb, const EnvDev& env) {
    return (int64_t)rb.num_links * env.num_obj <= kPairsMax && pair_lds(rb, env, false, 4).total <= 64 * 1024;
}

hipError_t launch_distance_pairs(const RobotDev& rb, const EnvDev& env, const QueryParams& qp, const float* q,
                                 const DistOut& out, const int32_t* idx, const uint32_t* count, int64_t n,
                                 int64_t max_waves, hipStream_t st, uint32_t* count_out) {
    // Lanes per configuration.  64 leave a shorter chain, 16 fill the waves
    // better once there are more waves than the SIMDs hold side by side.  Of
    // a batch in reference arithmetic, 64 against 16 lanes a call: xArm6 and
    // 40 boxes 1,000 configurations 42 / 58 us, 4,096 50 / 67, 8,192 70 / 74,
    // 16,384 103 / 102; 17 boxes 4,096 43 / 47 and 8,192 55 / 47; spatial10
    // and 28 boxes 16,384 113 / 116, 40 boxes 134 / 151: 64 lanes up to 4,096
    // configurations, and from 256 pairs a configuration on at any size.  A
    // bulk pass lists about one configuration in 60 to 300: a whole call on
    // spatial10 and 40 boxes, 65,536 190 / 208 us, 1,000,003 641 / 617;
    // 4 boxes 65,536 90 / 89, 200,000 119 / 113: 64 lanes up to 131,072.
    const bool wide = idx ? n <= 131072 : n <= 4096 || rb.num_links * env.num_obj >= 256;
    auto run = [&](auto shape) { return shape(rb, env, qp, q, out, idx, count, n, max_waves, count_out, st); };
    if (out.nearest) return env.use_obb ? run(launch_shape<true, true, 64>) : run(launch_shape<false, true, 64>);
    if (wide) return env.use_obb ? run(launch_shape<true, false, 64>) : run(launch_shape<false, false, 64>);
    return env.use_obb ? run(launch_shape<true, false, 16>) : run(launch_shape<false, false, 16>);
}

}  // namespace rvs
