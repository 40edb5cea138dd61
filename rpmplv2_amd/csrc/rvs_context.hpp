// Internal state of a context (shared by the C ABI layer rvs_capi.cpp and
// the request server rvs_server.cpp).  Not part of the public ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <initializer_list>
#include <map>
#include <utility>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/rvs.h"
#include "rvs_internal.hpp"

namespace rvs {

// A request that fails leaves no buffer and no error behind: the runtime keeps
// a call's error for hipGetLastError across later calls that succeed, and the
// launches that a caller goes on with, in less memory, report by it.
struct DevBuf {
    void* p = nullptr;
    size_t cap = 0;
    hipError_t ensure(size_t bytes) {
        if (bytes <= cap) return hipSuccess;
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
        size_t want = std::max<size_t>(bytes, 1 << 20);
        hipError_t e = hipMalloc(&p, want);
        if (e != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            return e;
        }
        cap = want;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

// Pinned host staging for the per-call tables of the edge search (copied to
// the device asynchronously; the call synchronizes before it returns).
struct PinnedBuf {
    void* p = nullptr;
    size_t cap = 0;
    hipError_t ensure(size_t bytes) {
        if (bytes <= cap) return hipSuccess;
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
        size_t want = std::max<size_t>(bytes, 1 << 20);
        hipError_t e = hipHostMalloc(&p, want, hipHostMallocDefault);
        if (e != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            return e;
        }
        cap = want;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
    }
};

struct RobotRec {
    RobotDev dev{};
    std::vector<void*> allocs;
    int num_dofs = 0, num_links = 0, num_pairs = 0;
    std::vector<float> radius;   // capsule radius per link (host copy)
};

struct EnvRec {
    EnvDev dev{};
    std::vector<void*> allocs;
    std::vector<rvs_box> boxes;
    std::vector<float> aabb, obb, cull;   // host copies of the device tables
    std::vector<int32_t> gorder;          // broad-phase walk order (host copy)
    std::vector<float> gcull;             // group boxes of the walk (host staging)
    int semantics = RVS_ENV_AABB;
    bool has_motion = false;              // rvs_env_set_motion_law was called
    EnvStepDev step{};                    // motion-law state on the device
};

// The launch shape of an RVS_PREC_FP32_REFINE batch of n configurations that
// nobody recorded one for: by the length of the walk and the batch (every shape
// gives the same bits, so the choice may follow n).  lists: whether the call
// can have the link-major pass's scratch (fast_links_bytes).
inline FastTuning default_shape(int32_t dofs, int32_t links, int32_t objects, int64_t n, bool lists) {
    if ((int64_t)links * objects < 1024) {
        // The walk order's four kernels (16 to 31 us) pay for themselves in
        // large batches, the earlier the longer the walk.  Sorted against
        // unsorted, us a call: xArm6 and 17 boxes 266 / 322 for 1,000,003
        // configurations, 120 / 101 for 260,000, 88 / 72 for 4,000; 80 boxes 233
        // / 228 for 260,000, 177 / 177 for 80,000; 120 boxes 189 / 197 for
        // 16,000, 242 / 282 for 200,000; 160 boxes 243 / 254 for 130,000; 14-DOF
        // chain and 70 boxes 412 / 419 and 473 / 546 for 130,000 and 200,000;
        // 10-DOF chain and 100 boxes 274 / 251 and 319 / 328.  Fewer than 32
        // pairs: never (xArm6 and 5 boxes 553 / 375 for 4,000,000, 22-DOF chain
        // and one box 737 / 533 for 1,000,000).
        // Where they order the whole pose (at most 3 joints) they pay early,
        // unless the walk is short: planar arm, 40 boxes 108 / 164 for 65,536;
        // 15 boxes 83 / 75 for 300,000 and 123 / 138 for 1,000,000; 4 boxes 130
        // / 102 for 1,000,003.
        const int64_t pairs = (int64_t)links * objects;
        int64_t from = INT64_MAX;
        if (dofs <= 3) {
            if (pairs >= 24) from = pairs >= 32 ? 1024 : 1 << 19;
        } else if (pairs >= 32) {
            from = objects >= 112 ? 1 << 14 : (pairs >= 700 ? 5 << 15 : 1 << 18);
        }
        return FastTuning{0, 64, 0, n >= from ? 5 : 0};
    }
    // Long walks: lane refill (1), the same with pair queues (3), or link-major
    // launches (4), whose lists take 128 bytes a configuration, at most 2 GiB.
    // A handful of configurations share nothing: lane refill for 1 and 10
    // among fewer than 400 boxes (or without lists) 133 and 187 against 164 and
    // 209 us with queues (10-DOF chain, 130 boxes), 257 and 607 against 288 and
    // 846 link by link (22-DOF chain, 256 boxes); among 512 boxes 427 and 1,340
    // against 344 and 1,260 link by link.
    const FastTuning refill{1, 256, 0, 5}, queues{3, 512, 0, 5}, by_link{4, 512, 0, 5};
    lists = lists && n <= (int64_t)1 << 24;
    if (n <= 16 && (objects < 400 || !lists)) return refill;
    // Refill, queues and link by link, us a call.  Arms of up to 7 links (6-DOF
    // arm): 200 boxes 307, 278 and 254 for 1,000 configurations, 482, 513 and
    // 506 for 400,000; 300 boxes 321, 337 and 282, and 941, 1,075 and 921 for
    // 1,000,000 (200,000: 467 and 441); 1,000 boxes 2,524, 2,672 and 969.
    if (links < 8) {
        if (lists && (objects >= 320 || (objects >= 200 && n < (int64_t)1 << 18))) return by_link;
        return n < (int64_t)1 << 18 ? queues : refill;
    }
    // 8 to 11 links (10-DOF chain): 130 boxes 229, 244 and 307 for 1,000, 957,
    // 1,042 and 1,224 for 1,000,000; 200 boxes 445, 420 and 395 for 30,000; 256
    // boxes 378, 464 and 419, and 1,331, 1,534 and 1,340 for 1,000,000; 700
    // boxes 972, 860 and 436 for 1,000, 3,372, 3,455 and 1,657 for 1,000,000.
    if (links < 12) {
        if (lists && objects >= 200) return by_link;
        return objects >= 600 && n < (int64_t)1 << 19 ? queues : refill;
    }
    // Longer chains:
    //                     1,000               130,000             400,000             1,000,000
    //   14 DOF,  80 boxes   389   331   452     502   449   636     845   791 1,126   1,574 1,639 1,937
    //   14 DOF, 160 boxes   628   540   617     752   653   790   1,238 1,145 1,379   2,403 2,287 2,401
    //   14 DOF, 256 boxes   763   678   647     952   850   889   1,490 1,517 1,484   3,068 2,961 2,484
    //   22 DOF,  96 boxes   830   633   804   1,038   835 1,116   1,614 1,433 1,932   3,269 3,279 3,491
    //   22 DOF, 128 boxes   855   748   902     976   899 1,146   1,620 1,623 2,008   3,383 3,519 3,578
    //   22 DOF, 200 boxes 1,319 1,128 1,111   1,420 1,234 1,403   2,240 2,157 2,297   4,742 4,128 3,865
    //   22 DOF, 512 boxes 2,770 2,287 1,922   2,974 2,503 2,405   5,516 4,579 3,657  10,955 8,794 6,458
    //   40 DOF, 256 boxes 2,475 2,225 2,172   2,801 2,519 2,834   4,540 4,148 4,029
    //   40 DOF, 400 boxes 3,703 3,148 2,958   3,863 3,422 3,617   6,443 5,577 4,881
    // so link by link from more obstacles on the longer the chain, and earlier
    // in batches that are large or too small to fill the card with queues (200
    // boxes, 300 configurations: 14 DOF 722, 589 and 556, 22 DOF 1,303, 1,012
    // and 956); queues in small batches and from 160 boxes on.
    if (lists && (objects >= 100 + 8 * links || (objects >= 176 && n >= (int64_t)1 << 19) ||
                  (objects >= 240 && n >= (int64_t)1 << 18) || (objects >= 200 && n <= 1024)))
        return by_link;
    if (n <= (int64_t)1 << 17 || objects >= 160) return queues;
    return refill;
}

}  // namespace rvs

// The opaque handle of include/rvs.h.
struct rvs_context {
    rvs_options opt{};
    hipStream_t stream = nullptr;
    std::mutex mu;
    // the last failure's message; err_mu guards it alone, since argument
    // checks fail before mu is taken
    mutable std::mutex err_mu;
    std::string err;
    std::vector<rvs::RobotRec> robots;
    std::vector<rvs::EnvRec> envs;
    rvs::DevBuf arena;
    rvs::PinnedBuf staging;
    int64_t last_refined = 0;
    // Asynchronous calls (rvs_*_async) enqueue on a caller's stream and
    // return; async_ev is recorded after each of them (each first waits for
    // the previous one, so the event covers them all).  Every other call
    // waits for it on the host before it touches the arena or the tables.
    hipEvent_t async_ev = nullptr;
    bool async_pending = false;
    void drain_async() {
        if (async_pending) {
            (void)hipEventSynchronize(async_ev);
            async_pending = false;
        }
    }
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    float stage_ms[3] = {0, 0, 0};
    int32_t nstages = 0;
    int32_t num_cus = 0;
    // FP32 bulk pass variant when no tuning is recorded: -1 = by walk length
    // and batch (tuning_for), otherwise the variant
    int32_t fast_variant = -1;
    // reference-arithmetic distance batches up to this many configurations
    // run 16 or 64 lanes per configuration (latency) instead of one
    int64_t wave_max = 16384;
    int32_t edge_waves_per_cu = 16;   // persistent first-collision kernel: resident waves per CU
    int32_t edge_spl = 0;             // ... and slots per lane in one 64-lane item (0: by the slots of the call)
    std::map<std::pair<int32_t, int32_t>, rvs::FastTuning> tuning;   // (robot, env) -> autotuned launch shape
    // captured FP32 + refinement pipelines of device-array rvs_distance calls
    struct Graph {
        int32_t robot, env;
        const void *q, *d, *profile, *verdict, *arena;
        int64_t n;
        rvs::FastTuning t;
        hipGraphExec_t exec;
        uint64_t used;
    };
    std::vector<Graph> graphs;
    uint64_t graph_clock = 0;
    uint32_t* count_host = nullptr;   // pinned, coherent: refinement count the graphs' refinement stores
    uint32_t* count_dev = nullptr;    // the same word's device address
    std::mutex tuning_mu;
    // The launch shape of an RVS_PREC_FP32_REFINE batch of n configurations:
    // the recorded one, else default_shape's.
    rvs::FastTuning tuning_for(int32_t robot, int32_t env, int32_t dofs, int32_t links, int32_t objects, int64_t n,
                               bool lists = true) {
        std::lock_guard<std::mutex> lk(tuning_mu);
        auto it = tuning.find({robot, env});
        if (it != tuning.end()) return it->second;
        // one lane per configuration: 64-thread workgroups measured fastest
        if (fast_variant >= 0) return rvs::FastTuning{fast_variant, fast_variant == 0 ? 64 : 256, 0, 5};
        return rvs::default_shape(dofs, links, objects, n, lists);
    }
    // Walk-order bits of the exact paths: a recorded shape's, else 5.
    int32_t order_bits(int32_t robot, int32_t env) {
        std::lock_guard<std::mutex> lk(tuning_mu);
        auto it = tuning.find({robot, env});
        return it != tuning.end() ? it->second.coh_bits : 5;
    }
    // Whether an isValid batch of n configurations runs in the walk order:
    // 16 to 31 us of sorting against fewer branches.  xArm6 and 17 boxes, REF32
    // (FP64): 204 against 235 us (246 / 318) for 1,000,003 configurations, 146
    // against 142 (174 / 193) for 524,288, 105 against 88 (126 / 124) for
    // 262,147; the planar arm among 4 boxes 80 against 59 us for 1,000,003.
    bool order_valid(int32_t robot, int32_t env, int64_t n) const {
        return n >= 1 << 19 && n <= INT32_MAX &&
               (int64_t)robots[robot].num_links * envs[env].dev.num_obj >= 32;
    }
    // Whether the launch shape of (robot, env) was recorded by a caller.
    bool tuned(int32_t robot, int32_t env) {
        std::lock_guard<std::mutex> lk(tuning_mu);
        return tuning.find({robot, env}) != tuning.end();
    }
};

namespace rvs {

// The context's lock for a synchronous call: it also waits for the
// asynchronous calls still in flight, which may use the arena and read the
// robot and obstacle tables.
struct CtxLock {
    std::lock_guard<std::mutex> lk;
    explicit CtxLock(rvs_context* c) : lk(c->mu) { c->drain_async(); }
};

// Sub-allocation of one device block, 256-byte aligned pieces.
struct Carve {
    char* base;
    size_t off = 0;
    explicit Carve(void* b) : base(static_cast<char*>(b)) {}
    template <typename T> T* take(size_t count) {
        off = (off + 255) & ~size_t(255);
        T* p = reinterpret_cast<T*>(base + off);
        off += count * sizeof(T);
        return p;
    }
    static size_t need(std::initializer_list<size_t> bytes) {
        size_t s = 0;
        for (size_t b : bytes) s += ((b + 255) & ~size_t(255));
        return s + 256;
    }
};


// FCL's world AABB of a box (and whether its rotation counts as identity)
// and the oriented-box table of the engine.
bool box_identity(const rvs_box& b);
void box_bounds(const rvs_box& b, float out[6]);
void box_obb(const rvs_box& b, float out[15]);
// Half extents of the tight world AABB of an oriented box (|R| h, rounded up
// by one part in 10^6 so that it contains the box despite float rounding).
void obb_extent(const float obb[15], float ext[3]);
QueryParams params_of(const rvs_context* c);

}  // namespace rvs
