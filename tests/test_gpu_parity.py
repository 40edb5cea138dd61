"""GPU parity: librvs.so on cuda:0 against the CPU oracle on the same inputs.

Bar: verdicts identical; REF32 distances and profiles bit-identical to the
oracle's reference arithmetic except where the device and host double sine /
cosine differ in the last bit (allowed: 2 float ulps); FP64 distances within
1e-12 m of the oracle's FP64 twin.
"""
import numpy as np
import pytest

from rpmplv2_amd import robots as R, rvs, workloads as W

pytestmark = pytest.mark.gpu


def ulps(a, b):
    a = np.ascontiguousarray(a, np.float32)
    b = np.ascontiguousarray(b, np.float32)
    ia = a.view(np.int32).astype(np.int64)
    ib = b.view(np.int32).astype(np.int64)
    ia = np.where(ia < 0, -(ia & 0x7FFFFFFF), ia)
    ib = np.where(ib < 0, -(ib & 0x7FFFFFFF), ib)
    return np.abs(ia - ib)


def check_ref32(oracle, engine, w, n=None):
    q = w.q if n is None else w.q[:n]
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, _ = engine.distance(rid, eid, q)
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene), q, 32)
    print(f"{w.name}: n={len(q)} valid={ver.mean():.4f} verdict mismatches={(ver != over).sum()}")
    assert (ver == over).all()
    assert ulps(d, od).max() <= 2
    assert ulps(prof, oprof).max() <= 2
    assert (d == od).mean() > 0.999
    return rid, eid


def test_workload1_ref32(oracle, engine):
    check_ref32(oracle, engine, W.workload1(65536))


def test_workload2_ref32(oracle, engine):
    check_ref32(oracle, engine, W.workload2(1 << 17))


def test_workload1_fp64(oracle, engine):
    w = W.workload1(65536)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver = engine.distance_f64(rid, eid, w.q)
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene), w.q, 64)
    assert (ver == over).all()
    assert np.abs(d - od).max() <= 1e-12
    assert np.abs(prof - oprof).max() <= 1e-12


def test_workload2_fp64(oracle, engine):
    w = W.workload2(1 << 16)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver = engine.distance_f64(rid, eid, w.q)
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene), w.q, 64)
    assert (ver == over).all()
    assert np.abs(d - od).max() <= 1e-12
    assert np.abs(prof - oprof).max() <= 1e-12


def test_nearest_points(oracle, engine):
    w = W.workload2(2048)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, npo = engine.distance(rid, eid, w.q, want_nearest=True)
    od, oprof, over, onp = oracle.distance(w.robot, oracle.scene_of(w.scene), w.q, 32, want_np=True)
    assert (ver == over).all()
    ok = ver == 1
    a, b = npo[ok], onp[ok]
    assert np.array_equal(np.isnan(a), np.isnan(b))
    m = ~np.isnan(a)
    assert np.abs(a[m] - b[m]).max() <= 1e-6


def test_is_valid(oracle, engine):
    w = W.workload2(1 << 16)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    v = engine.is_valid(rid, eid, w.q)
    ov = oracle.is_valid(w.robot, oracle.scene_of(w.scene), w.q)
    assert (v == ov).all()
    v64 = engine.is_valid(rid, eid, w.q, precision=rvs.PREC_FP64)
    ov64 = oracle.is_valid(w.robot, oracle.scene_of(w.scene), w.q, 64)
    assert (v64 == ov64).all()


def test_underestimation(oracle, engine):
    w = W.workload2(4096)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    sc = oracle.scene_of(w.scene)
    # nearest points of the first collision-free configuration, shared by all
    od, _, over, onp = oracle.distance(w.robot, sc, w.q, 32, want_np=True)
    k = int(np.argmax(over == 1))
    ref = onp[k]
    d, prof, st = engine.underestimation(rid, eid, w.q, ref)
    ud, uprof, ust = oracle.underestimation(w.robot, sc, w.q, ref)
    assert (st == ust).all()
    assert ulps(d, ud).max() <= 2
    assert ulps(prof[st == 1], uprof[st == 1]).max() <= 2
    # per-configuration sets
    d2, prof2, st2 = engine.underestimation(rid, eid, w.q[:512], onp[:512])
    ud2, uprof2, ust2 = oracle.underestimation(w.robot, sc, w.q[:512], onp[:512])
    assert (st2 == ust2).all()
    assert ulps(d2, ud2).max() <= 2


def _boxes_around(rng, rb, count, side_lo, side_hi, reach, clearance=0.02):
    """Boxes in a ball of `reach` around the middle of the zero pose's
    skeleton, their bounding balls clear of it."""
    P = R.skeleton_np(rb, np.zeros(rb.num_dofs))[0]
    t = np.linspace(0.0, 1.0, 21)[:, None, None]
    pts = (P[None, :-1] + t * (P[1:] - P[:-1])[None]).reshape(-1, 3)
    gap = np.max(rb.radius) + clearance
    rows = []
    while len(rows) < max(count, 1):
        sc = W._boxes(rng, 4 * count + 8, side_lo, side_hi, reach, center=P.mean(0))
        far = np.linalg.norm(sc.pos[:, None] - pts[None], axis=2).min(1) > 0.5 * np.linalg.norm(sc.dim, axis=1) + gap
        rows += [k for k in zip(sc.dim[far], sc.pos[far])]
    dim, pos = (np.array(x[:count]) for x in zip(*rows))
    return W.Scene(dim, pos, np.tile([1.0, 0.0, 0.0, 0.0], (count, 1)), np.zeros(count, np.uint8),
                   np.full(count, 1000.0, np.float32))


@pytest.mark.parametrize("dofs,boxes,n,far", [(6, 1, 1, False), (6, 16, 255, False), (10, 40, 257, False),
                                              (22, 100, 300, False), (22, 1000, 65, False), (6, 17, 257, True),
                                              (22, 100, 300, True), (22, 1000, 65, True)])
def test_underestimation_shared_set_sizes(oracle, engine, dofs, boxes, n, far):
    """One nearest-point set for all, from a single plane per link to sets
    of several tiles (2,200 and 22,000 planes), ragged batches, a NaN joint,
    a missing (NaN) pair and pairs the reference skips: stored flags equal,
    values within 2 ulp (the device's double sine and cosine), profiles of
    unstored configurations 0.  far: boxes out of the robot's reach, so that
    the configurations are stored."""
    rng = np.random.default_rng(90 + boxes)
    rb = R.xarm6() if dofs == 6 else R.chain(rng.uniform(0.05, 0.1, dofs), radius=0.02, ground_included=1)
    sc = W._boxes(rng, boxes, 0.02, 0.1, 2.5)
    if far:
        u = rng.normal(size=(boxes, 3))
        sc = W.Scene(sc.dim, 4.0 * u / np.linalg.norm(u, axis=1, keepdims=True), sc.quat, sc.is_ground,
                     sc.min_dist_tol)
    q = rng.uniform(-0.3, 0.3, (n, dofs)).astype(np.float32)
    q[n // 2, 1] = np.nan
    P = R.skeleton_np(rb, np.zeros(dofs))[0]
    ref = np.zeros((boxes, rb.num_links, 6), np.float32)
    ref[..., :3] = 0.5 * (P[:-1] + P[1:])
    ref[..., 3:] = np.clip(ref[..., :3], sc.aabb[:, None, :3], sc.aabb[:, None, 3:])
    ref[0, 0] = np.nan
    ref[-1, 1] = (0, 0, 0, 0, 0, -1000.0)
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    d, prof, st = engine.underestimation(rid, eid, q, ref)
    od, oprof, ost = oracle.underestimation(rb, oracle.scene_of(sc), q, ref)
    assert (st == ost).all()
    assert ulps(d, od).max() <= 2
    ok = st == 1
    assert (ok.mean() > 0.9) if far else True
    assert (prof[~ok] == 0).all() and (not ok.any() or ulps(prof[ok], oprof[ok]).max() <= 2)


def test_self_distance(oracle, engine):
    rb = R.chain(np.random.default_rng(5).uniform(0.1, 0.3, 22), radius=0.04, self_collision=True)
    q = np.random.default_rng(6).uniform(-np.pi, np.pi, (8192, 22)).astype(np.float32)
    rid = engine.load_robot(rb)
    sd = engine.self_distance(rid, q)
    osd = oracle.self_distance(rb, q, rb.self_pairs)
    assert ulps(sd, osd).max() <= 2
    assert ((sd < 0) == (osd < 0)).all()
    xa = R.xarm6()
    rid2 = engine.load_robot(xa)
    q2 = W.workload2(8192).q
    assert ulps(engine.self_distance(rid2, q2), oracle.self_distance(xa, q2, xa.self_pairs)).max() <= 2


def test_chain_ground(oracle, engine):
    rb = R.spatial(10, radius=0.025, ground_included=2)
    sc = W.ground_box().concat(W._boxes(np.random.default_rng(9), 5, 0.3, 0.3, 1.0, (0, 0, 0.1)))
    q = np.random.default_rng(10).uniform(-np.pi, np.pi, (16384, 10)).astype(np.float32)
    w = W.ConfigBatch("spatial10", rb, sc, q)
    check_ref32(oracle, engine, w)


def test_empty_and_single(oracle, engine):
    w = W.workload2(1)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, _ = engine.distance(rid, eid, w.q[:0])
    assert d.shape == (0,)
    d, prof, ver, _ = engine.distance(rid, eid, w.q[:1])
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene), w.q[:1], 32)
    assert ver[0] == over[0] and ulps(d, od).max() <= 2


@pytest.mark.parametrize("links,boxes", [(16, 16), (16, 17), (63, 4)])
def test_refinement_forms_at_their_limits(oracle, engine, links, boxes):
    """The exact refinement evaluates all pairs of a configuration at once up
    to 256 (link, obstacle) pairs and fewer than 64 links (16 x 16, 63 x 4),
    and link by link beyond (16 x 17): both give the oracle's reference
    arithmetic, on the FP32 path's flagged configurations and as the
    small-batch form of reference-arithmetic calls."""
    rng = np.random.default_rng(70 + links + boxes)
    rb = R.chain(rng.uniform(0.03, 0.06, links), radius=0.02)
    sc = W._boxes(rng, boxes, 0.05, 0.2, 0.9, (0, 0, 0.3))
    q = rng.uniform(-1.0, 1.0, (20000, links)).astype(np.float32)
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    osc = oracle.scene_of(sc)
    od, oprof, over, _ = oracle.distance(rb, osc, q, 32)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    print(f"{links} links x {boxes} boxes: collision-free {ver.mean():.3f}, refined {engine.last_refined()}")
    assert (ver == over).all() and np.abs(d - od).max() <= 1e-5
    d2, prof2, ver2, _ = engine.distance(rid, eid, q[:3000], precision=rvs.PREC_REF32)   # one wave per configuration
    assert (ver2 == over[:3000]).all() and ulps(d2, od[:3000]).max() <= 2 and ulps(prof2, oprof[:3000]).max() <= 2


@pytest.mark.parametrize("boxes", [0, 1, 5])
def test_fp32_refine_small_scenes_and_nan(oracle, engine, boxes):
    """The FP32 path (walk order, grouped broad phase) on scenes of 0, 1 and
    5 boxes (no group, one partial group, a full and a partial group), with
    non-finite joint values among the configurations: verdicts equal the
    oracle's, NaN distances where the oracle has them, the others within
    1e-5 m."""
    rng = np.random.default_rng(60 + boxes)
    rb = R.xarm6()
    sc = W._boxes(rng, boxes, 0.1, 0.4, 0.8, (0, 0, 0.4)) if boxes else W.Scene(
        np.zeros((0, 3)), np.zeros((0, 3)), np.zeros((0, 4)), np.zeros(0, np.uint8), np.zeros(0))
    q = W.workload2(50000).q.copy()
    q[::97, 1] = np.nan
    q[::89, 0] = np.inf
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    od, oprof, over, _ = oracle.distance(rb, oracle.scene_of(sc), q, 32)
    assert (ver == over).all()
    assert np.array_equal(np.isnan(d), np.isnan(od))
    m = ~np.isnan(d)
    assert np.abs(d[m] - od[m]).max() <= 1e-5


def test_fp32_screen_sends_nan_pairs_to_the_exact_pass(oracle, engine):
    """A link lying in the plane of a box face, with one end point projecting
    onto the opposite face and the other end point inside that face's span,
    makes the case tree return NaN (the reference reads nearest points it
    never set, CollisionAndDistance.cpp:476-574): the pair drops out of the
    minimum.  One rounding away the segment crosses the face and the pair is
    a hit.  Planar 2-DOF at q0 = 0 lies on y = 0, the box's lo.y face: the
    FP32 bulk pass must flag every such configuration for the exact pass,
    and the verdicts must be the reference arithmetic's on both sides of the
    discontinuity."""
    sc = W.Scene([[0.6, 0.5, 0.2]], [[0.5, 0.25, 0.0]], [[1, 0, 0, 0]], [0], [W.MAX_DISTANCE])
    assert sc.aabb[0, 1] == 0.0
    rb = R.planar_2dof(radius=0.02)
    osc = oracle.scene_of(sc)
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    # q0 = 0 exactly, any q1: link 0 takes the NaN path (the oracle drops it)
    q_on = np.zeros((256, 2), np.float32)
    q_on[:, 1] = np.linspace(-3.0, 3.0, 256, dtype=np.float32)
    od, oprof, over, _ = oracle.distance(rb, osc, q_on, 32)
    assert (oprof[:, 0] == W.MAX_DISTANCE).all()          # the NaN pair left link 0 at MAX_DISTANCE
    d, prof, ver, _ = engine.distance(rid, eid, q_on, precision=rvs.PREC_FP32_REFINE)
    refined = engine.last_refined()
    print(f"on the face plane: refined {refined} of {len(q_on)}, free {ver.mean():.3f}")
    assert refined == len(q_on)
    assert (ver == over).all() and ulps(d, od).max() <= 2 and ulps(prof, oprof).max() <= 2
    # one configuration alone
    d1, _, v1, _ = engine.distance(rid, eid, q_on[:1], precision=rvs.PREC_FP32_REFINE)
    assert engine.last_refined() == 1 and v1[0] == over[0] and ulps(d1, od[:1]).max() <= 2
    # across the discontinuity: q0 a few float steps either side of 0
    k = np.arange(-2000, 2001, dtype=np.float64)
    q0 = np.concatenate([k * 1e-10, k * 1e-8, np.float32(np.pi) * np.ones(1)]).astype(np.float32)
    q = np.stack([q0, np.tile(np.float32([0.0, 0.7, -1.3]), len(q0) // 3 + 1)[:len(q0)]], 1)
    od, oprof, over, _ = oracle.distance(rb, osc, q, 32)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    print(f"across it: refined {engine.last_refined()} of {len(q)}, free {ver.mean():.3f}, "
          f"oracle NaN pairs {(oprof[:, 0] == W.MAX_DISTANCE).sum()}")
    assert (ver == over).all()
    assert np.abs(d - od).max() <= 1e-5 and np.abs(prof - oprof).max() <= 1e-5
    assert 0 < over.mean() < 1


# A planar arm's first link crossing the face x = 0.5 of a box where one of
# the quirked corner tests of collisionCapsuleToRectangle
# (CollisionAndDistance.cpp:69, :71, :72) reports a hit although the capsule
# is 0.052-0.054 m from the box (r = 0.05); q1 turns the second link away.
# (box, q0, q1)
QUIRK_SCENES = [
    ((0.5, -1.0, 0.03, 1.0, 0.01, 1.0), float(np.arctan(0.11)), 1.5708),
    ((0.5, -0.1, 0.048, 1.0, 0.005, 1.0), float(np.arctan(-0.24)), -1.5708),
    ((0.5, -1.0, -0.035, 1.5, -0.045, -0.03), 0.0, 1.5708),
]


@pytest.mark.parametrize("case", [0, 1, 2])
def test_collision_tree_corner_quirk(oracle, engine, case):
    """isValid(q) on the quirked corner tests: the device reports the
    collision the reference's tree reports (FP32 and FP64 trees), and the
    distance paths report the positive distance the reference's
    computeDistance returns for the same configuration; around it, q0 swept
    across the edge of the quirk's region."""
    box, q0, q1 = QUIRK_SCENES[case]
    lo, hi = np.asarray(box[:3]), np.asarray(box[3:])
    sc = W.Scene([hi - lo], [(hi + lo) / 2], [[1, 0, 0, 0]], [0], [W.MAX_DISTANCE])
    assert np.abs(sc.aabb[0] - np.asarray(box)).max() < 1e-6
    rb = R.planar_2dof(radius=0.05)
    osc = oracle.scene_of(sc)
    q = np.stack([np.float32(q0) + np.linspace(-0.02, 0.02, 4001, dtype=np.float32),
                  np.full(4001, q1, np.float32)], 1).astype(np.float32)
    q[2000] = (q0, q1)
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    assert (engine.env_bounds(eid) == sc.aabb).all()
    ov = oracle.is_valid(rb, osc, q)
    ov64 = oracle.is_valid(rb, osc, q, 64)
    od, oprof, over, _ = oracle.distance(rb, osc, q, 32)
    assert ov[2000] == 0 and over[2000] == 1             # the tree's quirk hit; computeDistance: free
    v = engine.is_valid(rid, eid, q)
    v64 = engine.is_valid(rid, eid, q, precision=rvs.PREC_FP64)
    print(f"case {case}: tree collisions {int((ov == 0).sum())}, distance collisions {int((over == 0).sum())}, "
          f"tree hits at positive distance {int(((ov == 0) & (over == 1)).sum())}")
    assert (v == ov).all() and (v64 == ov64).all()
    d, prof, ver, _ = engine.distance(rid, eid, q)
    assert (ver == over).all() and ulps(d, od).max() <= 2
    d3, _, ver3, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    assert (ver3 == over).all() and np.abs(d3 - od).max() <= 1e-5


def test_nan_configurations(oracle, engine):
    w = W.workload2(256)
    q = w.q.copy()
    q[::7, 2] = np.nan
    q[::11, 0] = np.inf
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, _ = engine.distance(rid, eid, q)
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene), q, 32)
    assert (ver == over).all()
    assert np.array_equal(np.isnan(d), np.isnan(od))
    m = ~np.isnan(d)
    assert ulps(d[m], od[m]).max() <= 2
    v = engine.is_valid(rid, eid, q)
    assert (v == oracle.is_valid(w.robot, oracle.scene_of(w.scene), q)).all()


def test_edge_is_valid(oracle, engine):
    w = W.workload2(8192)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    q1, q2 = w.q[:4096], w.q[4096:]
    # short edges too, so both outcomes occur
    q2s = (q1 + 0.05 * (q2 - q1)).astype(np.float32)
    for b in (q2, q2s, q1):
        v = engine.edge_is_valid(rid, eid, q1, b)
        ov = oracle.edge_valid(w.robot, oracle.scene_of(w.scene), q1, b)
        assert (v == ov).all()
    assert 0 < engine.edge_is_valid(rid, eid, q1, q2s).mean() < 1


def test_edge_first_collision_workload3(oracle, engine):
    w3 = W.workload3(256)
    eid = engine.create_env(w3.scene)
    firsts = engine.edge_batches(eid, w3.batches)
    sc = oracle.scene_of(w3.scene)
    for b, f in zip(w3.batches, firsts):
        of = oracle.edge_first_collision(b.robot, sc, b.q1, b.dir, b.K, b.step)
        print(b.robot.name, "collide frac", (of >= 0).mean(), "mismatch", (f != of).sum())
        assert np.array_equal(f, of)


def test_edge_first_collision_planner_workload(oracle, engine):
    """Workload 3's four chains (10/14/18/22 DOF, self-collision on) with
    edges that start at collision-free states, as a planner's tree nodes
    are, in one persistent launch: the first colliding state of every edge
    equals the oracle's, for each (waves per CU, slots per lane) shape; the
    edges walk far past state 0 and many run to their last state."""
    w = W.workload3_planner(1024, oracle=oracle)
    eid = engine.create_env(w.scene)
    sc = oracle.scene_of(w.scene)
    expect = [oracle.edge_first_collision(b.robot, sc, b.q1, b.dir, b.K, b.step) for b in w.batches]
    allf = np.concatenate(expect)
    print(f"free {(allf < 0).mean():.3f}, median first collision {np.median(allf[allf >= 0])}")
    assert (allf != 0).all() and 0.1 < (allf < 0).mean() < 0.6 and np.median(allf[allf >= 0]) >= 5
    # judged by the engine's own one-state edges instead of the oracle, the
    # generator draws the same starts (the profile driver builds it that way)
    loaded = {}

    def judge(rb, scene, q):
        if id(rb) not in loaded:
            loaded[id(rb)] = engine.load_robot(rb)
        one = np.ones(len(q), np.int32)
        return engine.edge_first_collision(eid, np.full(len(q), loaded[id(rb)], np.int32), q, np.zeros_like(q),
                                           one) < 0

    wj = W.workload3_planner(1024, judge=judge)
    for a, b in zip(w.batches, wj.batches):
        assert np.array_equal(a.q1, b.q1) and np.array_equal(a.dir, b.dir), a.robot.name
    for wpc, spl in ((4, 2), (16, 1), (32, 4)):
        engine.set_edge_tuning(wpc, spl)
        got = engine.edge_batches(eid, w.batches)
        for b, g, e in zip(w.batches, got, expect):
            assert np.array_equal(g, e), (b.robot.name, wpc, spl, int((g != e).sum()))


def test_edge_first_collision_radii_ground_and_nan(oracle, engine):
    """xArm6 with a different radius on every link and the ground box
    skipped by its first two links, among the ground box and 16 boxes, from
    uniform starts with some NaN and infinite joint values: the first
    colliding state of every edge equals the oracle's (the axis-test tables
    hold one entry set per (radius, ground rule) and send NaN end points to
    the full test)."""
    w = W.workload2(4096)
    rb = R.xarm6(radius=[0.05, 0.045, 0.04, 0.035, 0.03, 0.02], ground_included=2)
    eid = engine.create_env(w.scene)
    rng = np.random.default_rng(23)
    n = 3000
    q1 = w.q[:n].copy()
    q1[::97, 2] = np.nan
    q1[5::101, 0] = np.inf
    q1[7::89, 4] = -np.inf
    u = rng.normal(size=(n, 6))
    u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    K = rng.integers(1, 80, n).astype(np.int32)
    b = W.EdgeBatch(rb, q1, u, K)
    of = oracle.edge_first_collision(rb, oracle.scene_of(w.scene), q1, u, K, 0.05)
    assert (of == 0).mean() < 0.9 and (of > 0).sum() > 100 and (of < 0).sum() > 20
    for wpc, spl in ((16, 2), (4, 1)):
        engine.set_edge_tuning(wpc, spl)
        f = engine.edge_batches(eid, [b])[0]
        bad = np.nonzero(f != of)[0]
        assert len(bad) == 0, (wpc, spl, bad[:10], f[bad[:10]], of[bad[:10]])


def test_edge_first_collision_folded_chains(oracle, engine):
    """Chains whose joints swing far (|q| up to 2 rad) fold onto
    themselves: many states have self pairs at or near contact, where the
    bounding-box bound of the self pairs must leave the verdict to the full
    segment-segment test.  Two box-free scenes far from the chains, so that
    self-collision alone ends the edges; first collisions equal the
    oracle's."""
    rng = np.random.default_rng(41)
    sc = W._boxes(rng, 4, 0.05, 0.1, 0.5, center=(10.0, 10.0, 10.0))
    eid = engine.create_env(sc)
    batches = []
    for n, r in ((8, 0.03), (12, 0.02)):
        rb = R.chain(rng.uniform(0.06, 0.12, n), radius=r, self_collision=True)
        m = 1500
        q1 = rng.uniform(-2.0, 2.0, (m, n)).astype(np.float32)
        u = rng.normal(size=(m, n))
        u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
        K = rng.integers(1, 40, m).astype(np.int32)
        batches.append(W.EdgeBatch(rb, q1, u, K))
    osc = oracle.scene_of(sc)
    expect = [oracle.edge_first_collision(b.robot, osc, b.q1, b.dir, b.K, b.step) for b in batches]
    allf = np.concatenate(expect)
    assert (allf == 0).mean() > 0.2 and (allf > 0).sum() > 400 and (allf < 0).sum() > 1000
    got = engine.edge_batches(eid, batches)
    for b, g, e in zip(batches, got, expect):
        assert np.array_equal(g, e), (b.robot.num_dofs, int((g != e).sum()))


def test_edges_many_obstacles(oracle, engine):
    """1,000 axis-aligned boxes (125 groups of 8 in the axis-test tables, the
    boxes of the full test read from global memory): first collisions of
    chain edges and isValid(q1, q2) of xArm6 edges equal the oracle's."""
    rng = np.random.default_rng(77)
    sc = W._boxes(rng, 1000, 0.015, 0.03, 3.0, (0.0, 0.0, 0.5))
    eid = engine.create_env(sc)
    osc = oracle.scene_of(sc)
    rb = R.chain(rng.uniform(0.08, 0.15, 10), radius=0.02, self_collision=True)
    m = 2000
    q1 = rng.uniform(-1.0, 1.0, (m, 10)).astype(np.float32)
    u = rng.normal(size=(m, 10))
    u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    K = rng.integers(1, 60, m).astype(np.int32)
    b = W.EdgeBatch(rb, q1, u, K)
    of = oracle.edge_first_collision(rb, osc, q1, u, K, 0.05)
    assert (of == 0).mean() < 0.5 and (of > 0).sum() > 200 and (of < 0).sum() > 200
    f = engine.edge_batches(eid, [b])[0]
    assert np.array_equal(f, of), int((f != of).sum())
    xa = R.xarm6()
    rid = engine.load_robot(xa)
    w = W.workload2(8192)
    qa, qb = w.q[:4096], (w.q[:4096] + 0.05 * (w.q[4096:] - w.q[:4096])).astype(np.float32)
    v = engine.edge_is_valid(rid, eid, qa, qb)
    ov = oracle.edge_valid(xa, osc, qa, qb)
    assert 0 < v.mean() < 1 and np.array_equal(v, ov), int((v != ov).sum())


@pytest.mark.parametrize("boxes", [0, 3])
def test_edge_first_collision_long_chain(oracle, engine, boxes):
    """A 40-link chain with self-collision (skeletons of 41 points in LDS)
    beside a 10-link one in the same launch, in an empty scene (no axis-test
    groups at all) and in a 3-box scene (one partial group): first
    collisions equal the oracle's."""
    rng = np.random.default_rng(90 + boxes)
    if boxes:
        sc = W._boxes(rng, boxes, 0.1, 0.3, 1.0, (0.0, 0.0, 0.5))
    else:
        sc = W.Scene(np.zeros((0, 3)), np.zeros((0, 3)), np.zeros((0, 4)), np.zeros(0, np.uint8),
                     np.zeros(0, np.float32))
    eid = engine.create_env(sc)
    osc = oracle.scene_of(sc)
    batches = []
    for n, m in ((40, 600), (10, 600)):
        rb = R.chain(rng.uniform(0.03, 0.06, n), radius=0.01, self_collision=True)
        q1 = rng.uniform(-1.2, 1.2, (m, n)).astype(np.float32)
        u = rng.normal(size=(m, n))
        u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
        batches.append(W.EdgeBatch(rb, q1, u, rng.integers(1, 40, m).astype(np.int32)))
    expect = [oracle.edge_first_collision(b.robot, osc, b.q1, b.dir, b.K, b.step) for b in batches]
    allf = np.concatenate(expect)
    assert (allf > 0).sum() > 20 and (allf < 0).sum() > 20
    got = engine.edge_batches(eid, batches)
    for b, g, e in zip(batches, got, expect):
        assert np.array_equal(g, e), (b.robot.num_dofs, int((g != e).sum()))


def test_edge_first_collision_sparse_scene(oracle, engine):
    # few, small obstacles so many edges run to their last state
    rng = np.random.default_rng(11)
    sc = W._boxes(rng, 8, 0.05, 0.1, 1.5)
    eid = engine.create_env(sc)
    rb = R.chain(rng.uniform(0.05, 0.1, 10), radius=0.01, self_collision=True)
    n = 512
    q1 = rng.uniform(-0.3, 0.3, (n, 10)).astype(np.float32)
    u = rng.normal(size=(n, 10)); u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    K = rng.integers(1, 200, n).astype(np.int32)
    b = W.EdgeBatch(rb, q1, u, K)
    f = engine.edge_batches(eid, [b])[0]
    of = oracle.edge_first_collision(rb, oracle.scene_of(sc), q1, u, K, 0.05)
    assert np.array_equal(f, of) and (of == -1).mean() > 0.1


def _engine_with_variant(v):
    import os
    old = os.environ.get("RVS_FAST_VARIANT")
    os.environ["RVS_FAST_VARIANT"] = v
    try:
        return rvs.Engine(device=0)
    finally:
        if old is None:
            del os.environ["RVS_FAST_VARIANT"]
        else:
            os.environ["RVS_FAST_VARIANT"] = old


@pytest.fixture(scope="module")
def engines_by_variant():
    """Engines whose FP32 bulk pass is the lane-refill ("pool"), the
    one-lane-per-configuration ("classic"), the lane-refill with per-lane
    pair queues ("lanes") or the link-major ("links") kernel."""
    e = {"pool": _engine_with_variant("1"), "classic": _engine_with_variant("0"), "lanes": _engine_with_variant("3"),
         "links": _engine_with_variant("4")}
    yield e
    for x in e.values():
        x.close()


@pytest.mark.parametrize("variant", ["pool", "classic", "lanes", "links"])
@pytest.mark.parametrize("wl", ["workload1", "workload2"])
def test_fp32_refine_verdict_exact(oracle, engines_by_variant, wl, variant):
    """FP32 bulk pass + exact refinement: verdicts identical to the reference
    arithmetic, distances within 1e-5 m of the FP64 oracle (and profiles of
    collision-free configurations too), for every bulk kernel."""
    engine = engines_by_variant[variant]
    w = W.workload1(65536) if wl == "workload1" else W.workload2(1 << 18)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, _ = engine.distance(rid, eid, w.q, precision=rvs.PREC_FP32_REFINE)
    refined = engine.last_refined()
    sc = oracle.scene_of(w.scene)
    od, oprof, over, _ = oracle.distance(w.robot, sc, w.q, 32)
    d64, prof64, ver64, _ = oracle.distance(w.robot, sc, w.q, 64)
    print(f"{wl}: refined {refined} of {len(w.q)}; verdict mismatches {(ver != over).sum()}")
    assert (ver == over).all()
    assert np.abs(d - d64).max() <= 1e-5
    ok = (ver == 1) & (ver64 == 1)
    assert np.abs(prof[ok] - prof64[ok]).max() <= 1e-5
    # collision configurations: same first colliding link, same partial profile
    bad = ver == 0
    assert np.abs(prof[bad] - oprof[bad]).max() <= 1e-5
    assert refined < 0.05 * len(w.q)


@pytest.mark.parametrize("variant", ["lanes", "links"])
def test_fp32_refine_queued_kernels_ragged(oracle, engines_by_variant, variant):
    """The per-lane-queue and link-major bulk kernels on ragged shapes: batch
    sizes that leave partial waves, workgroups and rounds (1, 63, 65, 1,000,
    70,001 configurations), robots of 1, 2 and 22 links (the link-major
    kernel launches once per link), scenes of 1, 5 and 40 boxes (a partial
    group, a group and a partial one, 10 groups), a ground box skipped for
    the first links, and non-finite joint values: verdicts equal the
    oracle's, distances and profiles within 1e-5 m, NaN where the oracle has
    NaN."""
    engine = engines_by_variant[variant]
    # (robot, boxes, side lo / hi, placement radius, centre): the 1-link
    # chain's link is fixed along z, crossed by its box in every configuration
    cases = [
        (R.chain([0.4], radius=0.03), 1, 0.05, 0.08, 0.01, (0.04, 0.0, 0.2)),
        (R.chain([0.3, 0.3], radius=0.03), 5, 0.05, 0.15, 0.5, (0.0, 0.0, 0.0)),
        (R.spatial(10, radius=0.025, ground_included=2), 40, 0.05, 0.2, 2.0, (0.0, 0.0, 0.3)),
        (W.workload5(16).robot, 40, 0.1, 0.3, 1.5, (0.0, 0.0, 0.0)),
    ]
    for k, (rb, nbox, lo, hi, rad, cen) in enumerate(cases):
        rng = np.random.default_rng(71 + k)
        sc = W._boxes(rng, nbox, lo, hi, rad, cen)
        if rb.ground_included:
            sc = W.ground_box().concat(sc)
        rid = engine.load_robot(rb)
        eid = engine.create_env(sc)
        osc = oracle.scene_of(sc)
        for n in (1, 63, 65, 1000, 70001):
            q = rng.uniform(-np.pi, np.pi, (n, rb.num_dofs)).astype(np.float32)
            if n > 100:
                q[::37, rb.num_dofs // 2] = np.nan
            print(f"{variant}: {rb.num_links} links, {sc.num_obj} boxes, {n} configurations", flush=True)
            d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
            od, oprof, over, _ = oracle.distance(rb, osc, q, 32)
            assert (ver == over).all(), (rb.num_links, nbox, n)
            assert np.array_equal(np.isnan(prof), np.isnan(oprof)) and np.array_equal(np.isnan(d), np.isnan(od))
            m = ~np.isnan(prof)
            assert np.abs(prof[m] - oprof[m]).max() <= 1e-5, (rb.num_links, nbox, n)
            m = ~np.isnan(d)
            assert np.abs(d[m] - od[m]).max() <= 1e-5, (rb.num_links, nbox, n)


@pytest.mark.parametrize("variant", ["pool", "classic", "lanes", "links"])
@pytest.mark.parametrize("scene", ["dense_overlap", "dense_overlap_wide"])
def test_fp32_refine_first_hit_in_obstacle_order(oracle, engines_by_variant, scene, variant):
    """Overlapping boxes make links cross several boxes, so the walk often
    finds a hit that is not the first in obstacle order; the first one's
    value (0 for a crossing, about -r for an inside end point) is the
    profile's.  Every bulk kernel (obstacle-order search before the hit, or
    the link-major kernel's search of the walk positions after it) gives the
    oracle's verdicts, and its profiles within 1e-5 m, with non-finite joint
    values among the configurations."""
    engine = engines_by_variant[variant]
    wide = scene == "dense_overlap_wide"
    rng = np.random.default_rng(23 if wide else 21)
    rb = R.chain([0.1] + [0.25] * 5, radius=0.03)
    sc = W._boxes(rng, 48, 0.2, 0.5, 0.9, (0, 0, 0.5)) if wide else W._boxes(rng, 24, 0.1, 0.4, 0.9, (0, 0, 0.5))
    q = rng.uniform(-np.pi, np.pi, (65536, 6)).astype(np.float32)
    q[::101, 2] = np.nan
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    print(f"{scene} {variant}: {len(q)} configurations", flush=True)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    od, oprof, over, _ = oracle.distance(rb, oracle.scene_of(sc), q, 32)
    assert (ver == over).all()
    assert np.array_equal(np.isnan(prof), np.isnan(oprof))
    m = ~np.isnan(prof)
    assert np.abs(prof[m] - oprof[m]).max() <= 1e-5
    assert (oprof <= 0).sum() > 10000 and len(np.unique(oprof[oprof <= 0])) > 100


@pytest.mark.parametrize("variant", ["classic", "links"])
def test_fp32_refine_joint_values_beyond_trig_range(oracle, engines_by_variant, variant):
    """The FP32 kinematics takes sines and cosines from the hardware
    functions, whose argument is rounded to turns: joint values beyond 4 pi
    give a NaN skeleton there, so such configurations go to the exact pass;
    values between 2 pi and 4 pi stay in the bulk pass.  Every configuration
    with its first joint beyond 4 pi is refined (one with a later joint beyond
    is refined when the walk reaches that joint: a hit before it ends the
    configuration).  Verdicts equal the reference arithmetic's, distances and
    profiles stay within 1e-5 m of FP64."""
    engine = engines_by_variant[variant]
    w = W.workload2(8192)
    q = w.q.copy()
    far = np.zeros(len(q), bool)
    far[::7] = True
    q[::7, 0] += np.float32(6 * np.pi)                   # 15.7 to 22.0 rad: beyond 4 pi
    q[3::11, 2] -= np.float32(2 * np.pi)                 # 6.1 to 10.2 rad in magnitude: within 4 pi
    q[5::13, 4] = np.float32(-4.2 * np.pi)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    refined = engine.last_refined()
    sc = oracle.scene_of(w.scene)
    od, oprof, over, _ = oracle.distance(w.robot, sc, q, 32)
    d64, prof64, _, _ = oracle.distance(w.robot, sc, q, 64)
    print(f"{variant}: refined {refined} of {len(q)} ({far.sum()} with the first joint beyond 4 pi)")
    assert refined >= far.sum()
    assert (ver == over).all()
    assert np.abs(d - d64).max() <= 1e-5
    ok = ver == 1
    assert np.abs(prof[ok] - prof64[ok]).max() <= 1e-5


@pytest.mark.parametrize("variant", ["pool", "classic", "lanes", "links"])
@pytest.mark.parametrize("far_boxes", [0, 199])
def test_fp32_refine_from_the_first_uncertain_link(oracle, engines_by_variant, far_boxes, variant):
    """The exact pass recomputes a flagged configuration from the first link
    whose decision was uncertain; the links before it keep the bulk pass's
    values.  Planar 2-DOF at q0 = 0: link 0 lies on the x axis, more than
    0.5 m from every box; link 1 ends within 8e-5 m of contact with the box
    above it (lo.y = 0.5), so every configuration is flagged at link 1 only.
    Link 1's value must be the reference arithmetic's (exact pass), link 0's
    within 1e-5 m of it, the verdicts and distances the reference's (d the
    smaller link value, or 0 at a hit).  With 199 far boxes the 400 pairs
    exceed the all-pairs refinement's limit, so the round-based form runs."""
    engine = engines_by_variant[variant]
    rb = R.planar_2dof(radius=0.02)
    dims = [[1.3, 0.5, 1.0]] + [[0.2, 0.2, 0.2]] * far_boxes
    pos = [[1.85, 0.75, 0.0]] + [[-3.0 + 0.3 * (k % 20), -3.0 + 0.3 * (k // 20), 4.0] for k in range(far_boxes)]
    sc = W.Scene(dims, pos, [[1, 0, 0, 0]] * (1 + far_boxes), [0] * (1 + far_boxes), [W.MAX_DISTANCE] * (1 + far_boxes))
    assert sc.aabb[0, 1] == np.float32(0.5)
    rng = np.random.default_rng(91 + far_boxes)
    delta = rng.uniform(-8e-5, 8e-5, 4096)
    q = np.stack([np.zeros(4096), np.arcsin(0.48 + delta)], 1).astype(np.float32)
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc)
    d, prof, ver, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    refined = engine.last_refined()
    od, oprof, over, _ = oracle.distance(rb, oracle.scene_of(sc), q, 32)
    print(f"{far_boxes} far boxes, {variant}: refined {refined} of {len(q)}, free {ver.mean():.3f}")
    assert refined == len(q)
    assert 0 < over.mean() < 1
    assert (ver == over).all()
    assert ulps(prof[:, 1], oprof[:, 1]).max() <= 2
    assert np.abs(prof[:, 0] - oprof[:, 0]).max() <= 1e-5 and (prof[:, 0] > 0.5).all()
    free = ver == 1
    assert np.array_equal(d[free], np.minimum(prof[free, 0], prof[free, 1])) and (d[~free] == 0).all()
    assert np.abs(d - od).max() <= 1e-5


@pytest.mark.parametrize("which", ["xarm6", "chain22", "planar2"])
def test_enclosing_radii(oracle, engine, which):
    if which == "xarm6":
        rb, q = R.xarm6(), W.workload2(8192).q
    elif which == "chain22":
        w = W.workload5(4096)
        rb, q = w.robot, w.q
    else:
        w = W.workload1(8192)
        rb, q = w.robot, w.q
    rid = engine.load_robot(rb)
    got = engine.enclosing_radii(rid, q)
    ref = oracle.enclosing_radii(rb, q)
    assert got.shape == ref.shape
    assert ulps(got, ref).max() <= 2
    assert (got == ref).mean() > 0.999


def _spine_inputs(which, n, seed):
    rng = np.random.default_rng(seed)
    if which == "xarm6":
        rb, q = R.xarm6(), W.workload2(n).q
    elif which == "chain22":
        w = W.workload5(n)
        rb, q = w.robot, w.q
    else:
        w = W.workload1(n)
        rb, q = w.robot, w.q
    u = rng.normal(size=q.shape)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    q_e = (q + np.pi * u).astype(np.float32)
    d = rng.uniform(0.005, 0.3, n).astype(np.float32)
    d[rng.random(n) < 0.02] = 0.0                                   # starts in contact: trapped
    prof = (d[:, None] + rng.uniform(0, 0.2, (n, rb.num_links))).astype(np.float32)
    return rb, q, d, prof, q_e


@pytest.mark.parametrize("which", ["xarm6", "chain22", "planar2"])
@pytest.mark.parametrize("num_iter,expanded", [(1, True), (5, True), (5, False)])
def test_extend_spines(oracle, engine, which, num_iter, expanded):
    """RBTConnect::extendSpine batch against the oracle: statuses and end
    states identical bit for bit on every spine."""
    rb, q, d, prof, q_e = _spine_inputs(which, 8192, 41)
    rid = engine.load_robot(rb)
    qn, st = engine.extend_spines(rid, q, d, prof, q_e, num_iter=num_iter, expanded=expanded)
    oqn, ost = oracle.extend_spines(rb, q, d, prof, q_e, num_iter=num_iter, expanded=expanded)
    same = (qn == oqn).all(1)
    print(f"{which} iter={num_iter} expanded={expanded}: status {np.bincount(st, minlength=4)[1:]}, "
          f"status mismatches {(st != ost).sum()}, states identical {same.mean():.5f}, "
          f"max diff {np.abs(qn - oqn).max():.3g}")
    bad = np.nonzero((st != ost) | ~same)[0]
    assert len(bad) == 0, f"spines differing from the oracle: {bad[:16].tolist()}"
    assert (st == 2).any() and (st == 1).any()


@pytest.mark.parametrize("dofs,n", [(16, 60001), (26, 1000), (30, 20000), (32, 30000), (64, 20000)])
def test_extend_spines_batch_forms(oracle, engine, dofs, n):
    """The joint distances in LDS (small batches) or worked out at each use
    (where they would cost resident workgroups), 64, 32 and 16 lanes a
    workgroup: a batch equals its parts bit for bit, and its head the oracle."""
    rng = np.random.default_rng(dofs)
    rb = R.chain(rng.uniform(0.05, 0.2, dofs), radius=0.03)
    q = rng.uniform(-0.5, 0.5, (n, dofs)).astype(np.float32)
    v = rng.normal(size=(n, dofs))
    q_e = (q + 2.0 * v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)
    d = rng.uniform(0.005, 0.5, n).astype(np.float32)
    prof = (d[:, None] + rng.uniform(0, 0.3, (n, dofs))).astype(np.float32)
    rid = engine.load_robot(rb)
    qn, st = engine.extend_spines(rid, q, d, prof, q_e, num_iter=3)
    parts = [engine.extend_spines(rid, q[k:k + 1900], d[k:k + 1900], prof[k:k + 1900], q_e[k:k + 1900], num_iter=3)
             for k in range(0, n, 1900)]
    assert np.array_equal(qn, np.concatenate([p[0] for p in parts]))
    assert np.array_equal(st, np.concatenate([p[1] for p in parts]))
    oqn, ost = oracle.extend_spines(rb, q[:300], d[:300], prof[:300], q_e[:300], num_iter=3)
    assert np.array_equal(qn[:300], oqn) and np.array_equal(st[:300], ost)
    assert (qn != q).any()


@pytest.mark.parametrize("dofs,boxes,n", [(16, 20, 60001), (22, 100, 40000), (64, 5, 20000)])
def test_extend_gen_spines_batch_forms(oracle, engine, dofs, boxes, n):
    """The same for underestimation layers."""
    rng = np.random.default_rng(dofs + boxes)
    rb = R.chain(rng.uniform(0.05, 0.2, dofs), radius=0.02)
    sc = _boxes_around(rng, rb, boxes, 0.05, 0.3, 0.08 * dofs, clearance=0.1)
    root = np.zeros(dofs, np.float32)
    v = rng.normal(size=(n, dofs))
    q_e = (np.pi * v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    kw = dict(num_layers=3, num_iter=2, d_crit=0.01)
    got = engine.extend_gen_spines(rid, eid, root, q_e, **kw)
    parts = [engine.extend_gen_spines(rid, eid, root, q_e[k:k + 3900], **kw) for k in range(0, n, 3900)]
    for i in range(3):
        assert np.array_equal(got[i], np.concatenate([p[i] for p in parts]))
    want = oracle.extend_gen_spines(rb, oracle.scene_of(sc), root, q_e[:200], **kw)
    for g, o in zip(got, want):
        assert np.array_equal(g[:200], o)
    assert (got[2] > 0).any() and (got[0] != root).any()


@pytest.mark.parametrize("use_real_dist", [False, True])
@pytest.mark.parametrize("num_iter", [1, 5])
def test_extend_gen_spines(oracle, engine, use_real_dist, num_iter):
    """RGBTConnect::extendGenSpine from one root towards 4096 targets (a
    generalized bur) against the oracle's composition of the same steps."""
    w = W.workload2(4096)
    sc = oracle.scene_of(w.scene)
    d, _, ver, _ = oracle.distance(w.robot, sc, w.q, 32)
    root = w.q[np.nonzero((ver == 1) & (d > 0.06))[0][0]]
    rng = np.random.default_rng(42)
    u = rng.normal(size=(4096, 6))
    q_e = (root + np.pi * u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    qn, st, dd = engine.extend_gen_spines(rid, eid, root, q_e, num_layers=5, num_iter=num_iter,
                                          use_real_dist=use_real_dist, d_crit=0.03)
    oqn, ost, odd = oracle.extend_gen_spines(w.robot, sc, root, q_e, num_layers=5, num_iter=num_iter,
                                             use_real_dist=use_real_dist, d_crit=0.03)
    same = (qn == oqn).all(1) & (dd == odd)
    print(f"real={use_real_dist} iter={num_iter}: status {np.bincount(st, minlength=4)[1:]}, "
          f"status mismatches {(st != ost).sum()}, identical {same.mean():.5f}")
    bad = np.nonzero((st != ost) | ~same)[0]
    assert len(bad) == 0, f"spines differing from the oracle: {bad[:16].tolist()}"
    # the root in contact: every target trapped at the root with d = 0
    root_bad = w.q[np.nonzero(ver == 0)[0][0]]
    qn, st, dd = engine.extend_gen_spines(rid, eid, root_bad, q_e[:64])
    assert (st == 2).all() and (qn == root_bad[None]).all() and (dd == 0).all()


@pytest.mark.parametrize("dofs,boxes,n,num_iter", [(6, 1, 1, 1), (10, 250, 65, 5), (22, 90, 70, 1), (22, 1000, 33, 2)])
def test_extend_gen_spines_plane_tiles(oracle, engine, dofs, boxes, n, num_iter):
    """Underestimation layers against plane sets of one tile and of several
    (down to one link a tile and fewer lanes a workgroup), ragged batches:
    identical to the oracle's composition."""
    rng = np.random.default_rng(95 + boxes)
    rb = R.xarm6() if dofs == 6 else R.chain(rng.uniform(0.05, 0.1, dofs), radius=0.02)
    u = rng.normal(size=(boxes, 3))
    sc = W._boxes(rng, boxes, 0.02, 0.1, 2.5)
    sc = W.Scene(sc.dim, 2.6 * u / np.linalg.norm(u, axis=1, keepdims=True), sc.quat, sc.is_ground, sc.min_dist_tol)
    root = np.zeros(dofs, np.float32)
    v = rng.normal(size=(n, dofs))
    q_e = (np.pi * v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    got = engine.extend_gen_spines(rid, eid, root, q_e, num_layers=4, num_iter=num_iter, d_crit=0.03)
    want = oracle.extend_gen_spines(rb, oracle.scene_of(sc), root, q_e, num_layers=4, num_iter=num_iter, d_crit=0.03)
    for g, o in zip(got, want):
        assert (g == o).all()
    assert (got[2] > 0).any()


@pytest.mark.parametrize("eps_step", [0.1, 0.02])
def test_edge_self_collision(oracle, engine, eps_step):
    """Capsule part of xArm6::checkSelfCollision(q1, q2) for 16384 edges
    against the oracle: verdicts identical, returned states identical."""
    rb = R.xarm6(radius=0.05)
    rng = np.random.default_rng(61)
    lim = np.asarray(rb.limits, np.float64)
    q1 = (lim[:, 0] + rng.random((16384, 6)) * (lim[:, 1] - lim[:, 0])).astype(np.float32)
    u = rng.normal(size=q1.shape)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    q2 = (q1 + rng.uniform(0.05, 3.0, len(q1))[:, None] * u).astype(np.float32)
    rid = engine.load_robot(rb)
    col, out = engine.edge_self_collision(rid, q1, q2, eps_step)
    ocol, oout = oracle.edge_self_collision(rb, q1, q2, eps_step)
    same = (out == oout).all(1)
    print(f"eps {eps_step}: collide {col.sum()} of {len(col)}, verdict mismatches {(col != ocol).sum()}, "
          f"states identical {same.mean():.5f}")
    bad = np.nonzero((col != ocol) | ~same)[0]
    assert len(bad) == 0, f"edges differing from the oracle: {bad[:16].tolist()}"
    assert col.sum() > 100


def _boxes_only(scene):
    keep = scene.is_ground == 0
    return W.Scene(scene.dim[keep], scene.pos[keep], scene.quat[keep], scene.is_ground[keep],
                   scene.min_dist_tol[keep])


def test_underestimation_moving(oracle, engine):
    """Moving-plane underestimation against the oracle, bit for bit."""
    w = W.workload2(1 << 15)
    sc = oracle.scene_of(w.scene)
    root = np.zeros(6, np.float32)
    _, _, _, np0 = oracle.distance(w.robot, sc, root[None], 32, want_np=True)
    rng = np.random.default_rng(81)
    q = (root + rng.uniform(-0.6, 0.6, (1 << 15, 6))).astype(np.float32)
    mv = rng.uniform(0, 0.5, w.scene.num_obj).astype(np.float32)
    mv[w.scene.is_ground == 1] = 0
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    d, prof, st = engine.underestimation_moving(rid, eid, q, np0[0], mv, 0.07)
    od, oprof, ost = oracle.underestimation_moving(w.robot, sc, q, np0[0], mv, 0.07)
    print(f"stored {st.mean():.3f}")
    assert (st == ost).all()
    assert ulps(d, od).max() <= 2 and (d == od).mean() > 0.999
    ok = st == 1
    assert ulps(prof[ok], oprof[ok]).max() <= 2


@pytest.mark.parametrize("self_collision", [False, True])
@pytest.mark.parametrize("v", [0.0, 0.1])
def test_trajectory_is_safe(oracle, engine, v, self_collision):
    """AbstractTrajectory::isSafe over 8192 straight candidate trajectories
    of 60 points from one current state, against the oracle."""
    w = W.workload2(64)
    scene = _boxes_only(w.scene)
    sc = oracle.scene_of(scene)
    rb = w.robot
    root = np.zeros(6, np.float32)
    _, p0, _, np0 = oracle.distance(rb, sc, root[None], 32, want_np=True)
    rng = np.random.default_rng(82)
    T, K = 8192, 60
    u = rng.normal(size=(T, 6))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    reach = rng.uniform(0.1, 2.5, T)
    s = np.linspace(0, 1, K + 1)[1:]
    pts = (root[None, None] + (reach[:, None, None] * s[None, :, None]) * u[:, None, :]).astype(np.float32)
    mv = np.full(scene.num_obj, v, np.float32)
    rid = engine.load_robot(rb)
    eid = engine.create_env(scene)
    safe = engine.trajectory_is_safe(rid, eid, pts, root, p0[0], np0[0], mv, t_iter=0.0, time_step=0.01,
                                     self_collision=self_collision)
    osafe = oracle.traj_safe(rb, sc, pts, root, p0[0], np0[0], mv, 0.0, 0.01,
                             pairs=rb.self_pairs if self_collision else None)
    print(f"v={v} self={self_collision}: safe {safe.sum()} of {T}, mismatches {(safe != osafe).sum()}")
    bad = np.nonzero(safe != osafe)[0]
    assert len(bad) == 0, f"trajectories differing from the oracle: {bad[:16].tolist()}"
    assert 0 < safe.sum() < T


@pytest.mark.parametrize("law", [0, 1, 2, 3])
def test_env_motion_laws(oracle, engine, law):
    """Environment::updateEnvironment on the GPU against the oracle: 300
    steps of 10 ms; the bounds the queries read follow the boxes, and a query
    on the moved environment equals one on a fresh environment built at the
    new positions."""
    rng = np.random.default_rng(95 + law)
    n = 24
    pos = np.zeros((0, 3))
    while len(pos) < n:
        c = np.stack([rng.uniform(-0.8, 0.8, 4 * n), rng.uniform(-0.8, 0.8, 4 * n), rng.uniform(0.05, 1.0, 4 * n)], 1)
        rr = np.linalg.norm(c - np.array([0, 0, 0.267]), axis=1)
        c = c[(rr < 0.95) & (rr > 0.35) & (np.hypot(c[:, 0], c[:, 1]) > 0.35)]
        pos = np.concatenate([pos, c])[:n]
    dim = rng.uniform(0.05, 0.2, (n, 3))
    quat = np.tile([1.0, 0, 0, 0], (n, 1))
    quat[::3] = [0.9238795, 0.0, 0.0, 0.3826834]        # some rotated boxes
    dyn = np.ones(n, np.uint8)
    dyn[::4] = 0
    scene = W.Scene(dim, pos, quat, np.zeros(n, np.uint8), np.full(n, W.MAX_DISTANCE), dynamic=dyn)
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    vel, vmax = (0.5 * u).astype(np.float32), np.full(n, 0.5, np.float32)
    eid = engine.create_env(scene)
    kw = dict(ws_center=(0, 0, 0.267), ws_radius=1.0, base_radius=0.15, robot_max_vel=3.0)
    engine.set_motion_law(eid, law, vel, vmax, **kw)
    m = oracle.MotionState(law, scene.pos, vel, vmax, dyn, **kw)
    gp, gv = engine.env_step(eid, 0.01, 150)
    gp, gv = engine.env_step(eid, 0.01, 150)
    op, ov = m.step(0.01, 300)
    err = np.abs(gp - op).max()
    print(f"law {law}: max position difference {err:.3g}, identical {(gp == op).all()}")
    if law == 1:
        assert err < 1e-4            # device and host sin / cos / atan2 may differ in the last bit
    else:
        assert (gp == op).all() and (gv == ov).all()
    moved = W.Scene(dim, gp, quat, np.zeros(n, np.uint8), np.full(n, W.MAX_DISTANCE))
    assert (engine.env_bounds(eid) == moved.aabb).all()
    rb = R.xarm6()
    rid = engine.load_robot(rb)
    q = W.workload2(4096).q
    d1, p1, v1, _ = engine.distance(rid, eid, q)
    d2, p2, v2, _ = engine.distance(rid, engine.create_env(moved), q)
    assert (d1 == d2).all() and (p1 == p2).all() and (v1 == v2).all()
    # the FP32 path's broad phase reads group boxes that the step recomputed
    d3, _, v3, _ = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    od, _, ov, _ = oracle.distance(rb, oracle.scene_of(moved), q, 32)
    assert (v3 == ov).all() and np.abs(d3 - od).max() <= 1e-5


def test_fp32_refine_after_env_update(oracle, engine):
    """Boxes moved in place (rvs_env_update) far across the scene: the FP32
    path's grouped broad phase keeps its walk order but rebuilds its group
    boxes, so verdicts stay identical to the oracle's on the moved scene and
    distances within 1e-5 m."""
    w = W.workload2(1 << 16)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    engine.distance(rid, eid, w.q, precision=rvs.PREC_FP32_REFINE)
    rng = np.random.default_rng(41)
    idx = np.arange(1, len(w.scene.dim), dtype=np.int32)          # every box but the ground
    pos = w.scene.pos.copy()
    pos[idx] = pos[idx][rng.permutation(len(idx))] + rng.uniform(-0.2, 0.2, (len(idx), 3))
    engine.update_env(eid, idx, pos[idx])
    moved = W.Scene(w.scene.dim, pos, w.scene.quat, w.scene.is_ground, w.scene.min_dist_tol)
    d, _, v, _ = engine.distance(rid, eid, w.q, precision=rvs.PREC_FP32_REFINE)
    od, _, ov, _ = oracle.distance(w.robot, oracle.scene_of(moved), w.q, 32)
    print(f"after update: collision-free {v.mean():.3f}, verdict mismatches {(v != ov).sum()}")
    assert (v == ov).all() and np.abs(d - od).max() <= 1e-5


@pytest.mark.parametrize("n", [1, 7, 300, 5000, 70000])
def test_small_batches_one_wave_per_configuration(oracle, engine, n):
    """Small reference-arithmetic batches run one wave per configuration;
    results (distances, profiles, verdicts, nearest points) are those of the
    one-lane-per-configuration kernel bit for bit (which walks batches of
    65,536 configurations or more in the walk order)."""
    w = W.workload2(n)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene)
    engine.set_small_batch(1 << 20)
    a = engine.distance(rid, eid, w.q, want_nearest=True)
    engine.set_small_batch(0)
    b = engine.distance(rid, eid, w.q, want_nearest=True)
    engine.set_small_batch(16384)
    for x, y in zip(a, b):
        assert np.array_equal(x, y, equal_nan=True)
    od, oprof, over, onp = oracle.distance(w.robot, oracle.scene_of(w.scene), w.q, 32, want_np=True)
    assert (a[2] == over).all() and ulps(a[0], od).max() <= 2


@pytest.mark.parametrize("oriented", [True, False])
def test_small_batches_many_obstacles(oracle, engine, oriented):
    """One wave per configuration over 512 boxes: the obstacles go in rounds
    of 64 with the wave's running minimum as the broad-phase bound, and a
    link ends after the first round with a hit.  Results equal the
    one-lane-per-configuration kernel's bit for bit (configurations free,
    colliding at link 0 and colliding further out, first hits beyond the
    first round)."""
    w = W.workload5(300)
    rid = engine.load_robot(w.robot)
    eid = engine.create_env(w.scene, rvs.ENV_OBB if oriented else rvs.ENV_AABB)
    engine.set_small_batch(1 << 20)
    a = engine.distance(rid, eid, w.q)
    engine.set_small_batch(0)
    b = engine.distance(rid, eid, w.q)
    engine.set_small_batch(16384)
    for x, y in zip(a[:3], b[:3]):
        assert np.array_equal(x, y, equal_nan=True)
    od, oprof, over, _ = oracle.distance(w.robot, oracle.scene_of(w.scene, oriented=oriented), w.q, 32)
    print(f"oriented={oriented}: collision-free {a[2].mean():.3f}")
    assert (a[2] == over).all() and ulps(a[0], od).max() <= 2 and ulps(a[1], oprof).max() <= 2


@pytest.mark.parametrize("oriented", [False, True])
@pytest.mark.parametrize("dofs,boxes,n", [(2, 0, 5), (6, 1, 1), (6, 16, 3), (6, 170, 67), (10, 102, 18), (10, 103, 18),
                                          (22, 46, 33), (40, 7, 9), (2, 1, 4097), (6, 16, 4099), (6, 40, 4101),
                                          (40, 6, 4098), (10, 25, 4097)])
def test_distances_by_pairs_sizes(engine, dofs, boxes, n, oriented):
    """16 or 64 lanes per configuration against one lane, bit for bit, with and
    without nearest points: from no obstacle to the row's 1,024 pairs and past
    them (103 boxes of ten links: link by link), more segments than lanes,
    ragged waves, contacts with several boxes, links that skip ground boxes,
    finite tolerances, NaN and infinite joints."""
    rng = np.random.default_rng(100 * dofs + boxes)
    rb = {2: R.planar_2dof, 6: R.xarm6}.get(dofs, lambda: R.chain(rng.uniform(0.05, 0.2, dofs), radius=0.03,
                                                                   ground_included=2))()
    sc = W._boxes(rng, boxes, 0.02, 0.3, 1.5, rotated=oriented)
    if boxes > 2:
        gnd, tol = sc.is_ground.copy(), sc.min_dist_tol.copy()
        gnd[::7] = 1
        tol[1::5] = 0.1
        sc = W.Scene(sc.dim, sc.pos, sc.quat, gnd, tol)
    q = rng.uniform(-np.pi, np.pi, (n, rb.num_dofs)).astype(np.float32)
    q[n // 2, 0] = np.nan
    q[n - 1, 1] = np.inf
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc, rvs.ENV_OBB if oriented else rvs.ENV_AABB)
    try:
        for near in ((False, True) if boxes else (False,)):
            engine.set_small_batch(1 << 20)
            a = engine.distance(rid, eid, q, want_nearest=near)
            engine.set_small_batch(0)
            b = engine.distance(rid, eid, q, want_nearest=near)
            for x, y in zip(a, b):
                assert (x is None and y is None) or np.array_equal(x, y, equal_nan=True)
    finally:
        engine.set_small_batch(16384)


@pytest.mark.parametrize("dofs,n,scale", [(6, 1, 1.0), (6, 63, 1.0), (3, 65, 1.0), (22, 200, 1.0), (40, 130, 1.0),
                                          (14, 70, 300.0), (14, 70, 1e-3), (7, 16, 1.0), (7, 17, 1.0), (9, 64, 1.0),
                                          (9, 65, 1.0), (9, 65536, 1.0)])
def test_self_collision_minimum_of_pairs(engine, dofs, n, scale):
    """The smallest pair distance, found without most of the pairs (or, with
    few, from every one: both sides of that rule's lines), against the
    smallest of all of them, bit for bit: one pair to 741, radii that
    differ, pairs in no order and twice, long and tiny links (coordinates of a
    kilometre, links below the equality threshold), NaN and infinite joints,
    ragged waves."""
    rng = np.random.default_rng(7 * dofs + n)
    if dofs == 6:
        rb = R.xarm6(radius=[0.08, 0.02, 0.05, 0.03, 0.06, 0.01])
    else:
        rb = R.chain(scale * rng.uniform(0.05, 0.3, dofs), radius=scale * rng.uniform(0.01, 0.06, dofs),
                     self_collision=True)
        pairs = [rb.self_pairs[k] for k in rng.permutation(len(rb.self_pairs))]
        rb.self_pairs = pairs + pairs[: len(pairs) // 3]
    q = rng.uniform(-np.pi, np.pi, (n, rb.num_dofs)).astype(np.float32)
    if n > 60:
        q[:20] *= 0.1
        q[n // 2, 0] = np.nan
        q[n - 1, 1] = np.inf
    rid = engine.load_robot(rb)
    lo, free = engine.self_collision(rid, q)
    all_pairs = engine.self_distance(rid, q)
    want = np.fmin.reduce(np.concatenate([np.full((n, 1), 1000.0, np.float32), all_pairs], 1), axis=1)
    assert np.array_equal(lo, want) and np.array_equal(free, (want >= 0).astype(np.uint8))


@pytest.mark.parametrize("dofs,boxes,points,traj", [(6, 1, 1, 5), (6, 16, 64, 70), (6, 70, 65, 40), (10, 9, 130, 30),
                                                    (22, 12, 20, 20), (2, 3, 1025, 9), (40, 5, 3, 7)])
@pytest.mark.parametrize("self_collision", [False, True])
def test_trajectory_is_safe_sizes(oracle, engine, dofs, boxes, points, traj, self_collision):
    """Chunks of 64 points and their remainders, more points than the time
    table holds, from two to forty joints (segments, radii rows and planes
    beyond a wave's lanes), moving obstacles: equal to the oracle's walk, with
    both outcomes where there are trajectories enough."""
    rng = np.random.default_rng(1000 * dofs + points)
    if dofs == 6:
        rb = R.xarm6()
    elif dofs == 2:
        rb = R.planar_2dof()
    else:
        rb = R.chain(rng.uniform(0.08, 0.15, dofs), radius=0.02, self_collision=True)
    sc = _boxes_around(rng, rb, boxes, 0.05, 0.2, {2: 1.2, 6: 0.7}.get(dofs, 0.07 * dofs + 0.1))
    osc = oracle.scene_of(sc)
    root = np.zeros(dofs, np.float32)
    _, p0, ok, np0 = oracle.distance(rb, osc, root[None], 32, want_np=True)
    assert ok[0] == 1
    v = rng.normal(size=(traj, dofs))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    s = np.linspace(0, 1, points + 1)[1:]
    pts = (rng.uniform(0.05, 2.5, traj)[:, None, None] * s[None, :, None] * v[:, None, :]).astype(np.float32)
    mv = rng.uniform(0, 0.05, boxes).astype(np.float32)
    dt = 1.0 / points
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    safe = engine.trajectory_is_safe(rid, eid, pts, root, p0[0], np0[0], mv, t_iter=0.1, time_step=dt,
                                     self_collision=self_collision)
    osafe = oracle.traj_safe(rb, osc, pts, root, p0[0], np0[0], mv, 0.1, dt,
                             pairs=rb.self_pairs if self_collision else None)
    assert traj < 20 or 0.05 < osafe.mean() < 0.95
    assert np.array_equal(safe, osafe)


@pytest.mark.parametrize("points", [1025, 2500])
def test_trajectory_points_past_the_time_table(oracle, engine, points):
    """More points than the time table holds, with reference states along the
    way: equal to the oracle's walk, both outcomes among them."""
    rng = np.random.default_rng(points)
    rb = R.xarm6()
    sc = _boxes_around(rng, rb, 12, 0.05, 0.2, 0.7)
    osc = oracle.scene_of(sc)
    root = np.zeros(6, np.float32)
    _, p0, ok, np0 = oracle.distance(rb, osc, root[None], 32, want_np=True)
    assert ok[0] == 1
    v = rng.normal(size=(40, 6))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    s = np.linspace(0, 1, points + 1)[1:]
    pts = (rng.uniform(0.05, 2.5, 40)[:, None, None] * s[None, :, None] * v[:, None, :]).astype(np.float32)
    mv = rng.uniform(0, 0.05, 12).astype(np.float32)
    dt = 1.0 / points
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    safe = engine.trajectory_is_safe(rid, eid, pts, root, p0[0], np0[0], mv, t_iter=0.1, time_step=dt)
    osafe = oracle.traj_safe(rb, osc, pts, root, p0[0], np0[0], mv, 0.1, dt)
    assert 0.1 < osafe.mean() < 0.9
    assert np.array_equal(safe, osafe)


def test_trajectory_cost_grows_with_its_points(engine):
    """Eight times the points of a trajectory that stays near its reference
    state take at most twenty times as long (64 times if every chunk added its
    times up from the start)."""
    import time

    rb = R.xarm6()
    sc = W._boxes(np.random.default_rng(3), 4, 0.05, 0.1, 0.2, center=(0.0, 0.0, 3.0))
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    root = np.zeros(6, np.float32)
    _, p0, _, np0 = engine.distance(rid, eid, root[None], want_nearest=True)

    def cost(points):
        pts = np.zeros((1, points, 6), np.float32)
        best = float("inf")
        for _ in range(4):
            t0 = time.perf_counter()
            safe = engine.trajectory_is_safe(rid, eid, pts, root, p0[0], np0[0], np.zeros(4, np.float32),
                                             time_step=1e-4)
            best = min(best, time.perf_counter() - t0)
            assert safe[0] == 1
        return best

    short, long = cost(4096), cost(32768)
    print(f"4,096 points {1e6 * short:.0f} us, 32,768 points {1e6 * long:.0f} us")
    assert long < 20 * short


@pytest.mark.parametrize("boxes", [1, 8, 9, 63, 64, 65, 130])
@pytest.mark.parametrize("dofs", [1, 6, 22])
def test_edge_first_collision_obstacle_marks(oracle, engine, boxes, dofs):
    """Obstacle counts at the edges of the table's batches, groups and 64-bit
    marks, robots of one joint to 22 with self pairs, ground boxes skipped by
    the first links, NaN rows, ragged waves: first indices and edge validity
    equal to the oracle's, with both outcomes among boxes enough."""
    rng = np.random.default_rng(10 * boxes + dofs)
    rb = R.xarm6(ground_included=2) if dofs == 6 else R.chain(rng.uniform(0.1, 0.4, dofs), radius=0.03,
                                                              ground_included=min(2, dofs), self_collision=dofs > 1)
    sc = _boxes_around(rng, rb, boxes, 0.05, 0.3, 0.8 if dofs == 6 else 0.15 * dofs + 0.4)
    sc = W.Scene(sc.dim, sc.pos, sc.quat, (rng.random(boxes) < 0.2).astype(np.uint8), sc.min_dist_tol)
    osc = oracle.scene_of(sc)
    n = 67
    q1 = rng.uniform(-0.5, 0.5, (n, dofs)).astype(np.float32)
    u = rng.normal(size=(n, dofs))
    u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    K = rng.integers(0, 40, n).astype(np.int32)
    q1[5, dofs - 1] = np.nan
    rid, eid = engine.load_robot(rb), engine.create_env(sc)
    got = engine.edge_first_collision(eid, np.full(n, rid, np.int32), q1, u, K)
    want = oracle.edge_first_collision(rb, osc, q1, u, K, 0.05)
    # (the single joint turns its link about its own axis)
    few = dofs == 1 or boxes < (8 if dofs == 6 else 30)
    assert few or ((want >= 0).mean() > 0.05 and (want < 0).mean() > 0.05 and (want > 0).any())
    assert np.array_equal(got, want)
    q2 = (q1 + 0.8 * u).astype(np.float32)
    ovalid = oracle.edge_valid(rb, osc, q1, q2)
    assert few or 0.02 < ovalid.mean() < 0.98
    assert np.array_equal(engine.edge_is_valid(rid, eid, q1, q2), ovalid)


@pytest.mark.parametrize("oriented", [False, True])
@pytest.mark.parametrize("dofs,boxes,n", [(2, 0, 3), (6, 1, 65), (6, 31, 300), (10, 32, 257), (10, 33, 64), (22, 64, 90),
                                          (6, 100, 513)])
def test_is_valid_obstacle_marks(oracle, engine, dofs, boxes, n, oriented):
    """Obstacle counts at the edges of the 32-bit marks and their remainders,
    both precisions, ground boxes skipped by the first links, ragged waves,
    NaN and infinite joints: flags equal to the oracle's, with both among
    boxes enough."""
    rng = np.random.default_rng(3 * boxes + dofs)
    rb = {2: R.planar_2dof, 6: lambda: R.xarm6(ground_included=2)}.get(
        dofs, lambda: R.chain(rng.uniform(0.1, 0.2, dofs), radius=0.03, ground_included=1))()
    sc = _boxes_around(rng, rb, boxes, 0.05, 0.25, 0.9 if dofs == 6 else 0.08 * dofs + 0.3)
    quat = rng.normal(size=(boxes, 4)) if oriented else sc.quat
    sc = W.Scene(sc.dim, sc.pos, quat / np.linalg.norm(quat, axis=1, keepdims=True),
                 (rng.random(boxes) < 0.2).astype(np.uint8), sc.min_dist_tol)
    q = rng.uniform(-np.pi, np.pi, (n, rb.num_dofs)).astype(np.float32)
    q[n // 2, 0] = np.nan
    q[n - 1, 1] = np.inf
    rid = engine.load_robot(rb)
    eid = engine.create_env(sc, rvs.ENV_OBB if oriented else rvs.ENV_AABB)
    osc = oracle.scene_of(sc, oriented=oriented)
    want = oracle.is_valid(rb, osc, q)
    assert boxes < 30 or 0.02 < want.mean() < 0.98
    assert np.array_equal(engine.is_valid(rid, eid, q), want)
    assert np.array_equal(engine.is_valid(rid, eid, q, precision=rvs.PREC_FP64), oracle.is_valid(rb, osc, q, 64))


@pytest.mark.parametrize("gripper", [0.0, 0.12])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_joint_that_is_no_number(oracle, engine, gripper, bad):
    """One joint of an xArm6 NaN or infinite, each in turn: verdicts, flags and
    first hits equal to the oracle's in every arithmetic."""
    rng = np.random.default_rng(77)
    rb = R.xarm6(gripper_length=gripper)
    sc = _boxes_around(rng, rb, 40, 0.05, 0.3, 0.8)
    osc = oracle.scene_of(sc)
    n = 600
    q = rng.uniform(-1.0, 1.0, (n, 6)).astype(np.float32)
    q[np.arange(n), np.arange(n) % 6] = bad
    rid, eid = engine.load_robot(rb), engine.create_env(sc, rvs.ENV_AABB)
    od, oprof, over, _ = oracle.distance(rb, osc, q, 32)
    assert all(0 < over[j::6].mean() < 1 for j in (4, 5))
    for prec in (rvs.PREC_REF32, rvs.PREC_FP64, rvs.PREC_FP32_REFINE):
        d, prof, ver, _ = engine.distance(rid, eid, q, precision=prec)
        assert np.array_equal(ver, over), prec
    assert np.array_equal(engine.is_valid(rid, eid, q), oracle.is_valid(rb, osc, q))
    u = rng.normal(size=(n, 6))
    u = (u / np.linalg.norm(u, axis=1, keepdims=True)).astype(np.float32)
    K = np.full(n, 20, np.int32)
    want = oracle.edge_first_collision(rb, osc, q, u, K, 0.05)
    assert np.array_equal(engine.edge_first_collision(eid, np.full(n, rid, np.int32), q, u, K), want)
    q2 = (q + 0.5 * u).astype(np.float32)
    assert np.array_equal(engine.edge_is_valid(rid, eid, q, q2), oracle.edge_valid(rb, osc, q, q2))


@pytest.mark.parametrize("n", [1, 17, 3639, 3640, 3700, 21500, 22700])
def test_host_arrays_in_place_and_copied(engine, n):
    """Host arrays up to 1 MiB are used in place, larger ones copied: both give
    the device arrays' bits, on each side of the line with the nearest points
    (288 bytes a configuration here) and without (about 46)."""
    import torch

    rng = np.random.default_rng(n)
    rb = R.xarm6()
    sc = W._boxes(rng, 2, 0.05, 0.3, 0.9)
    q = rng.uniform(-np.pi, np.pi, (n, 6)).astype(np.float32)
    rid, eid = engine.load_robot(rb), engine.create_env(sc, rvs.ENV_AABB)
    qd = torch.from_numpy(q).cuda()
    for prec in (rvs.PREC_REF32, rvs.PREC_FP32_REFINE):
        dd, pd, vd = (torch.empty(n, device="cuda"), torch.empty((n, 6), device="cuda"),
                      torch.empty(n, dtype=torch.uint8, device="cuda"))
        engine.distance_device(rid, eid, qd, dd, pd, vd, precision=prec)
        d, prof, ver, _ = engine.distance(rid, eid, q, precision=prec)
        assert np.array_equal(d, dd.cpu().numpy()) and np.array_equal(prof, pd.cpu().numpy())
        assert np.array_equal(ver, vd.cpu().numpy())
    m = min(n, 4000)
    _, _, _, near = engine.distance(rid, eid, q[:m], want_nearest=True)
    parts = [engine.distance(rid, eid, q[k:k + 500], want_nearest=True)[3] for k in range(0, m, 500)]
    assert np.array_equal(near, np.concatenate(parts), equal_nan=True)


@pytest.mark.parametrize("n", [17, 100, 3000, 5700])
def test_link_major_batches_of_host_arrays(engine, n):
    """Host arrays below 1 MiB of a batch that runs link by link: the device
    arrays' bits."""
    import torch

    rng = np.random.default_rng(n)
    rb = R.chain(rng.uniform(0.1, 0.3, 22), radius=0.04)
    sc = _boxes_around(rng, rb, 300, 0.02, 0.2, 2.0)
    q = rng.uniform(-np.pi, np.pi, (n, 22)).astype(np.float32)
    rid, eid = engine.load_robot(rb), engine.create_env(sc, rvs.ENV_AABB)
    out = (torch.empty(n, device="cuda"), torch.empty((n, 22), device="cuda"),
           torch.empty(n, dtype=torch.uint8, device="cuda"))
    engine.distance_device(rid, eid, torch.from_numpy(q).cuda(), *out, precision=rvs.PREC_FP32_REFINE)
    got = engine.distance(rid, eid, q, precision=rvs.PREC_FP32_REFINE)
    for a, b in zip(got, out):
        assert np.array_equal(a, b.cpu().numpy())


@pytest.mark.parametrize("boxes,points,parts", [(12, 10, 900), (200, 10, 900), (12, 1025, 9)])
def test_trajectories_in_place_and_copied(oracle, engine, boxes, points, parts):
    """4,500 trajectories of 10 points (1.1 MB, copied) against the same in
    parts that are used in place, with the current state's arrays in place (12
    boxes) and copied (200 boxes, 29 KB); long trajectories, copied whole: the
    oracle's walk, both outcomes among them."""
    rng = np.random.default_rng(5)
    rb = R.xarm6()
    sc = _boxes_around(rng, rb, boxes, 0.05, 0.2, 0.7)
    osc = oracle.scene_of(sc)
    rid, eid = engine.load_robot(rb), engine.create_env(sc, rvs.ENV_AABB)
    q = np.zeros(6, np.float32)
    _, prof, ok, near = oracle.distance(rb, osc, q[None], 32, want_np=True)
    assert ok[0] == 1
    n = 5 * parts
    u = rng.normal(size=(n, 6))
    u = rng.uniform(0.05, 2.5, (n, 1)) * u / np.linalg.norm(u, axis=1, keepdims=True)
    pts = (np.linspace(0, 1, points + 1)[1:, None] * u[:, None]).astype(np.float32)
    vel = np.full(boxes, 0.1, np.float32)
    dt = 0.1 / points

    def safe(p):
        return engine.trajectory_is_safe(rid, eid, p, q, prof[0], near[0], vel, time_step=dt)

    want = oracle.traj_safe(rb, osc, pts, q, prof[0], near[0], vel, 0.0, dt)
    print(f"safe {want.mean():.3f}")
    assert 0.05 < want.mean() < 0.95
    assert np.array_equal(safe(pts), want)
    assert np.array_equal(np.concatenate([safe(pts[k:k + parts]) for k in range(0, n, parts)]), want)
    assert np.array_equal(safe(pts[:1]), want[:1])
