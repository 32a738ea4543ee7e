"""Inputs at the edge of what the kernels take: configurations that are not
finite, models far from the origin, repeated self pairs, very large grids.

Verdicts are compared with the FP64 oracle outside its contact band, or bit
for bit with the same states in other company or on the general path.
"""
import numpy as np
import pytest
import torch

import pyoracle as PO
from prismplan_amd import _ppl
from prismplan_amd import substrate as S
from prismplan_amd import workloads as W
from prismplan_amd.planning_scene import HostScene
from prismplan_amd.robot_model_loader import load_robot_asset

pytestmark = pytest.mark.gpu
DEV = "cuda"


def up(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


@pytest.mark.parametrize("name,bad", [("panda", np.nan), ("fetch", np.nan), ("fetch", np.inf), ("fetch", 3e38)])
@pytest.mark.parametrize("n", [640, 33024])
def test_non_finite_states_leave_their_neighbours(name, bad, n):
    """A bad configuration at each place of a row of 16 states, rows with two
    and with nothing else, in launches with four lanes a state and with one: the
    others keep their verdicts, and a NaN configuration collides as in the
    oracle (its distance to any box counts as zero)."""
    rob = S.Robot(name)
    rng = np.random.default_rng(n)
    lo, hi = ((0.6, -0.9, 0.4), (1.3, 0.9, 1.6)) if name == "fetch" else (W.PANDA_BOX_LO, W.PANDA_BOX_HI)
    scene = W.random_obbs(rng, 20, lo, hi, half_hi=0.1 if name == "fetch" else 0.15)
    ds, plan = S.DeviceScene.from_host(scene), S.Plan.configs(rob, n)
    q = W.uniform_configs(rng, rob.arrays, n)
    clean = S.check_collision_batched(plan, ds, up(q)).cpu().numpy()
    is_bad = np.zeros(n, bool)
    is_bad[np.arange(16) * 17] = True                             # row r: its state r
    is_bad[16 * 16 + np.arange(16) * 16 + 8] = True               # rows 16-31: their middle state and one more
    is_bad[16 * 16 + np.arange(16) * 17] = True
    is_bad[32 * 16:33 * 16] = True                                # a whole row
    is_bad[-1] = True
    q[is_bad, 0] = bad
    got = S.check_collision_batched(plan, ds, up(q)).cpu().numpy()
    np.testing.assert_array_equal(got[~is_bad], clean[~is_bad])
    assert 0.02 < clean[~is_bad].mean() < 0.9
    if np.isnan(bad):
        ref, _ = PO.Oracle(rob.arrays, scene).check_collision(q[is_bad])
        np.testing.assert_array_equal(got[is_bad], ref)


@pytest.mark.parametrize("n", [300, 3000])
def test_edges_beside_one_without_an_end(n):
    """Edges whose end is NaN, among short edges that share their rows."""
    rob = S.Robot("panda")
    rng = np.random.default_rng(n)
    ds = S.DeviceScene.from_host(W.random_obbs(rng, 12, half_hi=0.12))
    a = W.uniform_configs(rng, rob.arrays, n)
    b = (a + rng.uniform(-0.2, 0.2, a.shape)).astype(np.float32)
    ns = rng.integers(3, 30, n).astype(np.int32)
    plan = S.Plan.edges(rob, ns)
    kw = dict(skip_resolved=False, state_hits=True)
    fh0, hits0 = (x.cpu().numpy() for x in S.edge_check_batched(plan, ds, up(a), up(b), **kw))
    bad = np.arange(n) % 3 == 1
    b[bad] = np.nan
    fh1, hits1 = (x.cpu().numpy() for x in S.edge_check_batched(plan, ds, up(a), up(b), **kw))
    np.testing.assert_array_equal(fh1[~bad], fh0[~bad])
    ok = ~np.repeat(bad, ns)
    np.testing.assert_array_equal(hits1[ok], hits0[ok])


def _millimetres(shift):
    """Panda in millimetres, its first moving link `shift` mm from the origin."""
    a = load_robot_asset("panda")
    ft = np.array(a["fixed_transforms"], np.float64).reshape(-1, 4, 4)
    ft[:, :3, 3] *= 1000.0
    ft[1, :3, 3] += shift
    a["fixed_transforms"] = ft.reshape(-1).tolist()
    for k in ("spheres_flat", "approx_spheres_flat"):
        a[k] = (1000.0 * np.array(a[k])).tolist()
    return a


@pytest.mark.parametrize("n,boxes", [(1, 12), (70, 20), (203, 70)])
@pytest.mark.parametrize("group", [1, 4, _ppl.PPL_COST_GROUPED])
def test_costs_far_from_the_origin(n, boxes, group):
    """Every state's links lie past 10 m in millimetres: boxes are found there
    as anywhere. FP32 places a sphere at 16,000 mm within 16,000 x 4.6e-7 =
    0.0074 mm of FP64 (parity_common's ratio), a box's face within as much
    again, so a hinge term is within 0.015 mm; weight 2. A gradient's direction
    turns by about 0.015 mm over the distance to the box, which is small for
    most states but has no bound at an edge of a box."""
    shift = np.array([16000.0, -300.0, 200.0])
    rob = S.Robot(_millimetres(shift))
    arr, rng = rob.arrays, np.random.default_rng(n + boxes)
    m = W.random_obbs(rng, boxes, half_hi=0.2)
    scene = W.random_obbs(np.random.default_rng(n + boxes), boxes, lo=1000 * np.array(W.PANDA_BOX_LO) + shift,
                          hi=1000 * np.array(W.PANDA_BOX_HI) + shift, half_lo=20.0, half_hi=200.0)
    assert m.n_obbs == scene.n_obbs
    q = W.uniform_configs(rng, arr, n)
    ds, plan = S.DeviceScene.from_host(scene), S.Plan.configs(rob, n)
    kw = dict(world_margin=50.0, weight=2.0, use_self=False, use_esdf=False)
    o, prm = PO.Oracle(arr, scene, nthreads=8), PO.cost_params(**kw)
    ref, g_ref, kink = o.hinge_grad(q, prm, tol=0.03)
    bar = 1e-5 * np.abs(ref) + 2.0 * 0.015 * np.maximum(o.hinge_terms(q, prm), 1)
    plan.set_cost_group(group)
    c0 = S.hinge_cost(plan, ds, up(q), S.cost_params(**kw))[0].cpu().numpy()
    assert np.all(np.abs(c0 - ref) < bar) and (n == 1 or (ref > 0).mean() > 0.5)
    plan.set_cost_group(group, grad=True)
    c1, _, g = S.hinge_cost(plan, ds, up(q), S.cost_params(**kw), grad=True)
    assert np.all(np.abs(c1.cpu().numpy() - ref) < bar)
    err = np.linalg.norm(g.cpu().numpy() - g_ref, axis=1) / np.maximum(np.linalg.norm(g_ref, axis=1), 1.0)
    assert np.mean(err[~kink] < 1e-2) > 0.95 or n == 1


@pytest.mark.parametrize("bad", [np.nan, np.inf, 3e38])
@pytest.mark.parametrize("group", [1, 4, _ppl.PPL_COST_GROUPED])
def test_costs_beside_non_finite_states(bad, group):
    """Costs, gradients, clearances and frames of the other states of a wave
    stay what they are without the bad ones (a prismatic joint, so that its
    place and not only its turn is lost)."""
    rob, n = S.Robot("fetch"), 130
    rng = np.random.default_rng(11)
    q = W.uniform_configs(rng, rob.arrays, n)
    ds = S.DeviceScene.from_host(W.random_obbs(rng, 40, W.FETCH_BOX_LO, W.FETCH_BOX_HI, half_hi=0.15))
    prm, pose = W.esdf_grid(center=(0.6, 0.0, 0.8), n=48, voxel=0.03)
    grid = S.DeviceScene.from_host(HostScene(voxel_params=prm, voxel_pose=pose, voxel_enable=np.ones(1, np.uint8), esdf_interp=1,
                                             voxel_features=rng.normal(0, 0.2, (1, 48 ** 3)).astype(np.float32)))
    plan = S.Plan.configs(rob, n)
    plan.set_cost_group(group)
    plan.set_cost_group(group, grad=True)
    cp = S.cost_params(world_margin=0.05, self_margin=0.05, weight=2.0)

    def run(x):
        x = up(x)
        out = [S.hinge_cost(plan, ds, x, cp)[0]] + [o for s in (ds, grid) for o in S.hinge_cost(plan, s, x, cp, grad=True)[::2]]
        out += [S.min_clearance_batched(plan, grid, x), *S.fk_batched(plan, x)]
        return [o.cpu().numpy() for o in out]

    is_bad = (np.arange(n) % 5 == 0) | (np.arange(n) >= 126)
    ref, keep = run(q), ~is_bad
    q[is_bad, 0] = bad
    for x, y in zip(run(q), ref):
        np.testing.assert_array_equal(x[keep], y[keep])


def _repeated_pairs():
    """Panda with every other self pair left out and the others named twice,
    as (i, j) and as (j, i)."""
    a = load_robot_asset("panda")
    r = np.array(a["self_cc_ranges_flat"], np.int64).reshape(-1, 3)
    pairs = [(i, j) for i, lo, hi in r.tolist() for j in range(lo, hi + 1) if (i + j) % 2 == 0]
    a["self_cc_ranges_flat"] = [v for i, j in pairs for v in (i, j, j, j, i, i)]
    return a


def _self_edges(rob, n, seed, skip, change=None):
    """The same edges in one plan of at least 65,536 states and in plans below
    that: (first hits, state verdicts) of either, and the states. change: applied
    to the edges' ends (start, end, random numbers)."""
    arr, rng = rob.arrays, np.random.default_rng(seed)
    a = W.uniform_configs(rng, arr, n)
    b = np.clip(a + rng.uniform(-0.8, 0.8, a.shape), arr.joint_lower, arr.joint_upper).astype(np.float32)
    if change:
        change(a, b, rng)
    ns = rng.integers(20, 64, n).astype(np.int32)
    ds = S.DeviceScene.from_host(HostScene())

    def run(lo, hi):
        plan = S.Plan.edges(rob, ns[lo:hi])
        out = S.edge_check_batched(plan, ds, up(a[lo:hi]), up(b[lo:hi]), check_self=True, skip_resolved=skip,
                                   state_hits=not skip)
        return (plan.n_states, *[x.cpu().numpy() for x in ((out,) if skip else out)])

    large, parts = run(0, n), [run(k, min(k + 700, n)) for k in range(0, n, 700)]
    assert large[0] >= 65536 and all(p[0] < 65536 for p in parts)
    return large[1:], [np.concatenate(x) for x in list(zip(*parts))[1:]], PO.edge_states(a, b, ns)


@pytest.mark.parametrize("skip", [False, True])
def test_self_pairs_named_twice(skip):
    """A pair counts once however often it is named: large and small edge sets
    agree with each other and with the oracle."""
    rob = S.Robot(_repeated_pairs())
    large, small, states = _self_edges(rob, 2000, 5, skip)
    for x, y in zip(large, small):
        np.testing.assert_array_equal(x, y)
    if not skip:
        ref, clr = PO.Oracle(rob.arrays).check_collision(states, check_self=True)
        assert not np.any((large[1] != ref) & (np.abs(clr) >= 1e-5)) and 0.02 < ref.mean() < 0.6


def test_esdf_grid_of_2_to_the_30_nodes():
    """A wide flat grid has more 64-lane workgroups than one launch takes: every
    node up to the last has its value."""
    n, voxel = 32768, 1.0 / 128
    box = HostScene.from_boxes(np.array([[3.0, 40.0, 2.0], [5.0, 5.0, 5.0]]),
                               np.array([[10.0, -20.0, 0.5], [-127.0, 125.0, 0.0]]),
                               np.array([[1.0, 0.0, 0.0, 0.0], [0.8, 0.0, 0.0, 0.6]]))
    prm = np.array([voxel * (n - 1), voxel * (n - 1), 0.0, voxel], np.float32)
    pose = np.array([0, 0, 0, 1, 0, 0, 0, 0], np.float32)
    got = S.esdf_from_obbs(S.DeviceScene.from_host(box), prm, pose)
    assert got.numel() == n * n
    k = np.unique(np.concatenate([np.random.default_rng(0).integers(0, n * n, 20000), [0, n - 1, n * n - n, n * n - 1]]))
    ix, iy = k // n, k % n
    p = np.stack([ix * voxel - 0.5 * float(prm[0]), iy * voxel - 0.5 * float(prm[1]), 0.0 * ix], 1)
    d = np.min([_box_distance(box, b, p) for b in range(2)], axis=0)
    # coordinates up to 128 m: FP32 resolves 1.5e-5 m there, the map to a box sums three such products
    assert np.abs(got[torch.from_numpy(k).to(DEV)].cpu().numpy() + d).max() < 2e-4


def _box_distance(scene, b, p):
    t, w, u = scene.obb_pose[b, :3].astype(float), float(scene.obb_pose[b, 3]), scene.obb_pose[b, 4:7].astype(float)
    s = 2.0 * np.cross(u, p)
    e = np.abs(p + w * s + np.cross(u, s) + t) - 0.5 * scene.obb_dims[b, :3]
    return np.linalg.norm(np.maximum(e, 0.0), axis=1) + np.minimum(e.max(1), 0.0)


def _branched():
    """Panda with link 5 hung on link 3: not a line of joints."""
    a = load_robot_asset("panda")
    a["joint_parents"] = [0, 0, 1, 2, 3, 3, 5, 6]
    a["t_memory_idx"] = [0, 1, 1, 1, 0, 1, 1, 1]
    return a


@pytest.mark.parametrize("skip", [False, True])
def test_rough_self_pass_of_a_tree(skip):
    """A joint whose parent is neither the root nor the joint before it: its
    parent's frame is read back from LDS. Large and small edge sets agree, and
    both with the oracle."""
    rob = S.Robot(_branched())
    large, small, states = _self_edges(rob, 2000, 8, skip)
    for x, y in zip(large, small):
        np.testing.assert_array_equal(x, y)
    if not skip:
        ref, clr = PO.Oracle(rob.arrays).check_collision(states, check_self=True)
        assert not np.any((large[1] != ref) & (np.abs(clr) >= 1e-5)) and 0.005 < ref.mean() < 0.9


def _solved(rob, ds, theta, T, step):
    """Validity of each of len(theta) trajectories of T waypoints, in one call."""
    plan = S.Plan.trajectories(rob, np.full(len(theta), T))
    opt = S.ChompOptimizer(plan, ds, up(theta.reshape(-1)), S.chomp_settings(collision_check_step=step)).step(0)
    return opt.solved().cpu().numpy()


@pytest.mark.parametrize("name,boxes", [("panda", 3), ("branched", 3), ("panda", 0)])
def test_densified_validity_alone_and_in_a_batch(name, boxes):
    """Forty trajectories at once take the two-step self pass over up to 600,000
    densified states, one alone the exact pass: the same verdicts."""
    rob = S.Robot(_branched() if name == "branched" else name)
    w = W.chomp(n_traj=40, n_wp=64, n_obbs=max(boxes, 1), seed=3 + boxes)
    ds = S.DeviceScene.from_host(w.scene if boxes else HostScene())
    theta = w.theta.reshape(40, -1)
    batch = _solved(rob, ds, theta, 64, 0.05)
    np.testing.assert_array_equal(batch, np.concatenate([_solved(rob, ds, theta[k:k + 1], 64, 0.05) for k in range(40)]))
    assert 0 < batch.sum() < 40


@pytest.mark.parametrize("n", [1, 2, 4, 5, 63, 65, 1100])
def test_spread_visit_reaches_every_chunk(n):
    """64 waypoints a trajectory and one state a segment: n chunks of 64 states,
    one to a trajectory, visited in spread order. Chunk counts of one, powers of
    two and one past and short of them; 1,100 take the two-step self pass."""
    rob = S.Robot("panda")
    w = W.chomp(n_traj=n, n_wp=64, n_obbs=3, seed=n)
    got = _solved(rob, S.DeviceScene.from_host(w.scene), w.theta.reshape(n, -1), 64, 100.0)
    D = rob.n_dof
    q = w.theta.reshape(n, D, 64).transpose(0, 2, 1).reshape(-1, D)
    hit, clr = PO.Oracle(rob.arrays, w.scene, nthreads=8).check_collision(q, check_self=True)
    sure = ~(np.abs(clr) < 1e-5).reshape(n, 64).any(1)
    np.testing.assert_array_equal(got[sure], ~hit.reshape(n, 64).any(1)[sure])
    assert n < 60 or 0.02 < got.mean() < 0.98


@pytest.mark.parametrize("skip", [False, True])
def test_self_check_of_edges_without_an_end(skip):
    """Edges with a NaN joint in the middle of the arm: the finite links' pairs
    decide, in large edge sets as in small ones."""
    rob = S.Robot("panda")

    def change(a, b, rng):
        b[rng.random(len(b)) < 0.3, 5] = np.nan

    large, small, states = _self_edges(rob, 2000, 6, skip, change)
    for x, y in zip(large, small):
        np.testing.assert_array_equal(x, y)
    if not skip:
        bad = np.isnan(states).any(1)
        assert large[1][bad].mean() > 0.001 and large[1][~bad].mean() > 0.02


@pytest.mark.parametrize("place", [300.0, 3e5, 1e30])
def test_self_check_far_off_the_limits(place):
    """A base rail run far off its limits, where FP32 resolves a sphere's place
    by less and less: the rough pass leaves to the exact one what it cannot
    prove there."""
    a = load_robot_asset("panda")
    a["joint_types"] = [3, 0] + a["joint_types"][2:]
    rob = S.Robot(a)

    def change(a, b, rng):
        a[rng.random(len(a)) < 0.5, 0] = place
        b[:, 0] = a[:, 0]

    large, small, _ = _self_edges(rob, 2000, 7, False, change)
    for x, y in zip(large, small):
        np.testing.assert_array_equal(x, y)
    assert 0.01 < large[1].mean() < 0.99


@pytest.mark.parametrize("name", ["panda", "baxter"])
def test_unobserved_grid_has_no_gradient(name):
    """A margin above the 1000 m of a sphere that no grid value applies to
    (outside, or beside an unobserved node): the hinge is margin - 1000 and has
    no gradient. The single-layer lookups equal the general ones, which a mask
    that masks nothing selects."""
    rob = S.Robot(name)
    arr, rng, n = rob.arrays, np.random.default_rng(9), 300
    prm, pose = W.esdf_grid(center=(0.5, 0.0, 0.5), n=48, voxel=0.03)
    src = W.random_obbs(rng, 8, half_hi=0.15)
    vals = PO.esdf_from_obbs(src.obb_dims, src.obb_pose, prm, pose).astype(np.float32).reshape(-1)
    vals[rng.random(vals.size) < 0.05] = -1000.0
    hs = lambda acm: HostScene(voxel_params=prm, voxel_pose=pose, voxel_enable=np.ones(1, np.uint8),
                               voxel_features=vals.reshape(1, -1), esdf_interp=1, sphere_acm=acm)
    q = up(W.uniform_configs(rng, arr, n))
    cp = S.cost_params(world_margin=1001.0, weight=1.0, use_self=False, use_obb=False)
    out = []
    for acm in (None, np.ones((arr.n_spheres, 1), np.uint8)):
        c, _, g = S.hinge_cost(S.Plan.configs(rob, n), S.DeviceScene.from_host(hs(acm)), q, cp, grad=True)
        out.append((c.cpu().numpy(), g.cpu().numpy()))
    np.testing.assert_allclose(out[0][0], out[1][0], rtol=5e-6)   # sums of up to 75 FP32 terms
    # sums of unit point gradients times arms of metres, over the model's spheres
    np.testing.assert_allclose(out[0][1], out[1][1], rtol=0, atol=1e-5 * arr.n_spheres)
    assert np.abs(out[0][1]).max() > 0.1


def test_grid_parameters_at_any_float():
    """Layer parameters and pose need no more than a float's alignment."""
    rob, n = S.Robot("panda"), 200
    rng = np.random.default_rng(10)
    prm, pose = W.esdf_grid(center=(0.5, 0.0, 0.5), n=48, voxel=0.03)
    vals = up(rng.normal(0, 0.2, 48 ** 3).astype(np.float32))
    one = torch.ones(1, dtype=torch.uint8, device=DEV)
    q, plan, out = up(W.uniform_configs(rng, rob.arrays, n)), S.Plan.configs(rob, n), []
    for shift in (0, 1, 3):
        at = lambda a: up(np.concatenate([np.zeros(shift, np.float32), a.reshape(-1)]))[shift:].reshape(a.shape)
        ds = S.DeviceScene(None, None, None, at(prm), at(pose), one, vals, esdf_interp=1)
        assert ds.view().voxel_params is not None and at(prm).data_ptr() % 16 == 4 * shift
        out.append((S.min_clearance_batched(plan, ds, q).cpu().numpy(),
                    S.hinge_cost(plan, ds, q, S.cost_params(use_self=False), grad=True)[2].cpu().numpy()))
    for x in out[1:]:
        np.testing.assert_array_equal(x[0], out[0][0])
        np.testing.assert_array_equal(x[1], out[0][1])


def test_tuning_entries_of_other_kernels_are_not_taken(tmp_path):
    """A cache file written for earlier kernels (keys without their revision)
    leaves the built-in shapes."""
    path = tmp_path / "tune.txt"
    S.tune_cache_file(path)
    try:
        rob, n = S.Robot("panda"), 4000
        rng = np.random.default_rng(2)
        ds = S.DeviceScene.from_host(W.random_obbs(rng, 64))
        q = up(W.uniform_configs(rng, rob.arrays, n))
        S.Plan.configs(rob, n).autotune_collide(ds, q, reps=2)
        assert S.Plan.configs(rob, n).collide_shape(64)[2] == 1
        lines = path.read_text().splitlines()
        old = ["/".join(w for w in l.split()[0].split("/") if not w.startswith("k")) + " 32 2 0.001" for l in lines
               if l.startswith("collide/")]
        assert old
        path.write_text("\n".join(old) + "\n")
        S.tune_cache_file(path)
        assert S.Plan.configs(rob, n).collide_shape(64) == (64, 0, 0)
    finally:
        S.tune_cache_file("")


@pytest.mark.parametrize("name,boxes,tile", [("panda", 212, 212), ("panda", 213, 128), ("baxter", 187, 128),
                                             ("fetch", 256, 128), ("branched", 300, 128)])
def test_many_boxes_pass_in_tiles(name, boxes, tile):
    """Past some 190 boxes (212 of Panda's, 186 of Baxter's) a launch of more waves than then fit the chip stages
    128 at a time, a small one all of them (up to 256): verdicts and first hits
    are those of any tile."""
    rob = S.Robot(_branched() if name == "branched" else name)
    arr, rng = rob.arrays, np.random.default_rng(boxes)
    ds = S.DeviceScene.from_host(W.random_obbs(rng, boxes, (0.5, -0.9, 0.3), (1.3, 0.9, 1.5), half_hi=0.04))
    a = W.uniform_configs(rng, arr, 3000)
    b = np.clip(a + rng.uniform(-0.6, 0.6, a.shape), arr.joint_lower, arr.joint_upper).astype(np.float32)
    ns = rng.integers(20, 80, len(a)).astype(np.int32)
    big, small = S.Plan.edges(rob, ns), S.Plan.edges(rob, ns[:300])
    assert small.collide_shape(boxes) == (min(boxes, 256), 0, 0) and small.collide_shape(128)[0] == 128
    assert big.collide_shape(boxes) == (tile, 0, 0) and big.collide_shape(170)[0] == 170
    x = S.edge_check_batched(big, ds, up(a), up(b)).cpu().numpy()
    y = S.edge_check_batched(small, ds, up(a[:300]), up(b[:300])).cpu().numpy()
    np.testing.assert_array_equal(x[:300], y)
    big.set_collide_shape(96, 0)
    np.testing.assert_array_equal(x, S.edge_check_batched(big, ds, up(a), up(b)).cpu().numpy())
    assert 0.02 < (x >= 0).mean() < 0.98
