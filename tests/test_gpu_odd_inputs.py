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
