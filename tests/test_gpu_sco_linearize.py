"""SCO's linearisation on both sides of its dispatch: a launch of few waypoints gives each a whole
wave and shares a trajectory among workgroups, one of many gives each eight lanes.  The small
launch against the FP64 oracle, then the same paths inside a large one against the small one, to
the bit: a path's result must not depend on how many others share its launch."""

import numpy as np
import pytest
import torch
from conftest import load_robot, random_cfgs

from pyroffi_amd.collision import RobotCollisionSpherized, Sphere
from pyroffi_amd.kernels._lib import check, lib
from pyroffi_amd.kernels.ops import _ptr, _stream
from pyroffi_amd.optimization_engines import ScoTrajOptConfig
from pyroffi_amd.optimization_engines._sco_optimization import BatchedSco

pytestmark = pytest.mark.gpu

MANY = 20000  # waypoints: past the whole-wave launches


def _linearize(robot, coll, geoms, trajs):
    opt = BatchedSco(robot, coll, geoms, trajs, ScoTrajOptConfig())
    opt.d.fill_(float("nan"))
    opt.J.fill_(float("nan"))
    st = lib().pk_traj_sco_linearize_f32(_stream(), opt.model.struct_ref(), _ptr(opt.x0), _ptr(opt.start), opt.B,
                                         opt.x0.shape[0], opt.max_len, 0, _ptr(opt.gstart), opt.G - 1, 0.05,
                                         _ptr(opt.d), _ptr(opt.J))
    check(st, "pk_traj_sco_linearize_f32")
    return opt.d.cpu().numpy(), opt.J.cpu().numpy()


@pytest.mark.parametrize("name,lens,split", [("panda", [1, 4, 5], (0, 1)), ("panda", [3, 129, 2], (63, 64, 65)),
                                             ("panda", [7, 6], (127, 128, 129)), ("fetch", [2, 31], (700,)),
                                             ("ur5", [8, 64, 7], (1, 256, 257)), ("baxter", [6, 9], (300,))])
def test_few_and_many_waypoints(oracle_mod, name, lens, split):
    robot, path = load_robot(name)
    coll = RobotCollisionSpherized.from_urdf(path)
    rng = np.random.default_rng(sum(lens))
    M = sum(split)
    world = np.concatenate([rng.uniform(-1, 1, (M, 3)), rng.uniform(0.02, 0.1, (M, 1))], 1).astype(np.float32)
    gstart = np.concatenate([[0], np.cumsum(split)]).astype(np.int32)
    geoms = tuple(Sphere.from_center_and_radius(world[a:b, :3], world[a:b, 3])
                  for a, b in zip(gstart[:-1], gstart[1:]))
    trajs = [random_cfgs(robot, T, seed=10 * i + T).astype(np.float32) for i, T in enumerate(lens)]
    d, J = _linearize(robot, coll, geoms, trajs)
    om = oracle_mod.TrajModel(oracle_mod.Tables.of(robot), oracle_mod.padded_spheres(coll), coll.active_idx_i,
                              coll.active_idx_j, world.astype(np.float64), 0.01, 1)
    rd, rJ = oracle_mod.sco_linearize(om, np.concatenate(trajs).astype(np.float64), gstart, 0.05)
    full = rd < 1e8  # an empty group has no distance
    # The tolerances of the oracle's own test of this kernel: FP32 distances at 2 m and their
    # gradients through weights exp(-d / 0.05), which turn 1e-6 m into 2e-5 of a weight.
    np.testing.assert_allclose(d[full], rd[full], atol=2e-5, rtol=0)
    np.testing.assert_allclose(J[full], rJ[full], atol=1e-4 * np.abs(rJ).max(), rtol=0)
    assert not np.isfinite(d[~full]).any() and not J[~full].any()
    n = len(d)
    copies = -(-MANY // n)
    d8, J8 = _linearize(robot, coll, geoms, trajs * copies)
    for c in (0, copies // 2, copies - 1):
        np.testing.assert_array_equal(d8[c * n:(c + 1) * n], d)
        np.testing.assert_array_equal(J8[c * n:(c + 1) * n], J)
