"""The trajectory cost's ways to find obstacles: a robot without spheres."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch
from conftest import load_robot, random_cfgs

from pyroffi_amd.collision import RobotCollisionSpherized
from pyroffi_amd.optimization_engines._lbfgs_trajopt_optimization import TrajModel, flatten_trajs, traj_cost

pytestmark = pytest.mark.gpu


def _world(M, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.uniform(-1, 1, (M, 3)), rng.uniform(0.02, 0.1, (M, 1))], 1).astype(np.float32)


@pytest.mark.parametrize("name,M", [("panda", 0), ("panda", 30), ("panda", 300), ("baxter", 300)])
def test_robot_without_spheres(name, M):
    """No collision term; smoothness and limits are the robot's own, to the bit."""
    robot, path = load_robot(name)
    coll = RobotCollisionSpherized.from_urdf(path)
    L = robot.links.num_links
    bare = SimpleNamespace(coll=SimpleNamespace(pose=SimpleNamespace(translation=lambda: np.zeros((L, 1, 3))),
                                                radius=np.full((L, 1), -1e9)),
                           active_idx_i=coll.active_idx_i, active_idx_j=coll.active_idx_j)
    paths = [random_cfgs(robot, T, seed=T, margin=0.1).astype(np.float32) for T in (5, 24, 33)]
    w = (1.0, 1.0, 0.5, 0.1, 1.0, 2.0)
    out = []
    for c in (bare, coll):
        model = TrajModel(robot, c, _world(M, 1), 0.05)
        out.append(traj_cost(model, *flatten_trajs(paths, model.device), w)[0])
    assert not out[0][:, 2].any()
    assert torch.equal(out[0][:, :2], out[1][:, :2])
