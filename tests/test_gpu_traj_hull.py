"""The trajectory cost's shared world search (paths of 24 waypoints and more, 128 obstacles and
more, four spheres a link and more: every case here meets all three) against the same waypoints
evaluated as short paths, which look every sphere up in the grid: path lengths around the
threshold, a wave's eight waypoints (whole and partly filled) and a workgroup's rounds, world
sizes around the threshold and a pass of 64 obstacles, obstacles crowded round the robot so that
the lists overflow, and robots of up to and of more than eight nodes."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch
from conftest import load_robot, random_cfgs

from pyroffi_amd.collision import RobotCollisionSpherized
from pyroffi_amd.optimization_engines._lbfgs_trajopt_optimization import TrajModel, flatten_trajs, traj_cost

pytestmark = pytest.mark.gpu


def _crowded(coll, L, per):
    """The collision model with `per` spheres on every link that has any: its own, then copies
    moved by a centimetre."""
    c = np.asarray(coll.coll.pose.translation()).reshape(L, -1, 3)
    r = np.asarray(coll.coll.radius).reshape(L, -1)
    rng = np.random.default_rng(0)
    centers, radii = np.zeros((L, per, 3)), np.full((L, per), -1e9)
    for k in range(L):
        own = np.flatnonzero(r[k] > 0)
        if len(own):
            i = own[np.arange(per) % len(own)]
            centers[k] = c[k, i] + rng.normal(0, 0.01, (per, 3)) * (np.arange(per) >= len(own))[:, None]
            radii[k] = r[k, i]
    return SimpleNamespace(coll=SimpleNamespace(pose=SimpleNamespace(translation=lambda: centers), radius=radii),
                           active_idx_i=coll.active_idx_i, active_idx_j=coll.active_idx_j)


@pytest.mark.parametrize("name,T,M,extent,mode", [
    ("panda", 24, 128, 1.0, 1), ("panda", 25, 129, 1.0, 0), ("panda", 33, 129, 1.0, 0), ("panda", 47, 200, 0.8, 1),
    ("panda", 65, 193, 0.5, 1), ("panda", 130, 300, 1.0, 0), ("panda", 40, 700, 0.4, 1), ("fetch", 24, 128, 1.0, 1),
    ("fetch", 47, 130, 0.8, 0), ("fetch", 63, 257, 0.6, 1), ("baxter", 25, 128, 1.0, 1), ("baxter", 31, 200, 0.6, 0)])
def test_long_path_equals_its_pieces(name, T, M, extent, mode):
    """Collision terms only.  Both sides add the same FP32 terms in another order: 1e-5 of the
    cost, 1e-4 of the gradient (whose terms cancel)."""
    robot, path = load_robot(name)
    coll = RobotCollisionSpherized.from_urdf(path)
    if name == "baxter":  # 14 nodes
        coll = _crowded(coll, robot.links.num_links, 8)
    rng = np.random.default_rng(T + M)
    world = np.concatenate([rng.uniform(-extent, extent, (M, 3)), rng.uniform(0.02, 0.1, (M, 1))], 1)
    model = TrajModel(robot, coll, world.astype(np.float32), 0.05, mode)
    assert T >= 24 and M >= 128 and len(model.t["spheres"]) >= 4 * robot.links.num_links
    paths = []
    for s in range(3):
        a, b = random_cfgs(robot, 2, seed=s)
        t = np.linspace(0, 1, T)[:, None]
        paths.append(((1 - t) * a + t * b).astype(np.float32))
    w = (0.0, 0.0, 0.0, 0.0, 0.0, 2.0)
    x, start, n = flatten_trajs(paths, model.device)
    comps, grad = traj_cost(model, x, start, n, w)
    alone, none = traj_cost(model, x, start, n, w, grad=False)
    assert none is None
    torch.testing.assert_close(alone[:, 2], comps[:, 2], rtol=1e-5, atol=1e-6)
    pieces = [p[i:i + 20] for p in paths for i in range(0, T, 20)]
    xs, ss, ns = flatten_trajs(pieces, model.device)
    pc, pg = traj_cost(model, xs, ss, ns, w)
    per = -(-T // 20)
    torch.testing.assert_close(comps[:, 2], pc[:, 2].reshape(3, per).sum(1), rtol=1e-5, atol=1e-6)
    assert torch.equal(x, xs)
    assert (grad - pg).norm() <= 1e-4 * pg.norm() + 1e-6
