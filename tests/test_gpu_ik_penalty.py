"""The wave-shared collision penalty of the multi-seed LM against the FP64 oracle, where
its culling can go wrong: world sizes around the 64 obstacles of a pass and the 256 held in
registers, obstacles crowded round the base (every pair in reach), radii that swallow the
robot, other obstacle kinds, and robots of six to fourteen joints; in the wave-per-seed kernel
(at most 1024 seeds) and in the 8-lane kernel with one, two and eight seeds a wave."""

import numpy as np
import pytest
import worlds
from conftest import load_robot, random_cfgs

from pyroffi_amd.collision import RobotCollisionSpherized
from pyroffi_amd.optimization_engines._ls_ik import ee_tables, ls_ik_run, prepare_ls_collision_buffers

pytestmark = pytest.mark.gpu

HAND = {"panda": "panda_hand", "ur5": "ee_link", "fetch": "gripper_link", "baxter": "left_gripper_base"}


@pytest.mark.parametrize("name,m,extent,r_hi", [
    ("panda", 1, 1.0, 0.15), ("panda", 63, 1.0, 0.15), ("ur5", 64, 1.0, 0.15), ("fetch", 65, 1.0, 0.15),
    ("fetch", 300, 0.4, 0.1), ("panda", 1000, 0.3, 0.05), ("ur5", 5, 1.0, 3.0), ("panda", 40, 1000.0, 0.1)])
def test_wave_penalty_matches_oracle(oracle_mod, name, m, extent, r_hi):
    def world(rng):
        s = np.concatenate([rng.uniform(-extent, extent, (m, 3)), rng.uniform(0.02, r_hi, (m, 1))], 1)
        return {"spheres": s.astype(np.float32)}

    _check(oracle_mod, name, 70, world)


@pytest.mark.parametrize("name,seeds,kinds", [
    ("fetch", 400, (257, 0, 0, 0)), ("panda", 400, (0, 40, 0, 0)), ("panda", 400, (0, 0, 30, 2)),
    ("ur5", 1000, (300, 10, 10, 1)), ("panda", 1001, (64, 0, 0, 0)), ("fetch", 3001, (70, 6, 0, 1)),
    ("baxter", 33, (300, 0, 0, 0)), ("baxter", 400, (65, 4, 4, 1))])
def test_eight_lane_penalty_matches_oracle(oracle_mod, name, seeds, kinds):
    names = ("spheres", "capsules", "boxes", "halfspaces")
    _check(oracle_mod, name, seeds, lambda rng: dict(zip(names, worlds.random_world(rng, *kinds, extent=0.8))))


def _check(oracle_mod, name, n_seeds, world):
    """Errors of the seeds (one point a wave) and after one step (five points of the line
    search).  FP32 sums of some thousand hinge terms: 1e-4 relative.  A step whose two best
    points tie to rounding may pick either, so 1% of the seeds may differ."""
    robot, path = load_robot(name)
    links = (robot.links.names.index(HAND[name]),)
    t = oracle_mod.Tables.of(robot)
    rng = np.random.default_rng(17)
    lo, hi = robot.joints.lower_limits, robot.joints.upper_limits
    tgt = oracle_mod.fk_links(t, random_cfgs(robot, 3, seed=18))[:, list(links)]
    seeds = rng.uniform(lo, hi, (3, n_seeds, len(lo))).astype(np.float32)
    world = world(rng)
    rs, rj, _, _ = prepare_ls_collision_buffers(robot, RobotCollisionSpherized.from_urdf(path),
                                                np.zeros((1, 4), np.float32))
    okw = dict(robot_spheres=rs, sphere_joint=rj, world=world["spheres"], world_capsules=world.get("capsules"),
               world_boxes=world.get("boxes"), world_halfspaces=world.get("halfspaces"), enable_collision=True,
               collision_weight=1e4, collision_margin=0.02)
    for iters in (0, 1):
        _, errs = ls_ik_run(robot, seeds, tgt, links, max_iter=iters, lambda_init=1e-2,
                            collision=(rs, rj, world, 1e4, 0.02))
        _, oerrs = oracle_mod.ls_ik(t, seeds, *ee_tables(robot, links), tgt, lo, hi, max_iter=iters,
                                    lambda_init=1e-2, **okw)
        close = np.isclose(errs.cpu().numpy(), oerrs, rtol=1e-4, atol=1e-5)
        assert close.all() if iters == 0 else close.mean() >= 0.99, (iters, close.mean())


@pytest.mark.parametrize("name,m", [("panda", 4), ("fetch", 2), ("baxter", 3)])
def test_shared_or_not_gives_the_same_bits(name, m):
    """Seeds among few others share the penalty over the wave, among many and few obstacles each
    lane tests for itself: the same sums."""
    robot, path = load_robot(name)
    links = (robot.links.names.index(HAND[name]),)
    rng = np.random.default_rng(m)
    lo, hi = robot.joints.lower_limits, robot.joints.upper_limits
    tgt = np.asarray(robot.forward_kinematics(random_cfgs(robot, 1, seed=2).astype(np.float32)))[:, list(links)]
    seeds = rng.uniform(lo, hi, (1, 12000, len(lo))).astype(np.float32)
    world = np.concatenate([rng.uniform(-0.6, 0.6, (m, 3)), np.full((m, 1), 0.3)], 1).astype(np.float32)
    rs, rj, ws, ok = prepare_ls_collision_buffers(robot, RobotCollisionSpherized.from_urdf(path), world)
    assert ok
    run = lambda s: ls_ik_run(robot, s, tgt, links, max_iter=5, collision=(rs, rj, ws, 1e4, 0.02))  # noqa: E731
    cfgs, errs = run(seeds)
    few_cfgs, few_errs = run(seeds[:, 3000:4100])
    assert (few_cfgs == cfgs[:, 3000:4100]).all() and (few_errs == errs[:, 3000:4100]).all()
