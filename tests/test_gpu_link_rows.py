"""Per-link distance rows against float64 numpy, where the kernels' table sorting and lane
strides can go wrong: interior and repeated padding, unsorted and repeated radii, links with
no sphere, NaN entries, one obstacle to several hundred, one configuration (its rows shared
among workgroups) to more than the launch has workgroups, and tables too large for the LDS.
Few configurations or obstacles take flat kernels; the others are reached by the same poses
many times over, every copy equal to the first."""

import numpy as np
import pytest
import torch
from conftest import load_robot, random_cfgs

from pyroffi_amd.collision import RobotCollisionSpherized, colldist_from_sdf
from pyroffi_amd.costs import self_collision_cost, world_collision_cost
from pyroffi_amd.kernels import ops

pytestmark = pytest.mark.gpu

TOL = 1e-5  # coordinates up to 3 m: 3e-7 a component, times the placement's dozen roundings


def _poses(rng, B, L):
    q = rng.normal(size=(B, L, 4))
    q /= np.linalg.norm(q, axis=-1, keepdims=True)
    return np.concatenate([q, rng.uniform(-1, 1, (B, L, 3))], -1).astype(np.float32)


def _table(rng, L, S, pad):
    t = np.concatenate([rng.normal(0, 0.2, (L, S, 3)), rng.choice([0.05, 0.1, 0.03, 0.07], (L, S, 1))], -1)
    drop = rng.random((L, S)) < 0.3
    drop[0], drop[-1] = False, True
    t[drop] = [0.0, 0.0, 0.0, pad]
    return t.astype(np.float32)


def _centres(poses, table):
    w, v = poses[:, :, None, :1].astype(np.float64), poses[:, :, None, 1:4].astype(np.float64)
    c = table[None, :, :, :3].astype(np.float64)
    u = 2 * np.cross(np.broadcast_to(v, v.shape[:2] + c.shape[2:]), np.broadcast_to(c, v.shape[:2] + c.shape[2:]))
    return c + w * u + np.cross(np.broadcast_to(v, u.shape), u) + poses[:, :, None, 4:]


def _copies(B, L, S, M, P=0):
    """Copies of B poses from which the rows (and self pairs, if any) are placed once."""
    n = -(-(1 << 23) // (B * L * S * M))
    return max(n, -(-(1 << 22) // (B * S * P)) if P else 0)


def _many(run, poses, n):
    """The rows of n copies of the poses; equal, so the first is returned."""
    out = []
    for x in run(torch.as_tensor(np.tile(poses, (n, 1, 1)), device="cuda")):
        if x is not None:
            x = x.reshape(n, len(poses), *x.shape[1:])
            assert torch.equal(x, x[:1].expand_as(x))
            x = x[0]
        out.append(x)
    return out


def _check(got, ref):
    big = ref >= 1e8
    np.testing.assert_array_equal(got >= 1e8, big)
    np.testing.assert_allclose(got[~big], ref[~big], atol=TOL, rtol=0)


@pytest.mark.parametrize("B,L,S,M", [(1, 1, 1, 1), (1, 5, 7, 600), (3, 13, 18, 63), (1100, 4, 5, 3),
                                     (2, 3, 700, 17), (70, 20, 9, 64)])
def test_rows_of_random_tables(B, L, S, M):
    rng = np.random.default_rng(B + 10 * L + S + M)
    poses = _poses(rng, B, L)
    world = np.concatenate([rng.uniform(-1, 1, (M, 3)), rng.uniform(0.02, 0.2, (M, 1))], 1).astype(np.float32)
    pi, pj = (rng.integers(0, L, 40).astype(np.int32) for _ in range(2))
    table = _table(rng, L, S, -1e9)
    c, r = _centres(poses, table), table[..., 3].astype(np.float64)
    d = np.full((B, L, M), np.inf)
    for s in range(S):
        e = world[None, None, :, :3] - c[:, :, s, None] + 1e-6
        d = np.minimum(d, np.linalg.norm(e, axis=-1) - (r[None, :, s, None] + world[None, None, :, 3]))
    own = np.full((B, 40), np.inf)
    for s in range(S):
        e = np.linalg.norm(c[:, pj, s] - c[:, pi, s] + 1e-6, axis=-1)
        own = np.minimum(own, e - (r[pi, s] + r[pj, s])[None])
    ow, osf = ops.sphere_distances_jax(*(torch.as_tensor(x, device="cuda") for x in (poses, table, world, pi, pj)))
    _check(ow.cpu().numpy(), d)
    _check(osf.cpu().numpy(), own)
    n = _copies(B, L, S, M, 40)
    dev = [torch.as_tensor(x, device="cuda") for x in (table, world, pi, pj)]
    mow, mosf = _many(lambda p: ops.sphere_distances_jax(p, *dev), poses, n)
    _check(mow.cpu().numpy(), d)
    _check(mosf.cpu().numpy(), own)
    mcost, mself = _many(lambda p: ops.sphere_distances_jax(p, *dev, cost=(0.2, 3.0)), poses, n)
    torch.testing.assert_close(mcost, colldist_from_sdf(mow, 0.2) * 3.0, rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(mself, colldist_from_sdf(mosf, 0.2) * 3.0, rtol=1e-5, atol=1e-6)
    cost, _ = ops.sphere_distances_jax(*(torch.as_tensor(x, device="cuda") for x in (poses, table, world, pi, pj)),
                                       self_pairs=False, cost=(0.2, 3.0))
    torch.testing.assert_close(cost, colldist_from_sdf(ow, 0.2) * 3.0, rtol=1e-5, atol=1e-6)
    # CUDA conventions: slots with r < 0 skipped, 1e9 without any.
    table[1 % L, 0, 3] = -0.01
    r = table[..., 3].astype(np.float64)
    d = np.full((B, L, M), 1e9)
    for s in range(S):
        e = np.linalg.norm(world[None, None, :, :3] - c[:, :, s, None], axis=-1)
        e = e - (r[None, :, s, None] + world[None, None, :, 3])
        d = np.minimum(d, np.where(r[None, :, s, None] < 0, np.inf, e))
    w = {"spheres": world, "capsules": np.zeros((0, 7)), "boxes": np.zeros((0, 15)), "halfspaces": np.zeros((0, 6))}
    ow, om = ops.sphere_world_links(torch.as_tensor(poses, device="cuda"), torch.as_tensor(table, device="cuda"), w)
    _check(ow.cpu().numpy(), d)
    _check(om.cpu().numpy(), d.reshape(B, -1).min(1))
    mow, _ = _many(lambda p: ops.sphere_world_links(p, torch.as_tensor(table, device="cuda"), w, world_min=False),
                   poses, n)
    _check(mow.cpu().numpy(), d)


def test_more_links_than_the_tables_hold():
    """Links without a slot, more than their words fit the LDS: no sphere anywhere."""
    L = 30000
    poses = torch.zeros((2, L, 7), device="cuda")
    poses[..., 0] = 1
    table = torch.zeros((L, 0, 4), device="cuda")
    world = torch.ones((3, 4), device="cuda")
    pi, pj = (torch.arange(k, k + 5, dtype=torch.int32, device="cuda") for k in (0, L - 5))
    ow, osf = ops.sphere_distances_jax(poses, table, world, pi, pj)
    assert torch.isinf(ow).all() and torch.isinf(osf).all()
    none = {"capsules": np.zeros((0, 7)), "boxes": np.zeros((0, 15)), "halfspaces": np.zeros((0, 6))}
    ow, _ = ops.sphere_world_links(poses, table, {"spheres": world, **none}, world_min=False)
    assert (ow == 1e9).all()


def test_nan_spheres_are_skipped():
    """A NaN centre or radius takes no part in a minimum, whatever its place in the table."""
    rng = np.random.default_rng(5)
    poses, table = _poses(rng, 6, 3), _table(rng, 3, 8, -1e9)
    world = np.concatenate([rng.uniform(-1, 1, (70, 3)), rng.uniform(0.02, 0.2, (70, 1))], 1).astype(np.float32)
    none = {"capsules": np.zeros((0, 7)), "boxes": np.zeros((0, 15)), "halfspaces": np.zeros((0, 6))}
    cuda = lambda x: torch.as_tensor(x, device="cuda")  # noqa: E731
    for place in (0, 3, 7):
        for col in (0, 3):
            bad, good = table.copy(), table.copy()
            bad[0, place, col] = np.nan
            good[0, place] = [0, 0, 0, -1e9]
            for n in (1, _copies(6, 3, 8, 70)):
                rows = lambda t: _many(lambda p: ops.sphere_world_links(p, cuda(t), {"spheres": world, **none}),  # noqa: E731
                                       poses, n)[0]
                torch.testing.assert_close(rows(bad), rows(good), rtol=0, atol=0)


@pytest.mark.parametrize("copies", [1, 100])
@pytest.mark.parametrize("name", ("panda", "baxter"))
def test_residuals_equal_activated_distances(name, copies):
    robot, path = load_robot(name)
    coll = RobotCollisionSpherized.from_urdf(path)
    q = torch.as_tensor(random_cfgs(robot, 37, seed=4).astype(np.float32), device="cuda").repeat(copies, 1)
    rng = np.random.default_rng(6)
    world = np.concatenate([rng.uniform(-1, 1, (50, 3)), rng.uniform(0.02, 0.2, (50, 1))], 1).astype(np.float32)
    for margin, weight in ((0.05, 2.0), (0.2, torch.tensor(3.0, device="cuda")), (np.float32(0.1), 1)):
        d = coll.compute_world_collision_distance(robot, q, world)
        got = world_collision_cost(q, robot, coll, None, world, margin, weight)
        torch.testing.assert_close(got, (colldist_from_sdf(d, margin) * weight).flatten(), rtol=1e-5, atol=1e-6)
        d = coll.compute_self_collision_distance(robot, q)
        got = self_collision_cost(q, robot, coll, None, margin, weight)
        torch.testing.assert_close(got, (colldist_from_sdf(d, margin) * weight).flatten(), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("kind,M", [(k, m) for k in ("capsules", "boxes") for m in (64, 65, 111, 112, 128, 129, 256, 300)])
def test_many_capsules_or_boxes(oracle_mod, kind, M):
    """Lane by lane and a wave per link (capsules from 65 of them, boxes where a pass of 128 is
    seven eighths full), point capsules and links without spheres among them."""
    rng = np.random.default_rng(M)
    B, L, S = 7, 6, 5
    poses, table = _poses(rng, B, L), _table(rng, L, S, -1e9)
    c = rng.uniform(-1, 1, (M, 3))
    if kind == "capsules":
        end = c + rng.normal(0, 0.3, (M, 3)) * (np.arange(M) % 7 != 0)[:, None]
        obs = np.concatenate([c, end, rng.uniform(0.02, 0.1, (M, 1))], 1).astype(np.float32)
    else:
        axes, _ = np.linalg.qr(rng.normal(size=(M, 3, 3)))
        obs = np.concatenate([c, axes.transpose(0, 2, 1).reshape(M, 9), rng.uniform(0.02, 0.3, (M, 3))], 1)
        obs = obs.astype(np.float32)
    world = {k: np.zeros((0, n), np.float32) for k, n in (("spheres", 4), ("capsules", 7), ("boxes", 15),
                                                          ("halfspaces", 6))}
    world[kind] = obs
    tab = torch.as_tensor(table, device="cuda")
    got, _ = _many(lambda p: ops.sphere_world_links(p, tab, world, world_min=False), poses, _copies(B, L, S, M))
    r = np.broadcast_to(table[None, :, :, 3], (B, L, S)).astype(np.float64)
    d = oracle_mod.obstacle_dist(_centres(poses, table).reshape(-1, 3), np.maximum(r, 0).reshape(-1),
                                 **{kind: obs.astype(np.float64)}).reshape(B, L, S, M)
    ref = np.minimum(np.where(r[..., None] < 0, np.inf, d).min(2), 1e9)
    _check(got.cpu().numpy(), ref)
