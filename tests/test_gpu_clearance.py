"""The configuration minimum of the sphere sweep, taken without rows, against float64 numpy and
against the rows' own minimum: one obstacle to several register chunks, one link to more links
than a wave has lanes, more candidates than a wave holds, links without spheres, and spheres,
obstacles and poses that no minimum takes."""

import numpy as np
import pytest
import torch

from pyroffi_amd.kernels import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL = 1e-5  # coordinates up to 3 m: 3e-7 a component, times the placement's dozen roundings


def _case(B, L, per_link, M, seed):
    rng = np.random.default_rng(seed)
    q = rng.normal(size=(B, L, 4))
    q /= np.linalg.norm(q, axis=-1, keepdims=True)
    poses = np.concatenate([q, rng.uniform(-1, 1, (B, L, 3))], -1).astype(np.float32)
    counts = rng.integers(0, per_link + 1, L)
    counts[0] = per_link
    start = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    spheres = np.concatenate([rng.normal(0, 0.15, (start[-1], 3)), rng.uniform(0.02, 0.1, (start[-1], 1))],
                             1).astype(np.float32)
    world = np.concatenate([rng.uniform(-1.5, 1.5, (M, 3)), rng.uniform(0.02, 0.2, (M, 1))], 1).astype(np.float32)
    return poses, start, spheres, world


def _reference(poses, start, spheres, world):
    link = np.repeat(np.arange(len(start) - 1), np.diff(start))
    p = poses.astype(np.float64)[:, link]
    c = np.broadcast_to(spheres[None, :, :3].astype(np.float64), p.shape[:2] + (3,))
    with np.errstate(all="ignore"):
        u = 2 * np.cross(p[..., 1:4], c)
        c = c + p[..., :1] * u + np.cross(p[..., 1:4], u) + p[..., 4:]
        d = np.linalg.norm(c[:, :, None] - world[None, None, :, :3].astype(np.float64), axis=-1)
        d = d - spheres[None, :, None, 3].astype(np.float64) - world[None, None, :, 3].astype(np.float64)
    return np.minimum(np.where(np.isnan(d), 1e9, d).min((1, 2)), 1e9)


def _sweep(poses, start, spheres, world, rows):
    t = [torch.as_tensor(x, device=DEV) for x in (poses, spheres, start, world, np.zeros(0, np.int32))]
    return ops.sphere_sweep(*t, 0, world=rows, world_min=True)[1].cpu().numpy()


@pytest.mark.parametrize("B,L,per_link,M", [(1, 1, 1, 1), (6, 2, 12, 1), (5, 3, 6, 64), (300, 13, 9, 65), (37, 13, 9, 129),
                                            (21, 65, 3, 256), (50, 2, 9, 256), (50, 2, 9, 257), (9, 65, 3, 1100), (2, 4, 250, 513)])
def test_minimum_of_random_scenes(B, L, per_link, M):
    case = _case(B, L, per_link, M, B + L + M)
    got, ref = _sweep(*case, rows=False), _reference(*case)
    np.testing.assert_allclose(got, ref, atol=TOL, rtol=0)
    np.testing.assert_allclose(got, _sweep(*case, rows=True), atol=TOL, rtol=0)


def test_obstacles_that_all_stay_candidates():
    """Every obstacle at one distance from every link: nothing is ruled out, so the wave's
    buffer is emptied many times."""
    poses, start, spheres, world = _case(7, 9, 4, 300, 3)
    poses[..., 4:] = 0
    world[:, :3] *= 2 / np.linalg.norm(world[:, :3], axis=1, keepdims=True)
    world[:, 3] = 0.1
    np.testing.assert_allclose(_sweep(poses, start, spheres, world, rows=False),
                               _reference(poses, start, spheres, world), atol=TOL, rtol=0)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("where", ["centre", "radius", "obstacle", "obstacle radius", "position", "quaternion"])
def test_values_that_are_not_finite(where, value):
    poses, start, spheres, world = _case(6, 5, 8, 70, 11)
    if where == "centre":
        spheres[1, 0] = value
    elif where == "radius":
        spheres[1, 3] = value
    elif where == "obstacle":
        world[::3, 1] = value
    elif where == "obstacle radius":
        world[::3, 3] = value
    else:
        poses[2, :, 5 if where == "position" else 1] = value  # one configuration
        poses[3, 1, 5 if where == "position" else 1] = value  # one link of another
    got, ref = _sweep(poses, start, spheres, world, rows=False), _reference(poses, start, spheres, world)
    rows = _sweep(poses, start, spheres, world, rows=True)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(rows))
    ok = np.isfinite(got)
    np.testing.assert_array_equal(got[~ok], rows[~ok])
    np.testing.assert_allclose(got[ok], ref[ok], atol=TOL, rtol=0)


def test_no_obstacles_and_no_spheres():
    poses, start, spheres, world = _case(4, 5, 3, 8, 5)
    assert (_sweep(poses, start, spheres, world[:0], rows=False) == np.float32(1e9)).all()
    assert (_sweep(poses, np.zeros(6, np.int32), spheres[:0], world, rows=False) == np.float32(1e9)).all()


@pytest.mark.parametrize("far", [100.0, 3000.0])
def test_scene_far_from_the_origin(far):
    """Robot and obstacles together at `far` metres, a power-of-two grid of 2^-12 m keeping the
    offsets exact: the distances are those of a scene at the origin, to the same tolerance."""
    poses, start, spheres, world = _case(200, 13, 9, 200, 17)
    poses[..., 4:] = np.round(poses[..., 4:] * 4096) / 4096 + np.round(far * 4096) / 4096
    world[:, :3] = np.round(world[:, :3] * 4096) / 4096 + np.round(far * 4096) / 4096
    assert (np.abs(poses[..., 4:]) < 2**12).all()  # 24 bits: exact
    got = _sweep(poses, start, spheres, world, rows=False)
    np.testing.assert_allclose(got, _reference(poses, start, spheres, world), atol=TOL, rtol=0)


@pytest.mark.parametrize("scale", [0.25, 0.999, 1.001, 1.5])
def test_quaternions_that_are_not_of_unit_length(scale):
    """The placement is linear in the sphere's offset, whatever the quaternion: the minimum is that
    of the rows' own formula.  Offsets up to 3 m: TOL."""
    poses, start, spheres, world = _case(300, 9, 12, 100, 23)
    poses[::2, :, :4] *= np.float32(scale)
    got, ref = _sweep(poses, start, spheres, world, rows=False), _reference(poses, start, spheres, world)
    np.testing.assert_allclose(got, ref, atol=TOL, rtol=0)
