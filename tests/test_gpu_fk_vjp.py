"""The FK adjoint's folded tree: the bound on the moving joints that sizes its tables (exact,
none, too small), ragged batches around a workgroup's 64 configurations, a tree whose
links hang from constant chains, mimic and offset-only joints, and trees as large as the LDS allows."""

import numpy as np
import pytest
import torch
from conftest import ROBOTS, load_robot, random_cfgs

from pyroffi_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ROBOTS + ("mimic_arm",))
@pytest.mark.parametrize("batch", [1, 63, 65, 200])
def test_bound_on_moving_joints(name, batch):
    robot, _ = load_robot(name)
    t = robot.device_tables()
    q = torch.as_tensor(random_cfgs(robot, batch, seed=3).astype(np.float32), device="cuda")
    rng = np.random.default_rng(batch)
    cot = torch.as_tensor(rng.normal(size=(batch, robot.links.num_links, 7)).astype(np.float32), device="cuda")
    args = (q, cot, *t.robot_buffers(), t.link_parent_joint)
    full = ops.fk_vjp(*args)
    torch.testing.assert_close(ops.fk_vjp(*args, max_moving=t.n_moving), full, rtol=0, atol=0)
    assert torch.isnan(ops.fk_vjp(*args, max_moving=t.n_moving - 1)).all()
    # Linear in the cotangent: 2 FP32 sums of up to 44 x 7 terms, 1e-5 of the largest entry.
    half = ops.fk_vjp(q, 0.5 * cot, *args[2:], max_moving=t.n_moving)
    torch.testing.assert_close(2 * half, full, rtol=1e-5, atol=1e-5 * float(full.abs().max()))


class _Tree:
    """Joint and link tables of a random tree whose every joint moves: the first A are actuated,
    the others follow one of them."""

    def __init__(self, J, A, seed):
        rng = np.random.default_rng(seed)
        j = np.arange(J)
        quat = rng.normal(size=(J, 4))
        quat /= np.linalg.norm(quat, axis=1, keepdims=True)
        axis = rng.normal(size=(J, 3))
        axis /= np.linalg.norm(axis, axis=1, keepdims=True)
        slides = (rng.random(J) < 0.2)[:, None]
        self.twists = np.concatenate([axis * slides, axis * ~slides], 1)
        self.parent_transforms = np.concatenate([quat, rng.uniform(-0.1, 0.1, (J, 3))], 1)
        self.parent_indices = np.where(rng.random(J) < 0.7, j - 1, rng.integers(-1, j))
        self.actuated_indices = np.where(j < A, j, -1)
        self.mimic_multiplier = np.where(j < A, 1.0, rng.uniform(-1, 1, J))
        self.mimic_offset = np.where(j < A, 0.0, rng.uniform(-1, 1, J))
        self.mimic_act_indices = np.where(j < A, -1, rng.integers(0, A, J))
        self._topo_sort_inv = j
        self.num_joints, self.num_actuated_joints = J, A
        self.parent_joint_indices = np.concatenate([[-1], j])  # as links: the base, then one a joint
        self.num_links = J + 1


def _vjp_of(t, q, cot):
    dev = lambda *v: [torch.as_tensor(np.ascontiguousarray(x), device="cuda") for x in v]  # noqa: E731
    tables = dev(t.twists, t.parent_tf, t.parent_idx, t.act_idx, t.mimic_mul, t.mimic_off, t.mimic_act_idx, t.topo_inv)
    return ops.fk_vjp(*dev(q, cot), *tables, *dev(t.link_parent_joint), max_moving=None)


@pytest.mark.parametrize("J,A", [(46, 16), (46, 10), (46, 9), (47, 3), (45, 16), (1, 1)])
def test_largest_trees(oracle_mod, J, A):
    """Trees near the limit of the LDS, against central differences of the float64 oracle.  FP32
    poses of a chain of up to 47 joints: 47 x 4 roundings of 6e-8, 1e-4 of the largest entry."""
    tree = _Tree(J, A, seed=J + A)
    t = oracle_mod.Tables(tree, tree)
    rng = np.random.default_rng(J)
    q = rng.uniform(-1, 1, (70, A)).astype(np.float32)
    cot = rng.normal(size=(70, J + 1, 7)).astype(np.float32)
    got = _vjp_of(t, q, cot).cpu().numpy()
    ref = np.zeros((70, A))
    h = 1e-5
    for a in range(A):
        step = np.zeros(A)
        step[a] = h
        ends = [oracle_mod.fk_links(t, q.astype(np.float64) + s * step) for s in (1, -1)]
        ref[:, a] = ((ends[0] - ends[1]) * cot).sum((1, 2)) / (2 * h)
    np.testing.assert_allclose(got, ref, rtol=0, atol=1e-4 * np.abs(ref).max())


def test_trees_past_the_limit_are_refused(oracle_mod):
    for J, A in ((48, 1), (64, 16)):
        tree = _Tree(J, A, seed=J)
        with pytest.raises(RuntimeError, match="LDS"):
            _vjp_of(oracle_mod.Tables(tree, tree), np.zeros((2, A), np.float32), np.zeros((2, J + 1, 7), np.float32))
