"""The FK adjoint's folded tree: the bound on the moving joints that sizes its tables (exact,
none, too small), ragged batches around a workgroup's 64 configurations, and a tree whose
links hang from constant chains, mimic and offset-only joints."""

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
