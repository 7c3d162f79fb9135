"""Time steps, times, step counter and failures where the stage kernels take the closing of a step along
(against the fused stage, which has a kernel of its own for it): bit for bit, over every stage variant, one-,
two- and four-stage tables, runs of uneven lengths, eager and as graphs, and with a given schedule."""
import numpy as np
import pytest
import torch

from pyhype_amd import workloads as W
from pyhype_amd.solvers import Euler2DBatch
from tests.helpers import bitwise_equal_blocks

pytestmark = pytest.mark.gpu

RUNS = [(1, True), (3, True), (2, False), (13, True), (1, False), (1, True)]


def history(variant, integrator, frozen=False):
    cfgs, meshes, _ = W.explosion_batch(seed=0, ncases=6, sizes=[24, 16, 33, 64, 70, 20], density_scaled=True)
    for c in cfgs:
        c.time_integrator = integrator
    cfgs[1].t_final = 1.0 / cfgs[1].fluid.far_field.a  # reached within the run: a last step is clipped to it
    s = Euler2DBatch(cfgs, meshes, rows_per_item=2)
    s.plan.set_launch(2 if variant == 0 else 1, 0, 2, variant=variant, rows_b=2)
    s.apply_initial_condition()
    if frozen:
        dt = s.plan.dt()
        s.plan.run_frozen(dt[None, :] * torch.linspace(0.1, 0.3, 5, dtype=dt.dtype, device=dt.device)[:, None],
                          check=False)
        return s.states(), [], s.plan.status()
    log = []
    for n, graph in RUNS:
        s.run_steps(n, use_graph=graph)
        log.append(s.plan.status())
    return s.states(), log, s.failed


@pytest.mark.parametrize("integrator", ["ExplicitEuler1", "RK2", "RK4"])
@pytest.mark.parametrize("variant", [1, 2, 3, 5, 6, 7, 8])
def test_folded_steps(variant, integrator):
    a, b = history(0, integrator), history(variant, integrator)
    assert a[2] == b[2] and (a[2] or integrator != "RK4")
    for x, y in zip(a[1], b[1]):
        for p, q in zip(x, y):
            np.testing.assert_array_equal(p, q)
    for x, y in zip(a[0], b[0]):
        assert bitwise_equal_blocks(x, y)


@pytest.mark.parametrize("variant", [1, 2, 3, 6])
def test_folded_steps_of_a_schedule(variant):
    a, b = history(0, "RK2", frozen=True), history(variant, "RK2", frozen=True)
    for p, q in zip(a[2], b[2]):
        np.testing.assert_array_equal(p, q)
    for x, y in zip(a[0], b[0]):
        assert bitwise_equal_blocks(x, y)
