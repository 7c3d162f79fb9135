"""Shared-halo stage on a mesh of both geometry kinds (one launch over both): residual and steps bit for bit
against the oracle, one and two rows per workgroup, odd rows, and strips at the ends of their columns."""
import numpy as np
import pytest

from oracle import pyhype_oracle as O
from pyhype_amd import Euler2D
from pyhype_amd import workloads as W
from tests.helpers import bitwise_equal_blocks, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("n", [3, 12, 61, 65])
def test_shared_halo_on_both_geometry_kinds(n, rows):
    cfg, mesh = W.double_mach_reflection(n)
    s = Euler2D(cfg, mesh)
    assert {e.cartesian for e in s.plan.blocks} == {True, False}
    s.plan.set_launch(rows, 0, 2, variant=2)
    s.apply_initial_condition()
    st = s.states()[0]
    R = s.plan.get_states(s.plan.residual())[0]
    sim = oracle_for(cfg, mesh, st)
    for k, b in sim.blocks.items():
        np.testing.assert_array_equal(R[k], O.residual(b, sim.flux_fn), err_msg=f"block {k}")
    s.run_steps(4)
    sim.run(4)
    assert bitwise_equal_blocks(s.states()[0], sim.states())
