"""The launch shape a plan reports is the one it runs: rows per workgroup of the shared-halo stage."""
import pytest

from pyhype_amd import Euler2D
from pyhype_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("asked, runs", [(1, 1), (2, 2), (3, 2), (6, 2)])
def test_rows_of_the_shared_halo_stage(asked, runs):
    P = Euler2D(*W.explosion_single(30)).plan
    P.set_launch(asked, variant=2)
    info = P.launch_info()
    assert info["variant"] == 2 and info["rows_per_item"] == runs
    assert info["items_cart"] == 30 // runs            # one strip of 30 rows
    P.set_launch(asked, variant=0)                     # the other stages take the rows as asked
    assert P.launch_info()["rows_per_item"] == asked
