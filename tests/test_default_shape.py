"""Launch shape of workloads without a tuned one: which stage each range of sizes gets."""
from types import SimpleNamespace

import pytest

from pyhype_amd import solvers


def plan(sizes, cartesian=True, flux="Roe", nq=1):
    kinds = cartesian if isinstance(cartesian, tuple) else (cartesian,) * len(sizes)
    blocks = [SimpleNamespace(nx=nx, ny=ny, cartesian=k) for (nx, ny), k in zip(sizes, kinds)]
    return SimpleNamespace(blocks=blocks, flux=flux, quadrature_points=nq,
                           cells=lambda: sum(b.nx * b.ny for b in blocks))


@pytest.mark.parametrize("p, variant, rows", [
    (plan([(1, 1)]), 2, 1), (plan([(60, 256)]), 2, 1), (plan([(61, 128)]), 2, 1), (plan([(60, 257)]), 2, 2),
    (plan([(61, 129)]), 2, 2), (plan([(60, 768)]), 2, 2), (plan([(60, 769)]), 6, 1),
    (plan([(50, 50)] * 4, (True, False, False, False), "HLLL"), 2, 1),
    (plan([(80, 100)] * 4, (True, False, False, False), "HLLL"), 6, 1),
    (plan([(60, 769)], False), 7, 1), (plan([(400, 400)]), 7, 1),
    (plan([(1000, 1000)]), 7, 1), (plan([(1000, 1001)]), 0, 8), (plan([(1000, 1001)], True, "HLLL"), 7, 1),
    (plan([(1600, 1600)], False, "HLLL"), 0, 10), (plan([(4000, 4000)]), 0, 64),
])
def test_default_shape(p, variant, rows):
    shape = solvers.default_shape(p)
    assert (shape.get("variant", 0), shape["rows_per_item"]) == (variant, rows)
    assert shape.get("xcd_chunk", 0) == (64 if variant == 7 and p.cells() > solvers.DEALT_CELLS else 0)


@pytest.mark.parametrize("n, rows_b", [(1, 1), (126, 1), (127, 2), (316, 2), (317, 3), (3000, 3)])
def test_default_shape_of_more_gauss_points(n, rows_b):
    shape = solvers.default_shape(plan([(n, n)], nq=2))
    assert (shape["variant"], shape["rows_per_item"], shape["rows_b"]) == (6, 1, rows_b)
