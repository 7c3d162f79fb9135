"""Plans and states outside the range of the short evaluations.  Lengths times 2^s leave every gradient's
increments and every flux alone and multiply the residual by 2^-s without any rounding, so the general
evaluations must give the short ones' bits.  A cell out of range sends its wave to the general evaluation:
the cells it does not reach must keep their bits.  States times 2^k, and a gas with gamma - 1 below 2^-20,
against the oracle."""
import numpy as np
import pytest

from oracle import pyhype_oracle as O
from pyhype_amd import Euler2D
from pyhype_amd import workloads as W
from pyhype_amd.fluids import Air
from pyhype_amd.solvers import mesh_dict
from pyhype_amd.states import ConservativeState, PrimitiveState
from tests.helpers import oracle_for, skewed_mesh

# mesh, flux, limiter, primitive, Gauss points, stage variants
PLANS = [("cart", "Roe", "Venkatakrishnan", False, 1, (0, 2, 6, 7)), ("skewed", "HLLL", "Venkatakrishnan", False, 1, (0, 2, 6, 7)),
         ("skewed", "Roe", "BarthJespersen", False, 1, (0, 2)), ("cart", "HLLL", "VanAlbada", True, 1, (2, 7)),
         ("cart", "Roe", "BarthJespersen", False, 2, (6,)), ("skewed", "HLLL", "Venkatakrishnan", False, 3, (6,)),
         ("ramp", "HLLL", "Venkatakrishnan", False, 1, (2, 7))]


def _setup(mesh, flux, limiter, primitive, nq, lengths=1.0):
    if mesh == "cart":
        cfg, m = W.explosion_single(70)
    elif mesh == "ramp":
        cfg, m = W.double_mach_reflection(12)
    else:
        cfg, m = W.explosion_single(20)[0], skewed_mesh()
    m = {n: dict(b, **{k: [float(v) * lengths for v in b[k]] for k in ("SW", "SE", "NW", "NE")})
         for n, b in mesh_dict(m).items()}
    cfg.fvm_flux_function_type, cfg.fvm_slope_limiter_type, cfg.fvm_num_quadrature_points = flux, limiter, nq
    cfg.reconstruction_type = PrimitiveState if primitive else ConservativeState
    return cfg, m


def _states(cfg, mesh, seed=9):
    rng, out = np.random.default_rng(seed), {}
    for n in mesh:
        shape = (cfg.ny, cfg.nx)
        r, p = (a * (1.0 + 0.1 * rng.standard_normal(shape)) for a in (1.2, 0.9))
        u, v = (0.3 * rng.standard_normal(shape) for _ in range(2))
        out[n] = np.stack([r, r * u, r * v, p / 0.4 + 0.5 * r * (u * u + v * v)], axis=-1)
        out[n][: cfg.ny // 4, : cfg.nx // 3] = [1.2, 0.0, 0.0, 2.25]   # still and uniform
    return out


def _residuals(plan_args, st, variants, lengths=1.0):
    """The residual of every stage variant, one plan."""
    cfg, m = _setup(*plan_args, lengths=lengths)
    s = Euler2D(cfg, m)
    s.set_state([st])
    out = []
    for v in variants:
        s.plan.set_launch(1 if v == 2 else 3, 0, 2, variant=v, rows_b=2)
        out.append(s.plan.get_states(s.plan.residual())[0])
    s.plan.close()
    return out


def _same(a, b, scale):
    for n in a:
        assert np.isfinite(a[n]).all()
        np.testing.assert_array_equal(a[n] * scale, b[n], err_msg=f"block {n}")


@pytest.mark.gpu
@pytest.mark.parametrize("plan", PLANS, ids=lambda p: "-".join(map(str, p[:5])))
@pytest.mark.parametrize("s", [-40, 66])
def test_lengths_out_of_range(plan, s):
    st = _states(*_setup(*plan[:5]))
    for a, b in zip(_residuals(plan[:5], st, plan[5]), _residuals(plan[:5], st, plan[5], lengths=2.0 ** s)):
        _same(a, b, 2.0 ** -s)


@pytest.mark.gpu
@pytest.mark.parametrize("plan", PLANS, ids=lambda p: "-".join(map(str, p[:5])))
@pytest.mark.parametrize("k", [-420, 110, 420])
def test_states_out_of_range_match_the_oracle(plan, k):
    cfg, m = _setup(*plan[:5])
    st = {n: a * 2.0 ** k for n, a in _states(cfg, m).items()}
    sim = oracle_for(cfg, m, st)
    with np.errstate(all="ignore"):
        ref = {n: O.residual(b, sim.flux_fn) for n, b in sim.blocks.items()}
    for R in _residuals(plan[:5], st, plan[5]):
        for n in ref:
            np.testing.assert_array_equal(R[n], ref[n], err_msg=f"block {n}")


BAD = {"nan": np.nan, "inf": np.inf, "negative": -1.0, "zero": 0.0, "huge": 2.0 ** 700, "tiny": 2.0 ** -700}


@pytest.mark.gpu
@pytest.mark.parametrize("plan", PLANS, ids=lambda p: "-".join(map(str, p[:5])))
def test_cells_out_of_range_leave_the_others_alone(plan):
    cfg, m = _setup(*plan[:5])
    st = _states(cfg, m)
    clean = _residuals(plan[:5], st, plan[5])
    at = [(cfg.ny // 2, cfg.nx // 2), (2, cfg.nx - 4)]
    for value in BAD.values():
        for var in (0, 1, 3):
            bad = {n: a.copy() for n, a in st.items()}
            first = next(iter(bad))
            for k, j in at:
                bad[first][k, j, var] = value
            for a, b in zip(clean, _residuals(plan[:5], bad, plan[5])):
                for n in a:
                    far = np.ones(a[n].shape[:2], dtype=bool)
                    if n == first:
                        for k, j in at:   # the residual's stencil: two cells along a row or a column
                            far[k, max(0, j - 2):j + 3] = False
                            far[max(0, k - 2):k + 3, j] = False
                            far[max(0, k - 1):k + 2, max(0, j - 1):j + 2] = False
                    np.testing.assert_array_equal(a[n][far], b[n][far], err_msg=f"block {n}, {value} in variable {var}")


@pytest.mark.gpu
@pytest.mark.parametrize("flux", ["Roe", "HLLL"])
@pytest.mark.parametrize("gamma", [1.0 + 2.0 ** -21, 1.0 + 2.0 ** -19])
def test_gas_out_of_range_matches_the_oracle(flux, gamma, monkeypatch):
    class Gas(Air):
        def gamma(self, *a, **kw):
            return gamma

    cfg, m = _setup("cart", flux, "Venkatakrishnan", False, 1)
    cfg.nx = cfg.ny = 30
    cfg.fluid = Gas(a_inf=1.0, rho_inf=1.0)
    st = _states(cfg, m)
    for a in st.values():     # pressures of the same size as before
        a[..., 3] = 0.9 / (gamma - 1) + 0.5 * (a[..., 1] ** 2 + a[..., 2] ** 2) / a[..., 0]
    for name, v in (("GAMMA", gamma), ("GM1", gamma - 1), ("ONE_OVER_GM1", 1.0 / (gamma - 1.0)),
                    ("G_OVER_GM1", gamma / (gamma - 1.0))):
        monkeypatch.setattr(O, name, v)
    sim = oracle_for(cfg, m, st)
    s = Euler2D(cfg, m)
    s.set_state([st])
    for v in (0, 2, 7):
        s.plan.set_launch(2, 0, 2, variant=v, rows_b=2)
        R = s.plan.get_states(s.plan.residual())[0]
        for n, b in sim.blocks.items():
            np.testing.assert_array_equal(R[n], O.residual(b, sim.flux_fn), err_msg=f"variant {v}, block {n}")
