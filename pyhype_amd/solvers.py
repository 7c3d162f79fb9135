"""Euler2D: the reference's solver API on top of the gfx950 backend.

``Euler2D(config, mesh_config)`` accepts the same ``SolverConfig`` and mesh dictionary / generator
as the reference (solvers/Euler2D.py:46-100, solvers/base.py:44-100).  ``solve()`` follows the
loop of ``Euler2D._solve`` (solvers/Euler2D.py:175-216): dt from the CFL condition clipped to the
final time, one explicit Runge-Kutta step of all blocks, a realizability check, ``t += dt`` --
with every step executed on the device.  ``run_steps(n)`` advances exactly ``n`` steps.
``Euler2DBatch`` advances many independent cases (each with its own dt) in the same launches.
"""
from __future__ import annotations

import logging
import pathlib
from typing import Dict, List, Optional, Sequence

import numpy as np

from .backend import CaseSpec, DevicePlan
from .mesh import MeshGenerator
from .states import ConservativeState, PrimitiveState
from .time_marching import butcher_table

_log = logging.getLogger("pyhype_amd")

SUPPORTED_FVM = ("MUSCL", "MUSCL-HIP")


class _Mesh:
    """The parts of QuadMesh an initial condition reads: centroids shaped (ny, nx, 1)."""

    def __init__(self, geom):
        self.x = geom.xc[:, :, None]
        self.y = geom.yc[:, :, None]
        self.nx, self.ny = geom.nx, geom.ny
        self.A = geom.A[:, :, None]
        self.geometry = geom


class HostBlock:
    """Host-side view of one block for the initial-condition protocol
    (initial_conditions/base.py:28-31): ``mesh.x/y``, ``config``, ``state``."""

    def __init__(self, config, entry):
        self.config = config
        self.global_block_num = entry.num
        self.mesh = _Mesh(entry.geom)
        self.state = ConservativeState(config.fluid, shape=(entry.ny, entry.nx, 4))
        self.entry = entry


def validate_config(config) -> List[List[float]]:
    """The construction-time checks of the reference factories, for the configuration space the
    backend implements (fvm/factory.py:33-65, fvm/SecondOrderMUSCL.py:49-52, flux/factory.py:30-47,
    limiters/factory.py:28-39, gradients/factory.py:26-37, time_marching/factory.py:29-62)."""
    if config.fvm_type not in SUPPORTED_FVM:
        raise ValueError(f"Specified finite volume method type {config.fvm_type} has not been specialized.")
    if config.fvm_spatial_order != 2:
        raise ValueError(f"No MUSCL finite volume method has been specialized with order {config.fvm_spatial_order}")
    if config.nghost != 1:
        raise ValueError("Number of ghost cells must be equal to 1 for this method.")
    if config.fvm_num_quadrature_points not in (1, 2, 3):
        # the _QUADS lookup of QuadraturePointData (mesh/quadratures.py:33-37,71)
        raise KeyError(config.fvm_num_quadrature_points)
    if config.fvm_gradient_type != "GreenGauss":
        raise ValueError(f"Gradient type {config.fvm_gradient_type} is not available.")
    if config.fvm_flux_function_type not in ("Roe", "HLLL"):
        raise ValueError(f"Flux function type {config.fvm_flux_function_type} is not available.")
    if config.fvm_slope_limiter_type not in ("VanLeer", "VanAlbada", "Venkatakrishnan", "BarthJespersen"):
        raise ValueError("MUSCL: Slope limiter type not specified.")
    if config.reconstruction_type not in (ConservativeState, PrimitiveState):
        raise ValueError("reconstruction_type must be ConservativeState or PrimitiveState")
    if config.interface_interpolation != "arithmetic_average":
        raise ValueError("Interface Interpolation method is not defined.")
    if not config.use_JIT:
        # the reference's use_JIT=False path evaluates other formulas (flux/HLLL.py:43-60,
        # flux/base.py:113-117, limiters/limiters.py:33-36); only the JIT arithmetic is implemented
        raise ValueError("use_JIT=False selects the reference's NumPy formulas, which this backend does not "
                         "implement; use use_JIT=True (the reference default)")
    return butcher_table(config.time_integrator, config)


# Launch shape of a workload without a tuned one (us per RK stage measured on an MI355X, 256 CUs, smooth
# flow, the alternatives beside it):
#  * The shared-halo stage (variant 2) while its workgroups, one per CU, fit the chip: with one row each up to
#    256 workgroups (120^2, 240 of them: 9.4 against 13.4 with the split stage and 26.7 fused; 64^2: 11.0,
#    14.6 and 25.7), with two rows beyond (160^2, 240: 10.7 against 13.8; 60 x 512, 256: 10.9 against 13.9; HLLL
#    14.2 against 19.8).  Between 257 and 384 workgroups of two rows, a second round, neither stage is the
#    faster one throughout.  A list whose length is no multiple of 8 gives some workgroup two items (an XCD's
#    share of the items and of the workgroups are rounded differently: 60 x 500, 250 workgroups, takes 17.3
#    where 256 take 10.9), which costs the split stage most, with its short items: six 93 x 61 HLLL quads,
#    372, 24.1 against 30.7; 60 x 700, 350, 18.6 against 19.8 (HLLL 23.2 and 26.0); 180^2, 270, 17.5 against
#    20.0.  Where its lists do divide by 8 the split stage takes 15 to 23 % less with Roe and 2 to 11 % less
#    with HLLL (60 x 768, 384: 18.8 against 14.6, HLLL 23.6 and 20.9; 5 x 64^2, 320: 18.3 against 14.1, 22.2
#    and 20.4; 4 x 70^2, 280: 18.8 against 16.0, 22.2 and 21.8).  The same happens below 256 where only the
#    shared-halo stage's own count does not divide (60 x 280, 140: 17.8 against 14.4; 180 x 168, 252: 16.7
#    against 13.8).  The fused stage takes 26 to 45 in all of these.
#    At 500 the shared-halo stage is behind in any case (5 x 100^2 HLLL: 26.3 against 22.5).
#  * The split stage with one y-face per wave up to the size where the states that pass between its
#    kernels no longer stay in the caches: strips (variant 6) while a Cartesian mesh has fewer than 10^5
#    cells (256^2: 18.2 against 20.4), row-major (variant 7) beyond (400^2: 26.6 against 27.4;
#    8 x 150^2: 29.5 against 33.8), up to 10^6 cells with Roe (1.1 x 10^6: 98 against 96 fused;
#    2.25 x 10^6: 220 against 167) and 2.5 x 10^6 with HLLL, whose fused kernel is bound by its
#    registers (1.1 x 10^6: 120 against 136; 2.8 x 10^6: 319 against 326).
#    From 2.5 x 10^5 cells the work lists are dealt to the XCDs in chunks of 64 items, which evens out flows
#    that cost more in one part of the mesh (a shock, HLLL: 5 x 240^2 38.8 -> 35.1, 5 x 450^2 82.7 -> 75.1,
#    4 x 640 x 240 64.9 -> 62.5; a blast or waves everywhere: between 4 % less and 3 % more from 2.9 x 10^5 to
#    10^6 cells).  Smaller meshes have too few chunks to spread evenly over 8 XCDs (400^2 has 41: 22.1 -> 25.9;
#    330^2 19.3 -> 21.6), or happen to have a good number (8 x 150^2, 46: 27.6 -> 27.2, shock 34.7 -> 33.5).
#  * The fused stage beyond, with items of 8 rows or more (1.1 x 10^6 cells: 4 rows 111.9, 8 rows 96.2;
#    2.4 x 10^6: 4 rows 221.6, 10 rows 201.0).
#  * More than one Gauss point per face: strips, one row per item (two take 33 to 180 % longer up to 1.2 x 10^5
#    cells, 0 to 5 % from 1.6 x 10^5), with 1, 2 or 3 rows of the update.  Two points with Roe and
#    Venkatakrishnan's limiter, with 1, 2, 3 rows: 100^2 23.9, 27.7, 27.8; 200 x 120 27.3, 25.7, 27.0; 400^2
#    59.1, 58.2, 56.0; 800 x 600 133, 128, 126.  HLLL, three points and general blocks order the same way
#    (100^2 HLLL 36.5, 42.5, 42.3; three points 30.1, 35.0, 35.8; 800 x 600 general HLLL with three 251, 235,
#    230); of 13 sizes only 4 x 61 x 55, whose list divides unevenly, is more than 4 % from the best of the
#    three (31.6, 28.1, 32.6).
SHARED_ITEMS = (256, 384)          # workgroups of the shared-halo stage with 1 and 2 rows
STRIP_CELLS = 100_000
DEALT_CELLS = 250_000
SPLIT_CELLS = {"Roe": 1_000_000, "HLLL": 2_500_000}
FUSED_ROWS = 8
GAUSS_CELLS = (16_000, 100_000)    # up to which the update of a plan with Gauss points takes 1 and 2 rows


def default_rows(cells: int) -> int:
    """Rows per item of the fused stage: about 4096 items of 60 columns."""
    return int(max(2, min(64, round(cells / (60 * 4096)))))


def default_shape(plan) -> dict:
    """``DevicePlan.set_launch`` arguments for a workload without a tuned shape (see above)."""
    cells = plan.cells()
    if plan.quadrature_points > 1:
        return {"rows_per_item": 1, "waves_per_simd": 3, "variant": 6,
                "rows_b": 1 if cells < GAUSS_CELLS[0] else (2 if cells < GAUSS_CELLS[1] else 3)}
    kinds = {e.cartesian for e in plan.blocks}
    strips = [(-(-e.nx // 60), e.ny) for e in plan.blocks]
    for rows, most in zip((1, 2), SHARED_ITEMS):
        if sum(n * -(-ny // rows) for n, ny in strips) <= most:
            return {"rows_per_item": rows, "variant": 2}
    if cells > SPLIT_CELLS[plan.flux]:
        return {"rows_per_item": max(FUSED_ROWS, default_rows(cells))}
    if cells < STRIP_CELLS and kinds != {False}:
        return {"rows_per_item": 1, "waves_per_simd": 3, "variant": 6, "rows_b": 1}
    return {"rows_per_item": 1, "waves_per_simd": 3, "variant": 7, "rows_b": 3,
            "xcd_chunk": 64 if cells > DEALT_CELLS else 0}


def mesh_dict(mesh_config) -> Dict[int, dict]:
    return mesh_config.dict if isinstance(mesh_config, MeshGenerator) else mesh_config


class _HostEntry:
    """The parts of a plan's block entry that HostBlock reads, for host-only set-ups."""

    def __init__(self, num, geom):
        self.num, self.geom, self.nx, self.ny = num, geom, geom.nx, geom.ny


def host_initial_states(config, mesh_config, initial_condition=None) -> Dict[int, np.ndarray]:
    """Initial conservative state of every block, computed on the host only (no device plan): the
    same IC protocol as Euler2D.apply_initial_condition (solvers/Euler2D.py:90-92) on blocks whose
    geometry follows the reference's mesh formulas."""
    from .mesh import BlockGeometry

    ic = config.initial_condition if initial_condition is None else initial_condition
    out = {}
    for n, d in mesh_dict(mesh_config).items():
        geom = BlockGeometry({k: d[k] for k in ("SW", "SE", "NW", "NE")}, config.nx, config.ny)
        hb = HostBlock(config, _HostEntry(n, geom))
        ic.apply_to_block(hb)
        out[n] = np.array(hb.state.data, dtype=np.float64)
    return out


class Euler2DBatch:
    """Independent cases advanced together.  All cases share flux, limiter, time integrator, CFL and
    fluid; each keeps its own block size, dt (CFL of its own blocks) and time."""

    def __init__(self, configs: Sequence, meshes: Sequence, *, rows_per_item: int = 0, grid_waves: int = 0,
                 force_general: bool = False, use_tuning_cache: bool = True):
        if len(configs) != len(meshes) or not configs:
            raise ValueError("need one mesh per config")
        c0 = configs[0]
        self.table = validate_config(c0)
        for c in configs[1:]:
            validate_config(c)
            for attr in ("fvm_flux_function_type", "fvm_slope_limiter_type", "reconstruction_type", "time_integrator",
                         "CFL", "fvm_num_quadrature_points"):
                if getattr(c, attr) != getattr(c0, attr):
                    raise ValueError(f"batched cases must share {attr}")
            if type(c.fluid) is not type(c0.fluid):
                raise ValueError("batched cases must share the fluid")
        self.configs = list(configs)
        self.fluid = c0.fluid
        specs = [CaseSpec(mesh_dict(m), c.nx, c.ny, c.t_final * c.fluid.far_field.a) for c, m in zip(configs, meshes)]
        self.plan = DevicePlan(specs, flux=c0.fvm_flux_function_type, table=self.table, fluid=c0.fluid,
                               cfl=c0.CFL, rows_per_item=rows_per_item, grid_waves=grid_waves,
                               force_general=force_general, limiter=c0.fvm_slope_limiter_type,
                               primitive=c0.reconstruction_type is PrimitiveState,
                               quadrature_points=c0.fvm_num_quadrature_points)
        self.tuned = False
        if rows_per_item == 0:
            from . import autotune

            self.tuned = use_tuning_cache and autotune.apply_cached(self.plan)
            if not self.tuned:
                # a persistent grid is asked for: the fused stage strides over its list with it
                shape = {"rows_per_item": default_rows(self.plan.cells())} if grid_waves else default_shape(self.plan)
                self.plan.set_launch(grid_waves=grid_waves, **shape)
        self.case_blocks: List[Dict[int, HostBlock]] = []
        for c, entries in enumerate(self.plan.case_blocks):
            self.case_blocks.append({n: HostBlock(self.configs[c], e) for n, e in entries.items()})
        self.t = np.zeros(len(configs))
        self.num_time_step = 0
        self.failed: Dict[int, int] = {}

    # ---------------------------------------------------------------- set-up
    def apply_initial_condition(self, initial_condition=None):
        """Euler2D.apply_initial_condition (solvers/Euler2D.py:90-92), then upload.  An explicit
        ``initial_condition`` replaces the configured one of every case."""
        for c, blocks in enumerate(self.case_blocks):
            ic = self.configs[c].initial_condition if initial_condition is None else initial_condition
            for blk in blocks.values():
                ic.apply_to_block(blk)
        self.upload()

    def upload(self):
        self.plan.set_states([{n: b.state.data for n, b in blocks.items()} for blocks in self.case_blocks])
        self.plan.reset(self.t, self.num_time_step)

    def set_state(self, states: Sequence[Dict[int, np.ndarray]]):
        for c, blocks in enumerate(self.case_blocks):
            for n, b in blocks.items():
                b.state.data = np.array(states[c][n], dtype=np.float64)
        self.upload()

    # ---------------------------------------------------------------- stepping
    strict = False  # raise on any unrealizable case (True for the single-case Euler2D)

    def run_steps(self, n: int, use_graph: bool = True):
        """Advance exactly n steps (dt per case from the CFL condition, clipped to t_final).

        A case whose state becomes unrealizable (rho <= 0 or E <= 0) is frozen at that step, as
        the reference aborts that run (solvers/Euler2D.py:144-152); ``failed`` maps case -> step.
        With ``strict`` a RealizabilityError is raised instead."""
        if n <= 0:
            return
        try:
            self.plan.run(n, use_graph=use_graph, check=False)
        finally:
            # also after a RealizabilityError: time, step counter and the failing step of each case
            # describe the state the plan holds
            bad, step, t, dt = self.plan.status()
            self.t = t
            self.dt_last = dt
            self.num_time_step = step
            self.failed = self.plan.failed_cases(bad)
        if self.strict:
            self.plan.check_realizable(bad)

    def autotune(self, steps: int = 10, **kw):
        """Tune the launch shape on the current state (state, time and step are restored)."""
        from . import autotune

        res = autotune.autotune(self.plan, steps=steps, **kw)
        self.tuned = True
        return res

    def states(self) -> List[Dict[int, np.ndarray]]:
        return self.plan.get_states()

    def sync_to_host(self):
        for c, st in enumerate(self.states()):
            for n, arr in st.items():
                self.case_blocks[c][n].state.data = arr

    def last_dt(self) -> np.ndarray:
        return self.plan.status()[3]


class Euler2D(Euler2DBatch):
    """Single-case solver with the reference's constructor, ``solve()`` and file output."""

    strict = True

    def __init__(self, config, mesh_config, **kw):
        super().__init__([config], [mesh_config], **kw)
        self.config = config
        self.t_final = config.t_final * config.fluid.far_field.a
        # Solver.__init__ (solvers/base.py:78-86)
        self.write_path = None
        if getattr(config, "write_solution", False):
            self.write_path = pathlib.Path(config.write_solution_base) / config.write_solution_name
            self.write_path.mkdir(exist_ok=True, parents=True)
            _log.info(self.write_path)

    @property
    def blocks(self):
        return self.case_blocks[0].values()

    def state(self, block_num: int) -> np.ndarray:
        return self.states()[0][block_num]

    # ---------------------------------------------------------------- file output
    def write_mesh(self):
        """Solver.write_mesh (solvers/base.py:142-155): cell centroids of every block as
        ``<write_path>/mesh/mesh_{x,y}_blk_<n>.npy`` with shape (ny, nx, 1)."""
        path = self.write_path / "mesh"
        path.mkdir(parents=True, exist_ok=True)
        for b in self.blocks:
            np.save(str(path / "mesh_x_blk_") + str(b.global_block_num), b.mesh.x)
            np.save(str(path / "mesh_y_blk_") + str(b.global_block_num), b.mesh.y)

    def write_solution(self):
        """Solver.write_solution (solvers/base.py:157-172): in mode ``every_n_timesteps`` and when
        ``num_time_step % write_every_n_timesteps == 0``, the conservative state of every block as
        ``<write_path>/<num_time_step>/<write_solution_name>_blk_<n>.npy`` (ny, nx, 4)."""
        cfg = self.config
        if cfg.write_solution_mode == "every_n_timesteps" and self.num_time_step % cfg.write_every_n_timesteps == 0:
            path = self.write_path / str(self.num_time_step)
            path.mkdir(parents=True, exist_ok=True)
            states = self.plan.get_states()[0]
            for b in self.blocks:
                np.save(str(path / cfg.write_solution_name) + "_blk_" + str(b.global_block_num),
                        states[b.global_block_num])

    def solve(self, chunk: int = 50, max_steps: Optional[int] = None):
        """Run to t_final (solvers/Euler2D.py:97-100,175-216).

        With ``config.write_solution`` the mesh is written first and the solution at the reference's
        points: ``write_solution`` runs after a step's update and before ``num_time_step`` is
        incremented, so the files in directory ``k`` (k a multiple of write_every_n_timesteps) hold
        the state after step k + 1.  Steps between output points run on the device in chunks."""
        self.apply_initial_condition()
        writing = self.write_path is not None
        if writing:
            self.write_mesh()
        every = max(1, int(getattr(self.config, "write_every_n_timesteps", 1) or 1))
        steps = 0
        while self.t[0] < self.t_final and (max_steps is None or steps < max_steps):
            if self.num_time_step % 50 == 0:
                _log.info("Simulation time: %s, Timestep number: %s", self.t[0] / self.fluid.far_field.a,
                          self.num_time_step)
            n = chunk if max_steps is None else min(chunk, max_steps - steps)
            last = float(getattr(self, "dt_last", [0.0])[0])
            if last <= 0.0 or self.t_final - self.t[0] < 1.5 * n * last:
                n = 1  # first step, or near t_final: single steps, so the count stops where the reference's does
            if writing and self.config.write_solution_mode == "every_n_timesteps":
                # the next output point: the step whose pre-increment counter is a multiple of `every`
                k = self.num_time_step
                nxt = k if k % every == 0 else k + (every - k % every)
                n = min(n, nxt - k + 1)
            self.run_steps(n)
            steps += n
            if writing:
                # run_steps advanced num_time_step by n; the reference writes with the counter of the
                # step just taken, before its increment
                self.num_time_step -= 1
                self.write_solution()
                self.num_time_step += 1
        self.sync_to_host()
