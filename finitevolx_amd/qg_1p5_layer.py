"""The reference's 1.5-layer QG double-gyre example on the GPU
(``scripts/qg_1p5_layer.py``), composed from the drop-in operators.

Each step is ``heun_step`` of

    dq/dt = -div(u q) - beta v + F - r zeta + nu lap(q),
    (lap - 1/Ld^2) psi = q  (DST-I, psi = 0 on the walls),

with upwind1 advection, u = -d_y(T_to_X psi), v = d_x(T_to_X psi) at the
U / V faces, zeta = lap(psi) and the wall (zero ghost ring) condition
re-applied before each tendency and after the step (``:420-497``).  The
tendency's operators are one HIP kernel of ``libfvx_hip.so`` (one kernel each
where the model's operators were replaced); the Helmholtz inversion is the
DST-I solve.  Snapshots are returned as arrays (the reference writes
them with xarray / Zarr, absent here).
"""

from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import torch

from finitevolx_amd import _lib
from finitevolx_amd.advection import Advection2D
from finitevolx_amd.boundary import pad_interior
from finitevolx_amd.grid import CartesianGrid2D
from finitevolx_amd.operators import Difference2D, Interpolation2D
from finitevolx_amd.solvers import dirichlet_field_solve, solve_helmholtz_dst
from finitevolx_amd.timestepping import heun_step, lincomb


@dataclass
class QuasiGeostrophicConfig:
    """Defaults of ``QuasiGeostrophicConfig`` (``scripts/qg_1p5_layer.py:280-300``)."""

    nx: int = 64
    ny: int = 64
    Lx: float = 5.12e6
    Ly: float = 5.12e6
    f0: float = 9.375e-5
    beta: float = 1.754e-11
    gravity: float = 9.81
    rossby_radius: float = 4.0e4
    drag: float = 5.0e-8
    viscosity: float = 5.0e4
    wind_curl_forcing: float = 2.0e-12
    dt: float = 4000.0
    spinup_steps: int = 5000
    steps: int = 10000
    snapshot_interval: int = 1000


def to_wall_field(interior) -> torch.Tensor:
    """Interior ``[ny, nx]`` -> full ``[ny+2, nx+2]`` with a zero ghost ring
    (``scripts/qg_1p5_layer.py:92-113``)."""
    t = _lib.as_field(interior)
    return torch.nn.functional.pad(t[None, None], (1, 1, 1, 1))[0, 0].contiguous()


_lib.extra_signatures({
    f"fvx_gyre_tendency_{s}": [_lib._vp] * 6 + [_lib._i] * 2 + [_lib._d] * 5 + [_lib._vp]
    for s in ("f32", "f64")
})


# The methods that the one-kernel path stands for, as this package defines them.
_METHODS = {cls: tuple((n, getattr(cls, n)) for n in names) for cls, names in (
    (Difference2D, ("diff_y_X_to_U", "diff_x_X_to_V", "laplacian", "_op")),
    (Interpolation2D, ("T_to_X", "V_to_T")), (Advection2D, ("__call__",)))}


def _unmasked(op, cls) -> bool:
    """Whether ``op`` is the package's own operator without a mask: no subclass, no
    method replaced on the class, and nothing set on the instance beyond its grid
    and mask (a method, say)."""
    return (type(op) is cls and op.mask is None and len(vars(op)) == 2
            and all(getattr(cls, n) is f for n, f in _METHODS[cls]))


def _gyre(q, psi, wind, grid, beta=0.0, drag=0.0, viscosity=0.0):
    """``(rhs, u, v)`` of the unmasked operators in one kernel; ``q`` None: no rhs."""
    u, v = torch.empty_like(psi), torch.empty_like(psi)
    rhs = None if q is None else torch.empty_like(q)
    ny, nx = psi.shape
    _lib.call(f"fvx_gyre_tendency_{_lib.suffix(psi)}", _lib.ptr(q), psi.data_ptr(),
              _lib.ptr(wind), _lib.ptr(rhs), u.data_ptr(), v.data_ptr(), ny, nx,
              float(grid.dx), float(grid.dy), float(beta), float(drag), float(viscosity),
              _lib.stream())
    return rhs, u, v


def geostrophic_velocity_from_streamfunction(psi_field, diff: Difference2D,
                                             interp: Interpolation2D):
    """T-point psi -> (u, v) at U / V faces through X points (``:115-145``)."""
    psi = _lib.as_field(psi_field)
    if psi.dim() == 2 and _unmasked(diff, Difference2D) and _unmasked(interp, Interpolation2D):
        return _gyre(None, psi, None, diff.grid)[1:]
    psi_on_x = interp.T_to_X(psi_field)
    return -diff.diff_y_X_to_U(psi_on_x), diff.diff_x_X_to_V(psi_on_x)


def initial_fields(config: QuasiGeostrophicConfig, grid: CartesianGrid2D):
    """PV anomaly, beta term and wind-curl forcing on the interior
    (``make_preprocessing_dataset``, ``:302-371``), as host arrays."""
    x = (np.arange(config.nx) + 0.5) * grid.dx
    y = (np.arange(config.ny) + 0.5) * grid.dy
    X, Y = np.meshgrid(x, y)
    q0 = 5.0e-9 * np.sin(2.0 * np.pi * X / config.Lx) * np.sin(np.pi * Y / config.Ly)
    beta_term = config.beta * (Y - 0.5 * config.Ly)
    wind_curl = -config.wind_curl_forcing * np.sin(2.0 * np.pi * Y / config.Ly)
    return q0, beta_term, wind_curl


class QG1p5LayerModel:
    """The example's state update on device arrays (FP64 by default)."""

    def __init__(self, config: QuasiGeostrophicConfig | None = None,
                 dtype: torch.dtype = torch.float64):
        self.config = config or QuasiGeostrophicConfig()
        c = self.config
        self.grid = CartesianGrid2D.from_interior(c.nx, c.ny, c.Lx, c.Ly)
        self.diff = Difference2D(self.grid)
        self.interp = Interpolation2D(self.grid)
        self.adv = Advection2D(self.grid)
        self.dtype = dtype
        q0, _, wind = initial_fields(c, self.grid)
        self.q0 = to_wall_field(torch.tensor(q0, dtype=dtype))
        self.wind_curl = to_wall_field(torch.tensor(wind, dtype=dtype))
        self.lam = 1.0 / c.rossby_radius**2

    def invert_streamfunction(self, q_field):
        """(lap - 1/Ld^2) psi = q on the interior, psi = 0 walls (``:432-452``)."""
        if q_field.dim() == 2 and min(q_field.shape) >= 4:
            return dirichlet_field_solve(q_field, self.grid.dx, self.grid.dy, self.lam)
        psi_i = solve_helmholtz_dst(q_field[1:-1, 1:-1].contiguous(), self.grid.dx,
                                    self.grid.dy, self.lam)
        return to_wall_field(psi_i)

    def tendency(self, q_field):
        """``(q_rhs, psi, u, v)`` of ``tendency`` (``:454-478``)."""
        c = self.config
        psi = self.invert_streamfunction(q_field)
        if self._plain_operators():
            q, p = _lib.as_field(q_field), _lib.as_field(psi)
            wind = _lib.as_field(self.wind_curl, q.dtype)
            if q.dim() == 2 and p.dtype == q.dtype and p.shape == q.shape == wind.shape:
                q_rhs, u, v = _gyre(q, p, wind, self.grid, c.beta, c.drag, c.viscosity)
                return q_rhs, psi, u, v
        u, v = geostrophic_velocity_from_streamfunction(psi, self.diff, self.interp)
        q_rhs = self.adv(q_field, u, v, method="upwind1")
        # V_to_T's ghost ring is zero, so the full-array combination adds
        # -beta v on the interior only, as the reference's ``.at[1:-1, 1:-1]``
        v_center = self.interp.V_to_T(v)
        q_rhs = lincomb(1.0, q_rhs, -c.beta, v_center, 1.0, self.wind_curl)
        zeta = self.diff.laplacian(psi)
        q_rhs = lincomb(1.0, q_rhs, -c.drag, zeta, c.viscosity, self.diff.laplacian(q_field))
        return q_rhs, psi, u, v

    def _plain_operators(self) -> bool:
        """Whether the tendency is that of the unmasked operators on one grid."""
        return (_unmasked(self.diff, Difference2D) and _unmasked(self.interp, Interpolation2D)
                and _unmasked(self.adv, Advection2D)
                and self.diff.grid is self.grid and self.adv.grid is self.grid)

    @staticmethod
    def apply_bc(q_field):
        """Zero ghost ring (``pad_interior``, ``:480-482``)."""
        return pad_interior(q_field, mode="constant")

    def pv_tendency(self, q_field):
        return self.tendency(self.apply_bc(q_field))[0]

    def step(self, q_field):
        """One Heun step and the diagnosed balanced state (``:484-497``)."""
        q_next = self.apply_bc(heun_step(q_field, self.pv_tendency, self.config.dt))
        psi_next = self.invert_streamfunction(q_next)
        u_next, v_next = geostrophic_velocity_from_streamfunction(psi_next, self.diff,
                                                                  self.interp)
        return q_next, psi_next, u_next, v_next

    def run(self, steps: int | None = None, snapshot_interval: int | None = None):
        """Integrate from the initial PV; returns the snapshot times and the
        q, psi, u, v snapshots as host arrays."""
        c = self.config
        steps = c.steps if steps is None else steps
        every = c.snapshot_interval if snapshot_interval is None else snapshot_interval
        q = self.q0.clone()
        out = {"time": [], "q": [], "psi": [], "u": [], "v": []}
        for n in range(1, steps + 1):
            q, psi, u, v = self.step(q)
            if n % every == 0 or n == steps:
                out["time"].append(n * c.dt)
                for k, t in (("q", q), ("psi", psi), ("u", u), ("v", v)):
                    out[k].append(t.cpu().numpy())
        return {k: np.asarray(v) for k, v in out.items()}
