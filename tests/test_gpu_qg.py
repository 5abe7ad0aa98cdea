"""GPU parity of the fused QG step against the oracle's composition.

Stage kernel: FP64 to 1e-12 relative (max-norm), FP32 tendency to 2e-5.  Full
steps: FP64 with tight solves matches the oracle (direct sparse Helmholtz
solves) to 1e-9; every solve is certified by its FP64 residual.  The
mixed-precision step (FP64 state, FP32 tendency and inner solves, FP64
refinement) stays within 1e-6 relative PV of the FP64 step over the 100 steps
of the 1024^2 basin configuration.
"""

import numpy as np
import pytest
import torch

import finitevolx_amd as fx
from finitevolx_amd import inputs
from finitevolx_amd.qg import QGModel
from oracle import fvx
from tests.gpu_util import assert_close_scaled, need_gpu, to_np

pytestmark = pytest.mark.gpu


def _params(nx, ny, L=5.12e6):
    return fvx.QGParams(nx, ny, L, L * ny / nx)


def _basin_mask(ny, nx, seed=3):
    return inputs.basin_mask(ny, nx, seed)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [(40, 72), (97, 64)])
def test_stage_kernel_matches_oracle(masked, shape):
    need_gpu()
    ny, nx = shape
    p = _params(nx, ny)
    wet = _basin_mask(ny, nx) if masked else np.ones((ny, nx), bool)
    rng = np.random.default_rng(0)
    qs = np.zeros((ny + 2, nx + 2))
    qs[1:-1, 1:-1] = rng.standard_normal((ny, nx)) * 1e-5 * wet
    qn = np.zeros_like(qs)
    qn[1:-1, 1:-1] = rng.standard_normal((ny, nx)) * 1e-5 * wet
    psi = np.zeros_like(qs)
    psi[1:-1, 1:-1] = rng.standard_normal((ny, nx)) * 1e4 * wet
    F = p.forcing()
    rhs = fvx.qg_rhs(qs, psi, p, F, wet)
    for prec, tol in (("float64", 1e-12), ("mixed", 2e-5), ("mixed32", 2e-5)):
        m = QGModel(nx, ny, p.Lx, p.Ly, mask=wet if masked else None, precision=prec)
        for (a, b, c) in ((0.0, 1.0, 1.0), (0.75, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3)):
            ref = a * qn + b * qs + c * p.dt * rhs
            got = m.stage(qs, psi, qn, a, b, c)
            assert_close_scaled(to_np(got), ref, tol, f"stage {prec} {(a, b, c)}")
        # the tendency alone (a=0, b=0, c=1/dt) isolates the rhs from the combination
        got = m.stage(qs, psi, qn, 0.0, 0.0, 1.0 / p.dt)
        assert_close_scaled(to_np(got), rhs, 10 * tol, f"rhs {prec}")


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("suffix", ["f64", "f64t32"])
def test_stage_with_certification_residual(masked, suffix):
    """The stage kernel's fused certification residual: block partials of
    ||q_s||^2 and ||q_s - (lap - lambda) psi||^2 (masked Dirichlet operator of
    the solve) sum to the oracle's norms; the stage output is unchanged."""
    import ctypes as C

    from finitevolx_amd import _lib

    need_gpu()
    ny, nx = 97, 130
    p = _params(nx, ny)
    wet = _basin_mask(ny, nx) if masked else np.ones((ny, nx), bool)
    rng = np.random.default_rng(4)
    qs = np.zeros((ny + 2, nx + 2))
    qs[1:-1, 1:-1] = rng.standard_normal((ny, nx)) * 1e-5 * wet
    psi = np.zeros_like(qs)
    psi[1:-1, 1:-1] = rng.standard_normal((ny, nx)) * 1e4 * wet
    b = qs[1:-1, 1:-1] * wet
    A, _ = fvx.dirichlet_helmholtz_matrix(wet, p.dx, p.dy, p.lambda_)
    m = wet > 0
    r = b[m] - A @ psi[1:-1, 1:-1][m]
    full = np.zeros((ny + 2, nx + 2), np.uint8)
    full[1:-1, 1:-1] = wet
    dev = torch.device("cuda")
    t_qs, t_psi = torch.tensor(qs, device=dev), torch.tensor(psi, device=dev)
    out = torch.zeros_like(t_qs)
    mask = torch.tensor(full, device=dev) if masked else None
    parts = torch.zeros(4096, dtype=torch.float64, device=dev)
    nblk = C.c_int(0)
    _lib.extra_signatures({f"fvx_qg_stage_cert_{suffix}": [_lib._vp] * 5 + [_lib._i, _lib._i]
                           + [_lib._d] * 10 + [_lib._vp, C.c_int64, C.POINTER(C.c_int), _lib._vp]})
    _lib.call(f"fvx_qg_stage_cert_{suffix}", t_qs.data_ptr(), t_psi.data_ptr(), t_qs.data_ptr(),
              out.data_ptr(), _lib.ptr(mask), ny + 2, nx + 2, p.dx, p.dy, p.beta, p.Ly, p.F0,
              p.nu4, 0.75, 0.25, 0.25 * p.dt, p.lambda_, parts.data_ptr(), parts.numel(),
              C.byref(nblk), _lib.stream())
    pv = parts.cpu().numpy()
    n = nblk.value
    assert 0 < n <= 2048
    np.testing.assert_allclose(pv[:n].sum(), (b * b).sum(), rtol=1e-12)
    np.testing.assert_allclose(pv[n:2 * n].sum(), (r * r).sum(), rtol=1e-10)
    ref = 0.75 * qs + 0.25 * qs + 0.25 * p.dt * fvx.qg_rhs(qs, psi, p, p.forcing(), wet)
    assert_close_scaled(to_np(out), ref, 1e-12 if suffix == "f64" else 2e-5, "stage output")


@pytest.mark.parametrize("masked", [False, True])
def test_fp64_steps_match_oracle(masked):
    need_gpu()
    ny, nx = 64, 96
    p = _params(nx, ny)
    wet = _basin_mask(ny, nx, 5) if masked else np.ones((ny, nx), bool)
    q0 = np.zeros((ny + 2, nx + 2))
    q0[1:-1, 1:-1] = inputs.qg_initial_pv(ny, nx, seed=2) * wet
    F = p.forcing()
    ref = q0.copy()
    for _ in range(3):
        ref = fvx.qg_step(ref, p, F, wet)
    m = QGModel(nx, ny, p.Lx, p.Ly, mask=wet if masked else None, precision="float64",
                rtol=1e-13)
    q = m.new_state(q0[1:-1, 1:-1])
    q, psi, info = m.step(q, nsteps=3)
    assert info["converged"] and info["solves"] == 9
    assert info["max_rel_residual"] <= 1e-13
    assert_close_scaled(to_np(q), ref, 1e-9, "3 QG steps fp64")
    # psi is the solve of the last stage state; check its residual in the oracle
    qi = to_np(q)  # final state differs from the last stage, so check the operator instead
    assert np.all(to_np(psi)[0, :] == 0) and np.all(to_np(psi)[:, -1] == 0)


@pytest.mark.parametrize("precision", ["mixed", "mixed32", "mixed64"])
def test_mixed_paths_track_fp64(precision):
    need_gpu()
    ny, nx = 128, 128
    p = _params(nx, ny)
    q0 = inputs.qg_initial_pv(ny, nx, seed=2)
    m64 = QGModel(nx, ny, p.Lx, p.Ly, precision="float64")
    mm = QGModel(nx, ny, p.Lx, p.Ly, precision=precision)
    q64, _, i64 = m64.step(m64.new_state(q0), nsteps=10)
    qm, _, im = mm.step(mm.new_state(q0), nsteps=10)
    assert i64["converged"] and im["converged"]
    assert im["max_rel_residual"] <= 1e-8 and i64["max_rel_residual"] <= 1e-8
    err = np.max(np.abs(to_np(qm) - to_np(q64))) / np.max(np.abs(to_np(q64)))
    assert err <= 1e-6, err


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("precision", ["float64", "mixed", "mixed32"])
def test_graph_replay_matches_host_driven_steps(precision, masked):
    """Steps 4-6 of the graph call are replays of the captured step graphs
    (the first three run eagerly to calibrate the budgets)."""
    need_gpu()
    ny, nx = 256, 192
    p = _params(nx, ny)
    wet = _basin_mask(ny, nx, 7) if masked else None
    q0 = inputs.qg_initial_pv(ny, nx, seed=4)
    tol = 1e-12 if precision == "float64" else 1e-9
    m1 = QGModel(nx, ny, p.Lx, p.Ly, precision=precision, rtol=tol, mask=wet)
    m2 = QGModel(nx, ny, p.Lx, p.Ly, precision=precision, rtol=tol, mask=wet)
    qa, _, ia = m1.step(m1.new_state(q0), nsteps=6, graph=False)
    qb, _, ib = m2.step(m2.new_state(q0), nsteps=6, graph=True)
    assert ia["converged"] and ib["converged"] and ib["solves"] == 18
    assert ib["max_rel_residual"] <= tol
    err = np.max(np.abs(to_np(qa) - to_np(qb))) / np.max(np.abs(to_np(qa)))
    assert err <= (1e-10 if precision == "float64" else 1e-6), err
    # a second call reuses the captured graphs
    qc, _, ic = m2.step(qb, nsteps=2, graph=True)
    assert ic["converged"] and ic["solves"] == 6


@pytest.mark.parametrize("precision", ["float64", "mixed"])
def test_graph_retry_after_a_jump_in_q(precision):
    """A jump in q between calls leaves the extrapolated warm starts poor,
    so the first replayed steps miss their budgets: each is redone from its
    untouched input with wider budgets (recaptured graphs), and the run
    matches host-driven steps from the same state."""
    need_gpu()
    ny, nx = 256, 192
    p = _params(nx, ny)
    q0 = inputs.qg_initial_pv(ny, nx, seed=4)
    tol = 1e-12 if precision == "float64" else 1e-9
    m1 = QGModel(nx, ny, p.Lx, p.Ly, precision=precision, rtol=tol)
    m2 = QGModel(nx, ny, p.Lx, p.Ly, precision=precision, rtol=tol)
    qa, pa, _ = m1.step(m1.new_state(q0), nsteps=8, graph=False)
    qb, pb, ib = m2.step(m2.new_state(q0), nsteps=8, graph=True)
    assert ib["converged"]
    jump = m1.new_state(inputs.qg_initial_pv(ny, nx, seed=9))
    qa += jump
    qb += jump
    qa, _, ia = m1.step(qa, pa, nsteps=5, graph=False)
    qb, _, ib = m2.step(qb, pb, nsteps=5, graph=True)
    print(f"[retry] {precision}: {ib}", flush=True)
    assert ib["retries"] >= 1, ib
    assert ia["converged"] and ib["converged"] and ib["solves"] == 15, ib
    assert ib["max_rel_residual"] <= tol
    err = np.max(np.abs(to_np(qa) - to_np(qb))) / np.max(np.abs(to_np(qa)))
    assert err <= (1e-10 if precision == "float64" else 1e-6), err


@pytest.mark.parametrize("masked", [False, True])
def test_chebyshev_smoothing_tracks_fp64(masked):
    """Mixed-precision steps whose inner V-cycles take Chebyshev weights
    (host-driven and replayed graphs) certify every solve and track the FP64
    steps; so do FP64 steps with the weights (off by default there)."""
    need_gpu()
    ny, nx = 256, 192
    p = _params(nx, ny)
    wet = _basin_mask(ny, nx, 7) if masked else None
    q0 = inputs.qg_initial_pv(ny, nx, seed=4)
    m64 = QGModel(nx, ny, p.Lx, p.Ly, precision="float64", mask=wet)
    q64, _, _ = m64.step(m64.new_state(q0), nsteps=6, graph=False)
    c64 = QGModel(nx, ny, p.Lx, p.Ly, precision="float64", mask=wet)
    assert c64.set_chebyshev(0.25)
    qc, _, ic = c64.step(c64.new_state(q0), nsteps=6, graph=True)
    assert ic["converged"] and ic["max_rel_residual"] <= 1e-8, ic
    assert np.max(np.abs(to_np(qc) - to_np(q64))) <= 1e-6 * np.max(np.abs(to_np(q64)))
    for graph in (False, True):
        mm = QGModel(nx, ny, p.Lx, p.Ly, precision="mixed", mask=wet)
        assert mm.set_chebyshev(0.1)
        qm, _, im = mm.step(mm.new_state(q0), nsteps=6, graph=graph)
        print(f"[chebyshev] masked={masked} graph={graph}: {im}", flush=True)
        assert im["converged"] and im["solves"] == 18 and im["max_rel_residual"] <= 1e-8, im
        err = np.max(np.abs(to_np(qm) - to_np(q64))) / np.max(np.abs(to_np(q64)))
        assert err <= 1e-6, err


def test_config2_basin_mixed_within_pv_gate():
    """The 1024^2 closed-basin configuration: f0 = 9.375e-5, beta = 1.754e-11,
    Ld = 4e4 m, nu4 = 1e9, dt = 1200 s, k^-3 PV (rms 1e-5, seed 2) with the
    double-gyre forcing, V(2,2) multigrid-PCG to 1e-8; 100 rk3_ssp_step steps
    all-FP64 against FP32 bulk with FP64 refinement.  Every solve is certified
    by its FP64 residual and the mixed PV stays within 1e-6 (max-norm
    relative) of the FP64 PV."""
    need_gpu()
    n, L, steps = 1024, 5.12e6, 100
    q0 = inputs.qg_initial_pv(n, n, rms=1e-5, seed=2)
    out = {}
    for prec in ("float64", "mixed"):
        m = QGModel(n, n, L, L, precision=prec, n_pre=2, n_post=2, dt=1200.0, rtol=1e-8)
        q, psi, info = m.step(m.new_state(q0), nsteps=steps)
        assert info["converged"] and info["solves"] == 3 * steps, (prec, info)
        assert info["max_rel_residual"] <= 1e-8, (prec, info)
        out[prec] = to_np(q)
        del m
    ref = out["float64"]
    err = np.max(np.abs(out["mixed"] - ref)) / np.max(np.abs(ref))
    l2 = np.linalg.norm(out["mixed"] - ref) / np.linalg.norm(ref)
    print(f"config-2 PV error after {steps} steps: max {err:.3e}, L2 {l2:.3e}")
    assert err <= 1e-6 and l2 <= 1e-6, (err, l2)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("ny,nx", [(3, 5), (4, 3), (17, 63), (62, 66), (24, 1511)])
def test_gyre_tendency_in_one_pass(ny, nx, dtype):
    """The one-kernel tendency and the field-to-field inversion against the
    oracle's step and against the operators one by one (whose grid is not the
    model's own object), with a ghost ring that holds anything.  24 x 1511 FP32
    inverts by FFT.  FP32: a velocity is a difference of psi, so 4 roundings are
    amplified up to n."""
    need_gpu()
    from finitevolx_amd.qg_1p5_layer import QG1p5LayerModel, QuasiGeostrophicConfig

    Ly = 5.12e6 * ny / nx
    model = QG1p5LayerModel(QuasiGeostrophicConfig(nx=nx, ny=ny, Ly=Ly), dtype)
    p = fvx.QGScriptParams(nx=nx, ny=ny, Ly=Ly)
    q_ref, wind = p.fields()
    rng = np.random.default_rng(nx)
    q_ref = q_ref + 1e-9 * rng.standard_normal(q_ref.shape)
    q = torch.tensor(q_ref, dtype=dtype, device="cuda")
    tol = 1e-11 if dtype == torch.float64 else max(1e-5, 4 * 6e-8 * max(ny, nx))
    for got, ref, name in zip(model.step(q), fvx.qg_script_step(q_ref, p, wind), ("q", "psi", "u", "v")):
        assert_close_scaled(to_np(got), ref, tol, f"{name} {ny}x{nx}")
    parts = QG1p5LayerModel(model.config, dtype)
    g = fx.CartesianGrid2D.from_interior(nx, ny, 5.12e6, Ly)
    parts.diff, parts.interp = fx.Difference2D(g), fx.Interpolation2D(g)
    assert model._plain_operators() and not parts._plain_operators()
    for got, ref, name in zip(model.tendency(q), parts.tendency(q), ("rhs", "psi", "u", "v")):
        assert got.shape == ref.shape and got.dtype == ref.dtype
        assert_close_scaled(to_np(got), to_np(ref), tol, f"{name} {ny}x{nx}")
    psi = to_np(model.invert_streamfunction(q))
    assert not psi[0].any() and not psi[-1].any() and not psi[:, 0].any() and not psi[:, -1].any()


@pytest.mark.parametrize("on_class", [False, True])
def test_replaced_operator_methods_are_used(on_class, monkeypatch):
    """A method replaced on one of the model's operators, or on its class, takes
    part in the tendency and in the velocities."""
    need_gpu()
    from finitevolx_amd import qg_1p5_layer as Q

    model = Q.QG1p5LayerModel(Q.QuasiGeostrophicConfig(nx=20, ny=16))
    psi = model.invert_streamfunction(model.q0)
    plain = model.tendency(model.q0)
    for name, op in (("laplacian", model.diff), ("diff_y_X_to_U", model.diff),
                     ("T_to_X", model.interp), ("V_to_T", model.interp)):
        own = getattr(op, name)
        calls = []
        if on_class:
            monkeypatch.setattr(type(op), name,
                                lambda self, f, own=own: calls.append(name) or 2.0 * own(f))
        else:
            setattr(op, name, lambda f, own=own: calls.append(name) or 2.0 * own(f))
        changed = model.tendency(model.q0)
        assert calls and not torch.equal(changed[0], plain[0]), name
        calls.clear()
        vel = Q.geostrophic_velocity_from_streamfunction(psi, model.diff, model.interp)
        assert bool(calls) == (name in ("diff_y_X_to_U", "T_to_X")), name
        if calls:
            assert_close_scaled(to_np(vel[0]), 2.0 * to_np(plain[2]), 1e-12, name)
        if on_class:
            monkeypatch.undo()
        else:
            delattr(op, name)
    for got, ref in zip(model.tendency(model.q0), plain):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("nx,ny", [(64, 64), (48, 80)])
def test_qg_1p5_layer_script_steps_match_oracle(nx, ny):
    """The reference example's composition (upwind1, X-point velocities, DST
    inversion, heun_step; scripts/qg_1p5_layer.py:420-497): 4 steps in FP64
    against the oracle's composition with exact Helmholtz solves."""
    need_gpu()
    from finitevolx_amd.qg_1p5_layer import QG1p5LayerModel, QuasiGeostrophicConfig

    cfg = QuasiGeostrophicConfig(nx=nx, ny=ny, Ly=5.12e6 * ny / nx)
    model = QG1p5LayerModel(cfg)
    p = fvx.QGScriptParams(nx=nx, ny=ny, Ly=5.12e6 * ny / nx)
    q_ref, wind = p.fields()
    assert_close_scaled(to_np(model.q0), q_ref, 1e-15, "q0")
    assert_close_scaled(to_np(model.wind_curl), wind, 1e-15, "wind curl")
    q = model.q0.clone()
    for n in range(4):
        q, psi, u, v = model.step(q)
        q_ref, psi_r, u_r, v_r = fvx.qg_script_step(q_ref, p, wind)
        for got, ref, name in ((q, q_ref, "q"), (psi, psi_r, "psi"), (u, u_r, "u"), (v, v_r, "v")):
            assert_close_scaled(to_np(got), ref, 1e-11, f"step {n} {name}")
    out = model.run(steps=6, snapshot_interval=3)
    assert out["q"].shape == (2, ny + 2, nx + 2) and list(out["time"]) == [3 * cfg.dt, 6 * cfg.dt]
