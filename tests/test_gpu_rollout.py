"""Runs of rollout steps (waam_rollout_forward, waam_adj_rollback, waam_cadj_rollback): the forward
bit-equal to the per-kernel entries step by step, and the gradients independent of how the run is
cut into segments, on odd extents, both storage orders, with and without the arc, and with a grid
that holds no liquid. (The gradients against binary64 differences: test_gpu_adjoint*.py.)"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

from tests.gpu_common import bits_equal, mismatch_report
from waam_solver_amd import kernels
from waam_solver_amd.field import tensor_of

THETA = (0.8, 1.2, 0.9)


def _twin(nx, ny, nz, layout, pool=True):
    from tests.step_cases import build_pair, torch_x

    tw, _ = build_pair("bead_mrt", layout=layout, nx=nx, ny=ny, nz=nz)
    g = tw.grid
    if not pool:
        tw.reset()
    T, H, fl = g.T.to_numpy(), g.H.to_numpy(), g.flags.to_numpy()
    plate = fl == 1
    T[plate] = 1700.0
    H[plate] = np.float32(tw.cp_rho) * np.float32(1700.0)
    g.T.from_numpy(T)
    g.H.from_numpy(H)
    if pool:
        for s in range(4):
            tw.step(torch_x(g.dx, g.nx, s, g.dt), (g.ny // 2) * g.dx, True)
    tw.sync()
    return tw, lambda n: (torch_x(g.dx, g.nx, 4 + n, g.dt), (g.ny // 2) * g.dx)


def _chain(tw, ro, flow: bool, welding: bool):
    """The same steps through the per-kernel entries: final (H, T, f_l)."""
    g, m = tw.grid, tw.mat
    eta, s_h, s_sig = THETA
    new = lambda t=None, lead=(): (  # noqa: E731
        lambda f: (tensor_of(f).copy_(t) if t is not None else None, f)[1])(
            g.field(torch.float32, leading=lead))
    dims = (g.nx, g.ny, g.nz)
    flags, phi = ro.flags, ro.phi
    H, H2, T, fl = new(tensor_of(ro.H0)), new(), new(), new()
    u = [new(x) if flow else new() for x in (ro.u0 if flow else (None,) * 3)]
    F, rho = [new() for _ in range(3)], new()
    norm = torch.zeros((), dtype=torch.float32, device=g.device)
    phase = lambda h: kernels.update_phase(h, T, fl, tw.cp_rho, tw.L_rho, m.T_solidus,  # noqa: E731
                                           m.T_liquidus)
    ceil = lambda h: kernels.clamp_enthalpy_ceiling_scalar(  # noqa: E731
        h, flags, tw.cp_rho, m.T_solidus, m.T_liquidus, tw.T_vapor_cap_K, tw.L_rho, g.FLAG_GAS)
    phase(H)
    if flow:
        fa, fb = new(ro.f0, (19,)), new(lead=(19,))
    for n in range(ro.n_steps):
        x, y = ro.path(n)
        ai, aj = x / g.dx, y / g.dx
        if welding:
            kernels.inject_arc_heat(H, flags, phi, fl, norm, ai, aj, ro.arc_k, tw.Q_w,
                                    ro.sigma0 * s_sig, g.dt, g.dx ** 3, eta,
                                    tw.arc_penetration_m / g.dx, int(tw.arc_surface_weighting),
                                    g.FLAG_SOLID, g.FLAG_GAS, scratch=g.scratch)
        ceil(H)
        kernels.advect_diffuse_temperature_into(H, H2, T, *u, flags, tw.alpha_lu, 1.0, tw.cp_rho,
                                                *dims)
        H, H2 = H2, H
        kernels.apply_thermal_boundary_losses(
            H, T, flags, tw.T_amb, ro.h_conv0 * s_h, ro.eps0 * s_h, 1, 1, tw.cp_rho, g.dt, g.dx,
            tw.sigma_sb, g.FLAG_SOLID, g.FLAG_GAS, *dims)
        kernels.clamp_enthalpy_floor_scalar(H, tw.cp_rho, flags, tw.T_amb, g.FLAG_GAS)
        phase(H)
        ceil(H)
        phase(H)
        if not flow:
            continue
        kernels.clear_forces(*F)
        kernels.compute_csf_tension(phi, flags, *F, tw.gamma_lu, g.FLAG_SOLID, g.FLAG_GAS, *dims,
                                    int(tw.enable_wetting), tw.theta_rad)
        kernels.compute_marangoni_force(T, phi, fl, *F, flags, tw.dgamma_dT_lu, g.dx,
                                        g.FLAG_SOLID, g.FLAG_GAS, *dims)
        if welding:
            from waam_solver_amd.physics import weld_forces

            kernels.apply_arc_pressure(F[2], flags, phi, ai, aj, ro.arc_k,
                                       weld_forces.arc_pressure_sigma_cells(tw),
                                       weld_forces.arc_pressure_peak_pa(tw), g.dt, g.dx, m.rho,
                                       g.FLAG_SOLID, g.FLAG_GAS)
        kernels.add_hydrostatic_gravity(F[2], fl, flags, 1.0, tw.g_lu, g.FLAG_SOLID, g.FLAG_GAS)
        kernels.add_buoyancy(T, F[2], fl, flags, tw.g_lu, tw.beta_T, m.T_liquidus, 1.0,
                             g.FLAG_SOLID, g.FLAG_GAS)
        kernels.clamp_body_force_magnitude(*F, flags, ro.F_cap, g.FLAG_SOLID, g.FLAG_GAS)
        kernels.collide_mrt(fa, fb, rho, *u, *F, fl, flags, None, None, None, None, None, tw.omega,
                            tw.omega_bulk, tw.C_darcy, g.FLAG_SOLID, g.FLAG_GAS, *dims)
        kernels.clamp_velocity_mach(*u, flags, ro.u_cap, g.FLAG_SOLID, g.FLAG_GAS)
        fa, fb = fb, fa
    return [tensor_of(t).cpu().numpy() for t in (H, T, fl)]


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,layout,welding,pool", [
    (33, 17, 19, 1, True, True), (64, 24, 20, 0, True, True), (65, 20, 21, 1, False, True),
    (40, 24, 20, 1, True, False)])
@pytest.mark.parametrize("mode", ["thermal", "none", "frozen", "flow"])
def test_runs_match_the_per_kernel_entries(hip_device, mode, nx, ny, nz, layout, welding, pool):
    from waam_solver_amd.adjoint import CoupledRollout, ThermalRollout

    print(f"[rollout] {mode} {nx}x{ny}x{nz} layout {layout} weld {welding} pool {pool}", flush=True)
    tw, path = _twin(nx, ny, nz, layout, pool)
    n = 9
    kw = {} if mode == "thermal" else dict(advection=mode)
    cls = ThermalRollout if mode == "thermal" else CoupledRollout
    g = torch.Generator(device="cuda").manual_seed(3)
    seeds, grads, lam0 = None, [], []
    for K in (1, 4, n, 50):  # segments of one step, a remainder, one segment, one unfilled
        ro = cls(tw, n, path, checkpoint_every=K, is_welding=welding, **kw)
        T, fl = ro.forward(THETA)
        if seeds is None:
            seeds = [torch.randn(T.shape, generator=g, device="cuda") for _ in range(2)]
            if mode in ("thermal", "none", "flow"):
                want = _chain(tw, ro, mode == "flow", welding)
                for name, a, b in zip(("H", "T", "f_l"), (ro.H_final, T, fl), want):
                    a = a.cpu().numpy()
                    assert bits_equal(a, b), mismatch_report(name, a, b)
        grads.append(ro.backward(*seeds))
        lam0.append(ro.lam0.cpu().numpy())
        assert np.isfinite(grads[-1]).all()
        # the segments only change which steps are recomputed; the scattered advection adjoint
        # adds up to a dozen binary64 terms a cell in no fixed order
        np.testing.assert_allclose(grads[-1], grads[0], rtol=1e-11, atol=0.0)
        np.testing.assert_allclose(lam0[-1], lam0[0], rtol=1e-9,
                                   atol=1e-12 * float(np.abs(lam0[0]).max()))


def test_struct_mirrors_have_the_c_layout(tmp_path):
    import shutil
    import subprocess
    from pathlib import Path

    from waam_solver_amd.adjoint import RollbackC, RolloutC

    cc = shutil.which("gcc")
    if cc is None:
        pytest.skip("no C compiler")
    inc = Path(__file__).resolve().parents[1] / "include"
    rows = [(c, py, f) for c, py in (("waam_rollout", RolloutC), ("waam_rollback", RollbackC))
            for f, _ in py._fields_]
    src = "#include <stddef.h>\n#include <stdio.h>\n#include \"waam_hip.h\"\nint main(void){\n"
    src += "".join(f'printf("%zu\\n", offsetof({c}, {f}));\n' for c, _, f in rows)
    src += 'printf("%zu %zu\\n", sizeof(waam_rollout), sizeof(waam_rollback));return 0;}\n'
    (tmp_path / "t.c").write_text(src)
    subprocess.run([cc, f"-I{inc}", str(tmp_path / "t.c"), "-o", str(tmp_path / "t")], check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True).stdout.split()
    assert [int(v) for v in out[:len(rows)]] == [getattr(py, f).offset for _, py, f in rows]
    assert [int(v) for v in out[len(rows):]] == [ctypes.sizeof(RolloutC), ctypes.sizeof(RollbackC)]


def test_rollout_calls_reject_bad_arguments():
    from waam_solver_amd._lib import WaamError, lib
    from waam_solver_amd.adjoint import RolloutC

    arcs = (ctypes.c_double * 2)()
    r = RolloutC(nx=4, ny=4, nz=4, layout=1)
    a = ctypes.addressof
    for change, match in (({}, "NULL|null"), (dict(nx=0), "waam_rollout_forward"),
                          (dict(slot0=2), "slot"), (dict(flow=3), "flow"),
                          (dict(nx=2000, ny=2000, nz=2000), "2\\^31")):
        q = RolloutC.from_buffer_copy(r)
        for k, v in change.items():
            setattr(q, k, v)
        with pytest.raises(WaamError, match=match):
            lib().call("waam_rollout_forward", a(q), a(arcs), a(arcs), 2, None)
    with pytest.raises(WaamError, match="steps"):
        lib().call("waam_rollout_forward", a(r), a(arcs), a(arcs), 0, None)
    with pytest.raises(WaamError, match="NULL"):
        lib().call("waam_rollout_forward", None, a(arcs), a(arcs), 1, None)


@pytest.mark.gpu
@pytest.mark.parametrize("eta", [math.nan, math.inf])
@pytest.mark.parametrize("mode", ["thermal", "flow"])
def test_a_bad_efficiency_is_not_swallowed(hip_device, mode, eta, monkeypatch):
    """An efficiency that is no number reaches every cell that the arc heats, as it does through
    the per-kernel entries."""
    from waam_solver_amd.adjoint import CoupledRollout, ThermalRollout

    tw, path = _twin(33, 17, 19, 1)
    ro = ThermalRollout(tw, 2, path) if mode == "thermal" else CoupledRollout(tw, 2, path)
    theta = (eta, 1.0, 1.0)
    monkeypatch.setitem(globals(), "THETA", theta)
    T, fl = ro.forward(theta)
    want = _chain(tw, ro, mode == "flow", True)
    assert np.isnan(want[0]).any() == math.isnan(eta)  # the ceiling bounds an infinite one
    for name, a, b in zip(("H", "T", "f_l"), (ro.H_final, T, fl), want):
        assert bits_equal(a.cpu().numpy(), b), mismatch_report(name, a.cpu().numpy(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("mode,fields", [("thermal", 5), ("none", 5), ("frozen", 6), ("flow", 35)])
def test_backward_memory(hip_device, mode, fields):
    """The backward holds so many fields for each step between two checkpoints, and a few more
    besides: two of each state and adjoint in turn, and work buffers in binary64."""
    from waam_solver_amd.adjoint import CoupledRollout, ThermalRollout

    tw, path = _twin(64, 40, 32, 1)
    n, field = 40, 4 * tw.grid.n_cells
    ro = (ThermalRollout(tw, n, path, checkpoint_every=n) if mode == "thermal" else
          CoupledRollout(tw, n, path, checkpoint_every=n, advection=mode))
    T, _ = ro.forward(THETA)
    seed = torch.ones_like(T)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    ro.backward(seed, seed)
    held = (torch.cuda.max_memory_allocated() - base - n * 6 * 1024 * 8) / field
    print(f"[rollout] {mode}: {held:.1f} fields over {n} steps", flush=True)
    # H and f_l at the last step, two of T; binary64 counts twice: the two seeds and dL/dH, dL/du
    # (three each), dL/df (nineteen), lamC, lamB, and the flow's T1, fl1 and G. The allocator may
    # hand out blocks up to 1 MiB (three fields) larger than asked: eight fields for those
    few = 8 + {"thermal": 6, "none": 16, "frozen": 28, "flow": 140}[mode]
    assert held < fields * n + few
