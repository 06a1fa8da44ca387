"""The rollouts' run entries against the step-by-step adjoint entries that they run as one
(waam_adj_arc_sums, waam_adj_thermal_step, waam_cadj_*): a whole rollback of nine steps, with
adjoints of the populations and velocity to start from, so that every term of the flow's adjoint
counts."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

from tests import test_gpu_rollout as rollout_tests
from tests.gpu_common import bits_equal, mismatch_report
from waam_solver_amd._lib import lib
from waam_solver_amd.field import P, tensor_of

pytestmark = pytest.mark.gpu

N_STEPS = 9
D64 = dict(dtype=torch.float64, device="cuda")


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _saved(ro, adv: bool, flow: bool) -> dict:
    """The state and saved fields of all the steps, as the backward lays them out."""
    n = ro.n_steps
    sv = {k: ro._new(2 if k == "T" and not flow else n + 1) for k in ("H", "T", "fl")}
    sv.update({k: ro._new(n) for k in (("A", "B", "E", "F") if adv else ("A", "E", "F"))})
    if flow:
        sv.update(u=ro._new(n + 1, 3), f=ro._new(n + 1, 19), Fr=ro._new(n, 3), Fc=ro._new(n, 3))
    elif adv:
        sv["u"] = ro._slots["u"]
    sv["sums"] = torch.zeros(2 * n, **D64)
    return sv


@pytest.mark.parametrize("nx,ny,nz,layout,welding", [
    (33, 17, 19, 1, True), (64, 24, 20, 0, True), (65, 20, 21, 1, False)])
def test_thermal_rollback_equals_its_entries(hip_device, nx, ny, nz, layout, welding):
    from waam_solver_amd.adjoint import ThermalRollout

    print(f"[rollback] thermal {nx}x{ny}x{nz} layout {layout} weld {welding}", flush=True)
    tw, path = rollout_tests._twin(nx, ny, nz, layout)
    g, n = tw.grid, N_STEPS
    ro = ThermalRollout(tw, n, path, checkpoint_every=n, is_welding=welding)
    ro.forward(rollout_tests.THETA)
    sv = _saved(ro, False, False)
    sv["H"][0].copy_(ro.ckpt[0])
    lib().call("waam_update_phase", P(sv["H"]), P(sv["T"]), P(sv["fl"]), tw.cp_rho, tw.L_rho,
               tw.mat.T_solidus, tw.mat.T_liquidus, g.n_cells, _stream())
    ro._run(0, n, sv, stack=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    seed = torch.randn(ro.shape, generator=gen, device="cuda")
    seed[tensor_of(ro.flags) == g.FLAG_GAS] = 0.0

    lam, grads = ro._new(2), torch.zeros(3, **D64)
    lam[0].copy_(seed)
    parts, totals = torch.empty(n * 6 * 1024, **D64), torch.empty(3 * n, **D64)
    r, (ai, aj) = ro._rollout(sv, True, 0), ro._arcs(0, n)
    lib().call("waam_adj_rollback", ctypes.addressof(r), ctypes.addressof(ai),
               ctypes.addressof(aj), n, P(lam), 0, P(parts), P(totals), P(grads), _stream())
    got, got_grads = lam[n & 1].cpu().numpy(), grads.cpu().numpy()

    a, b, lamC = seed.clone(), ro._new(), ro._new()
    grads, sums = torch.zeros(3, **D64), torch.zeros(2, **D64)
    for t in reversed(range(n)):
        c = ro._consts(t)
        if welding:
            lib().call("waam_adj_arc_sums", P(ro.flags), P(sv["fl"][t]), ctypes.addressof(c),
                       P(sums), nx, ny, nz, layout, P(g.scratch), _stream())
        lib().call("waam_adj_thermal_step", P(a), P(b), P(sv["H"][t]), P(sv["A"][t]),
                   P(sv["E"][t]), P(sv["F"][t]), P(sv["fl"][t]), P(ro.flags), P(sums),
                   ctypes.addressof(c), P(grads), P(lamC), nx, ny, nz, layout, P(g.scratch),
                   _stream())
        a, b = b, a
    # the same fp32 expressions; the arc's sums are binary64 totals that enter them rounded
    assert bits_equal(got, a.cpu().numpy()), mismatch_report("lam", got, a.cpu().numpy())
    np.testing.assert_allclose(got_grads, grads.cpu().numpy(), rtol=1e-12, atol=0.0)
    assert np.abs(got).max() > 0.0 and np.isfinite(got).all()


@pytest.mark.parametrize("nx,ny,nz,layout,welding", [
    (33, 17, 19, 1, True), (64, 24, 20, 0, True), (65, 20, 21, 1, False)])
@pytest.mark.parametrize("mode", ["none", "frozen", "flow"])
def test_coupled_rollback_equals_its_entries(hip_device, mode, nx, ny, nz, layout, welding):
    """Binary64 throughout, the coefficients of the flow's adjoint included, as the entries take
    them: what may differ is the order in which the advection adjoint's scattered terms add up."""
    from waam_solver_amd.adjoint import CoupledRollout

    print(f"[rollback] {mode} {nx}x{ny}x{nz} layout {layout} weld {welding}", flush=True)
    tw, path = rollout_tests._twin(nx, ny, nz, layout)
    g, n = tw.grid, N_STEPS
    ro = CoupledRollout(tw, n, path, checkpoint_every=n, is_welding=welding, advection=mode)
    ro.forward(rollout_tests.THETA)
    flow, adv = mode == "flow", mode != "none"
    sv = _saved(ro, adv, flow)
    ro._put(sv, *ro.ckpt[0])
    ro._run(0, n, sv, stack=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    N, shp = g.n_cells, ro.shape

    def start(*lead):
        """Random adjoints on the FLUID/IFACE cells (the rest of a grid has none to start with)."""
        t = torch.zeros(lead + shp, **D64)
        t.reshape(-1, N)[:, ro._cells] = torch.randn(
            (math.prod(lead), ro._cells.numel()), generator=gen, **D64)
        return t

    seed_H = torch.randn(shp, generator=gen, **D64)
    seed_H[tensor_of(ro.flags) == g.FLAG_GAS] = 0.0
    seed_u, seed_f = start(3), start(19)

    z = lambda *lead: torch.zeros(lead + shp, **D64)  # noqa: E731
    lam = {"lam_H": z(2), "lamC": z(), "lamB": z(), "parts": torch.empty(n * 6 * 1024, **D64),
           "step_totals": torch.empty(3 * n, **D64), "grads": torch.zeros(3, **D64)}
    lam["lam_H"][0].copy_(seed_H)
    if adv:
        lam["lam_u"] = z(2, 3)
        lam["lam_u"][0].copy_(seed_u)
    if flow:
        lam.update(lam_f=z(2, 19), lam_T1=z(), lam_fl1=z(), G=z(3))
        lam["lam_f"][0].copy_(seed_f)
    r, (ai, aj) = ro._rollout(sv, True, 0), ro._arcs(0, n)
    b = ro._rollback(lam, 0)
    lib().call("waam_cadj_rollback", ctypes.addressof(r), ctypes.addressof(b),
               ctypes.addressof(ai), ctypes.addressof(aj), n, _stream())
    names = ("lam_H",) + (("lam_u",) if adv else ()) + (("lam_f",) if flow else ())
    got = {k: lam[k][n & 1].cpu().numpy() for k in names}
    got["grads"] = lam["grads"].cpu().numpy()

    lam_H, lam_Ho, lam_u, lam_uo = seed_H.clone(), z(), seed_u.clone(), z(3)
    lam_f, lam_fin, lam_F, lam_Fr, G = seed_f.clone(), z(19), z(3), z(3), z(3)
    lamC, lamB, lam_T1, lam_fl1 = z(), z(), z(), z()
    grads, sums = torch.zeros(3, **D64), torch.zeros(2, **D64)
    for t in reversed(range(n)):
        c = ro._consts(t)
        fl1, H1 = sv["fl"][t + 1], sv["H"][t + 1]
        if flow:
            T1 = sv["T"][t + 1]
            lam_fl1.zero_()
            lam_T1.zero_()
            Fc, Fr = sv["Fc"][t], sv["Fr"][t]
            lib().call("waam_cadj_collide_mrt", P(sv["f"][t]), P(Fc[0]), P(Fc[1]), P(Fc[2]),
                       P(fl1), P(ro.flags), P(lam_f), P(lam_u), tw.omega, tw.omega_bulk,
                       tw.C_darcy, ro.u_cap, P(lam_fin), P(lam_F), P(lam_fl1), N, _stream())
            lib().call("waam_cadj_forces", P(Fr[0]), P(Fr[1]), P(Fr[2]), P(T1), P(fl1),
                       P(ro.flags), P(lam_F), ro.F_cap, tw.g_lu, tw.beta_T, tw.mat.T_liquidus,
                       int(bool(tw.enable_hydrostatic_gravity)), P(lam_Fr), P(lam_T1),
                       P(lam_fl1), N, _stream())
            lib().call("waam_cadj_marangoni", P(ro.phi), P(fl1), P(ro.flags), P(lam_Fr),
                       tw.dgamma_dT_lu, P(G), P(lam_T1), nx, ny, nz, layout, _stream())
            lib().call("waam_cadj_phase", P(H1), P(ro.flags), ctypes.addressof(c), P(lam_T1),
                       P(lam_fl1), P(lam_H), N, _stream())
            u = sv["u"][t]
        else:
            u = ro._slots["u"] if adv else torch.zeros((3,) + shp, device="cuda")
        if welding:
            lib().call("waam_adj_arc_sums", P(ro.flags), P(sv["fl"][t]), ctypes.addressof(c),
                       P(sums), nx, ny, nz, layout, P(g.scratch), _stream())
        # without advection the rollout saves no B: it is read where u is not 0 only
        B = sv["B"][t] if adv else sv["A"][t]
        lib().call("waam_cadj_thermal_step", P(lam_H), P(lam_Ho), P(lam_uo), P(sv["H"][t]),
                   P(sv["A"][t]), P(B), P(sv["E"][t]), P(sv["F"][t]), P(sv["fl"][t]), P(u[0]),
                   P(u[1]), P(u[2]), P(ro.flags), P(sums), ctypes.addressof(c), P(grads),
                   P(lamC), P(lamB), nx, ny, nz, layout, P(g.scratch), _stream())
        lam_H, lam_Ho, lam_u, lam_uo = lam_Ho, lam_H, lam_uo, lam_u
        lam_f, lam_fin = lam_fin, lam_f
    want = {"lam_H": lam_H, "lam_u": lam_u, "lam_f": lam_f, "grads": grads}
    for k, v in got.items():
        w = want[k].cpu().numpy()
        # a dozen binary64 terms in any order a step (12 * 2^-53 of the largest), nine steps,
        # and their amplification on the way; a coefficient rounded to fp32 is 1e-8 off
        np.testing.assert_allclose(v, w, rtol=0.0, atol=1e-12 * float(np.abs(w).max()), err_msg=k)
        assert np.abs(v).max() > 0.0
