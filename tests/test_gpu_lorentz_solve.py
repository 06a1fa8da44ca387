"""The Lorentz solve as one call against its single entries in solve order (which the oracle
covers): same arithmetic in the same order, so every field is the same bit for bit. Sizes around
the 8-cell tiles of the sweeps and the 1024-cell pieces of the force, sweep limits that end in
chunks of ten, of one (the potential changes its buffer) and of odd length, and tests that
converge in the first chunk, in a later one, or never."""

import numpy as np
import pytest
import torch

from waam_solver_amd import kernels as K
from waam_solver_amd.grid import WAAMGrid
from waam_solver_amd.materials import load_material

pytestmark = pytest.mark.gpu

MU0 = 4e-7 * np.pi
SCALARS = dict(sigma_cells=2.5, current_A=140.0, sigma_liquid=7e5, sigma_solid=9e5, omega_j=0.85,
               nz_solid=3, mu0=MU0, rho_ref=7800.0)


def _grid(dims, layout, seed):
    g = WAAMGrid(*dims, 2e-4, load_material("ER70S-6"), max_tracers=16, allocate_lorentz=True, layout=layout)
    rng = np.random.default_rng(seed)
    nz = dims[2]
    k = np.arange(nz)[None, None, :] * np.ones(dims)
    flags = np.where(k < nz // 2, 1, 2)
    flags = np.where(rng.random(dims) < 0.1, rng.choice([0, 1, 2, 4], dims), flags)
    g.flags.from_numpy(flags.astype(np.uint8))
    g.f_l.from_numpy(np.where(flags != 2, rng.random(dims), 0.0).astype(np.float32))
    g.phi_elec.from_numpy((rng.standard_normal(dims) * 1e-3).astype(np.float32))
    for n in ("Fx", "Fy", "Fz"):
        getattr(g, n).from_numpy(rng.standard_normal(dims).astype(np.float32))
    return g


def _by_entries(g, arc, dr, max_sweeps, tol, cold):
    s, n = SCALARS, (g.nx, g.ny, g.nz)
    K.elec_build_sigma(g.sigma_elec, g.f_l, g.flags, s["sigma_liquid"], s["sigma_solid"], 2)
    K.elec_clear_source(g.elec_source)
    K.elec_inject_arc_source(g.elec_source, *arc, s["sigma_cells"], s["current_A"], g.dx, g.nz)
    K.elec_normalize_source(g.elec_source, s["current_A"], g.dx, scratch=g.scratch)
    if cold:
        K.elec_init_ground(g.phi_elec, g.flags, s["nz_solid"], 1)
    done, conv = 0, False
    while done < max_sweeps and not conv:
        for it in range(min(10, max_sweeps - done)):
            K.elec_jacobi_step(g.phi_elec, g.phi_elec_tmp, g.sigma_elec, g.elec_source, g.flags,
                               g.dx, s["omega_j"], 2, 1, s["nz_solid"], *n)
            last = (g.phi_elec_tmp, g.phi_elec)
            g.phi_elec, g.phi_elec_tmp = last
        K.elec_l1_diff_into(*last, g.elec_l1_buf, g.scratch)
        done += it + 1
        res, norm = (float(v) for v in g.elec_l1_buf.to_numpy())
        conv = res / max(norm, 1e-30) < tol
    K.elec_compute_J(g.Jx, g.Jy, g.Jz, g.phi_elec, g.sigma_elec, g.flags, g.dx, 2, *n)
    K.elec_bin_axial_current(g.Jz, g.elec_rad_bins, arc[0], arc[1], g.dx, dr, g.n_elec_bins, g.nz)
    K.elec_prefix_bins(g.elec_rad_bins, g.n_elec_bins, g.nz)
    K.elec_B_axisymmetric(g.Bx, g.By, g.Bz, g.elec_rad_bins, arc[0], arc[1], g.dx, dr, s["mu0"],
                          g.n_elec_bins, g.nz)
    K.apply_lorentz_JxB(g.Fx, g.Fy, g.Fz, g.Jx, g.Jy, g.Jz, g.Bx, g.By, g.Bz, g.f_l, g.flags, g.dt,
                        g.dx, s["rho_ref"], 2)
    return done, conv


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("dims,max_sweeps,tol,cold", [
    ((8, 8, 8), 20, 1e-30, True),
    ((9, 7, 17), 21, 1e-30, False),    # ends on a chunk of one sweep
    ((9, 7, 17), 21, 1e30, False),     # converged before it: the potential is carried over
    ((33, 32, 31), 47, 1e-30, False),  # a last chunk of seven: four and three sweeps
    ((24, 43, 9), 60, 6e-2, True),     # converges on the way
    ((80, 40, 30), 41, 1e-30, True),   # more than one read by the host
    ((131, 67, 25), 23, 1e30, True),
    ((96, 96, 73), 22, 1e-30, False),  # single sweeps, a last chunk of two
    ((64, 64, 32), 41, 1e-30, False),  # as many tiles as are swept in LDS
    ((65, 64, 32), 41, 1e-30, False),  # a row of them more
    ((65, 64, 32), 60, 2e-1, True),    # converges on the way, read chunk by chunk
])
def test_solve_equals_its_entries(hip_device, layout, dims, max_sweeps, tol, cold):
    one, ref = _grid(dims, layout, 7), _grid(dims, layout, 7)
    arc = (dims[0] / 2 + 0.3, dims[1] / 2 - 0.2, dims[2] / 2 + 0.4)
    dr = max(float(max(dims[0], dims[1])) / (2.0 * one.n_elec_bins), 0.5)
    done, conv = _by_entries(ref, arc, dr, max_sweeps, tol, cold)
    r = K.lorentz_solve(one, arc, bin_dr_cells=dr, max_sweeps=max_sweeps, tol=tol, cold=cold,
                        **SCALARS)
    assert (r.sweeps, bool(r.converged)) == (done, conv)
    assert [r.res, r.norm] == one.elec_l1_buf.to_numpy().tolist()
    for n in ("elec_l1_buf", "sigma_elec", "elec_source", "phi_elec", "Jx", "Jy", "Jz",
              "elec_rad_bins", "Bx", "By", "Bz", "Fx", "Fy", "Fz"):
        a, b = getattr(one, n).to_numpy(), getattr(ref, n).to_numpy()
        assert np.array_equal(a, b), (n, float(np.abs(a - b).max()))
    assert float(torch.as_tensor(one.elec_source.to_numpy()).abs().sum()) > 0.0


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("name,overrides", [
    # droplets (steps that stay with the other engine), CTWD, an odd contiguous extent
    ("ctwd_srt", dict(enable_lorentz=True, nx=57, enable_recoil=True, enable_gas_shear=True)),
    # table material
    ("tables_mrt", dict(enable_lorentz=True, droplet_freq_hz=0.0)),
])
def test_fused_steps_equal_the_entries(hip_device, layout, name, overrides):
    """A twin with the Lorentz force in the fused engine against one in the reference-order
    engine: every field, the snapshot forces, the currents and the CTWD, bit for bit, over runs
    that switch the arc off and on."""
    from tests.step_cases import FIELDS, build_pair, torch_x

    twins = [build_pair(name, engine=e, layout=layout, **overrides)[0]
             for e in ("fused", "reference")]
    more = ("Fx_snap", "Fy_snap", "Fz_snap", "phi_elec", "sigma_elec", "elec_source", "Jx", "Jy",
            "Jz", "Bx", "By", "Bz", "elec_rad_bins", "f_src", "f_dst")
    fused_steps = 0
    for s in range(30):
        welding = not 12 <= s < 15
        for tw in twins:
            g = tw.grid
            tw.step(torch_x(g.dx, g.nx, s, g.dt), (g.ny // 2) * g.dx, welding)
        fused_steps += twins[0]._fused.pending
        if s not in (0, 1, 11, 13, 15, 29):
            continue
        for tw in twins:
            tw.sync()
        for n in FIELDS + more:
            a, b = (getattr(tw.grid, n).to_numpy() for tw in twins)
            assert np.array_equal(a, b), (s, n)
        a, b = twins
        assert (a.ctwd_m, a._bead_height_m) == (b.ctwd_m, b._bead_height_m)
        assert a._lorentz_unconverged == b._lorentz_unconverged
        if welding:
            assert np.float32(a._last_arc_ijk[2]) == np.float32(b._last_arc_ijk[2])
    assert fused_steps > 15


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n_bins,own_raw", [(4096, True), (100, False)])
def test_replaced_bins(hip_device, layout, n_bins, own_raw):
    """As many radial bins as the entries take, and a grid whose bins a program has replaced by
    more than ensure_lorentz_fields made (its second array is then too short, and the solve takes
    the entries' kernels): solved as by the entries."""
    from waam_solver_amd.field import DeviceField

    twins = []
    for _ in range(2):
        g = _grid((24, 43, 9), layout, 7)
        g.n_elec_bins = n_bins
        g.elec_rad_bins = DeviceField.zeros((g.nz, n_bins), torch.float32, g.device)
        if own_raw:
            g.elec_bins_raw = DeviceField.zeros((g.nz, n_bins), torch.float32, g.device)
        twins.append(g)
    one, ref = twins
    arc, dr = (12.3, 21.3, 4.9), 0.01
    _by_entries(ref, arc, dr, 20, 1e-30, True)
    K.lorentz_solve(one, arc, bin_dr_cells=dr, max_sweeps=20, tol=1e-30, cold=True, **SCALARS)
    for n in ("phi_elec", "Jx", "Jy", "Jz", "elec_rad_bins", "Bx", "By", "Bz", "Fx", "Fy", "Fz"):
        a, b = getattr(one, n).to_numpy(), getattr(ref, n).to_numpy()
        assert np.array_equal(a, b), (n, float(np.abs(a - b).max()))
