"""A run's first Lorentz solve starts from a grounded potential and may take as many sweeps as that
needs. A call that fails leaves the next one the first."""

from types import SimpleNamespace

from waam_solver_amd.physics import weld_forces


def test_a_failed_call_leaves_the_next_solve_cold():
    grid = SimpleNamespace(nx=9, ny=7, nz=5, n_elec_bins=64, ensure_lorentz_fields=lambda: None)
    twin = SimpleNamespace(
        lorentz_jacobi_iters=40, sigma_cells=2.0, welding_current_A=140.0, sigma_liquid_Sm=1e6,
        sigma_solid_Sm=1e5, lorentz_jacobi_omega=0.85, nz_solid=2, mat=SimpleNamespace(rho=7800.0))
    arc = (4.0, 3.0, 2.0)
    for _ in range(2):  # the first call's solve never ran
        args = weld_forces.lorentz_args(twin, grid, *arc)
        assert (args["cold"], args["max_sweeps"]) == (True, 2 * 9 * 9)
    weld_forces.note_lorentz(twin, SimpleNamespace(converged=1, res=0.0, norm=1.0), args)
    args = weld_forces.lorentz_args(twin, grid, *arc)
    assert (args["cold"], args["max_sweeps"]) == (False, 40)
