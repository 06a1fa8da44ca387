"""The cavity step on extents that end inside a wavefront or a block, bit-equal to the oracle's, in
both storage orders, with walls and lid cells inside the fluid as well."""

from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_common import bits_equal, mismatch_report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n,blocked", [(1, False), (5, False), (31, True), (62, True), (63, False)])
def test_cavity_sizes(hip_device, n, blocked, layout):
    from oracle.oracle import lib, ptr
    from waam_solver_amd.cavity import LID, WALL, LidDrivenCavity

    print(f"[cavity] n={n} blocked={blocked} layout={layout}", flush=True)
    cav = LidDrivenCavity(n=n, seed=5, device=hip_device, layout=layout)
    if blocked:
        fl = cav.flags.to_numpy().astype(np.uint8)
        rng = np.random.default_rng(2)
        inner = fl[1:-1, 1:-1, 1:-1]
        inner[rng.random(inner.shape) < 0.05] = WALL
        inner[rng.random(inner.shape) < 0.02] = LID
        fl[0, 1:3, 1] = 0  # fluid on the x edge: its sources wrap
        cav.flags.from_numpy(fl)
    L = lib(parallel=True)
    flags = cav.flags.to_numpy().astype(np.uint8)
    a, rho = cav.f.to_numpy(), cav.rho.to_numpy()
    b = a.copy()
    ux, uy, uz = (np.zeros(flags.shape, np.float32) for _ in range(3))
    cav.step(7)
    for _ in range(7):
        L.or_cavity_step(ptr(a), ptr(b), ptr(rho), ptr(ux), ptr(uy), ptr(uz), ptr(flags),
                         cav.omega, cav.omega, cav.u_lid, 0.0, 0.0, *flags.shape)
        a, b = b, a
    for name, got, want in (("rho", cav.rho, rho), ("ux", cav.ux, ux), ("uy", cav.uy, uy),
                            ("uz", cav.uz, uz), ("f", cav.f, a)):
        got = got.to_numpy()
        assert bits_equal(got, want), mismatch_report(name, got, want)
