"""Table material in the fused engine on both sides of the line between one thermal launch and
several (a count of row segments), against the reference-order engine, which the oracle covers: bit
for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(16, 208, 196), (16, 208, 197), (65, 40, 30)])
def test_table_steps_equal_the_other_engine(hip_device, dims):
    from tests.step_cases import FIELDS, build_pair

    nx, ny, nz = dims
    twins = [build_pair("tables_mrt", engine=e, layout=1, nx=nx, ny=ny, nz=nz)[0]
             for e in ("fused", "reference")]
    for s in range(12):
        for tw in twins:
            tw.step(nx // 2 * tw.grid.dx, (ny // 2 + 0.1 * s) * tw.grid.dx, True)
    for tw in twins:
        tw.sync()
    for n in FIELDS + ("f_src", "f_dst", "cp_rho_field"):
        a, b = (getattr(tw.grid, n).to_numpy() for tw in twins)
        assert np.array_equal(a, b), n
