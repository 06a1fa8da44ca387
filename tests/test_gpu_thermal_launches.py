"""A steady step's thermal kernels in one launch and in launches of their own, on grids on both sides
of each line between the two (plate-march blocks in the ZYX layout with constant material, row
segments elsewhere), against the sweeps of every cell: bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_common import bits_equal, mismatch_report
from tests.step_cases import FIELDS, build_pair, segment_record, torch_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,nx,ny,nz,layout", [
    ("bead_mrt", 16, 2728, 20, 1),    # 2046 plate-march blocks: the last grid that is together
    ("bead_mrt", 16, 2736, 20, 1),    # 2052
    ("bead_mrt", 64, 160, 24, 0),     # 10240 row segments
    ("bead_mrt", 64, 161, 24, 0),
    ("tables_mrt", 64, 256, 24, 0),   # 16384
    ("tables_mrt", 64, 257, 24, 0),
])
def test_both_sides_of_the_line(hip_device, name, nx, ny, nz, layout):
    print(f"[launches] {name} {nx}x{ny}x{nz} layout {layout}", flush=True)
    kw = dict(nx=nx, ny=ny, nz=nz, layout=layout)
    (tw, _), (ref, _) = build_pair(name, **kw), build_pair(name, **kw)
    g = tw.grid
    for s in range(14):
        for t in (tw, ref):
            if t._fused is not None:
                t._fused.quiet_skip = t is tw
            t.step(torch_x(g.dx, nx, s, g.dt), (ny // 2) * g.dx, True)
    nseg, listed, cold = segment_record(tw)
    print(f"[launches] {nseg} segments, {listed} listed, {cold} cold", flush=True)
    assert 0 < listed < nseg or layout == 0  # rows along z all cross the film
    if layout == 1:
        assert cold > nseg // 8
    for t in (tw, ref):
        t.sync()
    for f in FIELDS + ("f_src", "f_dst"):
        a, b = getattr(g, f).to_numpy(), getattr(ref.grid, f).to_numpy()
        assert bits_equal(a, b), mismatch_report(f, a, b)
    assert np.isfinite(g.T.to_numpy()).all()
