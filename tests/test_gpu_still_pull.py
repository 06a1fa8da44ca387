"""The steady step's pull moves only the directions of the row segments whose words can change
(the segment record's change words). Two fused twins from the same seeded pool, one with the
record off (every step sweeps and pulls everything): every field and both population buffers must
stay bit-equal, through the steps after a restart of the record, in the middle of a run and after
a host write, at the extents where segments end, wrap and clamp."""

from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_common import bits_equal, mismatch_report
from tests.step_cases import FIELDS, build_pair, torch_x

pytestmark = pytest.mark.gpu


def _align(n: int) -> int:
    return (n + 255) // 256 * 256


def _pulled(tw) -> tuple[int, int]:
    """(listed segments of the last steady step's pull, row segments)."""
    g = tw.grid
    fast, slow = (g.nx, g.nz) if g.layout == 1 else (g.nz, g.nx)
    nseg = -(-fast // 64) * g.ny * slow
    off = _align(nseg) + 256 + 4 * nseg + nseg          # bits, count, list, need
    off = _align(_align(off) + (g.n_cells + 1) // 2)    # the full pull's masks
    rec = g.quiet.to_numpy().view(np.uint8)
    return int(rec[off:off + 4].view(np.int32)[0]), nseg


def _bits(tw, bx: int, rows, k: int) -> list[int]:
    """The record bytes of segment bx of the rows j in slice k (rows along x)."""
    g = tw.grid
    nbx = -(-g.nx // 64)
    rec = g.quiet.to_numpy().view(np.uint8)
    return [int(rec[(k * g.ny + j) * nbx + bx]) for j in rows]


@pytest.mark.parametrize("nx,ny,nz,layout,pop", [
    (64, 40, 32, 1, "fp32"),     # one whole segment a row: it wraps onto itself
    (65, 24, 24, 1, "fp32"),     # the second segment is one cell: both its ends
    (63, 24, 24, 1, "bf16"),
    (200, 40, 32, 1, "fp16"),    # four segments, the last of eight cells
    (129, 31, 25, 1, "fp16"),
    (40, 24, 66, 0, "fp32"),     # rows along z: no record kept, every steady step pulls whole
    (33, 25, 64, 0, "fp16"),
])
def test_still_populations_are_left_alone(hip_device, nx, ny, nz, layout, pop):
    print(f"[still] {nx}x{ny}x{nz} layout {layout} {pop}", flush=True)
    kw = dict(nx=nx, ny=ny, nz=nz, layout=layout, population_storage=pop)
    (tw, _), (ref, _) = build_pair("bead_mrt", **kw), build_pair("bead_mrt", **kw)
    g = tw.grid
    done = 0
    for n, write in ((1, False), (2, False), (1, False), (36, True), (4, False), (30, False)):
        for s in range(done, done + n):
            for t in (tw, ref):
                if t._fused is not None:
                    t._fused.quiet_skip = t is tw
                t.step(torch_x(g.dx, g.nx, s, g.dt), (g.ny // 2) * g.dx, True)
        done += n
        if done > 8 and layout == 1:
            count, nseg = _pulled(tw)
            print(f"[still] step {done}: {count} of {nseg} segments pulled", flush=True)
            if done in (40, 74):
                assert count < nseg
        for t in (tw, ref):
            t.sync()
        for f in FIELDS:
            a, b = getattr(g, f).to_numpy(), getattr(ref.grid, f).to_numpy()
            assert bits_equal(a, b), f"step {done}: {mismatch_report(f, a, b)}"
        for f in ("f_src", "f_dst"):
            a, b = getattr(g, f).to_numpy(), getattr(ref.grid, f).to_numpy()
            assert bits_equal(a, b), f"step {done}: {mismatch_report(f, a, b)}"
        if layout == 1:
            # the warmed cell's row segments: cold plate before, not for some steps after, then again
            bits = _bits(tw, nx // 2 // 64, (1, 2), 1)
            print(f"[still] step {done}: record of the warmed rows {bits}", flush=True)
            if done == 40:
                assert all(b & 12 == 12 for b in bits)
            if done == 44:
                assert all(b & 4 == 0 for b in bits)
            if done == 74:
                assert bits[0] & 12 == 12  # the one that did not melt
        if write:  # hot gas populations and warm plate cells, as a host program may set them: one
            # above the record's limit (the lowest HAZ threshold), one that remelts
            for t in (tw, ref):
                p = t.grid.f_src.to_numpy()
                p[5, nx // 2, ny // 3, nz - 3] += np.float32(0.01)
                t.grid.f_src.from_numpy(p)
                T, H = t.grid.T.to_numpy(), t.grid.H.to_numpy()
                for j, warm, latent in ((1, 1200.0, 0.0), (2, t.mat.T_liquidus + 50.0, t.L_rho)):
                    T[nx // 2, j, 1] = warm
                    H[nx // 2, j, 1] = t.cp_rho * warm + latent
                t.grid.T.from_numpy(T)
                t.grid.H.from_numpy(H)
