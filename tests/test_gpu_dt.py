"""The time step's reduction at the edges of its tiles (64 x 4 of (i, j), 8
rows or 16 planes a pass) and on both sides of the 256 work-groups that one
launch reduces by itself, against the limit of one known velocity."""
from __future__ import annotations

import numpy as np
import pytest

import simplevofsolver_amd as sva
from simplevofsolver_amd.ic import random_fields

from parity_util import padded_shape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("glsizes", [(8, 4), (63, 5), (64, 32), (65, 36), (130, 9), (8, 4, 4), (64, 32, 4), (65, 36, 5),
                                     (130, 64, 40)])
def test_time_step_is_the_minimum(glsizes, tmp_path):
    """The only velocity stands in turn in the corners, at the tiles' edges
    and past them: the step is 0.4 h / (50 + 1e-8), two roundings from the
    number formed here (1e-15)."""
    nd, nx, ny = len(glsizes), glsizes[0], glsizes[1]
    ic = random_fields(glsizes, seed=3, uniformx=False)
    g = sva.solver_from_ic(ic, str(tmp_path / "a"))
    names = ["ux", "uy", "uz"][:nd]
    try:
        zero = {n: np.zeros(padded_shape(n, glsizes)) for n in names}
        for n in names:
            g.set(n, zero[n])
        for d, n in enumerate(names):
            for i in {2, min(64, nx), min(65, nx), nx}:
                h = ic.xc[i] - ic.xc[i - 1] if d == 0 else ic.lengths[d] / glsizes[d]
                for j in {1, min(32, ny), min(33, ny), ny}:
                    for k in [None] if nd == 2 else [1, glsizes[2]]:
                        a = zero[n].copy()
                        col = i - 1 if n == "ux" else i
                        a[(j, col) if k is None else (k, j, col)] = -50.0
                        g.set(n, a)
                        want = 0.4 * (h / (50.0 + 1e-8))
                        assert abs(g.decide_dt() - want) <= 1e-15 * want, (n, i, j, k)
            g.set(n, zero[n])
    finally:
        g.close()


@pytest.mark.parametrize("glsizes", [(4033, 270), (1000, 2025), (60, 2048), (1000, 36, 20), (8, 6, 48)])
def test_time_step_in_later_rows_and_passes(glsizes, tmp_path):
    """Grids of more than 512 tiles in 2D, whose threads take several rows, 8 a
    pass, up to a second pass with a clamped tail (4033 x 270: 8 row groups,
    256 rows a pass), and 3D grids of several plane groups: the only velocity
    stands on both sides of each thread's first, second, 8th and 9th row, of
    the last rows and of the first planes of each group."""
    nd, nx, ny = len(glsizes), glsizes[0], glsizes[1]
    gx, gy = -(-nx // 64), -(-ny // 4)
    rows = 4 * (min(gy, max(1, 512 // gx)) if nd == 2 else gy)
    js = sorted({j for j in (1, rows, rows + 1, 8 * rows, 8 * rows + 1, 8 * rows + 2, ny - 1, ny) if 1 <= j <= ny})
    gz = -(-glsizes[2] // 16) if nd == 3 else 1
    ks = [None] if nd == 2 else sorted({1, gz, gz + 1, 2 * gz, glsizes[2] - 1, glsizes[2]})
    ic = random_fields(glsizes, seed=3, uniformx=False)
    speed = 5000.0                # far below the diffusive limit of these grids
    g = sva.solver_from_ic(ic, str(tmp_path / "a"))
    names = ["ux", "uy", "uz"][:nd]
    try:
        for n in names:
            g.set(n, np.zeros(padded_shape(n, glsizes)))
        for d, n in enumerate(names):
            a = np.zeros(padded_shape(n, glsizes))
            for i in (2, nx):
                h = ic.xc[i] - ic.xc[i - 1] if d == 0 else ic.lengths[d] / glsizes[d]
                for j in js:
                    for k in ks:
                        at = (j, i - 1 if n == "ux" else i) if k is None else (k, j, i - 1 if n == "ux" else i)
                        a[at] = -speed
                        g.set(n, a)
                        a[at] = 0.0
                        want = 0.4 * (h / (speed + 1e-8))
                        assert abs(g.decide_dt() - want) <= 1e-15 * want, (n, i, j, k)
            g.set(n, a)
    finally:
        g.close()
