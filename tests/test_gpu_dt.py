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
