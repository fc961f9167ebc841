"""The marching source and interface kernels against the kernels of one row
and of blocks, bit for bit, on grids whose rows and planes are no multiples
of what a thread or work-group marches (the last march is partial), of more
than one tile in x and of fewer rows than one march.  Both sides are set, so
that the comparison does not depend on what the grid's size would choose."""
from __future__ import annotations

import numpy as np
import pytest

import simplevofsolver_amd as sva
from simplevofsolver_amd.ic import random_fields

pytestmark = pytest.mark.gpu

GRIDS = [(70, 45), (37, 27), (9, 6), (70, 45, 50), (33, 20, 27), (9, 12, 9)]
MARCHES = [("rhs_rows", 2), ("rhs_rows", 4), ("rhs_rows", 8), ("rhs_rows", 16), ("iface_planes", 4),
           ("iface_planes", 8), ("iface_planes", 16)]


@pytest.mark.parametrize("glsizes,march", [(g, m) for g in GRIDS for m in MARCHES
                                           if m[0] == "rhs_rows" or len(g) == 3])
def test_marches_match_one_row_and_blocks(glsizes, march, tmp_path):
    nd = len(glsizes)
    ic = random_fields(glsizes, seed=sum(glsizes), uniformx=False)
    one = sva.solver_from_ic(ic, str(tmp_path / "one"))
    many = sva.solver_from_ic(ic, str(tmp_path / "many"))
    try:
        for s in (one, many):
            s.set_tuning("rhs_rows", 1)
            if nd == 3:
                s.set_tuning("iface_planes", 0)
        many.set_tuning(*march)
        for step in range(2):
            assert one.integrate() == many.integrate()
            for n in ["ux", "uy", "t", "vof", "p", "psi", "curv"] + (["uz"] if nd == 3 else []):
                assert np.array_equal(many.get(n), one.get(n)), (step, n)
    finally:
        one.close()
        many.close()
