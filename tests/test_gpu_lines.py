"""The predictor's x-line solver (k_lines_lds) at the edges of its tiles: line
lengths around its 16-row segments, 64-row passes and load chunks, work-groups
of one line up to several sweeping wavefronts, groups that cross planes and
reach the periodic rows.  The recurrences are those of gtsv (src/tdm.c:17-50)
in its order, so the fields are compared bit for bit with the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from simplevofsolver_amd.ic import random_fields

from parity_util import copy_state, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("glsizes", [(4, 5), (16, 6), (17, 4), (18, 9), (33, 5), (49, 4), (64, 5), (65, 6), (66, 4),
                                     (129, 5), (193, 4), (257, 4), (1030, 4), (8191, 4), (5, 4, 5), (17, 4, 6),
                                     (65, 5, 4)])
def test_lines_match_oracle(glsizes, tmp_path):
    o, g = make_pair(random_fields(glsizes, seed=sum(glsizes), uniformx=glsizes[0] > 1000), tmp_path)
    names = ["ux", "uy", "t"] + (["uz"] if len(glsizes) == 3 else [])
    try:
        dt = o.decide_dt()
        want = None
        for lpb in (0, 1, 3, 16, 17, 40):
            g.set_tuning("lines_lpb", lpb)
            if want is None:
                copy_state(o, g)
                start = {n: o.get(n) for n in names + ["srcux_a", "srcux_b", "srcuy_a", "srcuy_b", "srct_a", "srct_b"]
                         + (["srcuz_a", "srcuz_b"] if len(glsizes) == 3 else [])}
                o.predict(0, dt)
                want = {n: o.get(n) for n in names}
            else:
                for n, v in start.items():
                    g.set(n, v)
            g.predict(0, dt)
            for n in names:
                assert np.array_equal(g.get(n), want[n]), (lpb, n)
    finally:
        g.close()


@pytest.mark.parametrize("lpb", [0, 17])
@pytest.mark.parametrize("glsizes", [(4, 5), (17, 4), (66, 4), (193, 4), (5, 4, 5), (65, 5, 4)])
def test_fused_lines_match_per_function_lines(glsizes, lpb, tmp_path):
    """The fused step reads ready increments and writes the halo images itself;
    the per-function step forms the increments and calls the boundary updates."""
    import simplevofsolver_amd as sva
    ic = random_fields(glsizes, seed=3, uniformx=False)
    a = sva.solver_from_ic(ic, str(tmp_path / "a"))
    b = sva.solver_from_ic(ic, str(tmp_path / "b"), schedule=0)
    try:
        a.set_tuning("lines_lpb", lpb)
        for _ in range(2):
            assert a.integrate() == b.integrate()
        for n in ["ux", "uy", "t"] + (["uz"] if len(glsizes) == 3 else []):
            assert np.array_equal(a.get(n), b.get(n)), n
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("lpb", [0, 5, 64])
@pytest.mark.parametrize("glsizes", [(4, 90), (16, 75), (32, 9), (47, 6), (48, 20), (49, 6), (80, 5), (96, 20), (97, 9),
                                     (6, 20, 16), (48, 9, 8), (81, 5, 6), (97, 6, 5)])
def test_lines_in_chunks_of_16_rows(glsizes, lpb, tmp_path):
    """Both sides of the limits between chunks of 16 and of 64 rows (nx 48 / 49
    and 96 / 97; ux has one row fewer), with the last access of a group partly
    past its last line: the fused step against the per-function one bit for
    bit, halo images included, and its line solves against the oracle's."""
    import simplevofsolver_amd as sva
    ic = random_fields(glsizes, seed=4, uniformx=False)
    o, a = make_pair(ic, tmp_path / "a")
    b = sva.solver_from_ic(ic, str(tmp_path / "b"), schedule=0)
    names = ["ux", "uy", "t"] + (["uz"] if len(glsizes) == 3 else [])
    try:
        a.set_tuning("lines_lpb", lpb)
        b.set_tuning("lines_lpb", lpb)
        for _ in range(2):
            assert a.integrate() == b.integrate()
        for n in names:
            assert np.array_equal(a.get(n), b.get(n)), n
        dt = o.decide_dt()
        copy_state(o, b)
        o.predict(0, dt)
        b.predict(0, dt)
        for n in names:
            assert np.array_equal(b.get(n), o.get(n)), n
    finally:
        a.close()
        b.close()
