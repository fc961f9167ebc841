"""The single case's step graph: every step of a solver that replays it against
one that issues plain launches (per-kernel timing on), bit for bit, with other
work and synchronisations between the replays, two solvers in turn, and the
tuning and precision switches that change the launches."""
from __future__ import annotations

import numpy as np
import pytest

import simplevofsolver_amd as sva
from simplevofsolver_amd.ic import random_fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("glsizes", [(32, 48), (20, 45), (300, 20), (16, 12, 20), (24, 20, 15)])
def test_graph_steps_match_plain_steps(glsizes, tmp_path):
    nd = len(glsizes)
    names = ["ux", "uy", "p", "t", "vof"] + (["uz"] if nd == 3 else [])
    pairs = []
    for k in range(2):
        ic = random_fields(glsizes, seed=5 + k, uniformx=k == 0)
        g = sva.solver_from_ic(ic, str(tmp_path / f"g{k}"))
        r = sva.solver_from_ic(ic, str(tmp_path / f"r{k}"))
        r.profile(True)
        pairs.append((g, r))
    switch = {4: lambda s: s.set_tuning("lines_lpb", 3), 6: lambda s: s.set_poisson_mixed(1),
              8: lambda s: s.set_poisson_mixed(-1), 9: lambda s: s.set_tuning("rhs_rows", 2)}
    try:
        for step in range(14):
            for g, r in pairs:
                for s in (g, r):
                    if step in switch:
                        switch[step](s)
                assert g.integrate() == r.integrate(), step
            for g, r in pairs:
                if step % 3 == 1:
                    assert g.diagnostics() == r.diagnostics()
                if step % 4 == 2:
                    # the program's own work on the fields between steps
                    for s in (g, r):
                        s.set("ux", 0.5 * s.get("ux"))
                        s.boundaries("ux")
                for n in names:
                    assert np.array_equal(g.get(n), r.get(n)), (step, n)
    finally:
        for g, r in pairs:
            g.close()
            r.close()


@pytest.mark.parametrize("glsizes", [(32, 48), (300, 20), (8191, 4), (16, 12, 20)])
def test_steps_are_replayed_and_switches_build_anew(glsizes, tmp_path):
    """The first step is issued launch by launch, the second builds the graph,
    all others replay it; a switch that changes the launches builds one graph,
    one that does not builds none, per-kernel timing replays none, and the
    runtime refuses nothing (8191: x lines of more than 64 KiB of LDS)."""
    g = sva.solver_from_ic(random_fields(glsizes, seed=5, uniformx=True), str(tmp_path / "g"))
    try:
        assert g.graph_counts() == (0, 0, 0)
        g.integrate()
        assert g.graph_counts() == (0, 0, 0)
        built, replayed = 0, 0
        for switch, builds, replays in [
                (lambda: None, 1, 1), (lambda: g.set("ux", 0.5 * g.get("ux")), 0, 1), (lambda: g.set_tuning("rhs_rows", 4), 1, 1),
                (lambda: g.set_poisson_mixed(1), 1, 1), (lambda: g.set_poisson_mixed(-1), 1, 1),
                (lambda: g.set_tuning("xcd_bands", 1), 0, 1), (lambda: g.profile(True), 0, 0),
                (lambda: g.profile(False), 0, 1)]:
            switch()
            for k in range(3):
                g.integrate()
                built += builds if k == 0 else 0
                replayed += replays
                assert g.graph_counts() == (built, replayed, 0), (k, builds)
    finally:
        g.close()
