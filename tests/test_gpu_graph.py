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


OPTIONS = {
    "one-kernel predictor": lambda s: s.set_fusion(127),
    "sequential x solve": lambda s: s.set_tuning("thomas_part", 0),
    "mixed radix": lambda s: (s.set_tuning("fft_radix", 4), s.set_tuning("fft_elems", 2048)),
    "two refinements": lambda s: s.set_poisson_mixed(2),
    "bands and rows": lambda s: (s.set_tuning("xcd_bands", 1), s.set_tuning("rhs_rows", 16), s.set_tuning("lines_lpb", 5)),
    "two streams for a while": lambda s: s.set_tuning("iface_overlap", 1),
}


@pytest.mark.parametrize("option", list(OPTIONS))
@pytest.mark.parametrize("glsizes", [(20, 45), (16, 256), (300, 20), (24, 20, 15)])
def test_graph_steps_with_options(glsizes, option, tmp_path):
    """The options that change a step's kernels or swap its buffers, set before
    the first step and taken back (two streams, after which the next step is
    the first on one stream) or repeated later on."""
    nd = len(glsizes)
    ic = random_fields(glsizes, seed=11, uniformx=False)
    g = sva.solver_from_ic(ic, str(tmp_path / "g"))
    r = sva.solver_from_ic(ic, str(tmp_path / "r"))
    try:
        r.profile(True)
        for s in (g, r):
            OPTIONS[option](s)
        for step in range(9):
            if step == 4:
                for s in (g, r):
                    if option == "two streams for a while":
                        s.set_tuning("iface_overlap", 0)
                    else:
                        OPTIONS[option](s)
            assert g.integrate() == r.integrate(), step
            for n in ["ux", "uy", "p", "t", "vof"] + (["uz"] if nd == 3 else []):
                assert np.array_equal(g.get(n), r.get(n)), (step, n)
        built, replayed, refused = g.graph_counts()
        assert refused == 0 and built == 1
        assert replayed == (4 if option == "two streams for a while" else 8)
    finally:
        g.close()
        r.close()


def test_graph_steps_in_threads(tmp_path):
    """Three solvers and a batch, each stepped by a thread of its own at the
    same time, against the same steps one after another."""
    import threading
    grids = [(32, 48), (20, 45), (40, 24), (24, 30), (48, 20), (16, 36)]

    def make(tag):
        ss = [sva.solver_from_ic(random_fields(z, seed=21 + k, uniformx=k % 2 == 0), str(tmp_path / f"{tag}{k}"))
              for k, z in enumerate(grids)]
        return ss, sva.Batch(ss[3:])

    def run(jobs, threads):
        if not threads:
            for j in jobs:
                j()
            return
        ts = [threading.Thread(target=j) for j in jobs]
        for t in ts:
            t.start()
        for t in ts:
            t.join(60)
            assert not t.is_alive()

    out = []
    for tag, threads in (("a", False), ("b", True)):
        ss, batch = make(tag)
        dts = {}

        def steps(k, f):
            dts[k] = [f() for _ in range(30)]

        try:
            run([lambda k=k: steps(k, ss[k].integrate) for k in range(3)] + [lambda: steps("batch", batch.integrate)],
                threads)
            batch.synchronize()
            out.append((dts, [[s.get(n) for n in ("ux", "uy", "p", "t", "vof")] for s in ss]))
            assert all(s.graph_counts() == (1, 29, 0) for s in ss[:3])
        finally:
            batch.close()
            for s in ss:
                s.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
