"""The Poisson x solves at the edges of their ranges (partitioned up to 256
rows; beyond, in sequence with kept factors, k_thomas_seq) against the same
discrete problem solved in extended precision on the host."""
from __future__ import annotations

import numpy as np
import pytest

from simplevofsolver_amd.ic import random_fields

from parity_util import interior, make_pair, read_mask

pytestmark = pytest.mark.gpu

GAMMA0 = 32.0 / 60.0


def solve_extended(ic, ux, uy, dt):
    """psi of the first stage's 2D problem (dft.c:406-468) in long double,
    modulo its mean."""
    ld = np.longdouble
    nx, ny = ic.glsizes
    dxf, dxc = np.diff(ic.xf).astype(ld), np.diff(ic.xc).astype(ld)
    dy = ld(ic.lengths[1]) / ny
    ux = ux.reshape(ny + 2, nx + 1)[1:-1].astype(ld)
    uy = uy.reshape(ny + 2, nx + 2)[1:, 1:-1].astype(ld)
    rhs = (np.diff(ux, axis=1) / dxf + np.diff(uy, axis=0) / dy) / (ld(GAMMA0) * ld(dt))
    ang = 2 * np.arctan2(ld(0), ld(-1)) * np.outer(np.arange(ny), np.arange(ny)) / ny
    c, s = np.cos(ang), np.sin(ang)
    re, im = c @ rhs, -s @ rhs                      # one spectral line per row
    lo, up = 1 / dxc[:-1] / dxf, 1 / dxc[1:] / dxf
    lam = -(2 / dy * np.sin(np.arctan2(ld(0), ld(-1)) * np.arange(ny) / ny)) ** 2
    q = np.stack([re, im], axis=-1)
    dg = -lo - up + lam[:, None]
    dg[:, 0] += lo[0]
    dg[:, -1] += up[-1]
    v = np.zeros((ny, nx), ld)
    for i in range(nx):
        den = dg[:, i] - (lo[i] * v[:, i - 1] if i else 0)
        if i == nx - 1:
            den[0] = 1                              # singular: its constant is removed below
        v[:, i] = up[i] / den
        q[:, i] = (q[:, i] - (lo[i] * q[:, i - 1] if i else 0)) / den[:, None]
    q[0, -1] = 0
    for i in range(nx - 2, -1, -1):
        q[:, i] -= v[:, i, None] * q[:, i + 1]
    psi = (c @ q[..., 0] - s @ q[..., 1]) / ny
    return psi - np.sum(psi * dxf) / np.sum(dxf) / ny


def error(g, ic, want):
    a = interior("psi", g.get("psi"), ic.glsizes).astype(np.longdouble)
    w = np.diff(ic.xf).astype(np.longdouble)
    a = a - np.sum(a * w) / np.sum(w) / a.shape[0]
    return float(np.max(np.abs(a - want)) / np.max(np.abs(want)))


@pytest.mark.parametrize("uniformx", [True, False])
@pytest.mark.parametrize("nx", [4, 7, 255, 256, 257, 300, 511, 512, 513, 700, 1023, 1024])
def test_x_solve_in_extended_precision(nx, uniformx, tmp_path):
    """The default elimination is within 1e-12 of long double, or where
    thomas_part 0 is not (the operator's condition grows as nx^2: 1e-12 to
    2.5e-12 from 700 stretched rows on) no further off than half again its
    error; the refined FP32 solve is within its 1e-8."""
    ic = random_fields((nx, 12), seed=nx, uniformx=uniformx)
    _, g = make_pair(ic, tmp_path)
    try:
        dt = g.decide_dt()
        want = solve_extended(ic, g.get("ux"), g.get("uy"), dt)
        err = {}
        for part in (0, 1):
            g.set_tuning("thomas_part", part)
            g.potential(0, dt)
            err[part] = error(g, ic, want)
        assert err[1] < max(1e-12, 1.5 * err[0]), err
        g.set_poisson_mixed(2)
        g.potential(0, dt)
        e = error(g, ic, want)
        assert e < 1e-8, e
    finally:
        g.close()


@pytest.mark.parametrize("glsizes", [(257, 5), (300, 48), (384, 20), (512, 6), (513, 9), (641, 32), (1100, 4), (260, 6, 5),
                                     (300, 8, 12)])
@pytest.mark.parametrize("refine", [-1, 0])
def test_kept_factors_change_nothing(glsizes, refine, tmp_path):
    """k_thomas_seq against k_thomas_spec (thomas_part 0) bit for bit: whole
    and partial passes of 128 rows, groups of fewer than 8 lines, the singular
    line's gauge, FP64 and FP32 spectra."""
    _, g = make_pair(random_fields(glsizes, seed=sum(glsizes), uniformx=False), tmp_path)
    try:
        g.set_poisson_mixed(refine)
        dt = g.decide_dt()
        psi = []
        for part in (1, 0):
            g.set_tuning("thomas_part", part)
            g.potential(1, dt)
            psi.append(g.get("psi")[read_mask("psi", glsizes).ravel()])
        assert np.all(np.isfinite(psi[0])) and np.array_equal(psi[0], psi[1])
    finally:
        g.close()
