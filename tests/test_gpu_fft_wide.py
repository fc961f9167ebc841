"""The transforms in work-groups of their full width (grids of thousands of
columns) with a partly empty last tile and an odd nx, whose last column has no
partner: the 256-point register kernels of 8 columns in y and 16 in z against
the mixed-radix ones, the mixed-radix kernels of 1024 against 2048 values per
LDS buffer."""
from __future__ import annotations

import numpy as np
import pytest

import simplevofsolver_amd as sva
from simplevofsolver_amd.ic import random_fields

from parity_util import demean, interior, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("glsizes", [(37, 256, 216), (37, 216, 256)])
def test_wide_transforms(glsizes, tmp_path):
    """psi of one pressure solve modulo its mean.  The paths differ by
    rounding, 1e-16 per transform, which the solve amplifies by its condition
    in x ((2 x 37 / pi)^2, below 1e3): 1e-11 leaves two digits.  The FP32
    passes of the refined solve leave 1e-7 times that, cubed by two
    refinements, and are held to the 1e-8 of the other refined solves."""
    ic = random_fields(glsizes, seed=7, uniformx=False)
    dxf = np.diff(ic.xf)
    g = sva.solver_from_ic(ic, str(tmp_path / "g"))

    def psi():
        g.potential(0, 1e-3)
        return interior("psi", demean("psi", g.get("psi"), glsizes, dxf), glsizes)

    try:
        want = psi()
        assert np.all(np.isfinite(want))
        g.set_poisson_mixed(2)
        refined = psi()
        assert rel(refined, want) < 1e-8
        g.set_tuning("fft_radix", 4)
        assert rel(psi(), refined) < 2e-8
        g.set_poisson_mixed(-1)
        assert rel(psi(), want) < 1e-11
        g.set_tuning("fft_elems", 2048)
        assert rel(psi(), want) < 1e-11
        # the equation itself, so that no fault that both paths share passes
        assert residual(g, ic, 1e-3) < 1e-9
    finally:
        g.close()


def residual(g, ic, dt):
    """max |lap psi - div u / (gamma dt)| / max |div u / (gamma dt)| with the
    first stage's gamma; rounding of the second differences is about
    eps (dy^-2 + dz^-2 + dx^-2) |psi| / |rhs|, 1e-10 on these grids."""
    nx, ny, nz = ic.glsizes
    gdt = 32.0 / 60.0 * dt
    ux = g.get("ux").reshape(nz + 2, ny + 2, nx + 1)[1:-1, 1:-1]
    uy = g.get("uy").reshape(nz + 2, ny + 2, nx + 2)[1:-1, 1:, 1:-1]
    uz = g.get("uz").reshape(nz + 2, ny + 2, nx + 2)[1:, 1:-1, 1:-1]
    dxf, dxc = np.diff(ic.xf), np.diff(ic.xc)
    dy, dz = ic.lengths[1] / ny, ic.lengths[2] / nz
    rhs = (np.diff(ux, axis=2) / dxf + np.diff(uy, axis=1) / dy + np.diff(uz, axis=0) / dz) / gdt
    p = interior("psi", g.get("psi"), ic.glsizes)
    grad = np.zeros((nz, ny, nx + 1))
    grad[:, :, 1:-1] = np.diff(p, axis=2) / dxc[1:-1]
    lap = np.diff(grad, axis=2) / dxf
    for a, d in ((1, dy), (0, dz)):
        lap = lap + (np.roll(p, 1, a) + np.roll(p, -1, a) - 2.0 * p) / d ** 2
    return float(np.max(np.abs(lap - rhs)) / np.max(np.abs(rhs)))
