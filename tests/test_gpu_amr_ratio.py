"""Hierarchies of refinement ratios 2, 3 and 4 against the AMR oracle: the flux
registers' lanes per face, and patches whose rows and columns leave lanes of
every tile shape idle.  Bit-exact on both levels, also where momenta of
2^-300 to 2^-700 and signed zeros send whole tiles to the IEEE sequences."""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
from amr_oracle import AmrOracle  # noqa: E402

import amr_cases as A  # noqa: E402
import finitevolumesolver_amd as fvs  # noqa: E402
from finitevolumesolver_amd.amr import AmrHierarchy  # noqa: E402

pytestmark = pytest.mark.gpu


def _small_momenta(i0, j0, rho, u):
    """rho u with momenta that no shared reciprocal serves, tiles in a row of
    each kind: 2^-300, -2^-500, 2^-700, zeros of either sign, and ordinary ones."""
    ny, nx = rho.shape
    kind = (i0 + np.arange(nx)) // 3 + (j0 + np.arange(ny))[:, None] // 2
    table = np.array([2.0 ** -300, -2.0 ** -500, 2.0 ** -700, 0.0, -0.0])
    return np.where(kind % 6 == 5, rho * u, table[kind % 6 % 5])


def _run(ratio, shape, small):
    n, dx0 = 18, 2.0 / 18
    layouts = [[(0, 0, 11, 18), (11, 0, 7, 18)],
               [(4 * ratio, 5 * ratio, 5 * ratio, 7 * ratio), (9 * ratio, 5 * ratio, 4 * ratio, 3 * ratio)]]

    def state(level, p):
        i0, j0, nx, ny = layouts[level][p]
        dx = dx0 / ratio ** level
        x = -1.0 + (i0 + np.arange(nx) + 0.5) * dx
        y = (-1.0 + (j0 + np.arange(ny) + 0.5) * dx)[:, None]
        rho = 1.0 + 0.4 * np.exp(-6.0 * (x * x + y * y))
        u, v = 0.3 * rho, -0.2 + 0.0 * rho
        # the small momenta stay small where the pressure is constant
        p = 1.0 + 0.8 * (x + y > (1.2 if small else 0.1))
        if small:
            mx, my = _small_momenta(i0, j0, rho, u), _small_momenta(j0, i0 + 1, rho, v)
            return np.stack([rho, mx, my, p / 0.4 + 0.5 * (mx * mx + my * my) / rho])
        return np.stack([rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)])

    fm = fvs.FluxMethod(fvs.PerfectGas(dim=2), base="HLLEM", reconstruction="MusclHancock")
    h = AmrHierarchy(fm, (n, n), layouts, dx0, ratio)
    o = AmrOracle((n, n), layouts, dx0, ratio, A.oracle_sweep(fm._h.desc), "reference")
    h.set_state(state)
    for l, lay in enumerate(layouts):
        for d in (0, 1):
            h.levels[l].set_shape(d, shape)
        for p in range(len(lay)):
            o.U[l][p][:, 2:-2, 2:-2] = state(l, p)
    h.average_down(1)
    o.average_down(1)
    for _ in range(2):
        dt = h.stable_dt()
        assert dt == o.stable_dt()
        h.advance(0.8 * dt)
        o.advance(0.8 * dt)
        for l in range(2):
            for p, g in enumerate(h.interiors(l)):
                assert np.array_equal(g, o.U[l][p][:, 2:-2, 2:-2]), (l, p)


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("ratio", [2, 3, 4])
def test_steps(cuda, ratio, shape):
    _run(ratio, shape, small=False)


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("ratio", [2, 3, 4])
def test_steps_of_small_momenta(cuda, ratio, shape):
    _run(ratio, shape, small=True)
