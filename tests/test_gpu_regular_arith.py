"""The sweeps' shared-reciprocal IEEE arithmetic: bit-exact with the oracle for
denominators whose reciprocals round hard, and across waves that fall back to
the general sequences (momenta below the guarded range, signed zeros)."""
from __future__ import annotations

import numpy as np
import pytest

from fields import rough_field
from sweep_ref import oracle_sweep

import finitevolumesolver_amd as fvs

pytestmark = pytest.mark.gpu


def _state(shape, kind):
    """(D + 2, nz, ny, nx) conservative states."""
    D = 2 if shape[0] == 1 else 3
    cons = rough_field(shape, seed=5 + shape[2], jumps=True)
    rng = np.random.default_rng(shape[2])
    rho = cons[0]
    if kind == "hard":
        # significands 2 - k 2^-52, k = 1 .. 6, on flat stretches: densities,
        # and through them the square roots' sums, next to powers of two
        ulps = rng.integers(1, 7, rho.shape)
        hard = np.ldexp(1.0, rng.integers(-1, 2, rho.shape)) * (2.0 - ulps * 2.0**-52)
        rho[:] = np.where(rng.random(rho.shape) < 0.7, hard, rho)
        cons[D + 1] += 10.0
    elif kind == "tiny":
        # momenta that the guard refuses, in half of the rows, and signed zeros
        m = cons[1:D + 1]
        tiny = np.ldexp(rng.standard_normal(m.shape), -rng.integers(150, 700, m.shape))
        pick = rng.integers(0, 4, m.shape)
        m[:] = np.choose(pick, [m, tiny, np.zeros_like(m), -np.zeros_like(m)])
        cons[1:D + 1, :, ::2] = np.where(pick == 0, 0.0, m)[:, :, ::2]
        cons[D + 1] += 2.0
    return cons


@pytest.mark.parametrize("limiter", ["MinMod", "VanLeer", "NoLimiter"])
@pytest.mark.parametrize("kind", ["hard", "tiny"])
@pytest.mark.parametrize("shape", [(1, 9, 61), (1, 70, 130), (7, 6, 63), (66, 5, 31)])
def test_bits(cuda, shape, kind, limiter):
    import torch
    D = 2 if shape[0] == 1 else 3
    if limiter == "NoLimiter" and kind == "hard":
        pytest.skip("central slopes across the jumps give negative pressures")
    cons = _state(shape, kind)
    if limiter == "NoLimiter":
        cons[0] = 1.0 + 0.1 * np.sin(np.arange(shape[2]) * 0.2)
        cons[1:D + 1] *= 0.05
        cons[D + 1] = 3.0
    fm = fvs.FluxMethod(fvs.PerfectGas(dim=D), base="HLLEM", limiter=limiter)
    dx = 1.0 / shape[2]
    for d in range(D):
        dt = 0.1 * dx
        ref, ref_dt, _ = oracle_sweep(fm._h.desc, cons, dt, dx, d)
        assert np.all(np.isfinite(ref))
        t_in = torch.from_numpy(cons).to(cuda)
        t_out = torch.empty_like(t_in)
        sdt = torch.empty(1, dtype=torch.float64, device=cuda)
        fvs.split_sweep(fm, t_in, t_out, dt, dx, d, sdt)
        torch.cuda.synchronize()
        got = t_out.cpu().numpy()
        # equal, zeros of either sign
        differ = np.argwhere(got != ref)
        first = tuple(differ[0]) if len(differ) else None
        assert first is None, (f"direction {d}: {len(differ)} values, the first at {first}: "
                               f"{float(got[first]).hex()} not {float(ref[first]).hex()}")
        assert sdt.item() == ref_dt
