"""The fused MUSCL-Hancock sweeps over the exact-Godunov base
(GodunovSweepX / GodunovSweepPencil with half-step states) against the
oracle's level driver: patches narrower than a stencil, widths around the X
sweep's 60-slot chunks and 64-lane waves, lengths around the pencils'
segments and the CFL pass's (one to four cells here), every limiter, both splittings, strong waves (whose CFL checks need
solved faces) and restarts; graphs and eager launches give the same bits.
Bar: 1e-12 per cell and 1e-13 for dt (tolerances.py), the exact solver's."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from fields import rough_field
from tolerances import tolerance_ratio

import finitevolumesolver_amd as fvs

pytestmark = pytest.mark.gpu


def _run(cuda, cons, shape, limiter, split, cfl, steps, graphs=True):
    import torch
    dim = len(shape)
    dx = tuple(1.0 / max(shape) for _ in shape)
    fm = fvs.FluxMethod(fvs.PerfectGas(dim=dim), base="Godunov", reconstruction="MusclHancock",
                        limiter=limiter)
    lvl = fvs.SinglePatchLevel(fm, shape, dx, splitting=split, cfl=cfl)
    lvl.set_graphs(graphs)
    lvl.set_state(torch.from_numpy(cons).to(cuda))
    done, fails, dts = lvl.advance(steps, batch=steps, return_dts=True)
    ref = O.level_run(fm._h.desc, cons, dx, steps,
                      splitting=O.L.SPLIT_STRANG if split == "Strang" else O.L.SPLIT_GODUNOV,
                      cfl=cfl)
    return done, fails, np.array(dts), lvl.get_state().cpu().numpy(), ref


@pytest.mark.parametrize("shape,limiter,split,cfl", [
    ((1, 1), "MinMod", "Godunov", 0.8),
    ((2, 3), "VanLeer", "Strang", 0.8),
    ((58, 33), "NoLimiter", "Godunov", 0.4),
    ((63, 31), "NoGradient", "Strang", 0.8),
    ((129, 64), "MinMod", "Strang", 0.8),
    ((70, 1501), "MinMod", "Godunov", 0.8),
    ((310, 1203), "VanLeer", "Godunov", 0.8),
    ((3, 1, 2), "MinMod", "Godunov", 0.8),
    ((31, 17, 5), "VanLeer", "Strang", 0.8),
    ((61, 6, 35), "NoLimiter", "Godunov", 0.4),
    ((20, 18, 22), "MinMod", "Strang", 1.6),
])
def test_fused_level_matches_oracle(cuda, shape, limiter, split, cfl):
    dim = len(shape)
    # unlimited slopes at jumps leave no gas: smooth data for NoLimiter
    cons = rough_field(((1,) if dim == 2 else ()) + tuple(reversed(shape)), seed=3 + sum(shape),
                       jumps=limiter != "NoLimiter")
    done, fails, dts, got, (ref, ref_dts, ref_fails) = _run(cuda, cons, shape, limiter, split, cfl, 5)
    print(shape, limiter, split, "fails", fails, "ratio", tolerance_ratio(got, ref), flush=True)
    assert done == 5 and fails == ref_fails
    assert np.max(np.abs(dts - ref_dts) / ref_dts) <= 1e-13
    assert tolerance_ratio(got, ref) <= 1.0
    eager = _run(cuda, cons, shape, limiter, split, cfl, 5, graphs=False)
    assert np.array_equal(eager[3], got) and list(eager[2]) == list(dts)


@pytest.mark.parametrize("base,recon", [("Godunov", "MusclHancock"), ("Godunov", "None"), ("HLLEM", "MusclHancock")])
def test_captures_within_a_run(cuda, base, recon):
    """By default a level launches its first eight steps and captures the later
    ones where it meets them, inside a run: same bits as eager launches."""
    import torch
    cons = rough_field((1, 40, 50), seed=8)
    runs = []
    for eager in (False, True):
        fm = fvs.FluxMethod(fvs.PerfectGas(dim=2), base=base, reconstruction=recon)
        lvl = fvs.SinglePatchLevel(fm, (50, 40), (0.02, 0.02), cfl=0.8)
        if eager:
            lvl.set_graphs(False)
        lvl.set_state(torch.from_numpy(cons).to(cuda))
        runs.append([lvl.advance(n, batch=b, return_dts=True) + (lvl.get_state().cpu().numpy(),)
                     for n, b in ((3, 3), (11, 11), (37, 37), (5, 2))])
    for a, b in zip(*runs):
        assert a[:2] == b[:2] and a[2] == b[2] and np.array_equal(a[3], b[3])
