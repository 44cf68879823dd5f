"""Exact-Godunov faces of states that are no gas: without pressure, with a
negative one, without density, with infinities and NaNs.  The sweeps, view
fluxes and stable dts have the oracle's numbers, infinities and NaNs: its
formulas, with which the kernels' shared quotients agree only for ordinary
operands.  Bar: equal special values, 1e-12 for numbers (the exact solver's)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from sweep_ref import oracle_sweep, padded_complete

import finitevolumesolver_amd as fvs

pytestmark = pytest.mark.gpu

INF, NAN = np.inf, np.nan


def _gas(rho, u, v, p):
    return [rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)]


KINDS = [_gas(1.0, 0.3, -0.2, 1.0), _gas(0.2, -1.0, 0.5, 40.0), _gas(1e-9, 0.1, 0.0, 1e-9),
         [1, 0, 0, 0], [1, 0.5, 0, 0.125], [1, -0.5, 0, 0.125],  # no pressure
         [1, 0.5, 0, 0.02], [2, 0.1, 0.1, -100],                 # a negative one
         [0, 0, 0, 0], [0, 1, 0, 1], [-1, 0.2, 0.1, 2],          # no density
         [1, 0.1, 0.2, NAN], [1, NAN, 0, 1], [NAN, 0.1, 0.1, 1], [1, INF, 0, 1], [1, 0.1, INF, 1],
         [1, 0.1, 0.2, INF]]


def _rows():
    """(4, 1, pairs, 2): a row of two cells per pair of kinds."""
    pairs = [(a, b) for a in KINDS for b in KINDS]
    return np.ascontiguousarray(np.array(pairs, dtype=float).transpose(2, 0, 1)[:, None])


def _assert_same(got, ref, what):
    special = ~np.isfinite(ref)
    assert np.array_equal(got[special], ref[special], equal_nan=True), what
    assert np.all(np.isfinite(got[~special])), what
    g, r = got[~special], ref[~special]
    assert np.all(np.abs(g - r) <= 1e-12 * np.maximum(1.0, np.abs(r))), what


@pytest.mark.parametrize("direction", [0, 1])
def test_first_order_sweep(cuda, direction):
    import torch
    fm = fvs.FluxMethod(fvs.PerfectGas(dim=2), base="Godunov", reconstruction="None")
    cons = _rows()
    if direction == 1:
        cons = np.ascontiguousarray(cons[[0, 2, 1, 3]].transpose(0, 1, 3, 2))
    t_out = torch.empty_like(torch.from_numpy(cons).to(cuda))
    sdt = torch.empty(1, dtype=torch.float64, device=cuda)
    with np.errstate(all="ignore"):
        fvs.split_sweep(fm, torch.from_numpy(cons).to(cuda), t_out, 1e-3, 1.0, direction, sdt)
        ref, _, _ = oracle_sweep(fm._h.desc, cons, 1e-3, 1.0, direction)
        _assert_same(t_out.cpu().numpy(), ref, "states")
        for k in range(cons.shape[2 + (direction == 1)]):
            at = (slice(None), slice(None)) + ((slice(k, k + 1),) if direction == 0 else (slice(None), slice(k, k + 1)))
            row = np.ascontiguousarray(cons[at])
            t_in = torch.from_numpy(row).to(cuda)
            fvs.split_sweep(fm, t_in, torch.empty_like(t_in), 1e-3, 1.0, direction, sdt)
            _, dt, _ = oracle_sweep(fm._h.desc, row, 1e-3, 1.0, direction)
            _assert_same(np.array([sdt.item()]), np.array([dt]), f"dt of pair {k}")


@pytest.mark.parametrize("recon", ["None", "MusclHancock"])
def test_view_fluxes(cuda, recon):
    import torch
    fm = fvs.FluxMethod(fvs.PerfectGas(dim=2), base="Godunov", reconstruction=recon)
    cons = _rows()
    gw = 2 * fm.GetStencilWidth()
    with np.errstate(all="ignore"):
        comp, g = padded_complete(cons, 2, gw)
    lo = (-g[0], -g[1], -g[2])
    shape = (4, 1, cons.shape[2], 3)
    t_flux = torch.zeros(shape, dtype=torch.float64, device=cuda)
    full = fvs.PatchView(torch.from_numpy(comp).to(cuda), lo)
    fm.ComputeNumericFluxes(fvs.PatchView(t_flux, (0, 0, 0)), full, 1e-3, 1.0, 0)
    ref = np.zeros(shape)
    fv, sv = O.host_view(ref), O.host_view(comp, lo)
    assert O.load().oracle_numeric_fluxes(C.byref(fm._h.desc), C.byref(fv), C.byref(sv), 1e-3, 1.0, 0) == 0
    _assert_same(t_flux.cpu().numpy(), ref, "fluxes")
