"""The single-precision speed bounds of the exact-Godunov CFL pass
(QuickSpeedBelow and SpeedBelow in fvs_godunov_bound.hpp), compiled for the
host, against the CPU oracle's signal speeds, and the iteration counts its wide
class rests on: no pair is certified to stay below its own speed, Newton
converges on the wide class (pressure ratios to 1e6, parting speeds to
min(1 / (2 (gamma - 1)), 1.25) and closing speeds to 1e3 times the root of
aL^2 + aR^2) well within the iteration cap from which it is used, and the
bounds are not empty (pairs are certified at 1.05 and 2 times their speed;
cells that are no gas never)."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import oracle_lib as O

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "finitevolumesolver_amd" / "csrc"

def _pairs(n, ratio_max, wide, seed, G):
    """Complete 2D states of pairs of the class, with its corners: the largest
    pressure ratio, the largest closing and parting speeds, equal states and
    weak jumps."""
    rng = np.random.default_rng(seed)
    rhoL, rhoR = 10.0 ** rng.uniform(-3, 3, n), 10.0 ** rng.uniform(-3, 3, n)
    pmin = 10.0 ** rng.uniform(-3, 3, n)
    ratio = 10.0 ** rng.uniform(0, np.log10(ratio_max), n)
    ratio[: n // 8] = ratio_max * (1 - 1e-7)
    ratio[n // 8: n // 4] = 1.0
    swap = rng.random(n) < 0.5
    pL, pR = np.where(swap, pmin * ratio, pmin), np.where(swap, pmin, pmin * ratio)
    aL, aR = np.sqrt(G * pL / rhoL), np.sqrt(G * pR / rhoR)
    uL = rng.uniform(-2, 2, n) * np.maximum(aL, aR)
    span = (np.sqrt(aL ** 2 + aR ** 2) if wide else np.minimum(aL, aR)) * (1 - 1e-6)
    part, close = (min(0.5 / (G - 1), 1.25) * span, 1e3 * span) if wide else (span, span)
    du = rng.uniform(-1, 1, n) * span
    du = np.where(du > 0, du * np.minimum(1.0, part / span), du)
    du[4::16] = -close[4::16] * 10.0 ** rng.uniform(-3, 0, du[4::16].size)
    du[::16], du[1::16], du[2::16] = -close[::16], part[1::16], 0.0
    du[3::16] *= 1e-6
    du = np.maximum(du, -1e7)
    slow = np.maximum(aL, aR) <= 1e6  # the class's sound speeds
    rhoL, rhoR, pL, pR, uL, du = (v[slow] for v in (rhoL, rhoR, pL, pR, uL, du))
    out = []
    for rho, u, p in ((rhoL, uL, pL), (rhoR, uL + du, pR)):
        cons = np.stack([rho, rho * u, 0.3 * rho, p / (G - 1) + 0.5 * rho * (u * u + 0.09)])
        out.append(O.complete_from_cons(cons, 2, G))
    return out


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
@pytest.mark.parametrize("cap,ratio,most,G", [
    (16, 4.0, 8, 1.4), (16, 4.0, 8, 1.1), (16, 4.0, 9, 5 / 3), (16, 4.0, 9, 2.0),
    (64, 1e6, 40, 1.4), (64, 1e6, 40, 1.1), (64, 1e6, 40, 5 / 3), (64, 1e6, 40, 2.0)])
def test_bound_holds_and_newton_converges_on_its_class(tmp_path, cap, ratio, most, G):
    n = 300_000
    Lq, Rq = _pairs(n, ratio, cap >= 64, seed=cap, G=G)
    n = Lq.shape[1]
    _, _, it, conv = O.exact_middle_state(Lq, Rq, 2, 0, max_it=cap, gamma=G)
    assert np.all(conv == 1) and int(it.max()) <= most, int(it.max())
    s0, s1 = O.exact_signals(Lq, Rq, 2, 0, G)
    speed = np.maximum(np.abs(s0), np.abs(s1))
    data = tmp_path / "pairs.bin"
    np.concatenate([Lq[:4], Rq[:4], speed[None]]).astype(np.float64).tofile(data)
    exe = tmp_path / "speed_below"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", f"-I{HERE / 'host_stub'}",
                    f"-I{CSRC}", str(HERE / "host_stub" / "speed_below.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe), str(data), str(cap), repr(G)], capture_output=True, text=True).stdout
    quick, tight = [[int(v) for v in line.split()] for line in out.splitlines()]
    assert quick[0] == 0 and tight[0] == 0, out
    assert quick[2] > 0.15 * n and tight[2] > 0.3 * n and tight[1] > 0.1 * n, out
    # cells that are no gas: none is certified at any speed
    bad = np.concatenate([Lq[:4], Rq[:4], np.full((1, n), 1e30)]).astype(np.float64)
    for k in range(5):
        bad[[0, 3, 0, 3, 4][k], k::5] = [0.0, -1.0, np.nan, np.inf, -2.0][k]
    bad.tofile(data)
    out = subprocess.run([str(exe), str(data), str(cap), repr(G)], capture_output=True, text=True).stdout
    assert out.split() == ["0"] * 6, out
