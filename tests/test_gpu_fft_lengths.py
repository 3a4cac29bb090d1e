"""Every transform length with a compile-time engine, on each axis of a mesh,
against the oracle: rhoofr, vpsi and vofrho.  Tolerances as in the parity tests
of those routines (1e-11 absolute for rho, 1e-11 of the largest force, 1e-12 of
the largest potential; FP32 transforms 2e-6)."""
import math
import re
from pathlib import Path

import numpy as np
import pytest

import oracle
from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu

_SRC = (Path(__file__).resolve().parent.parent / "cpmd_amd" / "csrc" / "fft_device.h").read_text()
LENGTHS = sorted({int(n) for n in re.findall(r"MC_FAST_SHAPE\((\d+),", _SRC)} - {16, 18})


def _system(n, axis, dual):
    """A cell whose mesh is n along `axis` and 16 or 18 along the others; with dual 3
    the wavefunction sphere passes a quarter of the mesh (no band to prune)."""
    ecut = 12.0
    edge = [(m - 0.6) * math.pi / math.sqrt(dual * ecut) for m in (16, 18, 16)]
    edge[axis] = (n - 0.6) * math.pi / math.sqrt(dual * ecut)
    nr = [16, 18, 16]
    nr[axis] = n
    cell = S.Cell(alat=edge[0], avec=np.diag(edge).astype(float), ecut=ecut, dual=dual, nr=tuple(nr))
    gs = S.gvectors(cell)
    tau = np.random.default_rng(n).uniform(0.0, 1.0, (2, 3)) * np.array(edge)
    return S.SyntheticSystem(cell=cell, gset=gs, tau=tau, nstate=3, f=np.array([2.0, 1.0, 0.5]))


@pytest.mark.parametrize("n", LENGTHS)
def test_length(gpu, n):
    for axis in range(3):
        for dual in (4.0, 3.0):
            sysm = _system(n, axis, dual)
            assert sysm.cell.nr[axis] == n
            gs, f = sysm.gset, sysm.f
            ctx = ops.Context(sysm.cell, gs)
            L = oracle.Layout(sysm.cell, gs)
            c = S.initial_coefficients(sysm, seed=n)
            v = S.real_space_potential(sysm, seed=n)
            rho_o, ek_o, cg_o, cr_o = oracle.rhoofr(L, c, f)
            c2_o = oracle.vpsi(L, c, np.zeros_like(c), f, v)
            for mode in ("fp64", "fp32"):
                ctx.set_precision(mode)
                rho, ek, cg, cr = ctx.rhoofr(c, f)
                c2 = ctx.vpsi(c, np.zeros_like(c), f, v)
                if mode == "fp64":
                    assert np.abs(rho - rho_o).max() < 1e-11
                    assert ek == pytest.approx(ek_o, rel=1e-12) and cr == pytest.approx(cr_o, rel=1e-12)
                    assert np.abs(c2 - c2_o).max() < 1e-11 * np.abs(c2_o).max()
                else:
                    assert np.abs(rho - rho_o).max() < 2e-6 * np.abs(rho_o).max()
                    assert np.abs(c2 - c2_o).max() < 2e-6 * np.abs(c2_o).max()
            if dual == 4.0:
                zv, rg, vps, rhops = S.local_pp_set(sysm, gs.hg)
                inyh, gk = gs.miller + np.array([m // 2 + 1 for m in sysm.cell.nr]), gs.miller @ sysm.cell.bvec
                ctx.set_density_gset(inyh, gs.hg, gk)
                ctx.set_local_pp([2], zv, rg, vps, rhops)
                ctx.set_ions(sysm.tau, sysm.cell.avec)
                pot, en, _ = ctx.vofrho(rho_o)
                frac = sysm.tau @ np.linalg.inv(sysm.cell.avec)
                pot_o, en_o, _, _ = oracle.vofrho(L, inyh, gs.hg, gk, [2], vps, rhops, frac, rho_o)
                assert np.abs(pot - pot_o).max() < 1e-12 * np.abs(pot_o).max()
                assert en["ehep"] == pytest.approx(en_o["ehep"], rel=1e-11)
