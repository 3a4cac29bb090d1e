"""The Ewald real-space sum over the ways its images and partners are dealt to
threads."""
import itertools
import math

import numpy as np
import pytest
import scipy.special

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


def _ewald_sums(zv, raggio, tau, ht, iesr):
    """The sums of oracle.ewald for one species with pairwise summation (the oracle
    adds its up to millions of positive terms one by one, which loses 1e-12)."""
    nat, rc = len(tau), math.sqrt(2.0) * raggio
    fr = (tau[:, None] - tau[None]) @ np.linalg.inv(ht)
    d = (fr - np.rint(fr)) @ ht
    esr, f = [], np.zeros((nat, 3))
    for img in itertools.product(range(-iesr, iesr + 1), repeat=3):
        r = d + np.array(img) @ ht
        x = np.linalg.norm(r, axis=2)
        off = ~np.eye(nat, dtype=bool)
        on = (x <= 20.0 * rc) & (off if not any(img) else True)
        x = np.where(on, x, 1.0)
        add = np.where(on, zv * zv * scipy.special.erfc(x / rc) / x, 0.0)
        esr.append(0.5 * add.sum())
        rep = np.where(on & off, add + 2.0 * zv * zv / math.sqrt(math.pi) * np.exp(-(x / rc) ** 2) / rc, 0.0) / x ** 2
        f += (rep[:, :, None] * r).sum(axis=1)
    return math.fsum(esr), f.T


@pytest.mark.parametrize("nat,iesr", [(1, 8), (2, 0), (2, 3), (23, 1), (60, 2), (257, 1), (300, 2), (725, 1), (2100, 0)])
def test_ewald_shares(gpu, nat, iesr):
    """Few atoms share the images of a pair among threads, many have a thread for
    several partners: one of each, and odd counts between.  All terms of esr are
    positive; nat (2 iesr + 1)^3 of them per atom keep it within 1e-12, and the
    forces within 1e-11 of the largest, as in the parity test of a small cell."""
    sysm = S.make_system(9.0, 1, 12.0, nstate=1, with_density=True)
    cell, gs = sysm.cell, sysm.gset
    ctx = ops.Context(cell, gs)
    zv, rg, vps, rhops = S.local_pp_set(sysm, gs.hg)
    ctx.set_density_gset(gs.miller + np.array([m // 2 + 1 for m in cell.nr]), gs.hg, gs.miller @ cell.bvec)
    ctx.set_local_pp([nat], zv, rg, vps, rhops)
    ht = np.array([[14.0, 0.0, 0.0], [2.0, 13.0, 0.0], [1.0, -2.0, 15.0]])
    tau = np.random.default_rng(nat).uniform(0.0, 14.0, size=(nat, 3))
    ctx.set_ions(tau, ht)
    esr, _, f = ctx.ewald(iesr=iesr)
    oesr, of = _ewald_sums(zv[0], rg[0], tau, ht, iesr)
    assert esr == pytest.approx(oesr, rel=1e-12)
    assert np.abs(f - of).max() <= 1e-11 * np.abs(of).max()
