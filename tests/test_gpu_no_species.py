"""Projectors of no species: any nhxs goes, it sizes nothing."""
import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nhxs", [0, 1, 40000])
def test_no_species(gpu, nhxs):
    sysm = S.make_system(9.0, 8, 30.0, nstate=1)
    ctx = ops.Context(sysm.cell, sysm.gset)
    ctx.set_projectors([], nhxs, [], np.zeros((nhxs, 0), np.int32), np.zeros((nhxs, nhxs, 0)),
                       np.zeros((sysm.gset.ngw, nhxs, 0)))
    assert ctx.nat == 0 and ctx.nhxs == nhxs
