"""Device memory that one test leaves in a reference cycle is gone before the next
begins, so that tests may compare the memory in use."""
import gc

import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S
from cpmd_amd._lib import McError

pytestmark = pytest.mark.gpu


def test_leaves_a_cycle(gpu):
    sysm = S.make_system(9.0, 8, 30.0, nstate=1)
    ctx = ops.Context(sysm.cell, sysm.gset)
    d = ctx.upload(np.zeros((sysm.gset.ngw, 4), np.complex128, order="F"))
    gc.disable()   # until the next test: nothing but its set-up collects
    with pytest.raises(McError) as e:
        ctx.rgs_dev(d, 4)
    assert "positive definite" in str(e.value)


def test_memory_in_use_is_settled(gpu):
    gc.enable()
    before = ops.mem_stats()[0]
    gc.collect()
    assert ops.mem_stats()[0] == before
