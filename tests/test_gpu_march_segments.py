"""The k-marching viscous kernels on partial tiles and uneven segments: nx one
past a 64-wide tile, ny below and past a 4-high one, nz below, at and past a
segment.  FP64 steps equal the oracle bit for bit; the mixed form stays within
the 1e-5 it is specified to and differs (its FP32 kernels ran)."""
import numpy as np
import pytest

import pyoracle
from ocfd import cases, native
from ocfd.config import PREC_MIXED
from util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 9, 65), (67, 9, 33), (34, 13, 129)])
@pytest.mark.parametrize("vis", ["CD6", "CD8"])
@pytest.mark.parametrize("iper,grid", [((1, 1, 1), "box"), ((1, 0, 1), "curv")])
def test_partial_tiles_and_segments(shape, vis, iper, grid):
    case = cases.random_case(shape=shape, seed=sum(shape), vis=vis, iperiodic=iper, grid=grid)
    ob = pyoracle.setup_oracle(case)
    ob.step(2)
    ref = ob.download_f()
    with native.setup_block(native.Block(case.cfg), case) as b:
        b.step(2)
        f = b.download_f()
    assert int(np.count_nonzero(f != ref)) == 0
    with native.setup_block(native.Block(case.cfg.replace(precision=PREC_MIXED)), case) as b:
        b.step(2)
        err = rel_l2(b.download_f(), ref)
    assert 0 < err <= 1e-5
