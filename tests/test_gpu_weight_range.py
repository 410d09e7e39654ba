"""The quotients of the WENO weights and of the characteristic basis leave out
the operand scaling of the general division.  One right-hand side near the ends
of the range where that is exact -- fluxes of some 1e75, whose smoothness
indicators squared come near the largest FP64 number, numerators down to some
1e-280, and exact zeros -- equals the oracle's, which divides, bit for bit: the
density, and with it every flux, is scaled by `scale`."""
import numpy as np
import pytest

import pyoracle
from ocfd import cases, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,split,char", [("WENO5", 2, 0), ("WENO7", 2, 0), ("WENO5", 1, 1), ("WENO7", 2, 1)])
@pytest.mark.parametrize("scale", [1e74, 1e40, 1e-100, 1e-285])
@pytest.mark.parametrize("still", [False, True])
def test_scaled_density(scheme, split, char, scale, still):
    case = cases.random_case(shape=(9, 11, 14), seed=90, scheme=scheme, split=split, char=char, jump=0.4)
    case.cfg = case.cfg.replace(if_viscous=0)
    case.prims[0] = case.prims[0] * scale
    if still:  # no flow along z in half of the block: numerators that are exactly zero
        case.prims[3][:, :, :7] = 0.0
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1)
    du = []
    for b in (native.setup_block(native.Block(case.cfg), case, use_uniform=True),
              pyoracle.setup_oracle(case)):
        b.exchange_primitives()
        (b.du_inviscous_character if char else b.du_inviscous)()
        du.append(b.download_du())
    assert np.isfinite(du[1]).all()
    bad = du[0] != du[1]
    assert int(np.count_nonzero(bad)) == 0, "%d values, first %r" % (
        np.count_nonzero(bad), list(zip(du[0][bad], du[1][bad]))[:3])
