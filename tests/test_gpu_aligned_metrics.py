"""Projecting sweeps on uniform grids: metric vectors along their own
coordinate take the reduced characteristic basis, all others the general one.
Both equal the same metrics given as fields (the general path) bit for bit."""
import numpy as np
import pytest

from ocfd import cases, native
from ocfd.config import METRIC_FIELD, METRIC_UNIFORM

pytestmark = pytest.mark.gpu

SKEWS = {
    "aligned": np.zeros(9),
    "skewed x": np.array([0, 0.2, -0.1, 0, 0, 0, 0, 0, 0]),
    "skewed": np.array([0, 0.1, 0.05, -0.2, 0, 0.1, 0.3, 0.1, 0]),
    "reversed y": np.array([0, 0, 0, 0, -2.0, 0, 0, 0, 0]),
}


@pytest.mark.parametrize("skew", SKEWS)
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme,split", [("WENO5", 1), ("WENO7", 2), ("OMP6", 2), ("UD7L", 1)])
def test_characteristic_sweeps(skew, precision, scheme, split):
    case = cases.random_case(shape=(18, 21, 70), seed=31, scheme=scheme, split=split, char=1, jump=0.3)
    cfg = case.cfg.replace(precision=precision)
    m = cases.uniform_box_metrics(cfg.nx, cfg.ny, cfg.nz)
    m[:9] += SKEWS[skew] * m[[0, 0, 0, 4, 4, 4, 8, 8, 8]]
    full = np.concatenate([m, m[:9] / m[9]])

    def du(mode, shapes):
        with native.Block(cfg.replace(metric_mode=mode)) as b:
            if mode == METRIC_UNIFORM:
                b.set_uniform_metrics(m)
                b.set_sweep_tiles(shapes)
            else:
                b.upload_metrics([np.full(cfg.halo_shape, v) for v in full])
            b.upload_primitives(case.halo_prims())
            b.exchange_primitives()
            b.du_inviscous_character()
            return b.download_du()

    ref = du(METRIC_FIELD, None)
    assert np.isfinite(ref).all()
    for shapes in ((0, 0, 0), (1, 1, 1), (2, 2, 2)):
        assert int(np.count_nonzero(du(METRIC_UNIFORM, shapes) != ref)) == 0, shapes
