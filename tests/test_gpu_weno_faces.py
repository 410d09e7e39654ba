"""The listed WENO faces of the hybrid scheme at list lengths around the
kernel's batches (64 faces, three batches per workgroup): none, a few, most
faces; all metric forms of the kernel, with and without projection, against
the oracle bit for bit (FP64)."""
import numpy as np
import pytest

import pyoracle
from ocfd import cases, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thresholds", [(1e9, 1e9), (0.05, 0.2), (1e-4, 1e-3), (-1.0, -1.0), (-1.0, 1e9)])
@pytest.mark.parametrize("char,split", [(1, 2), (0, 1)])
@pytest.mark.parametrize("form", ["uniform", "field", "walls", "skewed"])
def test_listed_faces(thresholds, char, split, form):
    kw = dict(iperiodic=(1, 0, 1), grid="curv") if form == "walls" else {}
    case = cases.random_case(shape=(9, 11, 23), seed=57, scheme="HYBRID", split=split, char=char, jump=0.5,
                             hybrid=thresholds, **kw)
    ob = pyoracle.setup_oracle(case)
    uniform = form in ("uniform", "skewed")
    if uniform:
        case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
        if form == "skewed":
            case.uniform_metrics[1] = 0.1 * case.uniform_metrics[0]
        case.cfg = case.cfg.replace(metric_mode=1)
        full = np.concatenate([case.uniform_metrics, case.uniform_metrics[:9] / case.uniform_metrics[9]])
        ob.upload_metrics([np.full(case.cfg.halo_shape, v) for v in full])
    ob.step(2)
    with native.setup_block(native.Block(case.cfg), case, use_uniform=uniform) as b:
        b.step(2)
        assert int(np.count_nonzero(b.download_f() != ob.download_f())) == 0
