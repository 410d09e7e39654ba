"""The right-hand side of a batch box that has stepped alone, whose whole
steps keep it in three parts: a batch call that advances no step leaves it as
it is, one that does replaces it."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_du_after_batch_steps(precision):
    case = cases.random_case(shape=(16, 16, 32), seed=83, scheme="WENO5")
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1, precision=precision)
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        b.step(1)
        want = b.download_du()
        b.step(1)
        want2, f2 = b.download_du(), b.download_f()
    with native.Batch([case.cfg, case.cfg]) as bt:
        for i in range(2):
            native.setup_block(bt.box(i), case, use_uniform=True)
        bt.box(1).step(1)
        bt.step(0)
        assert np.array_equal(bt.box(1).download_du(), want)
        bt.step(1)
        assert np.array_equal(bt.box(1).download_f(), f2)
        assert np.array_equal(bt.box(1).download_du(), want2)
