"""Which small blocks run their three sweeps in one launch: projecting schemes
on a uniform grid with one closed axis, whose two periodic sweeps are faster in
their own launches, only below 300 000 cells in FP64.  Steps are the same bits
either way."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def _step(case, shapes):
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        b.set_sweep_tiles(shapes)
        b.profile_enable(True)
        b.step(1)
        names = {n for n in b.profile_read() if n.startswith("inviscid")}
        return names, b.download_f()


# (nz, ny, nx)
@pytest.mark.parametrize("shape,per,scheme,char,precision,joined", [
    ((80, 80, 80), (1, 0, 1), "WENO7", 1, 0, False),
    ((48, 100, 120), (0, 1, 1), "WENO5", 1, 0, False),
    ((80, 80, 80), (1, 0, 1), "WENO7", 1, 1, True),
    ((64, 64, 64), (1, 0, 1), "WENO7", 1, 0, True),
    ((80, 80, 80), (1, 0, 1), "WENO7", 0, 0, True),
    ((80, 80, 80), (1, 0, 0), "WENO7", 1, 0, True),
    ((80, 80, 80), (1, 1, 1), "WENO7", 1, 0, True),
])
def test_rule(shape, per, scheme, char, precision, joined):
    case = cases.random_case(shape=shape, seed=92, scheme=scheme, split=2, char=char, iperiodic=per, dt=1e-7)
    case.uniform_metrics = cases.uniform_box_metrics(*shape[::-1])
    case.cfg = case.cfg.replace(metric_mode=1, precision=precision)
    names, f = _step(case, [0, 0, 0])
    assert (names == {"inviscid_xyz"}) == joined
    assert np.isfinite(f).all()
    # a shape for an axis: the sweeps one by one
    one, ref = _step(case, [1, 0, 0])
    assert len(one) == 3
    assert np.array_equal(f, ref)
