"""The x and y sweeps of the hybrid scheme in one march (blocks it fills the
chip with) against the two sweeps one after the other, bit for bit: columns
and rows that are no multiple of a wavefront, of a group of 8 rows or of a
segment, and WENO faces at the edges of a row."""
import numpy as np
import pytest

from ocfd import cases, native
from ocfd.config import METRIC_FIELD, METRIC_UNIFORM

pytestmark = pytest.mark.gpu


def _du(case, mode, m):
    with native.Block(case.cfg.replace(metric_mode=mode)) as b:
        if mode == METRIC_UNIFORM:
            b.set_uniform_metrics(m)
        else:
            full = np.concatenate([m, m[:9] / m[9]])
            b.upload_metrics([np.full(case.cfg.halo_shape, v) for v in full])
        b.upload_primitives(case.halo_prims())
        b.exchange_primitives()
        b.comput_rhybrid()
        b.profile_enable(True)
        b.du_inviscous_character()
        names = set(b.profile_read())
        return b.download_du(), names


# (nz, ny, nx)
@pytest.mark.parametrize("shape", [(90, 130, 192), (128, 119, 186), (224, 47, 254), (70, 250, 128)])
@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("precision", [0, 1])
def test_march(shape, split, precision):
    case = cases.random_case(shape=shape, seed=61, scheme="HYBRID", split=split, char=1, jump=0.3,
                             hybrid=(0.002, 0.02))
    case.cfg = case.cfg.replace(precision=precision)
    m = cases.uniform_box_metrics(*shape[::-1])
    got, names = _du(case, METRIC_UNIFORM, m)
    assert "inviscid_char_xy" in names
    ref, names = _du(case, METRIC_FIELD, m)  # the sweeps of metric fields
    assert "inviscid_char_xy" not in names
    assert np.isfinite(ref).all()
    assert int(np.count_nonzero(got != ref)) == 0
