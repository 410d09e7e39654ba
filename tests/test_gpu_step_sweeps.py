"""Whole steps of blocks whose sweeps run in their own launches (more than
600 000 cells): two steps, replayed from a graph, equal the steps composed of
the per-routine calls bit for bit: the x-y march and the z march, tuned tiles
and the default ones, halos filled for both buffers."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def _case(kw):
    kw = dict(kw)
    case = cases.random_case(shape=(90, 130, 192), seed=89, dt=1e-4, **kw)
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1)
    return case


@pytest.mark.parametrize("kw,tiles,names", [
    (dict(scheme="HYBRID", split=2, char=1, jump=0.3, hybrid=(0.002, 0.02)), (0, 0, 3),
     {"inviscid_char_xy", "inviscid_char_z"}),
    (dict(scheme="WENO7", split=2, char=1), (1, 2, 2), {"inviscid_char_x", "inviscid_char_y", "inviscid_char_z"}),
    (dict(scheme="WENO5", split=1, char=0), (0, 0, 0), {"inviscid_x", "inviscid_y", "inviscid_z"}),
], ids=["hybrid", "WENO7char", "WENO5"])
def test_step_against_routines(kw, tiles, names):
    case = _case(kw)
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        b.set_sweep_tiles(tiles)
        b.step(2)
        got = [b.download_f()] + b.download_primitives()
        b.profile_enable(True)
        b.step(1)
        assert {n for n in b.profile_read() if n.startswith("inviscid")} == names
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        b.step_by_routines(2)
        ref = [b.download_f()] + b.download_primitives()
    for a, r in zip(got, ref):
        assert np.isfinite(r).all()
        assert int(np.count_nonzero(a != r)) == 0
