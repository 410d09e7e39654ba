"""Statistics or a halo fill in the middle of a fused stage: they fill the
halos of the new u, v, w; the end of the stage still gives them back as the
stage began with, like every other stage."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("call", ["ana_box", "exchange_primitives"])
def test_inside_a_stage(precision, call):
    case = cases.random_case(shape=(16, 16, 32), seed=88, scheme="WENO5")
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1, precision=precision)
    out = []
    for filled in (False, True):
        with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
            b.set_stage_fusion(True)
            b.profile_enable(True)
            b.exchange_primitives()
            b.du_inviscous()
            b.du_viscous()
            b.save_fn()
            b.time_adv_rk3(1)
            fused = "stage_update_fused" in b.profile_read()
            if filled:
                getattr(b, call)()
            b.comput_duvwt()
            out.append(b.download_primitives())
    assert fused == bool(precision)
    for q, (a, b) in enumerate(zip(*out)):
        # (d always, and u, v, w without the fused update, have one buffer, which the call itself fills)
        if q == 0 or q == 4 or not fused:
            a, b = a[4:-4, 4:-4, 4:-4], b[4:-4, 4:-4, 4:-4]
        assert np.array_equal(a, b), q
