"""Whole steps of small blocks: the three sweeps in one launch, each into its
own part of du, joined by the stage update.  State and right-hand side equal
the routine-by-routine steps, whose sweeps run one by one, bit for bit; in the
mixed form, whose fused update rounds otherwise than the routines, the
right-hand side is left out of the comparison with a fused step."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def _run(case, how, nsteps=2):
    with native.setup_block(native.Block(case.cfg), case, use_uniform=case.cfg.metric_mode == 1) as b:
        if how == "step":
            b.profile_enable(True)
            b.step(1)
            assert "inviscid_xyz" in b.profile_read()
            b.profile_enable(False)
            b.step(nsteps - 1)
        else:
            b.set_stage_fusion(how == "fused routines")
            b.step_by_routines(nsteps)
        return b.download_du(), b.download_f()


def _same(case, how, du=True):
    got, ref = _run(case, "step"), _run(case, how)
    assert np.isfinite(ref[1]).all()
    for a, b in list(zip(got, ref))[0 if du else 1:]:
        assert int(np.count_nonzero(a != b)) == 0


@pytest.mark.parametrize("scheme,split,char", [("WENO5", 1, 0), ("WENO7", 2, 1), ("OMP6", 1, 0), ("UD7L", 1, 1),
                                               ("HYBRID", 2, 1), ("HYBRID", 1, 0)])
@pytest.mark.parametrize("shape", [(16, 16, 32), (9, 17, 33), (21, 40, 16)])
@pytest.mark.parametrize("metrics", ["uniform", "field", "closed"])
@pytest.mark.parametrize("precision", [0, 1])
def test_euler_steps(scheme, split, char, shape, metrics, precision):
    case = cases.random_case(shape=shape, seed=57, scheme=scheme, split=split, char=char, jump=0.2,
                             grid="box" if metrics == "uniform" else "curv", dt=1e-4,
                             iperiodic=(1, 1, 1) if metrics != "closed" else (0, 1, 0))
    case.cfg = case.cfg.replace(if_viscous=0, precision=precision)
    if metrics == "uniform":
        case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
        case.cfg = case.cfg.replace(metric_mode=1)
    _same(case, "routines" if precision == 0 else "fused routines")


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(16, 16, 32), (16, 24, 64), (19, 21, 35)])
@pytest.mark.parametrize("vis", ["CD6", "CD8"])
def test_viscous_steps(shape, vis, precision):
    case = cases.random_case(shape=shape, seed=58, scheme="WENO5", split=1, vis=vis)
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1, precision=precision)
    _same(case, "fused routines", du=False)


def test_mass_force_runs_the_sweeps_one_by_one():
    case = cases.random_case(shape=(16, 16, 32), seed=59, mass_force=(0.1, -0.2, 0.3))
    with native.setup_block(native.Block(case.cfg), case, use_uniform=False) as b:
        b.profile_enable(True)
        b.step(1)
        assert "inviscid_xyz" not in b.profile_read()
