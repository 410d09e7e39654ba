"""Halos of the two buffers of T (u, v, w): whole steps and fused stages of
periodic blocks fill both at once, the per-routine calls copy them after each
stage.  All halo'd primitives are alike bit for bit -- in the mixed form, whose
per-routine kernels round du differently, among the fused forms -- and edges
and corners keep what was uploaded."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def prims(case, how, nsteps, halos):
    with native.Block(case.cfg) as b:
        b.set_uniform_metrics(case.uniform_metrics)
        b.upload_primitives(halos)
        b.bc()
        if how == "step":
            b.step(nsteps)
        elif how == "mixed use":
            b.set_stage_fusion(True)
            b.step_by_routines(1)
            b.step(nsteps - 1)
        else:
            b.set_stage_fusion(how == "fused routines")
            b.step_by_routines(nsteps)
        return b.download_primitives()


@pytest.mark.parametrize("shape", [(16, 16, 32), (17, 19, 33)])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nsteps", [1, 2])
def test_halos(shape, precision, nsteps):
    case = cases.random_case(shape=shape, seed=77, scheme="WENO5")
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1, precision=precision)
    rng = np.random.default_rng(3)
    halos = []
    for a in case.prims:
        h = rng.uniform(0.5, 1.5, size=case.cfg.halo_shape)
        h[4:-4, 4:-4, 4:-4] = a
        halos.append(h)
    ref = prims(case, "routines" if precision == 0 else "step", nsteps, halos)
    inside = [np.zeros(n, bool) for n in ref[0].shape]
    for m in inside:
        m[4:-4] = True
    edge = sum(m.reshape([-1 if q == a else 1 for q in range(3)]).astype(int) for a, m in enumerate(inside)) < 2
    for h, r in zip(halos, ref):
        assert np.array_equal((h.astype(np.float32) if precision else h)[edge], r[edge])
    for how in ("step", "fused routines", "mixed use"):
        for a, r in zip(prims(case, how, nsteps, halos), ref):
            assert int(np.count_nonzero(a != r)) == 0, how
    with native.Batch([case.cfg, case.cfg]) as bt:
        for i in range(2):
            bt.box(i).set_uniform_metrics(case.uniform_metrics)
            bt.box(i).upload_primitives(halos)
            bt.box(i).bc()
        bt.step(nsteps)
        for a, r in zip(bt.box(1).download_primitives(), ref):
            assert int(np.count_nonzero(a != r)) == 0
