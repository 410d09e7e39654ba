"""Device memory of a batch: the arrays its steps use and no others (the
y and z parts of the right-hand side belong to whole steps of a box alone)."""
import ctypes

import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def _free():
    hip = ctypes.CDLL("libamdhip64.so")
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_footprint(precision):
    n, boxes = 80, 6
    case = cases.random_case(shape=(16, 16, 32), seed=84)
    cfg = case.cfg.replace(nx=n, ny=n, nz=n, metric_mode=1, precision=precision)
    with native.Batch([cfg]):  # (code objects and the runtime's own pools)
        pass
    before = _free()
    with native.Batch([cfg] * boxes) as bt:
        used = before - _free()
        halo, plane = (n + 8) ** 3, n ** 3
        # d, u, v, w, T, T2 (and u2, v2, w2 of the fused update); f, fn, du; Ev
        need = (9 * halo * 4 if precision else 6 * halo * 8) + (3 * 5 + 12) * plane * 8
        assert used <= boxes * need * 1.1, "%.1f MB of %.1f per box" % (used / boxes / 1e6, need / 1e6)
        # a box that steps alone takes the parts then, in the sweeps' type
        before1 = _free()
        box = bt.box(2)
        box.set_uniform_metrics(cases.uniform_box_metrics(n, n, n))
        box.profile_enable(True)
        box.step(1)
        assert "inviscid_xyz" in box.profile_read()
        parts = 10 * plane * (4 if precision else 8)
        assert before1 - _free() <= parts * 1.1 + (16 << 20)


@pytest.mark.parametrize("precision", [0, 1])
def test_first_step_of_a_block_allocates_nothing_large(precision):
    """A block alone takes the parts with its state, not inside its first step."""
    n = 80
    case = cases.random_case(shape=(16, 16, 32), seed=85)
    cfg = case.cfg.replace(nx=n, ny=n, nz=n, metric_mode=1, precision=precision)
    with native.Block(cfg) as b:
        b.set_uniform_metrics(cases.uniform_box_metrics(n, n, n))
        b.upload_primitives([np.ones(cfg.halo_shape)] * 5)
        b.bc()
        b.synchronize()
        before = _free()
        b.step(1)
        assert before - _free() < 10 * n ** 3 * (4 if precision else 8) // 2
        b.profile_enable(True)
        b.step(1)
        assert "inviscid_xyz" in b.profile_read()
