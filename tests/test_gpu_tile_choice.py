"""Tile shapes a caller sets are the ones that run: a block whose sweeps would
be joined in one launch (the three of a small block, x and y of a hybrid one)
runs the axes it set one by one; without a choice they are joined.  Results
are the same bits."""
import numpy as np
import pytest

from ocfd import cases, native

pytestmark = pytest.mark.gpu


def _step(case, shapes):
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        if shapes is not None:
            b.set_sweep_tiles(shapes)
            assert b.get_sweep_tiles() == list(shapes)
        b.profile_enable(True)
        b.step(1)
        names = {n for n in b.profile_read() if n.startswith("inviscid")}
        b.profile_enable(False)
        b.step(2)  # replayed from a graph
        return names, b.download_f()


def _uniform(**kw):
    case = cases.random_case(dt=1e-4, **kw)
    case.uniform_metrics = cases.uniform_box_metrics(case.cfg.nx, case.cfg.ny, case.cfg.nz)
    case.cfg = case.cfg.replace(metric_mode=1)
    return case


@pytest.mark.parametrize("scheme,char", [("WENO5", 0), ("WENO7", 1)])
def test_small_block(scheme, char):
    case = _uniform(shape=(20, 28, 40), seed=85, scheme=scheme, char=char)
    one = {"inviscid_char_" + a if char else "inviscid_" + a for a in "xyz"}
    names, f = _step(case, None)
    assert names == {"inviscid_xyz"}
    for shapes, want in (((0, 0, 0), {"inviscid_xyz"}), ((1, 0, 0), one), ((0, 2, 0), one), ((1, 2, 2), one),
                         ((0, 0, 1), one)):
        names, got = _step(case, shapes)
        assert names == want, (shapes, names)
        assert np.array_equal(got, f), shapes


def test_hybrid_march():
    # (nz, ny, nx): the march takes x and y of this block
    case = _uniform(shape=(90, 130, 192), seed=86, scheme="HYBRID", split=2, char=1, jump=0.3, hybrid=(0.002, 0.02))
    xy, one = {"inviscid_char_xy", "inviscid_char_z"}, {"inviscid_char_" + a for a in "xyz"}
    names, f = _step(case, None)
    assert names == xy
    for shapes, want in (((0, 0, 3), xy), ((1, 0, 0), one), ((0, 4, 4), one)):
        names, got = _step(case, shapes)
        assert names == want, (shapes, names)
        assert np.array_equal(got, f), shapes


@pytest.mark.parametrize("shape", [(20, 28, 40), (90, 130, 192)])
def test_autotune(shape):
    """The tuner's answer is what runs, also when it is set again later."""
    case = _uniform(shape=shape, seed=87, scheme="HYBRID", split=2, char=1, jump=0.3, hybrid=(0.002, 0.02))
    names, f = _step(case, None)
    with native.setup_block(native.Block(case.cfg), case, use_uniform=True) as b:
        shapes = b.autotune(reps=2)
        assert b.get_sweep_tiles() == shapes
        b.profile_enable(True)
        b.step(1)
        got = {n for n in b.profile_read() if n.startswith("inviscid")}
        if not any(shapes[:2]):
            assert got == names
        if names == {"inviscid_xyz"}:
            assert shapes == [0, 0, 0]
        b.profile_enable(False)
        b.step(2)
        assert np.array_equal(b.download_f(), f), shapes
    again, f2 = _step(case, shapes)
    assert again == got and np.array_equal(f2, f)
