"""The autotuner's choice of a launch knob (no GPU: the times are given)."""
from pyxtal_ff_amd import _native, autotune


def test_default_stays_unless_clearly_beaten():
    # five launch shapes that are the same kernel, apart from noise
    same = {4: 29.2e-3, 8: 29.0e-3, 16: 29.3e-3, 32: 28.9e-3, 64: 29.1e-3}
    assert autotune._pick(same, 16, same.get) == 16
    assert autotune._pick({0: 66.0, 48: 65.0, 112: 80.0}, 0, None) == 0
    # the default's one median an outlier: both timed again in turn
    looked = []

    def again(v):
        looked.append(v)
        return same[v]
    assert autotune._pick(dict(same) | {16: 31.5e-3}, 16, again) == 16
    assert looked == [32, 16] * 3
    # a real difference is taken
    real = {4: 30.0, 8: 29.0, 16: 40.0}
    assert autotune._pick(real, 16, real.get) == 8


def test_defaults_are_the_library_s():
    L = _native.load()
    assert {k: L.pxff_tune_get(k) for k in autotune.DEFAULTS} == autotune.DEFAULTS
    assert all(autotune.DEFAULTS[k] in v for k, v in autotune.CANDIDATES.items())
