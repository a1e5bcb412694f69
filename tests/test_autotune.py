"""The FFT plan sweep without a device: which knobs it times."""
import itertools

import pytest


@pytest.mark.parametrize("size,swept", [
    ((160, 192, 144), set()),                    # two radices on every axis
    ((256, 128, 64), set()),                     # kernels of their own
    ((181, 217, 31), set()),                     # dense products
    ((343, 96, 96), {"fft_order", "x_rt"}),      # 7^3: no two radices up to 32
    ((96, 514, 96), {"fft_order", "y_tx"}),      # 2 * 257, past the dense lengths: chirp-z
    ((96, 96, 640), {"fft_order", "z_tx"}),      # two radices only up to 424 along z
    ((1, 96, 96), {"x_rt"}),
])
def test_tune_fft_times_only_plans_that_differ(monkeypatch, size, swept):
    """A knob that no axis's plan reads is not timed and stays at its default, however the
    clock runs (here every timing is faster than the one before)."""
    from atlaswerks_amd import autotune, fluid
    made = []

    class Op:
        def __init__(self, g):
            made.append({k: autotune.get_knob(k) for k in autotune.PLAN_KNOBS})

        def ApplyInverseOperator(self, f):
            pass

    clock = (0.9 ** k for k in itertools.count())
    monkeypatch.setattr(fluid, "DiffOperGPU", Op)
    monkeypatch.setattr(autotune, "_time", lambda fn, reps: next(clock))
    saved = {k: autotune.get_knob(k) for k in autotune.PLAN_KNOBS}
    monkeypatch.setattr(autotune.torch, "randn", lambda *a, **k: None)
    try:
        for k in autotune.PLAN_KNOBS:
            autotune.set_knob(k, 0)
        chosen, timings = autotune.tune_fft(size, device="cpu")
        assert {k for k, t in timings.items() if t} == swept
        assert {k: autotune.get_knob(k) for k in chosen} == chosen
        assert all(chosen[k] == 0 for k in autotune.PLAN_KNOBS if k not in swept)
        assert all(chosen[k] == autotune.PLAN_KNOBS[k][-1] for k in swept)
        assert set(chosen) == set(timings) == set(autotune.PLAN_KNOBS)
        assert bool(made) == bool(swept)
    finally:
        for k, v in saved.items():
            autotune.set_knob(k, v)
