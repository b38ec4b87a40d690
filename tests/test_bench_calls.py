"""bench.py's reference_call_pattern issues the calls it names: fill, substep and swap three times a step; the
whole-step call is timed apart and reported under its own name."""
import numpy as np

import bench


class Recorder:
    """Stands for the library and its device, and notes each call."""
    np_real = np.float32

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append((name,) + a)


def test_reference_call_pattern_makes_the_separate_calls(monkeypatch):
    dev = Recorder()
    monkeypatch.setattr(bench, "make_device", lambda ac, prec, n, **kw: (dev, dev))
    out = bench.reference_call_pattern(None, 16, steps=2, warmup=1, dt=1e-3)
    dt = np.float32(1e-3)
    step = [c for s in range(3) for c in (("periodic",), ("substep", s, dt), ("swap",))]
    sync = [("sync",)]
    assert dev.calls == (sync + step + sync + sync + 2 * step + sync +  # warm-up, timed
                         sync + 2 * [("step", dt)] + sync + [("close",)])
    assert out["steps"] == 2 and out["cell_updates_per_s"] > 0
    assert "per substep" in out["calls"] and out["acDeviceIntegrateStep_cell_updates_per_s"] > 0
