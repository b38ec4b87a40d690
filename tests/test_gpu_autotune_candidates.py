"""Which launch shapes the autotuner times on FP32 grids that 64 columns divide: beside the role-split shape
the delay-line ones of 64 x 4 columns that give some CU its two workgroups (192^3 runs fastest with chunks of
64 planes, 432 workgroups), and no shape of one workgroup per CU or fewer."""
import re

import numpy as np
import pytest

from astaroth_amd import astaroth as ac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,chunks", [((192, 192, 192), {32, 64}), ((128, 128, 160), {32}), ((128, 128, 128), set()),
                                      ((192, 64, 384), {32, 64})])
def test_delay_line_shapes_timed(n, chunks, monkeypatch, capfd, require_gpu):
    print(f"case autotune candidates n={n}", flush=True)
    monkeypatch.setenv("ASTAROTH_AUTOTUNE_VERBOSE", "1")
    monkeypatch.delenv("ASTAROTH_AUTOTUNE_CACHE", raising=False)
    lib = ac.load("fp32")
    info = lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3,
                      AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True)
    with ac.Device(lib, info) as dev:
        dev.step(lib.np_real(1e-3))
        dev.sync()
    timed = re.findall(r"ish (\d+)x(\d+)x(\d+) kb=0 kind=(-?\d+)", capfd.readouterr().err)
    shapes = {tuple(int(v) for v in t) for t in timed}
    assert {s[2] for s in shapes if s[3] == 0} == chunks
    assert all(s[:2] == (64, 4) for s in shapes if s[3] == 0)
