"""The chunked compact lines (csrc/vv_lines.h) against the oracle, bit for
bit, where the split can go wrong: line lengths around the head, whole blocks
and one or more blocks per lane; noise and constant slopes, whose chunks meet
within the warm-up, and a single disturbance in zeros, whose chunks do not and
are run again."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _fields(kind, nr, np_, ld, seed):
    rng = np.random.default_rng(seed)
    k, i = np.meshgrid(np.arange(np_ + 1), np.arange(ld), indexing="ij")
    if kind == "random":
        C, th = 50 * rng.standard_normal((np_ + 1, ld)), rng.uniform(0, 1, (np_ + 1, ld))
    elif kind == "spot":        # zeros but for one point of each
        C, th = np.zeros((np_ + 1, ld)), np.zeros((np_ + 1, ld))
        C[np_ // 3, nr // 4 + 1], th[np_ // 2, nr // 2 + 1] = 3.7, 0.61
    else:                       # constant slopes, exactly representable
        C, th = i / 1024.0 + 0 * k, (3 * i + k) / 4096.0
    return {"C": C, "Cp": 0.5 * C, "th": th, "thp": th}


@pytest.mark.parametrize("kind", ["random", "spot", "slope"])
@pytest.mark.parametrize("nr,np_", [(8, 8), (16, 24), (25, 26), (26, 27), (32, 64), (66, 66), (73, 90), (74, 91), (130, 200),
                                    (255, 129), (512, 256), (700, 333), (2048, 40), (40, 1500)])
def test_chunked_lines_bitexact(nr, np_, kind):
    from codesthesis_dir_amd import BoxConfig, PeriodicBox
    print(f"[gpu] chunked lines nr={nr} np={np_} {kind}", flush=True)
    run = O.Run(nr, np_, 1e-5, 1e5, 1.0, width=3.0)
    box = PeriodicBox(BoxConfig(nr=nr, np=np_, width=3.0, dt=1e-5, Ra=1e5))
    for n, a in _fields(kind, nr, np_, run.ld, nr * np_).items():
        run[n][...] = a
        box.put(n, a)
    rng = np.random.default_rng(3)
    for n in ("uel", "vel"):
        a = rng.standard_normal(run["C"].shape)
        run[n][...] = a
        box.put(n, a)
    O.lib().vo_cvorticity(ctypes.byref(run.p), ctypes.byref(run.f), 0)
    O.lib().vo_temperature(ctypes.byref(run.p), ctypes.byref(run.f), 0)
    box.cvorticity(False)
    box.temperature(False)
    for name, hi in (("Cn", nr), ("thn", nr + 1)):
        g, o = box.get(name)[:, 1:hi], run[name][:, 1:hi]
        # the divisions' remainders underflow for operands below 1e-290; a
        # quotient there may be one denormal step (5e-324) off
        assert np.array_equal(g[np.abs(o) >= 1e-290], o[np.abs(o) >= 1e-290]), name
        assert np.max(np.abs(g - o)) <= 5e-324, name
    box.close()
