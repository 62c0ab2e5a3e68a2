"""The row solves' pivot tables where memory has room for two or one only
(csrc/vv_rlines.h): the same steps bit for bit, with the second stream (two
tables: one of them filled again for two of the operators) and without (one),
and single solves of every operator; a run is made and given back each time."""
import ctypes

import numpy as np
import pytest

import test_gpu_3d as T3
import test_gpu_sector as TS
import test_gpu_tank as TT

pytestmark = pytest.mark.gpu

MAKE = {
    "annulus": lambda: T3._gpu(34, 19, 16),
    "hor": lambda: T3._gpu(9, 7, 12, model=1),
    "sector": lambda: TS._gpu(34, 19, 18),
    "tank": lambda: TT._pair(34, 19, 16, seed=1)[0],
}


def _solve(run, which):
    if hasattr(run, "poisson1"):
        getattr(run, f"poisson{which}")()
    else:
        run.poisson(which)


@pytest.mark.parametrize("prog", list(MAKE))
def test_tables(prog, monkeypatch):
    fields = {}
    for tables in ("3", "2", "1"):
        print(f"[gpu] row tables {prog} {tables}", flush=True)
        monkeypatch.setenv("VV_RTABLES", tables)
        run = MAKE[prog]()
        rng = np.random.default_rng(7)
        for n in TT.NAMES:
            run.put(n, 1e-3 * rng.standard_normal(run.get(n).shape))
        run.step(3)
        for which in (3, 1, 2, 3):
            _solve(run, which)
        run.step(2)
        fields[tables] = {n: run.get(n) for n in TT.NAMES}
        run.close()
    for n, a in fields["3"].items():
        assert np.all(np.isfinite(a)), n
        assert np.array_equal(a, fields["2"][n]) and np.array_equal(a, fields["1"][n]), n


def test_memory(monkeypatch):
    """Two tables and both sets of work arrays fit where three tables do not:
    one table less is taken; one table leaves out the second set too."""
    from codesthesis_dir_amd.band import hip
    from codesthesis_dir_amd.sector import Sector, SectorConfig
    taken = {}

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    for tables in ("3", "2", "1"):
        print(f"[gpu] row tables memory {tables}", flush=True)
        monkeypatch.setenv("VV_RTABLES", tables)
        before = free()
        run = Sector(SectorConfig(nr=128, nz=128, np=128, dt=1e-5, Ra=1e4, Re=10.0, Ptl=1.0, Gr=0.0))
        taken[tables] = before - free()
        run.close()
    table, work = 8 * 127 * 128 * 128, 8 * 128 ** 3
    assert taken["3"] - taken["2"] >= 0.8 * table
    assert taken["2"] - taken["1"] >= 0.8 * (table + 2 * work)
