"""Compact lines whose chunks do not meet within the warm-up (csrc/vv_lines.h)
and are run again from the first such lane: wall layers and single disturbed
rows at either end before a core that is constant to the last bit, which fail
forward, back or both ways from different lanes; fields below the range of the
two-operation division; against the oracles, bit for bit.  And the time of
that path beside the proven one."""
from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest

import oracle as O
import oracle_merid as OM
import oracle_tank as OT

pytestmark = pytest.mark.gpu

KINDS = ["low", "high", "layers", "tiny"]


def _field(kind, shape, seed=0):
    """low, high: one disturbed row at that end of every axis; layers: erfc
    layers at both ends; tiny: noise of 1e-300; all before a flat core."""
    if kind in ("noise", "tiny"):
        return np.random.default_rng(seed).standard_normal(shape) * (1e-300 if kind == "tiny" else 1.0)
    f = np.full(shape, 0.25)
    for d, n in enumerate(shape):
        x = np.arange(n) / (n - 1)
        if kind == "layers":
            v = np.array([math.erfc(20 * t) + 0.5 * math.erfc(20 * (1 - t)) for t in x])
        else:
            v = (np.arange(n) == (2 if kind == "low" else n - 3)) * (1.0 + d + seed / 8)
        f = f + v.reshape([-1 if q == d else 1 for q in range(len(shape))])
    return f


def _same(g, o, what):
    # a quotient below 1e-290 may be one unit (its ulp, or the denormal step
    # 5e-324) off, as its remainder underflows; the next row takes 0.27 of
    # that over, so a row is off by under 1 / (1 - 0.27) units and a rounding
    off = np.abs(g - o) / np.maximum(2.0 ** -52 * np.abs(o), 5e-324)
    assert np.all(off[np.abs(o) >= 1e-290] == 0), what
    assert np.max(off) <= 2, what


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nr,np_", [(73, 90), (74, 91), (255, 129), (512, 700), (2048, 40), (40, 1500)])
def test_plane_bitexact(nr, np_, kind):
    from codesthesis_dir_amd import BoxConfig, PeriodicBox
    print(f"[gpu] line redo nr={nr} np={np_} {kind}", flush=True)
    run = O.Run(nr, np_, 1e-5, 1e5, 1.0, width=3.0)
    box = PeriodicBox(BoxConfig(nr=nr, np=np_, width=3.0, dt=1e-5, Ra=1e5))
    for q, n in enumerate(("C", "Cp", "th", "thp", "uel", "vel")):
        a = _field(kind if q < 4 else "noise", run["C"].shape, q)
        a[0] = a[-1]
        run[n][...] = a
        box.put(n, a)
    O.lib().vo_cvorticity(ctypes.byref(run.p), ctypes.byref(run.f), 0)
    O.lib().vo_temperature(ctypes.byref(run.p), ctypes.byref(run.f), 0)
    box.cvorticity(False)
    box.temperature(False)
    for name, hi in (("Cn", nr), ("thn", nr + 1)):
        _same(box.get(name)[:, 1:hi], run[name][:, 1:hi], name)
    box.close()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nr,nz,np_", [(74, 17, 90), (9, 130, 18), (17, 9, 258), (700, 6, 6), (6, 700, 7), (18, 6, 1300)])
def test_tank_bitexact(nr, nz, np_, kind):
    from codesthesis_dir_amd.tank import Tank, TankConfig
    print(f"[gpu] tank line redo {nr}x{nz}x{np_} {kind}", flush=True)
    cfg = TankConfig(nr=nr, nz=nz, np=np_, lx=1.0, lz=0.8, ly=2.5, dt=2e-4, Re=37.0, Ptl=5.0, Gr=11.0)
    run = Tank(cfg)
    ora = OT.Tank(nr, nz, np_, dt=cfg.dt, Re=cfg.Re, Ptl=cfg.Ptl, Gr=cfg.Gr, lx=1.0, lz=0.8, ly=2.5)
    for q, n in enumerate(("A", "B", "C", "th")):
        ora[n] = a = _field(kind, ora.shape, q)
        run.put(n, a)
    run.derivatives()
    for q, o in enumerate(ora.derivatives()):
        _same(run.derivative(q), o, q)
    run.close()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nr,nz,beta", [(90, 130, 1.5), (257, 300, 1.5), (600, 20, 1.5), (20, 700, 0.0)])
def test_merid_bitexact(nr, nz, beta, kind):
    from codesthesis_dir_amd.merid import Merid, MeridConfig
    print(f"[gpu] merid line redo {nr}x{nz} {kind}", flush=True)
    cfg = MeridConfig(nr=nr, nz=nz, beta=beta, dt=1e-5, Ra=3e4, Re=20.0, Pr=0.8)
    run = Merid(cfg)
    ora = OM.Merid(nr, nz, cfg.dt, cfg.Ra, cfg.Re, cfg.Pr, r=run.r, z=run.z)
    for q, n in enumerate(("w", "wp", "v", "vp", "th", "thp", "u", "ww")):
        a = _field(kind, ora.shape, q)
        ora.f[n][...] = a
        run.put(n, a)
    run.derivatives()
    ora.derivatives()
    for q in range(6):
        _same(run.derivative(q), ora.d[q], q)
    run.close()


def _time(run, put, go, keys, n=10):
    """Milliseconds of the kernels `keys` over n calls."""
    put()
    go()
    run.profile(True)
    for _ in range(n):
        go()
    p = run.profile_read()
    run.profile(False)
    return sum(p[k]["ms"] for k in keys)


@pytest.mark.parametrize("prog", ["plane", "tank", "merid"])
def test_time_of_flat_cores(prog):
    """A line done again is up to 2 N rows of one lane's chain out of LDS
    beside the chunks' 2 (40 + 8 mb) rows: 2.2, 2.3 and 3.3 times the kernel
    on a noisy field, where every entry is proven (so fields of noise must not
    take it).  From tables in memory it was 7 times."""
    print(f"[gpu] flat cores {prog}", flush=True)
    if prog == "plane":
        from codesthesis_dir_amd import BoxConfig, PeriodicBox
        run, names, keys = PeriodicBox(BoxConfig(nr=512, np=256, width=1.0, dt=1e-7, Ra=1e5)), ("C", "Cp", "th", "thp"), ["compact"]
        go = lambda: (run.cvorticity(False), run.temperature(False))
    elif prog == "tank":
        from codesthesis_dir_amd.tank import Tank, TankConfig
        run, names = Tank(TankConfig(nr=64, nz=384, np=384, dt=1e-7, Re=1e3, Ptl=5.0, Gr=1e6)), ("A", "B", "C", "th")
        keys, go = ["deriv_yz"], run.derivatives
    else:
        from codesthesis_dir_amd.merid import Merid, MeridConfig
        run, names = Merid(MeridConfig(nr=512, nz=256, dt=1e-7, Ra=1e5, Re=10.0, Pr=1.0)), ("w", "wp", "v", "vp", "th", "thp")
        keys, go = ["deriv"], run.derivatives
    shape = run.get(names[0]).shape

    def put(kind):
        if prog == "plane":
            run.start()   # the fields after it are the current ones again
        for q, n in enumerate(names):
            run.put(n, _field(kind, shape, q))

    t = {k: min(_time(run, lambda: put(k), go, keys) for _ in range(3)) for k in ("noise", "layers")}
    print("[gpu]", prog, t, flush=True)
    assert 1.3 * t["noise"] < t["layers"] < 4.5 * t["noise"]
    run.close()
