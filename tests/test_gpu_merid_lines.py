"""The meridional plane's chunked compact lines against the oracle, bit for
bit, at line lengths around the head, whole blocks and several blocks a lane,
and with fields whose chunks do not meet within the warm-up (a spot in zeros,
constants, by the rounding of their one-sided end rows), which are run again."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_merid as OM

pytestmark = pytest.mark.gpu

NAMES = ("w", "wp", "v", "vp", "th", "thp", "u", "ww")


@pytest.mark.parametrize("kind", ["random", "spot", "constant"])
@pytest.mark.parametrize("nr,nz,beta", [(8, 8, 0.0), (24, 26, 1.5), (33, 66, 1.5), (74, 57, 0.0), (90, 130, 1.5), (257, 300, 1.5),
                                        (600, 20, 1.5), (20, 700, 0.0)])
def test_chunked_lines_bitexact(nr, nz, beta, kind):
    from codesthesis_dir_amd.merid import Merid, MeridConfig
    print(f"[gpu] merid lines {nr}x{nz} {kind}", flush=True)
    cfg = MeridConfig(nr=nr, nz=nz, beta=beta, dt=1e-5, Ra=3e4, Re=20.0, Pr=0.8)
    run = Merid(cfg)
    ora = OM.Merid(nr, nz, cfg.dt, cfg.Ra, cfg.Re, cfg.Pr, r=run.r, z=run.z)
    rng = np.random.default_rng(nr * nz)
    for q, n in enumerate(NAMES):
        a = np.zeros(ora.shape)
        if kind == "random":
            a = rng.standard_normal(ora.shape)
        elif kind == "spot":
            a[nz // 3, nr // 2] = 3.7 + q
        else:
            a += 0.25 * (q + 1)
        ora.f[n][...] = a
        run.put(n, a)
    run.derivatives()
    ora.derivatives()
    for q in range(6):
        g, o = run.derivative(q), ora.d[q]
        # the divisions' remainders underflow for operands below 1e-290; a
        # quotient there may be one denormal step (5e-324) off
        assert np.array_equal(g[np.abs(o) >= 1e-290], o[np.abs(o) >= 1e-290]), q
        assert np.max(np.abs(g - o)) <= 5e-324, q
    run.close()
