"""The direct solves' row recurrences in chunks (csrc/vv_rlines.h) where the
split can go wrong: the shortest rows, one row past a chunk and past each
rule's bound (128 rows in chunks of 8, 1024 in chunks of 16, longer ones a
lane each), workgroups whose last lines are missing; by the residuals of the
solvers that use them, with their bounds."""
import numpy as np
import pytest

import oracle_tank as OT
import test_gpu_3d as T3
import test_gpu_sector as TS
import test_gpu_tank as TT

pytestmark = pytest.mark.gpu

NR = [4, 8, 9, 10, 17, 64, 127, 128, 129, 130, 255, 1024, 1025, 1026, 1100]


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("nr", NR)
def test_rot3d(which, nr):
    T3.test_poisson_residual_at_larger_sizes(which, (nr, 7, 10))


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("nr", NR)
def test_sector(which, nr):
    TS.test_poisson_residual_at_size_limits(which, (nr, 5, 7))


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("nr", [6] + NR[1:])
def test_tank(which, nr):
    nz, np_ = 7, 9
    print(f"[gpu] tank rows {which} {nr}", flush=True)
    run, ora = TT._pair(nr, nz, np_, seed=which)
    psi, _, rhs = OT.PSI[which]
    run.poisson(which)
    m, _ = ora.residual(which, run.get(psi), ora[rhs])
    assert m <= 1e-10 * np.max(np.abs(ora[rhs])) * max(nr, nz, np_) ** 2   # the solve test's bound
    run.close()


def test_time_of_long_rows():
    """Lines past a workgroup's threads, one a lane: a trip to memory for 16
    rows each way, 2 x 70 at 1100 rows, about 1.5 us each (measured 213 us a
    call; 485 where the coefficients were fetched row by row)."""
    import time
    print("[gpu] long rows", flush=True)
    run, _ = TS._pair(1100, 20, 20, seed=1)
    run.poisson(1)
    t = []
    for _ in range(20):
        s = time.perf_counter()
        run.poisson(1)
        t.append(time.perf_counter() - s)
    assert min(t) < 340e-6, min(t)
    run.close()
