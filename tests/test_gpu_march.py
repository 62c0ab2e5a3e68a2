"""The marching explicit kernels where their planes per workgroup can go
wrong: grids of fewer columns than a workgroup, planes that the last
workgroup of a column does not fill, and sizes that the rule gives one plane,
a few and many; by the bit-exact tests of the solvers that march."""
import numpy as np
import pytest

import oracle3 as O3
import test_gpu_3d as T3
import test_gpu_tank as TT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(6, 6, 6), (34, 33, 70), (66, 64, 139), (130, 127, 67)])
def test_tank(shape):
    TT.test_explicit_routines_bitexact(shape)


@pytest.mark.parametrize("shape", [(6, 6, 8), (34, 33, 70), (66, 64, 138), (130, 127, 66)])
def test_hor(shape):
    T3.test_hor_explicit_routines_match_oracle(shape)


@pytest.mark.parametrize("shape", [(4, 4, 4), (34, 33, 70), (66, 64, 138), (130, 127, 66)])
def test_rot(shape):
    print(f"[gpu] rot march {shape}", flush=True)
    run = T3._gpu(*shape)
    ora = O3.Run3(*shape, **T3.PARAMS)
    for n, a in T3._state(np.random.default_rng(sum(shape)), ora.shape, 150.0).items():
        run.put(n, a)
        ora[n] = a
    run.vorticity()
    for rt in ("avorticity", "bvorticity", "cvorticity"):
        ora.call(rt)
    for n in ("An", "Bn", "Cn"):
        assert np.array_equal(run.get(n), ora[n]), n
    run.close()
