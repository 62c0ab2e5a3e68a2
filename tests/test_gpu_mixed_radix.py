"""The mixed-radix FFT stages (csrc/vv_fft.h) in the four solvers that use
them: every odd prime with a stage of its own (3, 5, 7, 11, 13), repeated and
mixed primes, larger primes (formed several outputs per thread, or by GEMM in
the tank and the sector), one and several lines per workgroup; by the solve
tests of the solvers, with their bounds."""
import pytest

import test_gpu_3d as T3
import test_gpu_parity as T2
import test_gpu_sector as TS
import test_gpu_tank as TT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom,nr,np_", [(0, 520, 286), (1, 300, 90), (0, 24, 502), (1, 600, 34), (0, 1030, 182), (1, 20, 8190)])
def test_plane_poisson(geom, nr, np_):
    T2.test_poisson_default_direct_any_np(geom, nr, np_)


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(9, 7, 14), (7, 8, 22), (8, 6, 26), (7, 6, 34)])
def test_rot3d_poisson(which, shape):
    T3.test_poisson_matches_exact_solve(which, shape)


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(64, 48, 150), (33, 40, 374), (8, 6, 1430), (8, 6, 1458), (9, 6, 502)])
def test_rot3d_poisson_residual(which, shape):
    T3.test_poisson_residual_at_larger_sizes(which, shape)


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(6, 7, 9), (6, 6, 14), (6, 6, 22), (7, 6, 25), (6, 6, 26), (6, 6, 17), (6, 6, 30)])
def test_tank_poisson(which, shape):
    TT.test_poisson_matches_dense_solve(which, shape)


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(4, 5, 11), (5, 5, 21), (4, 5, 17)])
def test_sector_poisson(which, shape):
    TS.test_poisson_matches_dense_solve(which, shape)


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(33, 32, 160), (4, 4, 1001), (4, 5, 1430), (5, 4, 2000), (4, 4, 1458), (6, 5, 170)])
def test_sector_poisson_residual(which, shape):
    TS.test_poisson_residual_at_size_limits(which, shape)
