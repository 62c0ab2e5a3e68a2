"""Which way the tank's and the sector's side-wall modes are taken (FFTs in
LDS or matrix-core GEMMs, csrc/vv_ytrans.h) where the rule's lines lie, and
FFTs of 8 to 128 lines a workgroup with the last one cut short; by the solves'
residuals, with the bounds of their tests."""
import pytest

import test_gpu_sector as TS
import test_gpu_tank as TT

pytestmark = pytest.mark.gpu


# the plane and whether np planes of it go by FFT: a power of two; small odd
# np; up to 800000 points; lines of 384 and more; a prime above 13
@pytest.mark.parametrize("nr,nz,np_,fft", [
    (200, 200, 16, True), (20, 20, 9, False), (20, 20, 15, False), (20, 20, 33, True), (50, 42, 100, True), (66, 67, 10, True),
    (128, 128, 48, True), (128, 128, 50, False), (200, 200, 12, True), (200, 201, 20, False), (60, 60, 250, False),
    (60, 60, 390, True), (20, 20, 34, False)])
def test_tank(nr, nz, np_, fft):
    import oracle_tank as OT
    print(f"[gpu] tank transforms {nr}x{nz}x{np_}", flush=True)
    run, ora = TT._pair(nr, nz, np_, seed=np_)
    run.profile(True)
    for which in (1, 2, 3):
        run.poisson(which)
        psi, _, rhs = OT.PSI[which]
        m, _ = ora.residual(which, run.get(psi), ora[rhs])
        assert m <= 1e-10 * abs(ora[rhs]).max() * max(nr, nz, np_) ** 2, which   # the solve test's bound
    p = run.profile_read()
    assert (p["yfft_fwd"]["launches"] > 0, p["yfwd"]["launches"] > 0) == (fft, not fft)
    run.close()


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("shape", [(66, 67, 10), (50, 42, 100), (128, 66, 36), (90, 90, 110)])
def test_sector(which, shape):
    TS.test_poisson_residual_at_size_limits(which, shape)
