"""The transforms at the lengths where their first and last passes differ: one pass only (2, 3,
4, 5, 7, 8), two and more with every radix first and last, line counts that fill no tile, tiles
of one line and of many: the potential of a predicted field against the oracle, and the mixed
step's against the FP64 one."""
import numpy as np
import pytest

from harness import make_case, modulo_mean, oracle_for, rel_l2
from simpletcsolver_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(3, 4, 3), (5, 6, 4), (16, 10, 5), (17, 14, 7), (33, 16, 8), (64, 8, 32), (20, 12, 9),
                                      (7, 20, 10), (70, 28, 14), (129, 30, 49), (16, 70, 25), (10, 98, 21), (9, 42, 63),
                                      (31, 256, 6), (6, 4, 1024), (5, 512, 3)])
def test_potential_matches_oracle(need_gpu, nx, ny, nz):
    """FP64: the bound of the 16 x 12 x 8 potential (1e-12 relative), times the square of the
    grid's ratio to it in the directions the eigenvalues span (the smallest falls as the square of
    the length); mixed: the same in units of FP32's rounding over FP64's"""
    case = make_case(nx=nx, ny=ny, nz=nz, implicit=(1, 0, 0), amp=0.1)
    o = oracle_for(case)
    tol = 1e-12 * max(1.0, nx / 16., ny / 12., nz / 8.) ** 2
    o.predict(0, 1e-3)
    o.potential(0, 1e-3)
    want = modulo_mean(o.npy_fields()["psi"], case)
    for precision, t in (("fp64", tol), ("mixed", tol * 2.0 ** 29)):
        s = Solver(nx, ny, nz, case["xf"], case["xc"], precision=precision, **case["kw"])
        s.load_fields(case["fields"])
        s.predict(0, 1e-3)
        s.potential(0, 1e-3)
        psi = s.get_field("psi")
        assert np.isfinite(psi).all()
        assert rel_l2(modulo_mean(psi, case), want) <= t, precision
        # halo images and wall copies, through the host layout that includes them
        full = s.get_field_ref("psi")
        assert np.array_equal(full[1:-1, 0], full[1:-1, -2]) and np.array_equal(full[1:-1, -1], full[1:-1, 1])
        assert np.array_equal(full[0], full[-2]) and np.array_equal(full[-1], full[1])
        assert np.array_equal(full[..., 0], full[..., 1]) and np.array_equal(full[..., -1], full[..., -2])
        s.close()
    o.close()


@pytest.mark.parametrize("nx,ny,nz", [(64, 128, 2048), (128, 192, 1024), (96, 1024, 192), (128, 512, 256), (128, 256, 512)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_persistent_forms_compute_the_same_bits(need_gpu, nx, ny, nz, precision):
    """launches of enough tiles for the persistent axial (last radix 4, 2, 3, 4, 8) and inverse
    theta (8, 3, 8, 4, 2) transforms: the same potential as the one-tile forms, bit for bit, each
    repeated, with halo images and wall copies"""
    small = make_case(nx=nx, ny=ny, nz=4, Re=100.0, amp=0.0, uy_walls=(0.0, 0.0))
    rng = np.random.default_rng(5)
    f = {"ux": rng.random((nz, ny, nx + 1)), "uy": rng.random((nz, ny, nx + 2)), "uz": rng.random((nz, ny, nx + 2))}
    f["ux"][:, :, 0] = 0.0
    f["ux"][:, :, -1] = 0.0
    s = Solver(nx, ny, nz, small["xf"], small["xc"], precision=precision, **small["kw"])
    s.load_fields(f)
    want = None
    for mask in (0, 1, 4, 5, 5):
        s.tune("fft_exact", mask, 0)
        s.potential(1, 0.13)
        got = s.get_field_ref("psi")
        if want is None:
            want = got
            assert np.abs(want).max() > 0.0
        assert np.array_equal(got, want), mask
    s.close()
