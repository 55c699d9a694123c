"""The mixed step's line solves: the x forms (FP32 increment, final pass or not; one, two, four, eight
and sixteen rows per lane, several lines per wave) against the oracle, and the periodic images
that the final y and z passes write, in both precisions, read back bit for bit."""
import numpy as np
import pytest

from harness import make_case, oracle_for, rel_l2
from simpletcsolver_amd import Solver

pytestmark = pytest.mark.gpu


def _mixed_x(case, dt):
    o = oracle_for(case)
    s = Solver(case["nx"], case["ny"], case["nz"], case["xf"], case["xc"], precision="mixed", **case["kw"])
    s.load_fields(case["fields"])
    # right-hand sides and solves round to FP32: 6e-8 of the terms they add, the largest of which
    # is the second difference of strength a (test_gpu_psolve_lengths.py has the same bound)
    a = 2 * 0.5 * (8. / 15.) * dt / case["kw"]["Re"] / np.diff(case["xf"]).min() ** 2
    tol = 1e-6 + 16 * 6e-8 * (1 + 4 * a)
    f0 = o.npy_fields()
    o.predict(0, dt)
    s.predict(0, dt)
    of, sf = o.npy_fields(), s.fields()
    for n in ("ux", "uy", "uz", "t"):
        scale = max(1.0, np.linalg.norm(of[n] - f0[n]) / np.linalg.norm(of[n]))
        assert np.isfinite(sf[n]).all() and rel_l2(sf[n], of[n]) <= tol * scale, (n, a)
    s.close()
    o.close()


@pytest.mark.parametrize("implicit", [(1, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("nx", [3, 63, 64, 65, 129, 150, 256, 257, 512, 513, 1024])
def test_x_solves_match_oracle(need_gpu, nx, implicit):
    _mixed_x(make_case(nx=nx, ny=6, nz=5, implicit=implicit, t_amp=1e-2, Re=1e3, stretch=1.0), 1e-3)


@pytest.mark.parametrize("implicit", [(1, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("nx,ny,nz", [(3, 512, 512), (65, 128, 96), (150, 256, 70), (300, 128, 35)])
def test_x_solves_of_many_lines_match_oracle(need_gpu, nx, ny, nz, implicit):
    _mixed_x(make_case(nx=nx, ny=ny, nz=nz, implicit=implicit, t_amp=1e-2, Re=1e3, stretch=1.0), 1e-3)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("implicit", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 1, 1)])
@pytest.mark.parametrize("nx,ny,nz", [(3, 4, 3), (17, 32, 35), (40, 64, 35), (33, 98, 81), (5, 200, 6), (64, 6, 200)])
def test_images_of_the_final_pass(need_gpu, nx, ny, nz, implicit, precision):
    """a new solver's other buffers are zero, so an image that the predictor leaves out shows"""
    case = make_case(nx=nx, ny=ny, nz=nz, implicit=implicit, t_amp=1e-2, amp=0.1, Re=1e3)
    s = Solver(nx, ny, nz, case["xf"], case["xc"], precision=precision, **case["kw"])
    s.load_fields(case["fields"])
    for rk in range(2):
        s.predict(rk, 1e-3)
        for n in ("ux", "uy", "uz", "t"):
            a = s.get_field_ref(n)
            assert np.array_equal(a[1:-1, 0], a[1:-1, -2]) and np.array_equal(a[1:-1, -1], a[1:-1, 1]), (n, rk)
            assert np.array_equal(a[0], a[-2]) and np.array_equal(a[-1], a[1]), (n, rk)
            assert np.abs(a[1:-1, 0]).max() > 0.0, (n, rk)
    s.close()
