"""The periodic y and z line solves at the edges of their segments (32 rows per thread in FP64,
up to 64 in the mixed step): single segments, full ones, last ones of one row and of all but
one, factors that converge within a few rows and not before the line ends, against the oracle."""
import numpy as np
import pytest

from harness import gpu_for, make_case, oracle_for, rel_l2
from simpletcsolver_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("Re", [1e4, 1.0])
@pytest.mark.parametrize("nx,ny,nz", [(3, 4, 3), (5, 32, 35), (70, 64, 32), (6, 98, 63), (17, 126, 64), (5, 128, 81),
                                      (40, 192, 98), (33, 200, 125), (3, 256, 128), (4, 6, 512), (4, 540, 6), (3, 4, 1024)])
def test_periodic_solves_match_oracle(need_gpu, nx, ny, nz, Re, precision):
    dt = 1e-3
    for implicit in ((0, 1, 0), (0, 0, 1), (0, 1, 1)):
        case = make_case(nx=nx, ny=ny, nz=nz, implicit=implicit, Re=Re, t_amp=1e-2, amp=0.1)
        o = oracle_for(case)
        s = Solver(nx, ny, nz, case["xf"], case["xc"], precision=precision, **case["kw"])
        s.load_fields(case["fields"])
        # the systems are 1 + a second difference of strength a at most: condition 1 + 4 a, and
        # both sides solve them by some 16 roundings a row of the increment's precision
        lengths = case["kw"]["lengths"]
        h = min(lengths[1] * case["xf"][0] / ny, lengths[2] / nz)
        a = 2 * 0.5 * (8. / 15.) * dt / Re / h ** 2
        tol = 1e-14 + 16 * 2.2e-16 * (1 + 4 * a) if precision == "fp64" else 1e-6 + 16 * 6e-8 * (1 + 4 * a)
        f0 = o.npy_fields()
        o.predict(0, dt)
        s.predict(0, dt)
        of, sf = o.npy_fields(), s.fields()
        for n in ("ux", "uy", "uz", "t"):
            # the explicit directions may make the substep's increment larger than the field
            scale = max(1.0, np.linalg.norm(of[n] - f0[n]) / np.linalg.norm(of[n]))
            assert rel_l2(sf[n], of[n]) <= tol * scale, (n, implicit, a)
            # the periodic images, through what the next substep makes of them
        o.predict(1, dt)
        s.predict(1, dt)
        of, sf = o.npy_fields(), s.fields()
        if precision == "fp64":
            for n in ("ux", "uy", "uz", "t"):
                assert np.isfinite(sf[n]).all() and rel_l2(sf[n], of[n]) <= 1e3 * tol, (n, implicit, a)
        s.close()
        o.close()
