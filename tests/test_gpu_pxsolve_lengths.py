"""The radial Poisson solve at the lengths where its lines fill a wave's segments exactly, leave a
remainder or hold three rows (the least), with one line per wave and with several: the potential of a predicted
field against the oracle's."""
import numpy as np
import pytest

from harness import make_case, modulo_mean, oracle_for, rel_l2
from simpletcsolver_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(3, 4, 3), (63, 4, 4), (64, 4, 4), (65, 6, 4), (128, 4, 4), (129, 4, 4), (256, 4, 3), (257, 4, 4),
                                      (511, 4, 3), (512, 4, 3), (513, 4, 3), (1000, 4, 3), (1024, 4, 3), (4, 128, 128), (70, 128, 128)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_potential_matches_oracle(need_gpu, nx, ny, nz, precision):
    """the bound of the 16 x 12 x 8 potential (1e-12 relative) times the square of the grid's ratio
    to it in each direction (the smallest eigenvalue falls so), in FP32's rounding for the mixed
    step's transforms"""
    case = make_case(nx=nx, ny=ny, nz=nz, implicit=(1, 0, 0), amp=0.1)
    o = oracle_for(case)
    tol = 1e-12 * max(1.0, nx / 16., ny / 12., nz / 8.) ** 2 * (2.0 ** 29 if precision == "mixed" else 1.0)
    o.predict(0, 1e-3)
    o.potential(0, 1e-3)
    want = modulo_mean(o.npy_fields()["psi"], case)
    s = Solver(nx, ny, nz, case["xf"], case["xc"], precision=precision, **case["kw"])
    s.load_fields(case["fields"])
    s.predict(0, 1e-3)
    s.potential(0, 1e-3)
    assert rel_l2(modulo_mean(s.get_field("psi"), case), want) <= tol
    s.close()
    o.close()
