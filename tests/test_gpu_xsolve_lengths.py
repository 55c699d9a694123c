"""The x line solves at the edges of their forms (one, two, four, eight and sixteen rows per
lane: lines of 64, 128, 256, 512 and 1024 rows, and one more), as the last direction (the new
field written) and before y and z, against the oracle."""
import pytest

from harness import gpu_for, make_case, oracle_for, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("implicit", [(1, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("nx", [3, 63, 64, 65, 129, 150, 256, 257, 513, 1024])
def test_x_solves_match_oracle(need_gpu, nx, implicit):
    """the bound of the implicit substeps on other grids, 1e-14 (a few ulps of the field)"""
    case = make_case(nx=nx, ny=6, nz=5, implicit=implicit, t_amp=1e-2, Re=1e3)
    o, s = oracle_for(case), gpu_for(case)
    for rk in range(3):
        o.predict(rk, 1e-3)
        s.predict(rk, 1e-3)
    of, sf = o.npy_fields(), s.fields()
    for n in ("ux", "uy", "uz", "t"):
        assert rel_l2(sf[n], of[n]) <= 1e-14, n
    s.close()
    o.close()


@pytest.mark.parametrize("implicit", [(1, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("nx,ny,nz", [(3, 512, 512), (65, 128, 96), (150, 256, 70), (300, 128, 35)])
def test_x_solves_of_many_lines_match_oracle(need_gpu, nx, ny, nz, implicit):
    """several lines per wave, at launches of 2 to 16 blocks per CU; the same bound"""
    case = make_case(nx=nx, ny=ny, nz=nz, implicit=implicit, t_amp=1e-2, Re=1e3)
    o, s = oracle_for(case), gpu_for(case)
    o.predict(0, 1e-3)
    s.predict(0, 1e-3)
    of, sf = o.npy_fields(), s.fields()
    for n in ("ux", "uy", "uz", "t"):
        assert rel_l2(sf[n], of[n]) <= 1e-14, n
    s.close()
    o.close()
