"""The FP64 axial transforms at lengths of 513 to 568, 1025 to 1137 and 2049 to 2275 rows, whose tiles
are half as wide as their neighbours', and at the lengths beside them: a manufactured potential
comes back from the divergence of its gradient."""
import numpy as np
import pytest

from harness import make_case, oracle_for
from oracle import orc
from simpletcsolver_amd import Solver

pytestmark = pytest.mark.gpu


# enough lines that tiles keep their full width (two per CU), odd numbers of them, planes of a few rows
@pytest.mark.parametrize("nx,ny,nz", [(65, 256, 540), (66, 256, 512), (71, 256, 560), (67, 252, 576), (39, 256, 1080), (33, 256, 1120),
                                      (35, 250, 1152), (19, 256, 2100), (17, 256, 2187), (17, 256, 2304), (64, 256, 567)])
def test_manufactured_potential(need_gpu, nx, ny, nz):
    """bound: that of the 16 x 12 x 8 potential (1e-12 relative), times the square of the grid's
    ratio to it (the smallest eigenvalue falls as the square of the length)"""
    case = make_case(nx=nx, ny=ny, nz=4, Re=100.0, amp=0.0, uy_walls=(0.0, 0.0))
    o = oracle_for(case)
    hxxf, hyxc, hz = o.array("hxxf").copy(), o.array("hyxc").copy(), case["kw"]["lengths"][2] / nz
    o.close()
    psi = np.random.default_rng(nz).standard_normal((nz, ny, nx))
    rk, dt = 0, 0.3
    g = orc.rkcoefs()[rk, 2] * dt
    ux = np.zeros((nz, ny, nx + 1))
    ux[:, :, 1:nx] = g * (psi[:, :, 1:] - psi[:, :, :-1]) / hxxf[1:nx]
    uy = np.zeros((nz, ny, nx + 2))
    uy[:, :, 1:nx + 1] = g * (psi - np.roll(psi, 1, axis=1)) / hyxc[1:nx + 1]
    uz = np.zeros((nz, ny, nx + 2))
    uz[:, :, 1:nx + 1] = g * (psi - np.roll(psi, 1, axis=0)) / hz
    s = Solver(nx, ny, nz, case["xf"], case["xc"], **case["kw"])
    s.load_fields({"ux": ux, "uy": uy, "uz": uz})
    s.potential(rk, dt)
    d = s.get_field("psi")[:, :, 1:-1] - psi
    s.close()
    d -= d.mean()
    assert np.linalg.norm(d) <= 1e-12 * max(nx / 16., ny / 12., nz / 8.) ** 2 * np.linalg.norm(psi)
