"""psi's periodic images and wall copies as the persistent inverse theta transform leaves them, at
sizes that reach it with each last radix (8, 4, 3 and 2 rows apart).  The correction reads them,
so a missing one is a wrong flow.  psi is zero in a new solver, and the persistent form is the
first to write it here: an image that it leaves out stays zero and shows."""
import numpy as np
import pytest

from harness import make_case
from simpletcsolver_amd import Solver

SIZES = [(64, 128, 2048), (128, 192, 1024), (256, 384, 256), (96, 1024, 192), (128, 512, 256), (128, 256, 512)]


@pytest.mark.parametrize("radix", [2, 3, 4, 8])
@pytest.mark.parametrize("rows", [64, 96, 128, 192, 256, 288, 384, 512])
def test_the_thread_that_holds_the_last_row(radix, rows):
    """the transform of M packed rows gives a thread (row r0 of dr = M / 8, eight elements) the
    butterflies r0 + q dr < M / radix, and element M - 1, which holds row ny, is the last
    output of the last butterfly: the thread rows holding it are (M / radix - 1) mod dr alone"""
    if rows % (8 * radix):
        pytest.skip("not a length of this radix")
    dr, per = rows // 8, rows // radix
    nq = -(-8 // radix)
    holders = {r0 for r0 in range(dr) for q in range(nq) for r in range(radix)
               if r0 + q * dr < per and r0 + q * dr + r * per == rows - 1}
    assert holders == {(per - 1) % dr}


def _solver(nx, ny, nz, precision):
    small = make_case(nx=nx, ny=ny, nz=4, Re=100.0, amp=0.0, uy_walls=(0.0, 0.0))
    return Solver(nx, ny, nz, small["xf"], small["xc"], precision=precision, **small["kw"])


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz", SIZES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_first_potential_of_a_new_solver(need_gpu, nx, ny, nz, precision):
    rng = np.random.default_rng(7)
    f = {"ux": rng.random((nz, ny, nx + 1)), "uy": rng.random((nz, ny, nx + 2)), "uz": rng.random((nz, ny, nx + 2))}
    f["ux"][:, :, 0] = 0.0
    f["ux"][:, :, -1] = 0.0
    got = {}
    for mask in (5, 0):
        s = _solver(nx, ny, nz, precision)
        s.load_fields(f)
        s.tune("fft_exact", mask, 0)
        s.potential(1, 0.13)
        psi = s.get_field_ref("psi")
        s.close()
        assert np.array_equal(psi[1:-1, 0, 1:-1], psi[1:-1, -2, 1:-1]) and np.array_equal(psi[1:-1, -1, 1:-1], psi[1:-1, 1, 1:-1])
        assert np.array_equal(psi[0], psi[-2]) and np.array_equal(psi[-1], psi[1])
        assert np.array_equal(psi[..., 0], psi[..., 1]) and np.array_equal(psi[..., -1], psi[..., -2])
        got[mask] = psi
    assert np.abs(got[0]).max() > 0.0
    assert np.array_equal(got[5], got[0])


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz", [(128, 192, 1024), (256, 384, 256)])
def test_step_is_solenoidal_and_the_same_in_both_forms(need_gpu, nx, ny, nz):
    """two FP64 steps with the default forms and with the one-tile ones: the same bits, and a
    divergence at round-off (a face difference of velocities of 1 over the smallest spacing,
    and the solve's rounding over some log2 of the cells)"""
    got = []
    for mask in (None, 0):
        s = _solver(nx, ny, nz, "fp64")
        s.ic(seed=3, amp=0.1, nmodes=2, mode_amp=0.1)
        if mask is not None:
            s.tune("fft_exact", mask, 0)
        s.step()
        s.step()
        assert s.divergence() <= 2.2e-16 * 8 * max(nx, ny, nz) * 100
        got.append({n: s.get_field(n) for n in ("ux", "uy", "uz", "p")})
        s.close()
    for n in got[0]:
        assert np.array_equal(got[0][n], got[1][n]), n
