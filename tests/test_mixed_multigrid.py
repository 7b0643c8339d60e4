"""The coarse-grid correction in the mixed-precision solve's conjugate-gradient preconditioner
(les_mg.hip), at the sizes where its grids differ: odd and even halvings along i, periodic rows
whose half is odd, columns of one partial segment, of 8, 12 and 16 levels a segment and taller than
the segments.  The FP64 residual, which is evaluated apart from the
preconditioner, has to reach the tolerance, in the few iterations a working V-cycle takes (the
pass without it takes hundreds at 150x150x90); a relaxation other than 1 keeps the plain pass."""
import pytest

import common

pytestmark = pytest.mark.gpu

TOL = 1e-7


def _solve(dims, dx=4.0, dy=4.0, **kw):
    from les_halo_amd import LES, inputs
    from les_halo_amd.les import LES_PREC_MIXED
    L = LES(*dims, **common.REF_PHYS, omega=1.5, pjuge=0.0, nmaxp=50, precision=LES_PREC_MIXED,
            refine_tol=TOL, refine_max=40, refine_solver=1, **kw)
    L.load_case(inputs.make_case(*dims, seed=9, hmax=20.0, dx=dx, dy=dy))
    L.ifdata()
    out = []
    for n in (1, 2, 3):
        L.step(n)
        out.append(L.scalars())
    L.close()
    return out


@pytest.mark.parametrize("dims", [(40, 32, 20), (37, 30, 5), (61, 34, 64), (50, 46, 65), (33, 20, 97),
                                  (21, 12, 140), (150, 150, 90)])
def test_multigrid_reaches_tolerance_in_few_iterations(dims):
    print(dims, flush=True)
    for s in _solve(dims):
        assert s["resid_l2"] <= TOL, s
        assert s["cg_iters"] <= 40, s


def test_another_relaxation_keeps_the_plain_pass():
    for s in _solve((40, 32, 20), refine_omega=1.5):
        assert s["resid_l2"] <= TOL, s


@pytest.mark.parametrize("dx, dy", [(5.0, 3.0), (2.0, 10.0), (10.0, 2.0), (1.0, 20.0), (20.0, 1.0)])
@pytest.mark.parametrize("dims", [(61, 34, 64), (24, 96, 20)])
def test_multigrid_with_unequal_spacings(dims, dx, dy):
    print(dims, dx, dy, flush=True)
    for s in _solve(dims, dx, dy):
        assert s["resid_l2"] <= TOL, s
        assert s["cg_iters"] <= 40, s
