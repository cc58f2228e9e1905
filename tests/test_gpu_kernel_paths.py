"""The kernels' size-dependent paths at the edges of their ranges, against the oracle."""
import numpy as np
import pytest

import opf_oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu

# vel_nonlinear: two transforms of length L each way round by some 5 eps log2(L)
# of the field's size, below 1e-14 for every length here, and the products of
# two such fields by a few times that
TOL_NONLINEAR = 1e-13


@pytest.fixture(scope="module")
def opf():
    import opf as pkg
    return pkg


def _nonlinear_matches(opf, N, K, M):
    from opf import ic as icgen
    Re, alpha = 3000.0, 1.25
    ctx = opf.Context(N, K, M)
    ctx.setup(0, Re, alpha, 0.01)
    me = ctx.mesh()
    u = icgen.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, 7, 1e-2)
    ctx.put_state(0, *u)
    ctx.transform(0)
    ctx.nonlinear(0)
    got = ctx.get_nonlinear(0)
    oc = O.Ctx(N, K, M, Re=Re, alpha=alpha, dt=0.01)
    oc.set_state(*u)
    oc.transform()
    oc.nonlinear()
    scale = max(np.abs(f).max() for f in (oc.Nr, oc.Nt, oc.Nz))
    for c, ref in enumerate((oc.Nr, oc.Nt, oc.Nz)):
        assert np.abs(got[c] - ref).max() <= TOL_NONLINEAR * scale, c


# every transform length 2^a 3^b with its own radix sequence, as 3K and as 3M
@pytest.mark.parametrize("K,M", [(3, 9), (9, 3), (18, 18), (27, 27), (32, 32), (36, 36), (54, 54), (72, 72),
                                 (81, 81), (96, 96), (108, 4), (144, 4), (162, 4), (192, 4), (216, 4), (4, 108)])
def test_nonlinear_transform_lengths(opf, K, M):
    _nonlinear_matches(opf, 10, K, M)
