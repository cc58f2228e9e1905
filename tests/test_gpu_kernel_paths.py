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


def _one_step_matches(opf, N, K, M, Mp, gp, monkeypatch, tol):
    from opf import ic as icgen
    Re, alpha, dt = 2400.0, 1.25, 0.01
    monkeypatch.setenv("OPF_STEP_GP", str(gp))
    ctx = opf.Context(N, K, M, Mp)
    assert ctx.step_pairs() == gp
    ctx.setup(0, Re, alpha, dt)
    me = ctx.mesh()
    u = icgen.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, 3, 1e-2, Mp=Mp)
    ctx.put_state(0, *u)
    ctx.run(2, corr_fixed=1)
    got = ctx.get_state(0)
    oc = O.Ctx(N, K, M, Mp, Re=Re, alpha=alpha, dt=dt)
    oc.set_state(*u)
    oc.run(2, ncorr_fixed=1)
    for c, ref in enumerate((oc.ur, oc.ut, oc.uz)):
        assert rel_err(got[c], ref) <= tol, (N, c)
    ctx.close()


# The block elimination at every remainder of N by eight, at the edges of the
# ranges of its instantiations (N = 32, 64, 96) and at the smallest and largest
# N, for groups that do (K M = 12) and do not (18) fill the workgroups.  The
# pressure solves of the two differ by their forward errors, up to 1e-11 at
# N = 128 for the lowest modes; the velocity takes dt grad p of it.
@pytest.mark.parametrize("gp", [1, 2, 4])
@pytest.mark.parametrize("N,K,M,Mp", [(9, 4, 3, 1), (10, 3, 6, 2), (11, 4, 3, 1), (12, 3, 6, 3), (13, 4, 3, 1),
                                      (14, 4, 3, 4), (15, 4, 3, 1), (31, 4, 3, 1), (32, 3, 6, 1), (33, 4, 3, 2),
                                      (63, 4, 3, 1), (64, 3, 6, 1), (65, 4, 3, 1), (96, 3, 6, 1), (97, 4, 3, 1),
                                      (128, 3, 6, 1)])
def test_step_radial_sizes(opf, N, K, M, Mp, gp, monkeypatch):
    if gp == 4 and N > 96:
        pytest.skip("four pairs per workgroup need N <= 96")
    _one_step_matches(opf, N, K, M, Mp, gp, monkeypatch, 1e-12 if N <= 64 else 1e-11)


def test_step_with_a_replaced_factor_set(opf):
    """tim_lumesh_init into LDz (other c1, c2, the Neumann wall row): the next
    steps solve with it, and tim_lumesh_get returns its LAPACK factors; then
    vel_matrices rebuilds the set."""
    from opf import ic as icgen
    N, K, M, Re, alpha, dt = 20, 4, 3, 2400.0, 1.25, 0.01
    ctx = opf.Context(N, K, M)
    ctx.setup(0, Re, alpha, dt)
    before = ctx.lumesh_get(0, opf.LDZ)
    me = ctx.mesh()
    u = icgen.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, 3, 1e-2)
    ctx.lumesh_init(0, opf.LDZ, 0, 1, 130.0, -3e-4)
    ctx.put_state(0, *u)
    ctx.run(1, corr_fixed=1)
    got = ctx.get_state(0)
    oc = O.Ctx(N, K, M, Re=Re, alpha=alpha, dt=dt)
    oc.LDz = oc.lumesh_init(0, 1, 130.0, -3e-4)
    AB = oc.LDz[0][1:]
    assert np.abs(ctx.lumesh_get(0, opf.LDZ)[0][1:] - AB).max() <= 1e-13 * np.abs(AB).max()
    oc.set_state(*u)
    oc.run(1, ncorr_fixed=1)
    for c, ref in enumerate((oc.ur, oc.ut, oc.uz)):
        # harmonic 0 has a singular system under BC = 1, which the time step never meets
        assert rel_err(got[c][:, 1:], ref[:, 1:]) <= 1e-12, c
    ctx.vel_matrices(0, dt)
    after = ctx.lumesh_get(0, opf.LDZ)
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])


# theta lines of three passes whose sequence is not that of the z columns of
# their length, with requests of more than 64 KiB of LDS (M = 192)
@pytest.mark.parametrize("M", [128, 144, 162, 192, 216])
def test_nonlinear_long_theta_sequences(opf, M):
    _nonlinear_matches(opf, 10, 3, M)


# narrow and odd tile requests: a last tile of one line or one column, an odd
# number of z lines
@pytest.mark.parametrize("K,M,tm,tz", [(9, 16, 5, 2), (27, 6, 5, 0), (16, 9, 1, 0), (12, 8, 7, 2)])
def test_nonlinear_tiles(opf, K, M, tm, tz):
    from opf import ic as icgen
    res = []
    for shape in ((0, 0), (tm, tz)):
        ctx = opf.Context(10, K, M, tm=shape[0], tz=shape[1])
        ctx.setup(0, 3000.0, 1.25, 0.01)
        me = ctx.mesh()
        ctx.put_state(0, *icgen.seeded_perturbation(me["r"], me["intrdr"], K, M, 1.25, 7, 1e-2))
        ctx.transform(0)
        ctx.nonlinear(0)
        res.append(ctx.get_nonlinear(0))
        ctx.close()
    for c in range(3):
        assert np.array_equal(res[0][c], res[1][c]), c


# The plugins' batched transforms at odd numbers of z lines, at two and
# three passes: one step with the
# variable viscosity against the oracle, as close as the plugin's own test asks.
@pytest.mark.parametrize("K,M", [(9, 9), (3, 4), (27, 8), (16, 32), (32, 3), (54, 6)])
def test_viscosity_transform_lengths(opf, K, M):
    from opf import ic as icgen
    Re, alpha, dt = 2400.0, 1.25, 0.01
    prm = dict(rho=1000.0, radius=0.01, mu_0=0.056, mu_inf=0.0056, lam_CY=3e-3, n_CY=0.6, a_CY=2.0)
    ctx = opf.Context(10, K, M)
    ctx.nonnewtonian(0, **prm)
    ctx.setup(0, Re, alpha, dt)
    me = ctx.mesh()
    u = icgen.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, 3, 1e-2)
    ctx.put_state(0, *u)
    ctx.run(1)
    got = ctx.get_state(0)
    oc = O.Ctx(10, K, M, Re=Re, alpha=alpha, dt=dt)
    oc.nonnewtonian = prm
    oc.set_state(*u)
    oc.run(1, ncorr_fixed=1)
    for c, ref in enumerate((oc.ur, oc.ut, oc.uz)):
        assert rel_err(got[c], ref) <= 1e-12, c
    ctx.close()


# requests beyond what the kernels of the lengths hold (3K = 144: 8 columns; 3M =
# 48, 72: 8 lines, 432: 2 where the run-time plans hold one) and widths that
# split M unevenly
@pytest.mark.parametrize("K,M,tm,tz,runs", [(48, 16, 14, 14, (8, 8)), (48, 16, 7, 6, (6, 6)), (48, 16, 1, 2, (1, 2)),
                                            (48, 24, 13, 9, (8, 8)), (48, 24, 5, 0, (5, 8)), (3, 144, 0, 0, (14, 2)),
                                            (3, 144, 20, 1, (14, 2))])
def test_tile_config_names_the_tiles_that_run(opf, K, M, tm, tz, runs):
    """opf_tile_config gives the widths that the launches use, and a context made
    with those gives them again."""
    for _ in range(2):
        ctx = opf.Context(10, K, M, tm=tm, tz=tz)
        assert ctx.tile_config()[1:] == runs
        ctx.close()
        tm, tz = runs
