"""The factor sets of a slot (tim_lumesh_init / _invert / _get) and the time
step that solves with them."""
import numpy as np
import pytest

import opf_oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu

RE, ALPHA, DT = 2400.0, 1.25, 0.01


@pytest.fixture(scope="module")
def opf():
    import opf as pkg
    return pkg


def _field(rng, N, H):
    b = rng.standard_normal((N, H)) + 1j * rng.standard_normal((N, H))
    b[0] = b[-1] = 0.0
    return b


def test_factors_are_built_once_per_set(opf):
    """tim_lumesh_invert factors a set when it is first used and not again until
    the set changes: a repeated solve spends on the factors no more than half of
    what the first did (the launch finds nothing to do), with the same result,
    and the factors of one set take the memory of one set."""
    N, K, M = 48, 32, 24
    ctx = opf.Context(N, K, M, capacity=3)
    ctx.setup(0, RE, ALPHA, DT)
    H = ctx.H
    b = _field(np.random.default_rng(1), N, H)
    ctx.coll2phys(b)                       # the transforms' buffers
    bytes0 = _bytes(ctx)
    times, xs = [], []
    for _ in range(3):
        ctx.kernel_timing(True)
        xs.append(ctx.lumesh_invert(0, opf.LDZ, b))
        times.append(ctx.kernel_time("lapack_factor")[0])
        ctx.kernel_timing(False)
    assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])
    assert max(times[1:]) <= 0.5 * times[0], times
    assert _bytes(ctx) - bytes0 <= K * M * 129 * N + 8192
    # a change of the set is seen
    ctx.vel_matrices(0, 2.0 * DT)
    oc = O.Ctx(N, K, M, Re=RE, alpha=ALPHA, dt=2.0 * DT)
    ref = oc.lumesh_invert(oc.lumesh_init(0, 0, 1.0 / (2.0 * DT), -0.51 / RE), b)
    assert rel_err(ctx.lumesh_invert(0, opf.LDZ, b), ref) <= 1e-12


def _bytes(ctx):
    import ctypes as C
    n = C.c_size_t()
    opf_int = [C.c_int() for _ in range(6)]
    ctx.lib.opf_ctx_dims(ctx.h, *[C.byref(d) for d in opf_int], C.byref(n))
    return n.value


def test_factors_follow_the_device_loop(opf):
    """The factors that tim_lumesh_get returns are those of the matrices as the
    device loop left them (adaptive time step), also where they were asked for
    before."""
    N, K, M = 16, 6, 4
    from opf import ic
    me = opf.host_mesh(N)
    u = ic.seeded_perturbation(me["r"], me["intrdr"], K, M, ALPHA, 3, 1e-3)
    ctx = opf.Context(N, K, M)
    ctx.adaptive(0)
    ctx.setup(0, RE, ALPHA, DT)
    before = ctx.lumesh_get(0, opf.LDZ)[0]
    ctx.put_state(0, *u)
    ctx.run(4)
    dt = ctx.timestep(0)["dt"]
    assert dt != DT
    got = ctx.lumesh_get(0, opf.LDZ)
    fresh = opf.Context(N, K, M)
    fresh.setup(0, RE, ALPHA, dt)
    ref = fresh.lumesh_get(0, opf.LDZ)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    assert not np.array_equal(got[0], before)


def test_reading_a_singular_set_leaves_the_slot_alone(opf):
    """A set that tim_lumesh_init reported singular can be read and solved with
    without marking the slot's run as failed."""
    N, K, M = 16, 6, 4
    ctx = opf.Context(N, K, M)
    ctx.setup(0, RE, ALPHA, DT)
    with pytest.raises(opf.OpfError) as err:
        ctx.lumesh_init(0, opf.LDM, 0, 0, 0.0, 0.0)
    assert err.value.code == 3
    ctx.lumesh_get(0, opf.LDM)
    assert ctx.status(0)["status"] == 0
    ctx.lumesh_invert(0, opf.LDM, np.zeros((N, ctx.H), complex))
    assert ctx.status(0)["status"] == 0


# c1 that make a leading principal block (rows 0 .. 3 or 0 .. 7) of one pair's
# matrix c1 + c2 Lap (c2 = -3e-4, PM = 0, N = 20, alpha = 1.25) singular to a few
# 1e-14, while all whole matrices are regular (condition below 4e5): an
# elimination by blocks of four rows has nothing to divide by there.
@pytest.mark.parametrize("pairs", [1, 2, 4])
@pytest.mark.parametrize("c1", [-0.23272778313654063, -0.14513836407775046, -0.11507417760238585,
                                -0.35203654575952653])
def test_step_with_a_set_whose_leading_block_is_singular(opf, c1, pairs):
    """tim_lumesh_init takes such a set, and the time step solves with it as
    closely as tim_lumesh_invert does, while the context's other slots go on as
    without it; then vel_matrices takes it back."""
    from opf import ic
    N, K, M, c2 = 20, 4, 3, -3e-4
    ctx = opf.Context(N, K, M, capacity=2, pairs=pairs)
    me = ctx.mesh()
    u = ic.seeded_perturbation(me["r"], me["intrdr"], K, M, ALPHA, 3, 1e-2)
    for s in (0, 1):
        ctx.setup(s, RE, ALPHA, DT)
        ctx.put_state(s, *u)
    ctx.run(1, corr_fixed=1)
    plain = ctx.get_state(0)
    ctx.lumesh_init(0, opf.LDZ, 0, 0, c1, c2)
    for s in (0, 1):
        ctx.put_state(s, *u)
    ctx.run(1, corr_fixed=1)
    got = ctx.get_state(0)
    for a, b in zip(ctx.get_state(1), plain):
        assert np.array_equal(a, b)
    oc = O.Ctx(N, K, M, Re=RE, alpha=ALPHA, dt=DT)
    oc.LDz = oc.lumesh_init(0, 0, c1, c2)
    oc.set_state(*u)
    oc.run(1, ncorr_fixed=1)
    # the condition of the matrices, 4e5, times the rounding of the right-hand
    # sides, a few 1e-16
    for c, ref in enumerate((oc.ur, oc.ut, oc.uz)):
        assert rel_err(got[c], ref) <= 1e-9, c
    ctx.vel_matrices(0, DT)
    ctx.put_state(0, *u)
    ctx.run(1, corr_fixed=1, slots=[0])
    for a, b in zip(ctx.get_state(0), plain):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("amp", [1.0, 1e-10, 1e-20])
def test_explicit_step_of_small_states(opf, amp):
    """d_implicit = 0 (the matrices of the velocity are 1/dt I with the boundary
    rows) at any size of the state: the solves lose no digits to underflow."""
    from opf import ic
    N, K, M, dt = 20, 4, 3, 1e-4
    ctx = opf.Context(N, K, M)
    ctx.setup(0, RE, ALPHA, dt, implicit=0.0)
    me = ctx.mesh()
    u = [amp * f for f in ic.seeded_perturbation(me["r"], me["intrdr"], K, M, ALPHA, 3, 1e-2)]
    ctx.put_state(0, *u)
    ctx.run(2, corr_fixed=1)
    got = ctx.get_state(0)
    oc = O.Ctx(N, K, M, Re=RE, alpha=ALPHA, dt=dt, implicit=0.0)
    oc.set_state(*u)
    oc.run(2, ncorr_fixed=1)
    for c, ref in enumerate((oc.ur, oc.ut, oc.uz)):
        assert rel_err(got[c], ref) <= 1e-12, (amp, c)
