"""States that the corrector has to refuse."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, K, M, RE, ALPHA, DT = 16, 6, 4, 2400.0, 1.25, 0.01


def _state(opf, seed=3):
    from opf import ic
    me = opf.host_mesh(N)
    return ic.seeded_perturbation(me["r"], me["intrdr"], K, M, ALPHA, seed, 1e-3)


@pytest.mark.parametrize("pairs", [1, 2, 4])
@pytest.mark.parametrize("where", [(0, 5, 1), (1, 0, 7), (2, 3, -1), "all"])
def test_nan_state_is_reported(where, pairs):
    """A velocity with a NaN (in one coefficient of one component, or everywhere)
    makes tim_dterr a NaN: the run fails with status 4 instead of counting the
    corrector as converged, and the other slots of the run are as without it."""
    import opf
    ctx = opf.Context(N, K, M, capacity=2, pairs=pairs)
    u = [f.copy() for f in _state(opf)]
    if where == "all":
        for f in u:
            f[:] = np.nan
    else:
        c, n, h = where
        u[c][n, h] = np.nan
    v = _state(opf, 4)
    for s, f in ((0, u), (1, v)):
        ctx.setup(s, RE, ALPHA, DT)
        ctx.put_state(s, *f)
    with pytest.raises(opf.OpfError) as err:
        ctx.run(3)
    assert err.value.code == 4, err.value
    assert ctx.status(0)["status"] == 4 and ctx.status(0)["step"] == 0
    assert ctx.status(1)["status"] == 0 and ctx.status(1)["step"] == 3
    got = ctx.get_state(1)
    alone = opf.Context(N, K, M, pairs=pairs)
    alone.setup(0, RE, ALPHA, DT)
    alone.put_state(0, *v)
    alone.run(3)
    for a, b in zip(got, alone.get_state(0)):
        assert np.array_equal(a, b)


def test_nan_reaches_a_host_driven_corrector():
    """tim_dterr of a host-driven corrector on a state with a NaN is a NaN."""
    import opf
    ctx = opf.Context(N, K, M)
    u = [f.copy() for f in _state(opf)]
    u[1][4, 9] = np.nan
    ctx.setup(0, RE, ALPHA, DT)
    ctx.put_state(0, *u)
    for step in (ctx.predictor, ctx.corrector):
        ctx.transform(0)
        ctx.nonlinear(0)
        d = step(0)
    assert np.isnan(d)
