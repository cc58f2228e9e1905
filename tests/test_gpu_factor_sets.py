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
