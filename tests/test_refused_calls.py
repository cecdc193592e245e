"""A call that is refused leaves its replica as it was: the calls after it
give what they give in a context that never made it."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

BOX = [60.0, 60.0, 60.0]


def _system(dml, n=150):
    rng = np.random.default_rng(11)
    c = dml.Context(dml.dana_config(BOX, 2.0, 256, z0=30.0, zmax=60.0, integrator=dml.BROWNIAN,
                                    reservoir=dml.PISTON, seed=5))
    pos = rng.random((n, 3)) * (np.array(BOX) - 1.0) + 0.5
    c.set_state(pos, species=np.ones(n, np.int8))
    c.test_update()
    return c


def _refuse(dml, c, call):
    n = c.nslots()
    with pytest.raises(dml.DmlError) as e:
        if call == "box":  # all cell counts below four while cells are in use
            c.set_box([15.0, 15.0, 15.0])
        elif call == "order":  # a list that would do, and an index held twice
            c.set_order(ref_order=np.arange(n // 2), bkey=np.zeros(n, np.int32))
        elif call == "indices":
            c.set_order(bkey=np.full(n, -1, np.int32))
        else:  # more slots than the replica has
            c.reconfigure(dml.dana_config([15.0, 15.0, 15.0], 2.0, 4096), 0)
    return e.value.status


@pytest.mark.parametrize("call", ["box", "order", "indices", "slots"])
def test_refused_call_changes_nothing(dml, call):
    a, b = _system(dml), _system(dml)
    status = _refuse(dml, a, call)
    say("refused", call, status)
    assert status == {"box": -10, "order": -1, "indices": -1, "slots": -3}[call]
    for c in (a, b):
        c.set_zmax(58.0, 30.0)  # sends the replica's parameters
        c.update()
    np.testing.assert_array_equal(a.calc_rho(), b.calc_rho())
    np.testing.assert_array_equal(a.ref_order(), b.ref_order())
    for x, y in zip(a.cells() + a.lists() + a.slots(), b.cells() + b.lists() + b.slots()):
        np.testing.assert_array_equal(x, y)
    for c in (a, b):
        c.run(1, graph=False)
    sa, sb = a.state(), b.state()
    for k in sa:
        np.testing.assert_array_equal(sa[k], sb[k], err_msg=k)
    a.close()
    b.close()
