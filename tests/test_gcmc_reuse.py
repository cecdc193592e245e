"""Batched GCMC in a replica that is used again: another state, or another
configuration, gives what a new context gives (the marks that the calls before
left per cell and slot are not taken for the present call's)."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

BOX = [42.0, 42.0, 60.0]


def _config(dml):
    return dml.dana_config(BOX, 2.0, 512, z0=30.0, zmax=60.0, integrator=dml.BROWNIAN, h=1e-3,
                           reservoir=dml.GCMC, act=0.02, nadj=12, seed=40,
                           overlap_mode=dml.OVERLAP_ROUNDS, gcmc_mode=dml.GCMC_BATCHED)


def _result(c, seed):
    k = np.arange(180)
    pos = (np.column_stack([k % 6, k // 6 % 6, k // 36]) + 0.5) * [7.0, 7.0, 12.0] \
        + np.random.default_rng(seed).uniform(-0.5, 0.5, (180, 3))
    before = c.counters()
    c.set_state(pos, species=np.ones(len(pos), np.int8))
    c.test_update()
    for _ in range(2):
        c.gcmc(0.02, 12)
    after = c.counters()
    assert c.gcmc_outcomes(12) is not None  # in a batch
    s = c.state()
    s.update(order=c.gcmc_order(), ref=c.ref_order(), bkey=c.slots()[0], nn=c.lists()[0],
             rows=c.lists()[2], cells=c.cells()[3],
             moves=np.array([after[q] - before[q] for q in ("ins", "del_")]))
    return s


@pytest.mark.parametrize("again", ["state", "configuration"])
def test_replica_used_again(dml, again):
    c = dml.Context(_config(dml))
    _result(c, 1)
    if again == "configuration":
        c.reconfigure(_config(dml), 0)
    say("used once", again)
    got = _result(c, 1)
    new = dml.Context(_config(dml))
    want = _result(new, 1)
    say("moves", want["moves"])
    assert want["moves"][0] > 5
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    c.close()
    new.close()
