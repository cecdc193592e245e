"""The work lists of the overlap rounds: however a round is launched (grid or
one workgroup, whose list outgrows its LDS buffer here), with whatever lanes
per atom, the steps end in the same state bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [400, 3000, 12000])
def test_rounds_do_not_depend_on_their_launches(dml, n, monkeypatch):
    from dml import workloads as W
    sysd = W.system_replica(n, 5, reservoir_band=True)
    say("overlap lists", n)
    states = []
    for tail, lanes in (("0", 1), ("1", 16), ("2", 4), (None, 0)):
        if tail is None:
            monkeypatch.delenv("DML_OV_TAIL")
        else:
            monkeypatch.setenv("DML_OV_TAIL", tail)
        c = dml.Context(dml.dana_config(sysd["box"], sysd["skin"], len(sysd["pos"]) + 64, h=sysd["h"],
                                        z0=sysd["z0"], zmax=sysd["zmax"],
                                        integrator=dml.BROWNIAN, reservoir=dml.NO_RESERVOIR,
                                        overlap_mode=dml.OVERLAP_ROUNDS, prob=0.5))
        c.set_tuning(overlap_lanes=lanes, overlap_rounds=24)
        c.set_state(sysd["pos"], species=sysd["species"])
        c.run(3)
        cnt = c.counters()
        states.append((c.state(), [cnt[k] for k in ("try_", "depo", "choques", "passes",
                                                    "ov_unfinished")]))
        c.close()
    assert n < 1000 or states[0][1][2] > 100
    for st, cnt in states[1:]:
        assert cnt == states[0][1]
        for k, v in st.items():
            np.testing.assert_array_equal(v, states[0][0][k], err_msg=k)
