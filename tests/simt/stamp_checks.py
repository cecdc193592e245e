"""Overlap calls until the work-list stamps start over: STAMP_LIB is the CPU
build with so many stamps a call that some calls use them up.  Run by
test_simt_host.py in a process of its own."""
import os

import numpy as np
import pytest


@pytest.mark.parametrize("integrator", ["ermak", "brownian"])
def test_stamps_start_over(dml, integrator):
    rng = np.random.default_rng(9)
    n, box = 220, [30.0, 30.0, 40.0]
    k = np.arange(n)
    pos = (np.column_stack([k % 6, k // 6 % 6, k // 36]) + 0.5) * [5.0, 5.0, 5.6] \
        + rng.uniform(-1.2, 1.2, (n, 3))
    pos[:, 2] %= 40.0
    out = []
    for lib in (dml.LIB_PATH, os.environ["STAMP_LIB"]):
        dml.LIB_PATH, dml._lib = lib, None
        c = dml.Context(dml.dana_config(box, 2.0, 256, integrator=getattr(dml, integrator.upper()),
                                        reservoir=dml.NO_RESERVOIR, h=1e-2, z0=40.0, zmax=40.0,
                                        prob=0.5, seed=5, overlap_mode=dml.OVERLAP_ROUNDS))
        c.set_state(pos, species=np.where(k < 36, 2, 1).astype(np.int8))
        steps = []
        for _ in range(20):
            c.run(1, graph=False)
            steps.append((c.state(), c.counters()))
        out.append(steps)
        c.close()
    assert out[0][-1][1]["choques"] > 0
    for q, ((a, ka), (b, kb)) in enumerate(zip(*out)):
        assert ka == kb, q
        for x in a:
            np.testing.assert_array_equal(a[x], b[x], err_msg="step %d %s" % (q, x))
