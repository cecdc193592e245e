"""A replica whose GCMC mode changes between two runs of captured steps: its
trials are those of steps launched one by one."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

BOX = [42.0, 42.0, 60.0]


def _config(dml, batched, seed):
    return dml.dana_config(BOX, 2.0, 512, z0=30.0, zmax=60.0, integrator=dml.BROWNIAN, h=1e-3,
                           reservoir=dml.GCMC, act=0.02, nadj=12, seed=seed,
                           overlap_mode=dml.OVERLAP_ROUNDS,
                           gcmc_mode=dml.GCMC_BATCHED if batched else 0)


def _state(rng, n=180):
    k = np.arange(n)
    return (np.column_stack([k % 6, k // 6 % 6, k // 36]) + 0.5) * [7.0, 7.0, 12.0] \
        + rng.uniform(-0.5, 0.5, (n, 3))


def _set(dml, c, rep, batched):
    c.reconfigure(_config(dml, batched, 40 + rep), rep)
    pos = _state(np.random.default_rng(rep))
    c.set_state(pos, species=np.ones(len(pos), np.int8), rep=rep)
    c.set_step_limit(0, rep)
    c.set_active(True, rep)


@pytest.mark.parametrize("modes", [[True, False, True], [False, True, False]])
def test_mode_changes_between_captured_runs(dml, modes):
    out = []
    for graph in (True, False):
        c = dml.Context([_config(dml, True, 40), _config(dml, True, 41)])
        _set(dml, c, 0, True)
        for batched in modes:
            _set(dml, c, 1, batched)
            c.run(3, graph=graph)
            k = c.counters(1)
            say("graph", graph, "batched", batched, "insertions", k["ins"], "deletions", k["del_"])
            s = c.state(1)
            out.append((graph, k["ins"], k["del_"], c.replica_status(1), s))
        c.close()
    m = len(modes)
    for a, b in zip(out[:m], out[m:]):
        assert a[1:4] == b[1:4] and a[1] > 0
        for k in a[4]:
            np.testing.assert_array_equal(a[4][k], b[4][k], err_msg=k)
