"""Replicas that sit a run out: what they are configured for does not change
the others, and they go on when they are released."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

BOX = [30.0, 30.0, 40.0]


def _config(dml, rep):
    return dml.dana_config(BOX, 2.0, 256, integrator=dml.BROWNIAN if rep else dml.ERMAK,
                           reservoir=dml.NO_RESERVOIR, h=1e-2, z0=40.0, zmax=40.0, prob=0.5,
                           seed=5 + rep, overlap_mode=dml.OVERLAP_EXACT if rep == 1
                           else dml.OVERLAP_ROUNDS)


def _set(c, rep, at=0):
    k = np.arange(200)
    pos = (np.column_stack([k % 6, k // 6 % 6, k // 36]) + 0.5) * [5.0, 5.0, 5.6] \
        + np.random.default_rng(rep).uniform(-1.2, 1.2, (200, 3))
    pos[:, 2] %= 40.0
    c.set_state(pos, species=np.where(k < 36, 2, 1).astype(np.int8), rep=at)


@pytest.mark.parametrize("graph", [True, False])
def test_paused_and_released(dml, graph):
    c = dml.Context([_config(dml, r) for r in range(3)])
    for r in range(3):
        _set(c, r, r)
    steps = [0, 0, 0]
    for paused in ([1], [], [0, 2], [1, 2], []):
        for r in range(3):
            c.set_active(r not in paused, r)
            steps[r] += 0 if r in paused else 3
        c.run(3, graph=graph)
    say("steps", steps)
    for r in range(3):
        alone = dml.Context(_config(dml, r))
        _set(alone, r)
        alone.run(steps[r], graph=False)
        ka, kb = c.counters(r), alone.counters()
        if r != 1:  # the rounds count a paused replica's calls too
            ka.pop("passes"), kb.pop("passes")
        assert ka == kb
        a, b = c.state(rep=r), alone.state()
        for k in a:
            np.testing.assert_array_equal(a[k], b[k], err_msg="%d %s" % (r, k))
        alone.close()
    c.close()


def test_pool_counts_what_it_reserves(dml):
    """the pool's own figure against the device memory it takes: the rest is
    cells (some 10,000 entries of 44 bytes) and rounding to 2 MB of the few
    arrays that are not a multiple of it"""
    from dml import serve

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert dml.lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    serve.SlotPool([(256, 1, [60.0, 60.0, 60.0])]).close()  # the runtime's own
    before = free()
    pool = serve.SlotPool([(1 << 20, 1, [60.0, 60.0, 60.0])])
    used = before - free()
    say("reserved", used, "counted", pool.hbm_bytes())
    assert pool.hbm_bytes() - (2 << 20) <= used <= pool.hbm_bytes() + (32 << 20)
    pool.close()
