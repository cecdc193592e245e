"""What a setter leaves on the stream is waited for by the calls that read
device memory with a plain copy.  Run by test_simt_host.py in a process of its
own, with fills that happen no earlier than they must."""
import numpy as np


def _context(dml):
    return dml.dana_config([40.0, 40.0, 60.0], 2.0, 256, z0=30.0, zmax=60.0,
                           integrator=dml.BROWNIAN, reservoir=dml.PISTON, seed=5)


def _used(dml):
    c = dml.Context(_context(dml))
    c.set_state(np.random.default_rng(6).random((60, 3)) * [39.0, 39.0, 58.0] + 0.5)
    c.run(1, graph=False)
    assert c.counters()["particle_steps"] == 60
    return c


def test_counters_of_a_replica_set_up_again(dml):
    c = _used(dml)
    c.reconfigure(_context(dml), 0)
    assert not any(c.counters().values())
    c = _used(dml)
    c.reconfigure(_context(dml), 0)
    assert c.list_stats() == (0.0, 0, 0)


def test_setters_one_after_the_other(dml):
    c = _used(dml)
    c.set_box([40.0, 40.0, 200.0])  # other cells, cleared on the stream
    nc, cell, use, of = c.cells()
    assert nc[2] == 38 and (of == -1).all()
    c.reconfigure(_context(dml), 0)
    c.set_state(np.random.default_rng(7).random((50, 3)) * [39.0, 39.0, 58.0] + 0.5)
    c.test_update()
    d = dml.Context(_context(dml))
    d.set_state(np.random.default_rng(7).random((50, 3)) * [39.0, 39.0, 58.0] + 0.5)
    d.test_update()
    for x, y in zip(c.cells() + c.lists(), d.cells() + d.lists()):
        np.testing.assert_array_equal(x, y)
