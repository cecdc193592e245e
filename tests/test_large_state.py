"""States larger than the staging block that a context keeps: set and read
back bit for bit, and no device memory held afterwards."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

KEPT = 64 << 20  # most bytes of device staging a context keeps


def _free(dml):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert dml.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("given", [("vel", "acel", "pos_old", "old_cg"), ("old_cg",)])
def test_large_state(dml, given):
    rng = np.random.default_rng(2)
    per = 24 * (1 + len(given)) + 14
    n = KEPT // per * 2 + 777  # three pieces, the last one small
    box = [400.0, 400.0, 400.0]
    cfg = dml.dana_config(box, 2.0, n + 300, z0=200.0, zmax=400.0, reservoir=dml.GCMC,
                          integrator=dml.BROWNIAN, max_neighbors=16,
                          overlap_mode=dml.OVERLAP_ROUNDS)
    d = {k: rng.random((n, 3)) * 400.0 for k in ("pos",) + given}
    species = rng.integers(1, 3, n).astype(np.int8)
    flags = np.where(rng.random(n) < 0.9, dml.FL_ALIVE, 0).astype(np.uint8)
    flags |= np.where((flags > 0) & (rng.random(n) < 0.7), dml.FL_REF, 0).astype(np.uint8)
    flags |= np.where((flags > 0) & (rng.random(n) < 0.5), dml.FL_GCMC, 0).astype(np.uint8)
    kw = {k: d[k] for k in given}
    first = dml.Context(cfg)  # (the runtime's own copy buffers come with the first large copies)
    first.set_state(d["pos"], species=species, flags=flags, **kw)
    first.state()
    first.close()
    c = dml.Context(cfg)
    free = _free(dml)
    c.set_state(d["pos"], species=species, flags=flags, **kw)
    s = c.state()
    held = free - _free(dml)
    say("atoms", n, "bytes", per * n, "held", held)
    assert held <= KEPT + (4 << 20)
    for k in ("pos", "vel", "acel", "pos_old", "old_cg"):
        want = d[k] if k in d else {"vel": 0.0, "acel": 0.0, "old_cg": 1e8}.get(k, d["pos"])
        np.testing.assert_array_equal(s[k], np.broadcast_to(want, (n, 3)), err_msg=k)
    np.testing.assert_array_equal(s["species"], species)
    np.testing.assert_array_equal(s["flags"], flags)
    np.testing.assert_array_equal(c.ref_order(), np.nonzero(flags & dml.FL_REF)[0])
    np.testing.assert_array_equal(c.gcmc_order(), np.nonzero(flags & dml.FL_GCMC)[0])
    bk, pid, seq = c.slots()
    for a in (bk, pid, seq):
        np.testing.assert_array_equal(a, np.arange(n))
    assert c.observables()[0, 3] == np.count_nonzero(flags & dml.FL_ALIVE)
    # a smaller state in the same slots: nothing of the larger one is left
    c.set_state(d["pos"][:100])
    assert c.nslots() == 100 and c.observables()[0, 3] == 100
    np.testing.assert_array_equal(c.ref_order(), np.arange(100))
    c.close()
