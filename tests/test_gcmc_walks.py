"""The ordered walks of a batched GCMC call at the edges of their 64-trial
batches: calls of 1 to 200 trials, with points freed and taken again inside
one batch and across two, against the trials run one after the other."""
import numpy as np
import pytest

from test_gcmc_batch import _gcmc_system, _state_equal
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nadj,at", [(1, 0), (2, 0), (63, 5), (64, 57), (65, 60), (130, 61),
                                     (200, 122)])
@pytest.mark.parametrize("p_ins", [0.2, 0.7])
def test_batches_decide_as_one_after_the_other(dml, nadj, at, p_ins):
    rng = np.random.default_rng(1000 + nadj)
    box = np.array([40.0, 40.0, 60.0])
    pos, z, ions = _gcmc_system(rng, box, 11, 330)
    z0, zmax = 14.0, box[2] - 0.5
    vol = box[0] * box[1] * (zmax - z0)
    inside = ions[(ions[:, 2] >= z0) & (ions[:, 2] <= zmax)]
    say("gcmc walks", nadj, at, p_ins, len(inside))
    u = rng.random((nadj, 5))
    u[:, 0] = np.where(rng.random(nadj) < p_ins, 0.25, 0.75)
    special = at + 8 <= nadj
    if special:
        def point(p):
            return [0.25, 0.0, p[0] / box[0], p[1] / box[1], (p[2] - z0) / (zmax - z0)]
        # before the block only rejected trials: the list is the start's
        u[:at, 0], u[:at, 1] = 0.75, 1e30
        n, k = len(inside), 7
        last = [0.75, 0.0, 1.0 - 1e-12, 0.5, 0.5]
        first = [0.75, 0.0, 1e-12, 0.5, 0.5]
        u[at:at + 8] = [point(inside[k]),                       # taken
                        [0.75, 0.0, (k + 0.5) / n, 0.5, 0.5],   # frees it
                        point(inside[k]),                       # now free
                        point(inside[k]),                       # taken by the one before
                        last,                                   # which leaves again
                        point(inside[k]),
                        first,
                        point(inside[0])]
    g = rng.standard_normal((2, nadj, 3))
    u2 = rng.random((nadj, 5))
    ctx = []
    for mode in (0, dml.GCMC_BATCHED):
        c = dml.Context(dml.dana_config(box, 2.0, len(pos) + 1024, h=5e-5, z0=z0, zmax=zmax,
                                        integrator=dml.BROWNIAN, reservoir=dml.GCMC,
                                        overlap_mode=dml.OVERLAP_ROUNDS, gcmc_mode=mode, seed=3))
        c.set_state(pos, species=z)
        c.test_update()
        ctx.append(c)
    for it, uu in enumerate((u, u2)):
        for c in ctx:
            c.gcmc(len(inside) / vol, nadj, uu, g[it])
        out = ctx[1].gcmc_outcomes(nadj)
        # (a later call whose list could empty runs trial by trial)
        assert out is not None or it, "ran trial by trial"
        _state_equal(ctx[0], ctx[1], "call %d" % it)
        if special and it == 0:
            assert not out["accepted"][:at].any()
            assert out["accepted"][at:at + 8].tolist() == [0, 1, 1, 0, 1, 1, 1, 1]
    for c in ctx:
        c.run(2)
    _state_equal(ctx[0], ctx[1], "steps")
    for c in ctx:
        c.close()
