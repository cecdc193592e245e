"""Replicas of up to 4,096 slots take most phases of a step in one workgroup
each; the same atoms in a context of one slot more take the grid-wide kernels.
Whole runs of both, bit for bit, for each integrator, reservoir and overlap
order, with sizes around a workgroup's pass of 1,024 entries, and replicas of
different kinds (one of them empty) in one context."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

SMALL = 4096  # most slots of a small replica


def _ions(rng, n, box):
    m = int(np.ceil(n ** (1.0 / 3.0)))
    k = np.arange(n)
    cell = np.column_stack([k % m, k // m % m, k // (m * m)])
    pos = (cell + 0.5) * (box / m) + rng.uniform(-0.6, 0.6, (n, 3))
    return pos[rng.permutation(n)]


def _config(dml, kind, n, box, capacity, seed):
    integrator, reservoir, overlap = kind
    res = {"piston": dml.PISTON, "gcmc": dml.GCMC, "batched": dml.GCMC, "chunks": dml.CHUNKS,
           "none": dml.NO_RESERVOIR}[reservoir]
    top = box[2]
    return dml.dana_config(
        box, 2.0, capacity, h=1e-2 if integrator == "ermak" else 1e-3,
        z0=0.6 * box[2] if reservoir != "none" else top, zmax=top,
        integrator=dml.ERMAK if integrator == "ermak" else dml.BROWNIAN, reservoir=res,
        precision=dml.FP64, act=0.008, nadj=8, seed=seed,
        overlap_mode=dml.OVERLAP_EXACT if overlap == "exact" else dml.OVERLAP_ROUNDS,
        gcmc_mode=dml.GCMC_BATCHED if reservoir == "batched" else 0)


def _set(c, rep, kind, pos, box):
    if kind[1] == "chunks":
        # the lower part of the box and, above z0, the template's place
        c.set_chunk(pos[:40] * [1.0, 1.0, 0.2], 0.2 * box[2] + 3.2, 0.9 * box[2], rep=rep)
    c.set_state(pos, species=np.ones(len(pos), np.int8), rep=rep)


def _same(a, b, nrep):
    for r in range(nrep):
        sa, sb = a.state(rep=r), b.state(rep=r)
        for k in sa:
            m = min(len(sa[k]), len(sb[k]))
            np.testing.assert_array_equal(sa[k][:m], sb[k][:m], err_msg="%d %s" % (r, k))
        np.testing.assert_array_equal(a.ref_order(rep=r), b.ref_order(rep=r))
        assert a.replica_status(r) == b.replica_status(r)
        np.testing.assert_array_equal(a.zmax(rep=r), b.zmax(rep=r))


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 3000, 3700])
@pytest.mark.parametrize("kind", [("ermak", "piston", "exact"), ("ermak", "none", "rounds"),
                                  ("ermak", "gcmc", "rounds"), ("brownian", "gcmc", "exact"),
                                  ("brownian", "batched", "rounds"),
                                  ("brownian", "chunks", "exact")])
def test_small_equals_grid_wide(dml, kind, n):
    rng = np.random.default_rng(n)
    side = max((n / 0.006) ** (1.0 / 3.0), 24.0)
    box = np.array([side, side, side])
    pos = _ions(rng, n, box)
    say("small replicas", kind, n)
    ctx = []
    for capacity in (SMALL, SMALL + 1):
        c = dml.Context(_config(dml, kind, n, box, capacity, 5))
        _set(c, 0, kind, pos, box)
        c.run(8)
        ctx.append(c)
    _same(ctx[0], ctx[1], 1)
    for c in ctx:
        c.close()


def test_small_replicas_of_every_kind(dml):
    rng = np.random.default_rng(3)
    kinds = [("ermak", "piston", "rounds"), ("brownian", "chunks", "rounds"),
             ("ermak", "gcmc", "exact"), ("brownian", "batched", "exact"),
             ("ermak", "none", "rounds")]
    sizes = [900, 1500, 2100, 1200, 0]
    boxes = [np.full(3, max((n / 0.006) ** (1.0 / 3.0), 24.0)) for n in sizes]
    pos = [_ions(rng, n, b) if n else np.zeros((0, 3)) for n, b in zip(sizes, boxes)]
    say("small replicas of every kind")
    ctx = []
    for capacity in (SMALL, SMALL + 1):
        c = dml.Context([_config(dml, k, n, b, 3072 if q else capacity, 5 + q)
                         for q, (k, n, b) in enumerate(zip(kinds, sizes, boxes))])
        for q, k in enumerate(kinds):
            _set(c, q, k, pos[q], boxes[q])
        c.run(8)
        ctx.append(c)
    _same(ctx[0], ctx[1], len(kinds))
    for c in ctx:
        c.close()
