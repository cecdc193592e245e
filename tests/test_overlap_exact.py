"""overlap_moveback in the reference's order (dana.F90:849-943) where its
device form can go wrong: ref lists around the 64 positions of a mask word,
more entries to meet than an atom's list holds, reverts that put atoms back
before and behind the walk, and more ref atoms than the masks in LDS take.
State, marks and counters equal the oracle's exactly."""
import numpy as np
import pytest

from test_gpu_parity import electrode, pair, say

pytestmark = pytest.mark.gpu


def _lattice(rng, n, lo, box, step, jitter):
    """n points of a jittered lattice above lo, at least step - 2 jitter apart"""
    nx, ny = int(box[0] // step), int(box[1] // step)
    k = np.arange(n)
    p = np.column_stack([k % nx, k // nx % ny, k // (nx * ny)]) * step
    p = p + jitter * rng.uniform(-1, 1, p.shape) + [step / 2, step / 2, lo]
    return p


def _compare(s, c):
    so, sd = s.state(), c.state()
    for k in ("pos", "vel", "species", "flags"):
        np.testing.assert_array_equal(sd[k], so[k], err_msg=k)
    cnt = c.counters()
    assert (cnt["try_"], cnt["depo"], cnt["choques"], cnt["passes"]) == (
        s.c.try_, s.c.depo, s.c.choques, s.c.passes)
    return cnt


@pytest.mark.parametrize("n,crowd", [(1, 1), (63, 4), (64, 24), (65, 24), (200, 40), (700, 3)])
def test_crowded_moves_match_oracle(orc, dml, n, crowd):
    """groups of `crowd` ions are thrown onto one place each, some of them
    onto the electrode; contacts deposit with probability 0.6"""
    rng = np.random.default_rng(1000 + n)
    box = np.array([44.0, 44.0, 70.0])
    el = electrode(3.51, 12, 12, 2, 1.755)
    ions = _lattice(rng, n, 8.0, box, 4.2, 0.45)
    pos = np.vstack([el, ions])
    z = np.array([2] * len(el) + [1] * len(ions), np.int8)
    say("overlap exact", n, crowd)
    h, dif = 1e-3, 250.0
    s, c = pair(orc, dml, box, 10.0, pos, z, ermak=False, zmax=70.0, z0=60.0, h=h, prob=0.6,
                overlap_mode=dml.OVERLAP_EXACT)
    s.test_update(); c.test_update()
    for _ in range(3):
        so = s.state()
        ref = s.ref_order()
        p = so["pos"][ref]
        place = p[rng.integers(0, len(p), len(p) // crowd + 1)] * [1, 1, rng.choice([0.2, 1.0])]
        goal = place[rng.integers(0, len(place), len(p))] + 0.8 * rng.standard_normal(p.shape)
        move = np.where(rng.random((len(p), 1)) < 0.7, goal - p, 0.3 * rng.standard_normal(p.shape))
        move = np.clip(move, -6, 6)
        nz = (move / np.sqrt(2 * dif * h)).reshape(-1)
        ud = rng.random(len(p))
        assert s.brownian(nz, ud) == 0
        c.brownian(nz, ud)
        assert s.test_update()[0] == 0
        c.test_update()
        u = rng.random(8192)
        st, _ = s.overlap(u)
        assert st == 0
        c.overlap(u)
        _compare(s, c)
        s.f_to_cg(False); c.f_to_cg()
        if s.nref == 0:
            break
    c.close()


def test_masks_beyond_lds_match_oracle(orc, dml):
    """131,200 ref atoms: one word more than LDS holds and a remainder"""
    rng = np.random.default_rng(77)
    n = 131072 + 128
    box = np.array([210.0, 210.0, 240.0])
    pos = _lattice(rng, n, 2.0, box, 4.1, 0.3)
    z = np.ones(n, np.int8)
    say("overlap exact", n)
    h, dif = 5e-5, 250.0
    s, c = pair(orc, dml, box, 2.0, pos, z, ermak=False, zmax=240.0, z0=239.0, h=h,
                overlap_mode=dml.OVERLAP_EXACT)
    s.test_update(); c.test_update()
    nz = rng.standard_normal(3 * n) * 1.5
    ud = rng.random(n)
    assert s.brownian(nz, ud) == 0
    c.brownian(nz, ud)
    assert s.test_update()[0] == 0
    c.test_update()
    st, _ = s.overlap(rng.random(64))
    assert st == 0
    c.overlap(rng.random((1, 64)))
    assert _compare(s, c)["choques"] > 100
    c.close()
