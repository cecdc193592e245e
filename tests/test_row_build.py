"""Rows of the register-resident build (k_listbuild_wr) against the oracle's
ngroup_cells, entry for entry, where its split can go wrong: a single atom, a
cell with fewer ref atoms than parts, cells of several hundred atoms (more
than one load of centre atoms, many passes of candidates), and systems on both
sides of each bound on the waves per cell."""
import numpy as np
import pytest

from test_gpu_parity import assert_lists_equal, pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,side,skin", [(1, 60.0, 10.0), (7, 60.0, 10.0), (500, 60.0, 10.0),
                                         (2000, 60.0, 10.0), (30000, 90.0, 2.0),
                                         (205000, 165.0, 2.0)])
def test_rows_by_size_match_oracle(orc, dml, n, side, skin):
    """n atoms at 0.05 / A^3 packed into a corner of the box, a tenth of them
    electrode atoms (candidates without a row)"""
    rng = np.random.default_rng(n)
    step = 0.05 ** (-1.0 / 3.0)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    k = np.arange(n)
    pos = np.column_stack([k % m, k // m % m, k // (m * m)]) * step + 0.5
    pos += 0.9 * rng.uniform(-0.5, 0.5, pos.shape)
    pos = pos[rng.permutation(n)]
    box = np.array([side, side, side + 5.0])
    z = np.where(rng.random(n) < 0.1, 2, 1).astype(np.int8)
    z[0] = 1
    say("row build", n)
    s, c = pair(orc, dml, box, skin, pos, z, zmax=box[2])
    assert s.test_update()[0] == 0
    c.test_update()
    assert_lists_equal(c, s)
    c.close()
