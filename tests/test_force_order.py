"""The force kernel's cell-ordered list of ref atoms (systems of 200,000 slots
and more) against the ref order, which the other row builds keep: the same
steps, bit for bit, with atoms deposited, inserted and deleted between two
rebuilds, on both sides of the size from which the list is used."""
import numpy as np
import pytest

from test_gcmc_batch import _state_equal
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

REGISTER_ROWS, WAVE_ROWS = 5, 4  # list kernels: the first keeps the list, the other does not


@pytest.mark.parametrize("n,mode", [(199900, 0), (200000, 0), (203000, 0), (203000, 1)])
def test_cell_order_equals_ref_order(dml, n, mode):
    rng = np.random.default_rng(n + mode)
    step = 4.64
    m = int(np.ceil(n ** (1.0 / 3.0)))
    k = np.arange(n)
    pos = np.column_stack([k % m, k // m % m, k // (m * m)]) * step + step / 2
    pos += rng.uniform(-0.9, 0.9, pos.shape)
    pos = pos[rng.permutation(n)]
    z = np.where(rng.random(n) < 0.1, 2, 1).astype(np.int8)
    z[pos[:, 2] > 0.5 * m * step] = 1  # the insertion volume holds ions only
    box = np.array([m * step, m * step, m * step + 20.0])
    say("force order", n, mode)
    out = []
    for kernel in (REGISTER_ROWS, WAVE_ROWS):
        c = dml.Context(dml.dana_config(
            box, 2.0, n + 4096, h=1e-2, z0=0.5 * box[2], zmax=box[2], integrator=dml.ERMAK,
            reservoir=dml.GCMC, precision=dml.FP64, overlap_mode=dml.OVERLAP_ROUNDS, act=0.01,
            nadj=300 if mode else 12, seed=11,
            gcmc_mode=(dml.GCMC_BATCHED | dml.GCMC_ALTERNATE) if mode else 0))
        c.set_tuning(list_kernel=kernel)
        c.set_state(pos, species=z)
        c.test_update()
        c.forces()
        first = c.state()["force"]
        c.run(5)
        out.append((c, first))
    np.testing.assert_array_equal(out[0][1], out[1][1])
    _state_equal(out[0][0], out[1][0], "steps")
    for c, _ in out:
        c.close()
