"""Checks of the host side that need the CPU build of libdml: its hipMalloc
fails on request.  Run by test_simt_host.py in a process of its own."""
import ctypes

import numpy as np
import pytest


def _fail_malloc(dml, k):
    """the k-th hipMalloc from now fails (0: none)"""
    ctypes.c_int.in_dll(dml.lib(), "simt_fail_malloc").value = k


def _left(dml):
    return ctypes.c_int.in_dll(dml.lib(), "simt_fail_malloc").value


def _chunks(dml, zmax=60.0, overlap=None):
    box = [40.0, 40.0, zmax]
    return dml.dana_config(box, 2.0, 256, z0=30.0, zmax=zmax, integrator=dml.BROWNIAN,
                           reservoir=dml.CHUNKS, seed=5,
                           overlap_mode=dml.OVERLAP_ROUNDS if overlap is None else overlap)


def _system(dml):
    rng = np.random.default_rng(3)
    c = dml.Context(_chunks(dml))
    block = rng.random((20, 3)) * [40.0, 40.0, 9.0]
    c.set_chunk(block, 9.0 + 3.2, 55.0)
    c.set_state(rng.random((60, 3)) * [39.0, 39.0, 58.0] + 0.5, species=np.ones(60, np.int8))
    c.test_update()
    return c


def _fail(dml, c, call):
    rng = np.random.default_rng(4)
    k = 0
    while True:  # each allocation of the call in turn
        k += 1
        _fail_malloc(dml, k)
        try:
            if call == "chunk":
                c.set_chunk(rng.random((50, 3)) * 9.0, 30.0, 40.0)
            elif call == "exact":
                c.reconfigure(_chunks(dml, 50.0, dml.OVERLAP_EXACT), 0)
            else:  # wider rows
                g = _chunks(dml, 50.0)
                g.max_neighbors = 4096
                c.reconfigure(g, 0)
        except dml.DmlError as e:
            assert e.status == -3
            continue
        finally:
            left = _left(dml)
            _fail_malloc(dml, 0)
        assert left > 0  # the call allocates k - 1 times
        return k - 1


@pytest.mark.parametrize("call", ["chunk", "exact", "rows"])
def test_out_of_memory_changes_nothing(dml, call):
    n = _fail(dml, _system(dml), call)
    assert n > 0
    for k in sorted({1, n}):
        a, b = _system(dml), _system(dml)
        _fail_malloc(dml, k)
        with pytest.raises(dml.DmlError):
            if call == "chunk":
                a.set_chunk(np.random.default_rng(4).random((50, 3)) * 9.0, 30.0, 40.0)
            else:
                g = _chunks(dml, 50.0, dml.OVERLAP_EXACT if call == "exact" else None)
                if call == "rows":
                    g.max_neighbors = 4096
                a.reconfigure(g, 0)
        _fail_malloc(dml, 0)
        for c in (a, b):
            c.set_zmax(58.0, 30.0)
            c.update()
            c.bloques()
        np.testing.assert_array_equal(a.calc_rho(), b.calc_rho())
        sa, sb = a.state(), b.state()
        for q in sa:
            np.testing.assert_array_equal(sa[q], sb[q], err_msg="%s %d %s" % (call, k, q))
        a.close()
        b.close()


def test_out_of_memory_box_can_be_set_again(dml):
    """no memory for the cells of a taller box: the old box stays, and the call
    can be made again"""
    rng = np.random.default_rng(6)
    pos = rng.random((60, 3)) * [39.0, 39.0, 58.0] + 0.5
    out = []
    for k in (0, 1, 9):
        c = dml.Context(dml.dana_config([40.0, 40.0, 60.0], 2.0, 256, z0=30.0, zmax=60.0,
                                        integrator=dml.BROWNIAN, reservoir=dml.PISTON, seed=5))
        c.set_state(pos, species=np.ones(60, np.int8))
        c.test_update()
        if k:
            _fail_malloc(dml, k)
            with pytest.raises(dml.DmlError):
                c.set_box([40.0, 40.0, 200.0])
            _fail_malloc(dml, 0)
            c.set_zmax(60.0, 30.0)
            c.update()
            assert c.cells()[0][2] == 11  # int(60 / 5.2)
        c.set_box([40.0, 40.0, 200.0])
        c.update()
        assert c.cells()[0][2] == 38
        out.append(c.lists())
        for x, y in zip(out[0], out[-1]):
            np.testing.assert_array_equal(x, y)
        c.close()


def test_reconfigure_before_the_larger_cells_are_there(dml):
    """dml_set_chunk asks for the cells of the tallest box its blocks can make;
    a box that needs them all, set before any call that sorts cells"""
    c = dml.Context(_chunks(dml))
    c.set_chunk(np.random.default_rng(3).random((4, 3)) * [40.0, 40.0, 9.0], 12.2, 55.0)
    g = dml.dana_config([40.0, 40.0, 700.0], 2.0, 256, z0=30.0, zmax=700.0,
                        integrator=dml.BROWNIAN, reservoir=dml.NO_RESERVOIR)
    c.reconfigure(g, 0)
    pos = np.random.default_rng(6).random((60, 3)) * [39.0, 39.0, 690.0] + 0.5
    c.set_state(pos, species=np.ones(60, np.int8))
    c.test_update()
    fresh = dml.Context(g)
    fresh.set_state(pos, species=np.ones(60, np.int8))
    fresh.test_update()
    for x, y in zip(c.lists(), fresh.lists()):
        np.testing.assert_array_equal(x, y)
    c.close()
    fresh.close()


def test_cells_that_are_not_in_place_hold_nothing(dml):
    c = dml.Context(_chunks(dml))
    pos = np.random.default_rng(6).random((60, 3)) * [39.0, 39.0, 58.0] + 0.5
    c.set_state(pos)
    c.test_update()
    sorted_now = c.cells()[3]
    assert (sorted_now >= 0).all()
    c.set_chunk(np.random.default_rng(3).random((4, 3)) * [40.0, 40.0, 9.0], 12.2, 55.0)
    np.testing.assert_array_equal(c.cells()[3], sorted_now)  # the box is what it was
    c.reconfigure(dml.dana_config([40.0, 40.0, 600.0], 2.0, 256, z0=30.0, zmax=600.0,
                                  integrator=dml.BROWNIAN, reservoir=dml.NO_RESERVOIR), 0)
    c.set_state(pos)
    nc, cell, use, of = c.cells()
    assert nc[2] == 115 and use and (of == -1).all()
    c.test_update()
    assert (c.cells()[3] >= 0).all()
    c.close()


def test_state_is_read_without_memory_to_stage_it(dml):
    c = dml.Context(dml.dana_config([40.0, 40.0, 60.0], 2.0, 4096, z0=30.0))
    pos = np.random.default_rng(8).random((4096, 3)) * 39.0
    c.set_state(pos)  # 38 bytes an atom staged, 170 to read it back
    _fail_malloc(dml, 1)
    got = c.state()
    assert _left(dml) == 0  # an allocation was asked for and refused
    np.testing.assert_array_equal(got["pos"], pos)
    np.testing.assert_array_equal(got["pos_old"], pos)
    np.testing.assert_array_equal(got["vel"], np.zeros((4096, 3)))
    np.testing.assert_array_equal(got["old_cg"], np.full((4096, 3), 1e8))
    np.testing.assert_array_equal(got["species"], np.ones(4096, np.int8))
    np.testing.assert_array_equal(got["flags"], np.full(4096, dml.FL_ALIVE | dml.FL_REF))
    c.close()


@pytest.mark.parametrize("call", ["brownian", "ermak_a", "overlap", "overlap_rounds"])
def test_no_memory_for_injected_numbers(dml, call):
    """the call fails, and does not draw numbers of its own instead"""
    rng = np.random.default_rng(3)
    c = dml.Context(dml.dana_config([40.0, 40.0, 60.0], 2.0, 256, z0=60.0, zmax=60.0, seed=5,
                                    integrator=dml.ERMAK if call == "ermak_a" else dml.BROWNIAN,
                                    reservoir=dml.NO_RESERVOIR,
                                    overlap_mode=dml.OVERLAP_EXACT if call == "overlap"
                                    else dml.OVERLAP_ROUNDS))
    c.set_state(rng.random((60, 3)) * [39.0, 39.0, 58.0] + 0.5)
    c.test_update()
    before = c.state()
    args = {"brownian": (np.zeros(180), np.zeros(60)), "ermak_a": (np.zeros(360), np.zeros(60)),
            "overlap": (np.zeros((1, 64)),), "overlap_rounds": (np.zeros((4, 256)), 4)}[call]
    for k in (1, 2)[:1 if call.startswith("overlap") else 2]:
        _fail_malloc(dml, k)
        with pytest.raises(dml.DmlError) as e:
            getattr(c, call)(*args)
        assert e.value.status == -3 and _left(dml) == 0
        after = c.state()
        for x in before:
            np.testing.assert_array_equal(after[x], before[x], err_msg=x)
    c.close()


def test_failed_allocation_is_not_reported_by_a_later_call(dml):
    c = _system(dml)
    _fail_malloc(dml, 1)
    with pytest.raises(dml.DmlError):
        c.set_chunk(np.random.default_rng(4).random((50, 3)) * 9.0, 30.0, 40.0)
    pts = np.array([[1.0, 2.0, 3.0], [20.0, 20.0, 20.0]])
    du, hard = c.gcmc_trial_energy(pts, noalloc=True)
    want, hard2 = c.gcmc_trial_energy(pts)
    np.testing.assert_array_equal(du, want)
    np.testing.assert_array_equal(hard, hard2)
    c.close()
