"""Tests of the host side and of the launch-shape edges on the CPU, against the
SIMT build of the same sources under AddressSanitizer (see test_simt.py)."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def simt():
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    sys.path.insert(0, os.path.join(HERE, "simt"))
    import sim
    sim.build(asan=True)
    return sim


def _run(sim, name, order="forward", pick="", **env):
    e = sim.env(asan=True)
    e.update(DML_SIMT="1", SIMT_ORDER=order, **env)
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", os.path.join(HERE, name), "-q", "-x",
                        "-s", "-p", "no:cacheprovider", "-k", pick],
                       env=e, cwd=ROOT, capture_output=True, text=True, timeout=1200)
    tail = (r.stdout + r.stderr)[-4000:]
    assert r.returncode == 0, tail
    assert "AddressSanitizer" not in r.stdout + r.stderr, tail


@pytest.mark.parametrize("name", ["test_refused_calls.py", "test_gcmc_reuse.py",
                                  os.path.join("simt", "host_checks.py")])
def test_host_side(simt, name):
    _run(simt, name)


def test_overlap_stamps_start_over(simt, tmp_path):
    lib = str(tmp_path / "libdml_stamps.so")
    simt.build(asan=True, SIMT_OUT=lib, SIMT_FLAGS="-DOV_STAMPS=0x10000000")
    _run(simt, os.path.join("simt", "stamp_checks.py"), STAMP_LIB=lib)


def test_reads_wait_for_the_stream(simt):
    _run(simt, os.path.join("simt", "wait_checks.py"), SIMT_LAZY="1")


# sizes on both sides of a wave's 64 trials or positions, split and whole
# cells, and replicas that take a workgroup each
EDGES = [("test_overlap_exact.py", "crowded"),
         ("test_gcmc_walks.py", "0.2-64-57 or 0.2-65-60 or 0.7-130-61"),
         ("test_row_build.py", "500-60 or 2000-60"),
         ("test_small_replicas.py", "kind1-1025 or kind0-1] or kind3-1]")]


@pytest.mark.parametrize("order", ["forward", "reverse"])
@pytest.mark.parametrize("name,pick", EDGES)
def test_launch_shape_edges(simt, name, pick, order):
    _run(simt, name, order, pick)
