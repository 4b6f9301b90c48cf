"""Launches of the C entry points (grids, LDS, kernels) recorded on the host, without a GPU (host_launches.py)."""

import json
import os
import shutil
import subprocess
import sys

import pytest

from jqmc_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH) or shutil.which("gcc") is None,
                                reason="library not built, or no C compiler")


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("shim") / "hip_host_shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(HERE, "hip_host_shim.c")], check=True)
    return so


def _scenario(shim, name):
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_launches.py"), shim, name], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.splitlines()[-1])


def test_large_lds_is_allowed_on_every_device(shim):
    """The permission for more than 64 KiB of dynamic LDS belongs to a kernel on a device: a system on a second
    device in the same process gets it too, and no launch is refused."""
    rec = _scenario(shim, "large_lds")
    for dev in (0, 1):
        large = {k for k, *_, lds, d, _ in rec if d == dev and lds > 65536}
        assert {"k_el_kinetic", "k_fr_orbital"} <= large, large
    assert not [r for r in rec if r[-1]]


def test_what_the_set_up_takes_is_taken_by_the_other_calls(shim):
    """A launch of 2^32 work-items or more along one dimension is refused: no call of a walker set that the set-up
    takes runs into that."""
    rec = _scenario(shim, "many_walkers")
    assert {"k_init_rows", "k_el_prep", "k_lrdmc_move", "k_dlnpsi_small", "k_rank_narrow"} <= {r[0] for r in rec}
    assert not [r for r in rec if r[-1]]


def test_forces_are_taken_in_equal_parts(shim):
    """One walker more than fit a part does not cost a chain of launches of its own, nor a larger workspace."""
    (one, b1), (two, b2) = _scenario(shim, "long_forces")
    assert len(one) == 1 and len(two) == 2 and abs(two[0] - two[1]) <= 1
    assert b2 == b1
