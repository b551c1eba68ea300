"""Device buffers and the cache of scene blocks, on a stand-in for the HIP
runtime (tests/cpu_emul/mem.cpp)."""
from __future__ import annotations

import ctypes as C
import os

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def mem():
    return C.CDLL(os.path.join(ROOT, "tests", "_build", "libmem.so"))


@pytest.mark.parametrize("fits", [1, 0], ids=["after making room", "no room at all"])
def test_allocation_leaves_no_stored_error(mem, fits):
    assert mem.mem_no_stored_error(fits) == 0
