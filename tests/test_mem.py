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


@pytest.mark.parametrize("how", [0, 1, 2], ids=["allocated anew", "temporary of a build", "wait succeeds"])
def test_blocks_that_may_be_in_use_are_not_kept(mem, how):
    assert mem.mem_refused_wait(how) == 0


@pytest.mark.parametrize("thread_device", [0, 3])
def test_waits_for_the_device_of_its_blocks(mem, thread_device):
    assert mem.mem_waits_for_its_device(thread_device) == 0


@pytest.mark.parametrize("megabytes,allocations", [(1, 1), (6, 1), (512, 1), (513, 5)])
def test_full_cache_makes_way_for_the_sizes_in_use(mem, megabytes, allocations):
    """Five rounds of one size after 512 MB of another: allocated once and kept
    (513 MB fit no cache: allocated each time)."""
    f = mem.mem_moves_on
    f.argtypes = [C.c_int, C.c_ulonglong]
    assert f(5, megabytes << 20) == allocations


def test_small_blocks_count_as_pages(mem):
    assert mem.mem_small_blocks_kept(140000) == (512 << 20) // 4096
