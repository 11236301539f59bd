"""Allocations made on first use where one fails: the sampled step's scratch (ksearch_amd/csrc/sample.cpp) and the buffers
of a prompt pass or a decode round (alloc_together) never look as if they held what they do not, so that the call after a
failed one asks again instead of launching over null pointers.  Host-only build against mock allocations; no GPU work."""
import ctypes as C

import pytest

from tests import host_mock


@pytest.fixture()
def scratch():
    lib = C.CDLL(host_mock.build())
    lib.mock_sample_create.restype = C.c_void_p
    lib.mock_sample_destroy.argtypes = [C.c_void_p]
    lib.mock_sample_reserve.argtypes = [C.c_void_p, C.c_int, C.c_int, C.POINTER(C.c_int)]
    before, h = lib.mock_allocated(), lib.mock_sample_create()
    out = (C.c_int * 4)()

    def reserve(rows, n, fail_after=-1):
        lib.mock_fail_alloc(fail_after)
        rc = lib.mock_sample_reserve(h, rows, n, out)
        lib.mock_fail_alloc(-1)
        return rc, *out

    yield reserve
    lib.mock_sample_destroy(h)
    assert lib.mock_allocated() == before


@pytest.mark.parametrize("fail_after", [0, 1])
def test_a_failed_allocation_is_asked_for_again(scratch, fail_after):
    rc, rows, n, lists, heads = scratch(4, 1000, fail_after)
    assert rc == 1 and (lists and heads or (rows, n) == (0, 0))
    assert scratch(4, 1000) == (0, 4, 1000, 1, 1)


def test_a_failed_growth_leaves_nothing_behind_that_the_sizes_claim(scratch):
    assert scratch(2, 1000) == (0, 2, 1000, 1, 1)
    assert scratch(16, 1000, 0) == (1, 0, 0, 0, 1)
    assert scratch(1, 500) == (0, 1, 500, 1, 1)
    assert scratch(2, 400) == (0, 2, 500, 1, 1) and scratch(1, 500) == (0, 2, 500, 1, 1)


@pytest.mark.parametrize("fail_after", [0, 1, 2])
def test_buffers_needed_together_are_there_together_or_not_at_all(fail_after):
    lib = C.CDLL(host_mock.build())
    three, n, before = (C.c_void_p * 3)(), C.c_int(), lib.mock_allocated()
    lib.mock_fail_alloc(fail_after)
    assert lib.mock_together(three, C.byref(n)) == 1 and n.value == 0 and lib.mock_allocated() == before
    assert lib.mock_together(three, C.byref(n)) == 0 and n.value == 3 and lib.mock_allocated() == before + 3


def test_a_buffer_grows_in_steps_and_survives_a_failure():
    lib = C.CDLL(host_mock.build())
    lib.mock_grow.restype, lib.mock_grow.argtypes = C.c_uint64, [C.c_uint64]
    step, before = 16 << 20, lib.mock_allocated()
    assert [lib.mock_grow(n) for n in (1, step, 5, step + 1, 2 * step)] == [step, step, step, 2 * step, 2 * step]
    assert lib.mock_allocated() == before + 1
    lib.mock_fail_alloc(0)
    assert lib.mock_grow(5 * step) == 0 and lib.mock_allocated() == before
    assert lib.mock_grow(7) == step and lib.mock_allocated() == before + 1
