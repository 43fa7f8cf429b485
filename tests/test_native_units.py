"""Parts of the native code that no call of the C ABI reaches by itself,
through tests/native (built with the library)."""
import ctypes
import os

import pytest

MB = 1 << 20


@pytest.fixture(scope="module")
def unit():
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_build", "libtrc_unit.so")
    if not os.path.exists(path):
        from tensorray_amd import build
        build.build_tests()
    return ctypes.CDLL(path)


def _fit(unit, first, total, per_item, per_window, kept, may_alloc, free):
    out = (ctypes.c_uint64 * 3)()
    c = ctypes.c_uint64
    unit.unit_fit_window(c(first), c(total), c(per_item), c(per_window), c(kept), ctypes.c_int(may_alloc), c(free), out)
    return tuple(out)


KEPT, ALLOCATED = 1, 2
WINDOW = 2 << 20  # paths
DEEP = 124        # bytes per path at 8 bounces


def test_window_choice(unit):
    # small requests take the stream's memory, large ones the whole window
    assert _fit(unit, 1000, 1000, DEEP, 0, 32 * MB, 1, 1 << 40) == (1000, KEPT, 0)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 1 << 40) == (WINDOW, ALLOCATED, WINDOW * DEEP)
    # half of it where the whole cannot be had
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 200 * MB)[:2] == (WINDOW // 2, ALLOCATED)
    # nothing to be had, or a captured call: the largest the stream's memory holds
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 0)[:2] == (WINDOW // 8, KEPT)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 0, 1 << 40) == (WINDOW // 8, KEPT, 0)
    # not even that: small windows, down to half a megabyte
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 0, 1, MB)[:2] == (8192, ALLOCATED)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 0, 1, 0)[:2] == (4096, 0)
    # odd sizes stay multiples of 64, and a request below the smallest window is asked for once
    w, how, asked = _fit(unit, 1_000_001, 1_000_001, DEEP, 0, 0, 1, 70 * MB)
    assert how == ALLOCATED and w % 64 == 0 and w * DEEP == asked <= 70 * MB < 1_000_001 * DEEP
    assert _fit(unit, 100, 100, DEEP, 0, 0, 1, 0) == (100, 0, 100 * DEEP)


def test_window_choice_ends_when_counters_outgrow_it(unit):
    """Queues keep a kilobyte of counters per chunk: with billions of samples
    no chunk fits the stream's memory, and the search ends."""
    w, how, _ = _fit(unit, 1 << 22, 1 << 33, 90, 1024, 32 * MB, 0, 1 << 40)
    assert how == 0 and w == 4096
