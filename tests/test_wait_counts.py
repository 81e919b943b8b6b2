"""spg_wait_counts: the host's wait for counts that a kernel stores to pinned memory (no GPU needed: a thread stores them here)."""
import os
import threading
import time

import numpy as np
import pytest

from spargeattn_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")


@pytest.mark.parametrize("n", [0, 1, 139, 5000])
def test_sum_of_counts_that_are_there(n):
    counts = np.arange(n, dtype=np.int32) * 400000          # (the sum needs 64 bits)
    assert _lib.load().spg_wait_counts(counts.ctypes.data, n, 0.0) == counts.astype(np.int64).sum()


def test_gives_up_in_time():
    counts = np.array([3, -1, 4], np.int32)
    t = time.monotonic()
    assert _lib.load().spg_wait_counts(counts.ctypes.data, 3, 0.02) == -1
    assert 0.015 < time.monotonic() - t < 5.0
    assert _lib.load().spg_wait_counts(None, 3, 0.02) == -1


def test_a_long_wait_gives_the_core_back():
    counts = np.array([-1], np.int32)
    t = time.process_time()
    assert _lib.load().spg_wait_counts(counts.ctypes.data, 1, 0.2) == -1
    assert time.process_time() - t < 0.1                    # (half a millisecond, and a few microseconds in every 50)


def test_waits_for_counts_in_any_order():
    counts = np.full(64, -1, np.int32)

    def store():
        for i in np.random.default_rng(0).permutation(64):
            counts[i] = i
            time.sleep(1e-4)
    t = threading.Thread(target=store)
    t.start()
    assert _lib.load().spg_wait_counts(counts.ctypes.data, 64, 10.0) == 64 * 63 // 2
    t.join()
