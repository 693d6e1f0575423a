"""The path tracer's queue segments and traversal chunks, walked on the CPU as
the kernels walk them (pathtrace.hip: queue_walk, first_chunks, k_trace's
chunks): every entry is taken once, and no segment gets more entries than it
holds."""
import ctypes as C

import numpy as np
import pytest

import hostemu_bind as hb

BLOCK = 256


def segment(n):
    f = hb.lib().wlh_pt_segment
    f.restype, f.argtypes = C.c_uint32, [C.c_uint64]
    return f(n)


SIZES = (1, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 4095, 12345, 65537, (1 << 20) + 3)


@pytest.mark.parametrize("n", SIZES)
def test_first_queue_is_walked_once_and_fits_the_segments(n):
    """Blocks of 256 entries dealt to the XCDs in turn: each appends at most
    one entry per entry it walks to its XCD's segment."""
    seen = np.zeros(n, np.int32)
    for x in range(8):
        walked = 0
        for at in range(x * BLOCK, n, 8 * BLOCK):
            seen[at:at + BLOCK] += 1
            walked += min(BLOCK, n - at)
        assert walked <= segment(n), (n, x)
    assert (seen == 1).all()
    # later queues: an XCD walks its own segment only, so it appends at most
    # as many as it read; all segments together fit the queue's allocation
    assert n <= 8 * segment(n) < n + 8 * BLOCK + 8 * BLOCK


@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("n", SIZES)
def test_first_trace_chunks(n, chunk):
    seen = np.zeros(n, np.int32)
    per = BLOCK // chunk
    for x in range(8):
        c, empty = 0, False
        while c < n // chunk + 16:
            s0 = ((c // per) * 8 + x) * BLOCK + (c % per) * chunk
            lo, hi = min(s0, n), min(s0 + chunk, n)
            # the schedule stops at the first empty chunk: none may follow it
            assert not (empty and lo < hi)
            empty = empty or lo >= hi
            seen[lo:hi] += 1
            c += 1
    assert (seen == 1).all()


@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("nrays,nshadow", [(0, 0), (0, 1), (1, 0), (64, 64), (65, 127), (1000, 0),
                                           (0, 1000), (777, 888)])
def test_ray_chunks_then_shadow_chunks(nrays, nshadow, chunk):
    rays, shadow = np.zeros(nrays, np.int32), np.zeros(nshadow, np.int32)
    ray_chunks = (nrays + chunk - 1) // chunk
    total = ray_chunks + (nshadow + chunk - 1) // chunk
    for c in range(total + 3):
        is_shadow = c >= ray_chunks
        n = nshadow if is_shadow else nrays
        s0 = (c - ray_chunks if is_shadow else c) * chunk
        lo, hi = min(s0, n), min(s0 + chunk, n)
        assert (lo < hi) == (c < total)
        (shadow if is_shadow else rays)[lo:hi] += 1
    assert (rays == 1).all() and (shadow == 1).all()


def test_segment_of_the_largest_batches():
    for n in (1 << 27, (1 << 32) - 1):
        assert 8 * segment(n) >= n
