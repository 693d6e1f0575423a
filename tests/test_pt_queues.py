"""The path tracer's queue segments and traversal chunks, walked on the CPU with
the kernels' own index arithmetic (traverse_device.h: QueueWalk, DealtChunks,
SegmentChunks): every entry is taken once, and no segment gets more entries
than it holds."""
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
    """Each XCD appends at most one entry per entry it walks to its segment."""
    seen = np.zeros(n, np.int32)
    for x in range(8):
        walked, k = 0, 0
        while True:
            lo, hi = hb.chunk("dealt_block", n, x, k)
            if lo >= hi:
                break
            assert hi - lo <= BLOCK
            seen[lo:hi] += 1
            walked += hi - lo
            k += 1
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
        empty = False
        for c in range(n // chunk // 8 + 2 * per + 3):
            lo, hi = hb.chunk("dealt_chunk", n, x, chunk, c)
            # the schedule stops at the first empty chunk: none may follow it
            assert lo <= hi <= n and not (empty and lo < hi)
            empty = empty or lo >= hi
            seen[lo:hi] += 1
        assert empty
    assert (seen == 1).all()


@pytest.mark.parametrize("lo", [0, 77 * 256])
@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("nrays,nshadow", [(0, 0), (0, 1), (1, 0), (64, 64), (65, 127), (1000, 0),
                                           (0, 1000), (777, 888), (4096, 4096)])
def test_ray_chunks_then_shadow_chunks(nrays, nshadow, chunk, lo):
    rays, shadow = np.zeros(nrays, np.int32), np.zeros(nshadow, np.int32)
    total = (nrays + chunk - 1) // chunk + (nshadow + chunk - 1) // chunk
    for c in range(total + 3):
        b, e, is_shadow = hb.chunk("segment_chunk", lo, nrays, nshadow, chunk, c)
        assert (b < e) == (c < total) and lo <= b <= e
        (shadow if is_shadow else rays)[b - lo:e - lo] += 1
        assert e - lo <= (nshadow if is_shadow else nrays)
    assert (rays == 1).all() and (shadow == 1).all()


def test_segment_of_the_largest_batches():
    for n in (1 << 27, (1 << 32) - 1):
        assert 8 * segment(n) >= n
