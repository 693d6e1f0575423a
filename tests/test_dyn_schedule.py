"""The run-time chunk schedule of the persistent trace kernels
(traverse_persistent.h, XcdChunks) against a brute-force simulation of its
fetch rule, over the raw traces' chunks as the kernels compute them
(traverse_device.h, EighthChunks).  An XCD's W waves (W = 4 per workgroup, grid /
8 workgroups per XCD) start on its chunks 0 .. W - 1; a wave that got a chunk
asks at once for its next, which is W + k, k the value its fetch returned from
the XCD's counter (less the launch's base), and an empty chunk ends it.  For
every interleaving of the fetches, each ray must be taken exactly once and the
counter must advance by EighthChunks::count, the amount the host adds to the
base it keeps for the next launch on the stream.
"""
import ctypes as C

import numpy as np
import pytest

import hostemu_bind as hb

WAVES_PER_BLOCK = 4


def simulate(n, grid, chunk, rng):
    taken = np.zeros(n, np.int32)
    advance = []
    for x in range(8):
        wavesx = (grid // 8) * WAVES_PER_BLOCK
        counter = 0
        ahead = []  # per wave that holds a chunk: its next chunk

        def take(c):
            nonlocal counter
            b, e = hb.chunk("eighth_chunk", n, x, chunk, c)
            if b >= e:
                return None
            taken[b:e] += 1
            counter += 1
            return wavesx + counter - 1

        for wx in range(wavesx):  # static first chunks
            nxt = take(wx)
            if nxt is not None:
                ahead.append(nxt)
        while ahead:  # chunks are used up in a random order of the waves
            i = int(rng.integers(len(ahead)))
            nxt = take(ahead[i])
            if nxt is None:
                ahead.pop(i)
            else:
                ahead[i] = nxt
        advance.append(counter)
    return taken, advance


@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("grid", [8, 16, 1536, 1544])
def test_every_ray_once_and_counter_advance(grid, chunk):
    L = hb.lib()
    rng = np.random.default_rng(grid)
    for n in (1, 7, 8, 255, 256, 257, 2047, 2048, 2049, 65537, 1 << 20, 3 << 20):
        taken, advance = simulate(n, grid, chunk, rng)
        assert (taken == 1).all(), (n, grid)
        for x in range(8):
            assert advance[x] == L.wlh_eighth_count(n, x, chunk), (n, grid, x)


@pytest.mark.parametrize("chunk", [64, 128])
def test_largest_launches_stay_in_range(chunk):
    """The launches of up to 2^32 - 1 rays: their first and last chunks, and those
    past them.  A wave's next index, up to 64 past its last ray, fits 32 bits."""
    f = hb.lib().wlh_launch_rays
    f.restype, f.argtypes = C.c_uint32, [C.c_uint32]
    for total in ((1 << 31) + 5, (1 << 32) - 70, (1 << 32) - 9, (1 << 32) - 7, (1 << 32) - 1):
        left = total
        while left:
            n = f(left)
            assert 0 < n <= left and n % 32 * (left - n) == 0  # any-hit words are not shared
            left -= n
            n8 = (n + 7) // 8
            for x in range(8):
                lo, hi = min(x * n8, n), min((x + 1) * n8, n)
                assert hi + 64 < 1 << 32
                count = hb.lib().wlh_eighth_count(n, x, chunk)
                assert count == (hi - lo + chunk - 1) // chunk
                if count:
                    assert hb.chunk("eighth_chunk", n, x, chunk, 0)[0] == lo
                    assert hb.chunk("eighth_chunk", n, x, chunk, count - 1)[1] == hi
                b, e = hb.chunk("eighth_chunk", n, x, chunk, count + 7)
                assert b == e == hi
