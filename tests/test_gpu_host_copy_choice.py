"""Which host copies of the buffer take the library's pinned chunks: not a
program's first small ones, which would pay for 32 MiB of pinned memory, and
not those of memory that the caller pinned.  Seen by the address space that a
copy adds; the bytes come whole either way."""

import ctypes as C
import json
import mmap

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def renderer(ffr, mib):
    return ffr.BufferRenderer(json.dumps({
        "dimensions": 2, "size": [1024, mib * 128], "bounds": [[0, 1], [0, 1]],
        "xforms": [{"weight": 1, "variations": [{"name": "linear", "weight": 1.0}],
                    "pre_affine": {"A": [[0.5, 0], [0, 0.5]], "b": [0.2, 0.1]}}]}),
        precision="fp64", seed=1)


def address_space():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[0]) * mmap.PAGESIZE


def copies(ffr, mib, reads, writes, pinned=False):
    """how much each copy adds to the address space, MiB"""
    r = renderer(ffr, mib)
    lib, n = ffr.lib(), mib * MIB
    words = np.arange(n // 8, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    if pinned:
        p = C.c_void_p()
        assert lib.hipHostMalloc(C.byref(p), C.c_size_t(n), C.c_uint(0)) == 0
        host = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_uint64)), (n // 8,))
    else:
        host = np.empty(n // 8, dtype=np.uint64)
    host[:] = words
    grown = []
    for k in range(writes + reads):
        before = address_space()
        if k < writes:
            assert lib.ffr_write_buffer(r._h, host.ctypes.data_as(C.c_void_p), C.c_size_t(n)) == 0
        else:
            host[:] = 0
            assert lib.ffr_read_buffer(r._h, host.ctypes.data_as(C.c_void_p), C.c_size_t(n)) == 0
        grown.append((address_space() - before) / MIB)
        assert np.array_equal(host, words)
    r.close()
    if pinned:
        assert lib.hipHostFree(p) == 0
    return grown


@pytest.mark.parametrize("mib, reads, writes, pinned, made", [
    (8, 2, 2, False, False),    # small ones
    (32, 1, 1, False, False),   # one that does not win the memory back
    (32, 3, 1, False, True),    # its repetition does
    (64, 1, 1, False, True),    # a large one
    (64, 2, 2, True, False),    # the caller's pinned memory
])
def test_pinned_chunks_are_made_where_they_pay(ffr_mod, mib, reads, writes, pinned, made):
    copies(ffr_mod, 4, 1, 1)  # (the runtime's own staging)
    grown = copies(ffr_mod, mib, reads, writes, pinned)
    print(f"host copies {mib} MiB pinned={pinned}: {grown}", flush=True)
    assert (max(grown) >= 32) == made
