"""A destroyed server gives its device memory back: the records of cell
updates past the LDS cell cache that its passes kept (a pass of 2^24 samples
or more of a flame that misses the cache) among it."""

import ctypes as C

import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu


def free_memory(ffr):
    free, total = C.c_size_t(), C.c_size_t()
    # (of the HIP runtime that the library is linked with)
    assert ffr.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_servers_give_their_memory_back(ffr_mod):
    text = read_flame("batch/flame_1069.json")  # 2.4 missed words a sample

    def serve():
        print("serve", flush=True)
        with ffr_mod.Server() as s:
            job = s.submit(text, 1 << 28, precision="fp32", seed=5)
            s.wait(job)
            assert s.job(job).state == ffr_mod.JOB_DONE
            s.release(job)

    free = []
    for _ in range(4):
        serve()
        free.append(free_memory(ffr_mod))
    # (the runtime's own first allocations come with the first server; the
    # records of a pass take 2.7 GB)
    for before, after in zip(free[1:], free[2:]):
        assert before - after < 64 << 20, free
