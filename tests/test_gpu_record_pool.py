"""Record memory that renders can do without (miss records, split walkers) is
lent for a render: a device's renderers, batches and servers share it, it
makes way for an allocation that a call needs, one of at most 10 GiB stays
after the last of them, and free_idle frees it."""

import ctypes as C
import json
import threading

import numpy as np
import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu

GB = 1 << 30


def free_memory(ffr):
    free, total = C.c_size_t(), C.c_size_t()
    # (of the HIP runtime that the library is linked with)
    assert ffr.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def spread(ffr, k=0, **kw):
    return ffr.BufferRenderer(read_flame("batch/flame_1069.json"), precision="fp32", seed=k, **kw)


def with_records(ffr, k):
    r = spread(ffr, k, binned=0)
    assert r.render(1 << 28) and r.record_use[0] > 0
    return r


def split(ffr, k):
    r = spread(ffr, k, batch_size=65536)
    assert r.render(1 << 26) and r.last_stats.atomics == 0
    return r


@pytest.mark.parametrize("render", [with_records, split])
def test_renderers_share_it(ffr_mod, render):
    print(f"record pool {render.__name__}", flush=True)
    after = []
    for _ in range(3):
        ffr_mod.free_idle()
        free, rs, held = free_memory(ffr_mod), [], []
        for k in range(5):
            rs.append(render(ffr_mod, k))
            held.append(free - free_memory(ffr_mod) -
                        sum(r.cells * r.cell_words * r.word_bytes for r in rs))
        assert held[0] > GB and held[-1] < 1.1 * held[0], held
        for r in rs:
            r.close()
        assert free - free_memory(ffr_mod) < 10 * GB + (256 << 20)
        ffr_mod.free_idle()
        after.append(free_memory(ffr_mod))
    # (the runtime keeps a few MB per stream from the first time on)
    assert after[1] - after[2] < 64 << 20, after


def test_it_outlives_the_last_renderer(ffr_mod):
    """a program that makes one renderer after another does not allocate and
    free gigabytes with each"""
    print("record pool of renderers in turn", flush=True)
    for _ in range(2):
        with_records(ffr_mod, 0).close()
    idle = free_memory(ffr_mod)
    for k in range(3):
        r = with_records(ffr_mod, k)
        assert idle - free_memory(ffr_mod) < r.cells * r.cell_words * r.word_bytes + (64 << 20)
        r.close()
        assert abs(idle - free_memory(ffr_mod)) < 64 << 20
    ffr_mod.free_idle()
    assert free_memory(ffr_mod) - idle > 4 * GB


def test_batches_share_it(ffr_mod):
    print("record pool of batches", flush=True)
    rs = [spread(ffr_mod, k) for k in range(4)]
    batches = [ffr_mod.Batch([r]) for r in rs]
    for b in batches:
        assert all(b.render([1 << 28]))
    free = free_memory(ffr_mod)
    for rep in range(2):  # (graphs replayed after others used the memory)
        for b, r in zip(batches, rs):
            assert all(b.render([1 << 28])) and r.record_use[0] > 0
    assert free - free_memory(ffr_mod) < 64 << 20
    for r in rs:
        alone = spread(ffr_mod, rs.index(r))
        for _ in range(3):
            assert alone.render(1 << 28)
        assert np.array_equal(alone.counts(alone.read_buffer()), r.counts(r.read_buffer()))
        alone.close()
    for b in batches:
        b.close()
    for r in rs:
        r.close()


def test_it_makes_way(ffr_mod):
    print("record pool makes way", flush=True)
    a = spread(ffr_mod, binned=0)
    assert a.render(1 << 30) and a.record_use[0] > 0  # (8 GB of record memory)
    cells = (free_memory(ffr_mod) + 3 * GB) // 8
    text = json.dumps({
        "dimensions": 3, "size": [4096, 4096, cells >> 24], "bounds": [[0, 1]] * 3,
        "xforms": [{"weight": 1, "variations": [{"name": "linear", "weight": 1.0}]}]})
    b = ffr_mod.BufferRenderer(text, precision="fp64")
    b.close()
    assert a.render(1 << 28)
    a.close()


def test_threads_render_with_their_own(ffr_mod):
    """more renderers at a time than idle memories are kept"""
    print("record pool of threads", flush=True)
    n, renders, errors = 6, 3, []
    rs = [spread(ffr_mod, k, binned=0) for k in range(n)]

    def work(r):
        try:
            for _ in range(renders):
                assert r.render(1 << 26)
        except Exception as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(r,)) for r in rs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for k, r in enumerate(rs):
        alone = spread(ffr_mod, k, binned=0)
        for _ in range(renders):
            assert alone.render(1 << 26)
        assert np.array_equal(alone.counts(alone.read_buffer()), r.counts(r.read_buffer()))
        alone.close()
        r.close()
