"""What a render learns about its misses comes from renders through the LDS
cell cache alone: an uncached batch, whose every sample goes past the cache, does
not make the next cached one take records.  (FP64 renders of a flame that
misses 0.12 words a sample keep their atomics; the first render of a renderer,
which knows nothing, takes records.)"""

import pytest

from conftest import read_flame

pytestmark = pytest.mark.gpu

SAMPLES = 1 << 27  # 131072 walkers


def known(ffr, **kw):
    r = ffr.BufferRenderer(read_flame("batch/flame_1159.json"), precision="fp64", seed=3, **kw)
    assert r.render(SAMPLES) and r.record_use[0] > 0
    assert r.render(SAMPLES) and r.record_use[0] == 0
    return r


def test_uncached_batch(ffr_mod):
    print("misses after an uncached batch", flush=True)
    r = known(ffr_mod)
    with ffr_mod.Batch([r]) as batch:
        assert all(batch.render([1 << 20]))  # 1024 walkers: no cache
    assert r.render(SAMPLES) and r.record_use[0] == 0
    r.close()


def test_uncached_kind(ffr_mod):
    print("misses of a kind after an uncached pass", flush=True)
    r = ffr_mod.BufferRenderer(read_flame("batch/flame_1159.json"), precision="fp64", seed=3)
    with ffr_mod.Batch([r]) as batch:
        for n, records in ((SAMPLES, True), (SAMPLES, False), (1 << 20, False), (SAMPLES, False)):
            assert all(batch.render([n]))
            assert (r.record_use[0] > 0) == records, n
    r.close()
