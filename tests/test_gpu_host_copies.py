"""Host copies of a renderer's buffer through the pinned chunks: written,
added and read back exactly, at sizes on both sides of the 8 MB from which
they are taken and of whole chunks, and by several threads at once (one has
the chunks, the others take the runtime's copy)."""

import threading

import numpy as np
import pytest

import flames as TF

pytestmark = pytest.mark.gpu


def renderer(ffr, cells_x, cells_y):
    text = TF.color_flame(3, size=64)
    assert '"size": [64, 64]' in text
    return ffr.BufferRenderer(text.replace('"size": [64, 64]', f'"size": [{cells_x}, {cells_y}]'),
                              precision="fp64", seed=1)


def words(r, seed):
    rng = np.random.default_rng(seed)
    n = r.cells * r.cell_words
    w = rng.integers(0, 1 << 20, n, dtype=np.uint64)
    c = w.reshape(r.cells, r.cell_words)
    c[:, 1:] = c[:, 1:].astype(np.float64).view(np.uint64)
    return w


def roundtrip(r, seed):
    a, b = words(r, seed), words(r, seed + 1)
    r.write_buffer(a)
    assert np.array_equal(r.read_buffer(), a)
    r.add_buffer(b)
    s = r.read_buffer()
    assert np.array_equal(r.counts(s), r.counts(a) + r.counts(b))
    assert np.array_equal(r.colors(s), r.colors(a) + r.colors(b))  # whole numbers: exact


# 32 bytes a cell: 8 MiB is 262144 cells, a chunk 65536
@pytest.mark.parametrize("size", [(512, 511), (512, 512), (512, 513), (1024, 1025), (1917, 1079)])
def test_sizes(ffr_mod, size):
    print(f"host copies {size}", flush=True)
    with renderer(ffr_mod, *size) as r:
        roundtrip(r, 3)


def test_threads(ffr_mod):
    rs = [renderer(ffr_mod, 900, 700 + k) for k in range(4)]
    errors = []

    def run(r, seed):
        try:
            for k in range(4):
                roundtrip(r, seed + k)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=run, args=(r, 100 * k)) for k, r in enumerate(rs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    for r in rs:
        r.close()
